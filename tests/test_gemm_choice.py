"""The kernel a MATMUL node takes, on the CPU (lbr_gemm_choice: nothing is launched)."""

import pytest

from runtime.ir import OpType
from test_fusion import _lib, _node

BASE = 1 << 40


def _choice(M, N, K, batches=1, trans_b=1):
    shape = (1, M, N) if batches == 1 else (batches, M, N)
    return _lib().gemm_choice(_node(OpType.MATMUL, [BASE, 2 * BASE], 3 * BASE, shape,
                                    (K, trans_b, int(batches == 1), 0)))


@pytest.fixture(autouse=True)
def _no_overrides(monkeypatch):
    for e in ("LBR_GEMM_TILE", "LBR_GEMM_KSPLIT", "LBR_GEMM_SPLIT"):
        monkeypatch.delenv(e, raising=False)


@pytest.mark.parametrize("K,ks", [(20, 2), (20, 16), (200, 5), (200, 6), (712, 16), (1036, 16)])
def test_ragged_k_with_ranges_it_does_not_give(monkeypatch, K, ks):
    """A K that does not cut into the forced number of whole 32-wide ranges has no split tile: the
    register-staged kernel runs, never an fp32 DMA tile, which would drop the columns past K/32·32."""
    monkeypatch.setenv("LBR_GEMM_KSPLIT", str(ks))
    assert _choice(300, 70, K)[:3] == ("gemm_mfma_f32_nt", "", False)


def test_ragged_k_with_a_tile_the_split_kernel_lacks(monkeypatch):
    for name in ("32x48b3", "nonsenseb3", "b3"):
        monkeypatch.setenv("LBR_GEMM_TILE", name)
        assert _choice(300, 70, 200)[:3] == ("gemm_mfma_f32_nt", "", False), name


@pytest.mark.parametrize("K,ks", [(712, 2), (712, 3), (100, 4), (1036, 11)])
def test_ragged_k_with_ranges_it_gives(monkeypatch, K, ks):
    monkeypatch.setenv("LBR_GEMM_KSPLIT", str(ks))
    name, tile, split, got = _choice(300, 70, K)
    assert name == "gemm_mfma_f32_nt" and tile and split and got == ks


@pytest.mark.parametrize("M,N,K,batches,split", [
    (512, 3072, 768, 1, False), (1023, 1909, 768, 1, False), (1024, 1909, 768, 1, True), (2, 1 << 13, 1 << 13, 12, True),
    (1024, 2304, 768, 1, False),   # measured: an fp32 tile is faster
    (1024, 2304, 768, 2, True), (1024, 3072, 768, 1, True), (1024, 768, 3072, 1, True)])
def test_family_of_a_gemm(monkeypatch, M, N, K, batches, split):
    """Above 1.5e9 multiply-adds the split-bf16 kernel, but for sizes measured to be faster without."""
    name, tile, got, _ = _choice(M, N, K, batches)
    assert (name, got) == ("gemm_dma_f32_nt", split) and tile
    for force in (0, 1):
        monkeypatch.setenv("LBR_GEMM_SPLIT", str(force))
        assert _choice(M, N, K, batches)[2] == bool(force)


@pytest.mark.parametrize("K,force,split", [(200, None, True), (4, None, True), (200, "1", True), (200, "0", False),
                                           (202, None, False), (202, "1", False)])
def test_family_of_a_ragged_k(monkeypatch, K, force, split):
    """A K that is a multiple of 4 but not of 32 takes the split kernel at any size unless that is
    switched off; one that is no multiple of 4 has the register-staged kernel alone."""
    if force is not None:
        monkeypatch.setenv("LBR_GEMM_SPLIT", force)
    assert _choice(30, 70, K)[::2] == ("gemm_mfma_f32_nt", split)


def test_transposed_b_only():
    assert not _choice(2048, 2048, 2048, trans_b=0)[2]


@pytest.mark.parametrize("K", [96, 100])
@pytest.mark.parametrize("tile", ["256x256", "256x128", "128x256", "128x128", "128x64", "64x128", "64x64"])
def test_forced_tile(monkeypatch, tile, K):
    """A tile name ending in b3 gives the split kernel's tile, one without the fp32 kernel's."""
    monkeypatch.setenv("LBR_GEMM_TILE", tile + "b3")
    assert _choice(300, 70, K)[1:3] == (tile, True)
    if tile not in ("256x128", "128x256"):   # split tiles alone
        monkeypatch.setenv("LBR_GEMM_TILE", tile)
        assert _choice(300, 70, K)[1:3] == ((tile, False) if K % 32 == 0 else ("", False))
