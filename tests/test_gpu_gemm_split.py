"""The split-bf16 GEMM (gemm_split.hip): every tile at its edges against a float64 closed form, its
epilogues, operands of every exponent, and the results it hands to the fp32 matrix cores (infinities,
NaN, the largest values).

Tolerance: the sum rounds six times per 16 terms and once at the end, each time by less than 2⁻²³ of a
partial sum and by a random part of it (standard deviation 2⁻²³/√12).  Partial sums stay within three
times the root of their terms' squares (σ); √n·2⁻²³ of that, for all n roundings, is 3.5 standard
deviations were every partial sum so large: 2.2e-6 σ at K = 96, 7e-6 at 1036.  A kernel without one of its
six products would be 1.1e-5 σ or more off (emulated)."""

import numpy as np
import pytest

import test_gpu_fused_epilogues as epilogues
from conftest import normwise_rel
from helpers import one_node_graph, randn, rng, run_gpu
from runtime.ir import OpType
from test_gpu_ops import _gemm_case

pytestmark = pytest.mark.gpu



def _case(M, N, K, batches, with_bias, tile=None, ks=None, name="gemm_dma_f32_nt"):
    """A GEMM that has to run on the split kernel, with that tile (None: any) and K ranges."""
    from runtime.executor.compiled import CompiledExecutor
    from runtime.planner import plan
    r = rng(M * 7 + N + K)
    a, b = randn(r, batches, M, K), randn(r, *((N, K) if batches == 1 else (batches, N, K)))
    a64, bt64 = a.astype(np.float64), np.swapaxes(b, -2, -1).astype(np.float64)
    ref, size = a64 @ bt64, 3 * np.sqrt((a64 ** 2) @ (bt64 ** 2)).max()
    consts, attrs = {"b": b}, {"transpose_b": True}
    if with_bias:
        consts["bias"] = randn(r, N)
        ref, size = ref + consts["bias"], size + np.abs(consts["bias"]).max()
    else:
        attrs["alpha"] = 0.3
        ref, size = ref * np.float32(0.3), size * 0.3
    g = one_node_graph(OpType.MATMUL_ADD if with_bias else OpType.MATMUL, {"a": a}, (batches, M, N), attrs, consts)
    ex = CompiledExecutor()
    ex.compile(plan(g))
    try:
        step, = ex.step_params()
        y = ex.run({"a": a})["out"]
    finally:
        ex.close()
    assert step["name"] == name and step["split"], step
    assert (tile is None or step["tile"] + "b3" == tile) and (ks is None or step["ksplit"] == ks), step
    assert np.abs(y - ref).max() <= np.sqrt(6 * -(-K // 16) + 1) * 2.0 ** -23 * size


TILES = ["256x256", "256x128", "128x256", "128x128", "128x64", "64x128", "64x64"]


@pytest.mark.parametrize("tile", [t + "b3" for t in TILES])
@pytest.mark.parametrize("M,N,K,batches", [(300, 520, 96, 1), (513, 257, 64, 1), (2, 3, 32, 1), (257, 130, 160, 3)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_split_tiles(monkeypatch, tile, M, N, K, batches, with_bias):
    monkeypatch.setenv("LBR_GEMM_TILE", tile)
    monkeypatch.setenv("LBR_GEMM_KSPLIT", "1")
    _case(M, N, K, batches, with_bias, tile, 1)


@pytest.mark.parametrize("tile,ks,M,N,K", [("256x256b3", 3, 200, 300, 960), ("64x64b3", 2, 70, 130, 64)])
def test_split_ksplit(monkeypatch, tile, ks, M, N, K):
    monkeypatch.setenv("LBR_GEMM_TILE", tile)
    monkeypatch.setenv("LBR_GEMM_KSPLIT", str(ks))
    _case(M, N, K, 1, True, tile, ks)


@pytest.mark.parametrize("tile", ["256x256b3", "128x128b3", "64x128b3"])
def test_split_epilogues(monkeypatch, tile):
    epilogues.test_gemm_activation_epilogue(monkeypatch, OpType.GELU, True, tile, "1", 300, 520, 96)
    epilogues.test_gemm_gated_epilogue(monkeypatch, tile, "silu", True, 0, True)
    epilogues.test_transpose_gemm(monkeypatch, tile, "1", 12, 70, 8, 100, False, True)
    epilogues.test_transpose_gemm(monkeypatch, tile, "1", 4, 300, 64, 200, True, True)


@pytest.mark.parametrize("tile", [None, "256x256b3", "64x64b3"])
@pytest.mark.parametrize("M,N,K,batches", [(231, 200, 712, 1), (300, 70, 100, 1), (2, 5, 4, 1), (130, 260, 20, 3),
                                           (70, 130, 1036, 1)])
def test_split_ragged_k(monkeypatch, tile, M, N, K, batches):
    """K a multiple of 4 that is none of 16 or 32 (a tile forces the shape, None is the default
    choice, in K ranges where it takes them); neighbours of the last columns are another row's."""
    if tile:
        monkeypatch.setenv("LBR_GEMM_TILE", tile)
        monkeypatch.setenv("LBR_GEMM_KSPLIT", "1")
    _case(M, N, K, batches, True, tile, 1 if tile else None, "gemm_mfma_f32_nt")


@pytest.mark.parametrize("K", [20, 200, 712])
@pytest.mark.parametrize("ks", [2, 6, 16])
def test_ragged_k_under_forced_ranges(monkeypatch, K, ks):
    """Every column of a ragged K counts, whether K gives that many ranges or not."""
    monkeypatch.setenv("LBR_GEMM_KSPLIT", str(ks))
    _gemm_case(300, 70, K, True, 1, True, False)


def _run(a, b):
    M, K = a.shape
    g = one_node_graph(OpType.MATMUL, {"a": a[None]}, (1, M, b.shape[0]), {"transpose_b": True}, {"b": b})
    return run_gpu(g, {"a": a[None]})[0]


@pytest.mark.parametrize("tile", ["256x256b3", "64x64b3"])
def test_split_is_exact_where_fp32_is(monkeypatch, tile):
    """One term a result.  Times a power of two: each operand's three planes add up to its fp32 value,
    to the last bit.  Two 12-bit significands (two planes each, and an exact fp32 product): so do the
    products of their planes."""
    monkeypatch.setenv("LBR_GEMM_TILE", tile)
    monkeypatch.setenv("LBR_GEMM_KSPLIT", "1")
    b = randn(rng(5), 130, 96) * np.exp2(rng(6).integers(-20, 20, (130, 96))).astype(np.float32)
    two = np.exp2(rng(7).integers(-20, 20, 96)).astype(np.float32)
    np.testing.assert_array_equal(_run(np.diag(two), b), two[:, None] * b.T)
    np.testing.assert_array_equal(_run(b, np.diag(two)), b * two)
    d, e = (rng(s).integers(1 << 11, 1 << 12, n).astype(np.float32) for s, n in ((8, 96), (9, (130, 96))))
    np.testing.assert_array_equal(_run(np.diag(d), -e), -(d[:, None] * e.T))


@pytest.mark.parametrize("tile", ["256x256b3", "64x64b3"])
def test_split_outside_range(monkeypatch, tile):
    """Infinities, NaN, the largest finite values (infinite as scaled bf16) and tiny operands (whose
    low planes, unscaled, are no normal bf16 values) give what the fp32 kernel gives."""
    monkeypatch.setenv("LBR_GEMM_KSPLIT", "1")
    r = rng(11)
    a, b = randn(r, 200, 96), randn(r, 150, 96)
    a[3, 7] = np.inf
    a[4, 9] = -np.inf
    a[5, [1, 2]] = [np.inf, -np.inf]
    a[70, 5] = np.nan
    b[9, 40] = np.inf
    b[9, :40] = 1.0
    a[100] = 0.0
    a[100, 11] = np.finfo(np.float32).max
    b[:, 11] = np.sign(b[:, 11]) * 0.5
    a[101] *= np.float32(1e-33)
    a[102] *= np.float32(1e-36)
    outs = {}
    for t in (tile, "64x64"):
        monkeypatch.setenv("LBR_GEMM_TILE", t)
        outs[t] = _run(a, b)
    x, y = outs[tile], outs["64x64"]
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    np.testing.assert_array_equal(x[np.isinf(y)], y[np.isinf(y)])
    np.testing.assert_array_equal(np.isinf(x), np.isinf(y))
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    for rows in ([100], [101], [102], [0, 1, 2, 60, 199]):   # each range by its own size
        ok = np.isfinite(y[rows])
        assert normwise_rel(x[rows][ok], ref[rows][ok]) <= 1e-5


@pytest.mark.parametrize("tile", ["256x256b3", "64x64b3"])
def test_split_operand_range(monkeypatch, tile):
    """Operands of every exponent, subnormals included, against small and large ones: no bit of an
    operand is lost.  Bound: 6 roundings down (2⁻²³ of the partial sum each) per 16 terms, and the
    products left out (2⁻²⁴ of a product); results below the fp32 range to its last bit."""
    monkeypatch.setenv("LBR_GEMM_TILE", tile)
    monkeypatch.setenv("LBR_GEMM_KSPLIT", "1")
    r, K = rng(21), 96
    ea = np.repeat([-145, -140, -136, -134, -130, -125, -120, -111, -100, -60, 0, 60, 100, 120], 5)
    eb = np.repeat([-140, -120, -60, 0, 15, 40, 50, 51, 80, 100, 110, 122], 11)
    a, b = (np.ldexp(r.standard_normal((len(e), K)), e[:, None]).astype(np.float32) for e in (ea, eb))
    y = _run(a, b).astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    ref, size = a @ b.T, np.abs(a) @ np.abs(b).T
    tol = (6 * K / 16 + 1) * 2.0 ** -23 * size + K * 2.0 ** -149
    fits = size < 2.0 ** 127
    assert fits.sum() > 8000
    bad = fits & ~(np.abs(y - ref) <= tol)
    assert not bad.any(), sorted({(int(ea[i]), int(eb[j])) for i, j in zip(*np.nonzero(bad))})


@pytest.mark.parametrize("K", [64, 128, 200, 256])
def test_split_mean_error_of_short_k(monkeypatch, K):
    """The sum changes sign within a short K too, so that its roundings down do not add up: the mean
    error of 512x512 results, whose own spread is 2.4e-7 / 512 = 5e-10 of their rms, is within 7e-9 of
    it (one sign throughout gives 7e-9 at K = 64, 1.3e-8 at 200, 1.5e-8 at 256)."""
    monkeypatch.setenv("LBR_GEMM_TILE", "64x64b3")
    monkeypatch.setenv("LBR_GEMM_KSPLIT", "1")
    r = rng(K)
    a, b = randn(r, 512, K), randn(r, 512, K)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    err, rms = _run(a, b) - ref, np.sqrt((ref ** 2).mean())
    assert abs(err.mean()) <= 7e-9 * rms
    assert np.sqrt((err ** 2).mean()) <= 3e-7 * rms
