"""A layer on one token: the GEMV's fused epilogues against the node-by-node plan (the same bits) and
a float64 closed form, and the one-row attention against the closed form and the tiled kernel."""

import numpy as np
import pytest

from conftest import normwise_rel
from helpers import cf_attention, cf_gelu_tanh, cf_silu, one_node_graph, randn, rng, run_gpu
from runtime.ir import Graph, OpType

pytestmark = pytest.mark.gpu


def _gemv(K, N, bias, r):
    """A one-row MATMUL_ADD, or without `bias` a MATMUL with an alpha that is no power of two."""
    g = Graph()
    a, w = randn(r, 1, 1, K), randn(r, N, K, scale=0.1)
    g.add_tensor("a", (1, 1, K))
    g.inputs.append("a")
    g.add_tensor("w", (N, K)).buffer = w
    g.constants.append("w")
    ins, c = ["a", "w"], a.astype(np.float64) @ w.T.astype(np.float64)
    if bias:
        b = randn(r, N)
        g.add_tensor("b", (N,)).buffer = b
        g.constants.append("b")
        ins, c = ins + ["b"], c + b
    else:
        c = c * 0.3
    g.add_tensor("c", (1, 1, N))
    g.add_node(OpType.MATMUL_ADD if bias else OpType.MATMUL, ins, "c",
               {"transpose_b": True, **({} if bias else {"alpha": 0.3})})
    return g, a, c


def _check(g, feed, ref, name):
    from runtime.executor.compiled import CompiledExecutor
    from runtime.planner import plan
    ys, names = [], []
    for fuse in (True, False):
        ex = CompiledExecutor(fuse=fuse)
        ex.compile(plan(g))
        try:
            ys.append(ex.run(feed)[g.outputs[0]])
            names.append(ex.kernel_names())
        finally:
            ex.close()
    assert names[0][0] == name and names[1][0] == "gemv_t", names
    np.testing.assert_array_equal(ys[0], ys[1])
    assert normwise_rel(ys[0], ref) <= 1e-5


@pytest.mark.parametrize("K,N,bias", [(256, 130, True), (33, 7, False), (2560, 4, True), (256, 1000, False)])
def test_gemv_residual(K, N, bias):
    r = rng(K + N)
    g, a, c = _gemv(K, N, bias, r)
    x = randn(r, 1, 1, N)
    g.add_tensor("x", (1, 1, N))
    g.inputs.append("x")
    g.add_tensor("y", (1, 1, N))
    g.add_node(OpType.ADD, ["c", "x"], "y", {})
    g.outputs.append("y")
    _check(g, {"a": a, "x": x}, c + x, "gemv_t+resid")


@pytest.mark.parametrize("op,cf", [(OpType.GELU, cf_gelu_tanh), (OpType.SILU, cf_silu)])
@pytest.mark.parametrize("K,N,bias", [(256, 130, True), (33, 7, False)])
def test_gemv_activation(op, cf, K, N, bias):
    g, a, c = _gemv(K, N, bias, rng(K))
    g.add_tensor("y", (1, 1, N))
    g.add_node(op, ["c"], "y", {})
    g.outputs.append("y")
    _check(g, {"a": a}, cf(c), "gemv_t+act")


@pytest.mark.parametrize("K,F,bias,gbias,order", [(256, 130, False, False, 0), (33, 7, True, True, 1),
                                                  (2560, 1, False, True, 0)])
def test_gemv_gated(K, F, bias, gbias, order):
    r = rng(K + F)
    g, a, c = _gemv(K, 2 * F, bias, r)
    for k in (0, 1):
        g.add_tensor(f"s{k}", (1, 1, F))
        g.add_node(OpType.SLICE, ["c"], f"s{k}", {"dim": 2, "start": k * F, "end": (k + 1) * F})
    halves = [c[..., :F], c[..., F:]]
    x, up = halves[order], halves[1 - order]
    ins = [f"s{order}", f"s{1 - order}"]
    if gbias:
        gb = randn(r, F)
        g.add_tensor("gb", (F,)).buffer = gb
        g.constants.append("gb")
        ins.insert(1, "gb")
        x = x + gb
    g.add_tensor("y", (1, 1, F))
    g.add_node(OpType.GATED_ACT, ins, "y", {"has_bias": gbias, "act": "silu"})
    g.outputs.append("y")
    _check(g, {"a": a}, cf_silu(x) * up, "gemv_t+gated")


@pytest.mark.parametrize("bh,group,hd,causal", [(32, 4, 128, True), (5, 1, 8, False), (3, 3, 40, True), (1, 1, 64, False)])
def test_attention_one_row(monkeypatch, bh, group, hd, causal):
    r = rng(bh + hd)
    q, k, v = randn(r, 1, bh, 1, hd), randn(r, 1, bh // group, 1, hd), randn(r, 1, bh // group, 1, hd)
    q[0, 0, 0, 0] = np.inf if bh > 3 else q[0, 0, 0, 0]   # a score that is not finite: the row is NaN
    attrs = {"causal": causal, **({"group_size": group} if group > 1 else {})}
    g = one_node_graph(OpType.ATTENTION, {"q": q, "k": k, "v": v}, q.shape, attrs)
    names = []
    y = run_gpu(g, {"q": q, "k": k, "v": v}, kernels=names)
    assert names == ["attn_one_f32"]
    monkeypatch.setenv("LBR_ATTN_FOLD", "0")
    np.testing.assert_array_equal(y, run_gpu(g, {"q": q, "k": k, "v": v}))
    ok = np.isfinite(y)
    assert ok.all() or bh > 3
    assert normwise_rel(y[ok], cf_attention(q, k, v, causal=causal, group=group)[ok]) <= 1e-6


@pytest.mark.parametrize("H,Hkv,hd,K", [(4, 2, 32, 96), (3, 3, 20, 33)])
def test_gemv_heads(H, Hkv, hd, K):
    r = rng(K)
    g, a, c = _gemv(K, (H + 2 * Hkv) * hd, True, r)
    col, qkv = 0, []
    for k, h in enumerate((H, Hkv, Hkv)):
        wd = h * hd
        g.add_tensor(f"s{k}", (1, 1, wd))
        g.add_node(OpType.SLICE, ["c"], f"s{k}", {"dim": 2, "start": col, "end": col + wd})
        g.add_tensor(f"h{k}", (1, 1, h, hd))
        g.add_node(OpType.RESHAPE, [f"s{k}"], f"h{k}", {"shape": (1, 1, h, hd)})
        g.add_tensor(f"t{k}", (1, h, 1, hd))
        g.add_node(OpType.TRANSPOSE, [f"h{k}"], f"t{k}", {"dim0": 1, "dim1": 2})
        qkv.append(c[..., col:col + wd].reshape(1, h, 1, hd))
        col += wd
    g.add_tensor("y", (1, H, 1, hd))
    g.add_node(OpType.ATTENTION, ["t0", "t1", "t2"], "y", {"causal": True, **({"group_size": H // Hkv} if H > Hkv else {})})
    g.outputs.append("y")
    _check(g, {"a": a}, cf_attention(*qkv, causal=True, group=H // Hkv), "gemv_t+heads")
