"""The RoPE window in any order its nodes can run in: the matcher takes every one, and a model that
exports another order than transformers' gives, fused, what it gives node by node."""

from itertools import permutations

import numpy as np
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from conftest import normwise_rel
from test_fusion import MB, _rope_chain, _windows


def test_rope_window_in_every_order():
    nodes = _rope_chain(0, 8 * MB)
    head, (mc, s1, s2, ng, ct, ms, ad) = nodes[:3], nodes[3:]
    before = [(2, 3), (1, 4), (3, 4), (4, 5)]   # s2 → neg, s1 → cat, neg → cat, cat → ·sin
    seen = 0
    for p in permutations(range(6)):
        if any(p.index(a) > p.index(b) for a, b in before):
            continue
        win = [(mc, s1, s2, ng, ct, ms)[k] for k in p]
        assert _windows(head + win + [ad]) == [(0, 10, "head_prologue")], p
        seen += 1
    assert seen == 18
    # CAT where x was (x is dead by then): its product is the one that reads it last
    over = _rope_chain(0, 8 * MB)
    x = over[2].output
    over[7].output = x
    over[8].inputs[0] = x
    assert _windows(over) == [(0, 10, "head_prologue")]
    # ... but not before q·cos has read x
    assert _windows(over[:3] + [over[k] for k in (4, 5, 6, 7, 3, 8, 9)]) == [(0, 3, "head_prologue")]
    # the same slice twice, or a NEG too many, is no window
    assert _windows(head + [mc, s2, s2, ng, ct, ms, ad]) == [(0, 3, "head_prologue")]
    assert _windows(head + [mc, s1, ng, ng, ct, ms, ad]) == [(0, 3, "head_prologue")]


class _Layer(nn.Module):
    """Grouped-query attention with per-head Q/K norm; rotate_half negates between its slices."""

    def __init__(self, width, heads, kv, hd, seq):
        super().__init__()
        self.heads, self.kv, self.hd = heads, kv, hd
        self.q, self.k, self.v = (nn.Linear(width, h * hd, bias=False) for h in (heads, kv, kv))
        self.qn, self.kn = nn.Parameter(torch.rand(hd) + 0.5), nn.Parameter(torch.rand(hd) + 0.5)
        a = torch.arange(seq)[:, None] / 1e4 ** (torch.arange(0, hd, 2) / hd)
        a = torch.cat((a, a), -1)[None, None]
        self.register_buffer("cos", a.cos())
        self.register_buffer("sin", a.sin())

    def forward(self, x):
        b, s, _ = x.shape

        def head(lin, w, n):
            h = lin(x).view(b, s, n, self.hd)
            h = w * (h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-6))
            h = h.transpose(1, 2)
            half = self.hd // 2
            return h * self.cos + torch.cat((-h[..., half:], h[..., :half]), -1) * self.sin
        q, k = head(self.q, self.qn, self.heads), head(self.k, self.kn, self.kv)
        v = self.v(x).view(b, s, self.kv, self.hd).transpose(1, 2)
        y = F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=self.kv != self.heads)
        return y.transpose(1, 2).reshape(b, s, self.heads * self.hd)


@pytest.mark.gpu
@pytest.mark.parametrize("S,hd,H,kv,batch", [(1, 128, 8, 2, 1), (70, 64, 6, 6, 2), (200, 128, 4, 2, 1)])
def test_rope_other_order_fused_equals_unfused(monkeypatch, S, hd, H, kv, batch):
    from runtime.exporter import export_model
    from runtime.session import Session
    torch.manual_seed(S + hd)
    m = _Layer(256, H, kv, hd, S).eval()
    x = torch.randn(batch, S, 256)
    ys, kinds = [], []
    for fuse in ("1", "0"):
        monkeypatch.setenv("LBR_FUSE", fuse)
        g = export_model(m, (x,))
        s = Session(g)
        s.create()
        ys.append(s.run({g.inputs[0]: x.numpy()})[g.outputs[0]])
        kinds.append([k for _, _, k in s.executor.fused_runs()])
        s.close()
    assert {"head_prologue", "gemm_head_prologue"} & set(kinds[0]) and not kinds[1], kinds
    with torch.no_grad():
        ref = m.double()(x.double()).numpy()
    assert normwise_rel(ys[0], ref) <= 1e-5 and normwise_rel(ys[1], ref) <= 1e-5
