"""Timed cases of the executor: the layers and calls of the fp32 transformers it runs.

Each case is a PyTorch model exported to a graph and compiled by ``Session``, as a user's
program does it once.  A pass is then either ``Session.run`` (host arrays in, host arrays out:
``"call": "session"``) or one launch of the compiled plan on inputs that are resident on the
GPU (``"call": "resident"``, the executor's ``upload_inputs`` / ``launch``), whose outputs are
the plan's own output buffers.

Layers come in the two styles the workloads have: "gpt" (LayerNorm, biases, tanh-GELU,
multi-head causal attention) and "qwen" (RMSNorm, no biases, per-head Q/K RMSNorm, RoPE,
grouped K/V heads, SiLU-gated feed-forward).
"""

import math
import os
import sys

import numpy as np
import torch
import torch.nn as nn
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "lets-build-a-runtime_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from runtime.exporter import export_model  # noqa: E402
from runtime.session import Session  # noqa: E402

EPS = {"gpt": 1e-5, "qwen": 1e-6}
THETA = 1e6


# ---------------------------------------------------------------- the models

class RMSNorm(nn.Module):
    def __init__(self, width, eps):
        super().__init__()
        self.weight = nn.Parameter(torch.empty(width))
        self.eps = eps

    def forward(self, x):
        return self.weight * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + self.eps))


def norm_of(style, width):
    return nn.LayerNorm(width, eps=EPS[style]) if style == "gpt" else RMSNorm(width, EPS[style])


def rotate_half(x):
    half = x.shape[-1] // 2
    return torch.cat((-x[..., half:], x[..., :half]), dim=-1)


class Attention(nn.Module):
    """x + O(attention(norm(x))): causal, or with an additive mask given as an input."""

    def __init__(self, c):
        super().__init__()
        self.style, self.heads, self.kv, self.hd = c["style"], c["heads"], c["kv_heads"], c["head_dim"]
        self.masked = c["mask"]
        bias = self.style == "gpt"
        self.norm = norm_of(self.style, c["width"])
        self.q = nn.Linear(c["width"], self.heads * self.hd, bias=bias)
        self.k = nn.Linear(c["width"], self.kv * self.hd, bias=bias)
        self.v = nn.Linear(c["width"], self.kv * self.hd, bias=bias)
        self.o = nn.Linear(self.heads * self.hd, c["width"], bias=bias)
        if self.style == "qwen":
            self.q_norm, self.k_norm = RMSNorm(self.hd, EPS["qwen"]), RMSNorm(self.hd, EPS["qwen"])
            self.register_buffer("cos", torch.empty(1, 1, c["seq"], self.hd))
            self.register_buffer("sin", torch.empty(1, 1, c["seq"], self.hd))

    def forward(self, x, mask=None):
        b, s = x.shape[0], x.shape[1]
        h = self.norm(x)
        q = self.q(h).view(b, s, self.heads, self.hd)
        k = self.k(h).view(b, s, self.kv, self.hd)
        v = self.v(h).view(b, s, self.kv, self.hd).transpose(1, 2)
        if self.style == "qwen":
            q, k = self.q_norm(q).transpose(1, 2), self.k_norm(k).transpose(1, 2)
            q = q * self.cos + rotate_half(q) * self.sin
            k = k * self.cos + rotate_half(k) * self.sin
        else:
            q, k = q.transpose(1, 2), k.transpose(1, 2)
        if self.masked:
            a = F.scaled_dot_product_attention(q, k, v, attn_mask=mask)
        elif self.kv != self.heads:
            a = F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True)
        else:
            a = F.scaled_dot_product_attention(q, k, v, is_causal=True)
        return x + self.o(a.transpose(1, 2).reshape(b, s, self.heads * self.hd))


class Mlp(nn.Module):
    """x + W2(act(W1(norm(x)))), or the SiLU-gated form."""

    def __init__(self, c):
        super().__init__()
        self.style = c["style"]
        self.norm = norm_of(self.style, c["width"])
        bias = self.style == "gpt"
        self.up = nn.Linear(c["width"], c["hidden"], bias=bias)
        if self.style == "qwen":
            self.gate = nn.Linear(c["width"], c["hidden"], bias=False)
        self.down = nn.Linear(c["hidden"], c["width"], bias=bias)

    def forward(self, x):
        h = self.norm(x)
        if self.style == "qwen":
            return x + self.down(F.silu(self.gate(h)) * self.up(h))
        return x + self.down(F.gelu(self.up(h), approximate="tanh"))


class AddNorm(nn.Module):
    """A residual add and the norm of the sum; both are wanted."""

    def __init__(self, c):
        super().__init__()
        self.norm = norm_of(c["style"], c["width"])

    def forward(self, x, r):
        s = x + r
        return s, self.norm(s)


class Block(nn.Module):
    def __init__(self, c):
        super().__init__()
        self.attention, self.mlp = Attention(c), Mlp(c)

    def forward(self, x):
        return self.mlp(self.attention(x))


class Head(nn.Module):
    """The last norm and the vocabulary projection."""

    def __init__(self, c):
        super().__init__()
        self.norm = norm_of(c["style"], c["width"])
        self.out = nn.Linear(c["width"], c["vocab"], bias=False)

    def forward(self, x):
        return self.out(self.norm(x))


class LanguageModel(nn.Module):
    """Token ids in, logits out: embeddings, blocks, last norm, tied vocabulary projection."""

    def __init__(self, c):
        super().__init__()
        self.style = c["style"]
        self.tokens = nn.Embedding(c["vocab"], c["width"])
        if self.style == "gpt":
            self.positions = nn.Parameter(torch.empty(c["seq"], c["width"]))
        self.blocks = nn.ModuleList(Block(c) for _ in range(c["layers"]))
        self.norm = norm_of(self.style, c["width"])

    def forward(self, ids):
        x = self.tokens(ids)
        if self.style == "gpt":
            x = x + self.positions
        for b in self.blocks:
            x = b(x)
        return F.linear(self.norm(x), self.tokens.weight)


MODELS = {"attention": Attention, "mlp": Mlp, "norm": AddNorm, "block": Block, "head": Head, "lm": LanguageModel}


# ---------------------------------------------------------------- the cases

def _case(layer, style, seq, width, batch=1, heads=0, kv_heads=0, head_dim=0, hidden=0, mask=False, layers=0,
          vocab=0, call="resident", **name):
    return {"layer": layer, "style": style, "batch": batch, "seq": seq, "width": width, "heads": heads,
            "kv_heads": kv_heads or heads, "head_dim": head_dim, "hidden": hidden, "mask": mask, "layers": layers,
            "vocab": vocab, "call": call, **name}


def listed():
    return [
        # the smallest whole call: one short block, host arrays in and out; latency and launches
        _case("block", "gpt", 32, 64, heads=4, head_dim=16, hidden=256, call="session", name="block_toy_session"),
        # three ragged sequences through a block whose widths are no multiples of a tile
        _case("block", "gpt", 77, 200, batch=3, heads=5, head_dim=40, hidden=712, name="block_ragged"),
        # the layers of a GPT-2-width block at a short context
        _case("attention", "gpt", 512, 768, heads=12, head_dim=64, name="attention_512x768"),
        _case("mlp", "gpt", 512, 768, hidden=3072, name="mlp_512x768"),
        # two padded sequences: the pattern comes as an additive mask
        _case("attention", "gpt", 333, 768, batch=2, heads=12, head_dim=64, mask=True, name="attention_masked"),
        # the layers of a 4B grouped-query model over a 1024-token prompt
        _case("attention", "qwen", 1024, 2560, heads=32, kv_heads=8, head_dim=128, name="attention_gqa_1024x2560"),
        _case("mlp", "qwen", 1024, 2560, hidden=9728, name="mlp_gated_1024x2560"),
        # the same model's block on a single token: every weight read for one row
        _case("block", "qwen", 1, 2560, heads=32, kv_heads=8, head_dim=128, hidden=9728, name="block_one_token"),
        # residual add and norm over long rows, the memory-bound part of every layer
        _case("norm", "gpt", 4096, 4096, batch=4, name="add_norm_16384x4096"),
        # a 7B model's layers at a 4096-token context, the largest work
        _case("attention", "gpt", 4096, 4096, heads=32, head_dim=128, name="attention_4096x4096"),
        _case("mlp", "gpt", 4096, 4096, hidden=16384, name="mlp_4096x4096"),
        # a whole model call: 128 token ids in, logits of the full vocabulary out, on the host
        _case("lm", "gpt", 128, 768, heads=12, head_dim=64, hidden=3072, layers=2, vocab=50257, call="session",
              name="lm_128_session"),
    ]


def _spread(rng, low, high):
    """A whole number from low to high, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        layer = rng.choice(("attention", "attention", "mlp", "mlp", "norm", "block", "head", "lm"))
        style = rng.choice(("gpt", "qwen"))
        batch = rng.choice((1, 1, 1, 2, 3))
        seq = _spread(rng, 1, 4096 // batch)
        head_dim = rng.choice((16, 24, 32, 40, 64, 64, 80, 96, 128, 128))
        heads = _spread(rng, 1, min(32, 4096 // head_dim))
        kv = heads // rng.choice([g for g in (1, 2, 4) if heads % g == 0]) if style == "qwen" else heads
        mask = layer == "attention" and batch * heads * seq * seq <= 1 << 26 and rng.random() < 0.25
        if layer == "norm":
            c = _case(layer, style, seq, _spread(rng, 64, 8192), batch=batch)
        elif layer == "head":
            c = _case(layer, style, seq, heads * head_dim, batch=batch, vocab=_spread(rng, 1000, 64000))
        else:
            width = heads * head_dim
            hidden = rng.randint(2 * width, 4 * width) if rng.random() < 0.4 else 4 * width
            c = _case(layer, style, seq, width, batch=batch, heads=heads, kv_heads=kv, head_dim=head_dim,
                      hidden=0 if layer == "attention" else hidden, mask=mask,
                      layers=rng.randint(1, 3) if layer == "lm" else 0,
                      vocab=_spread(rng, 1000, 50257) if layer == "lm" else 0,
                      call=rng.choice(("resident", "session")) if layer in ("block", "lm") else "resident")
        w = work(c)
        if w["flops"] <= most and w["bytes"] <= 2e9:
            return c


def _sizes(c):
    """(elements of the weights, elements in and out, flops) of one pass."""
    rows, d, bias = c["batch"] * c["seq"], c["width"], c["style"] == "gpt"
    qo, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    norm = d * (2 if bias else 1)
    att_w = norm + d * (2 * qo + 2 * kv) + ((qo + 2 * kv + d) if bias else 2 * c["head_dim"])
    pairs = c["seq"] ** 2 if c["mask"] else c["seq"] * (c["seq"] + 1) // 2
    att_f = 2 * rows * d * (2 * qo + 2 * kv) + 4 * c["batch"] * qo * pairs
    mlp_w = norm + c["hidden"] * d * (2 if bias else 3) + (c["hidden"] + d if bias else 0)
    mlp_f = 2 * rows * c["hidden"] * d * (2 if bias else 3)
    io = 2 * rows * d
    if c["layer"] == "attention":
        return att_w, io + (c["batch"] * c["heads"] * c["seq"] ** 2 if c["mask"] else 0), att_f
    if c["layer"] == "mlp":
        return mlp_w, io, mlp_f
    if c["layer"] == "block":
        return att_w + mlp_w, io, att_f + mlp_f
    if c["layer"] == "norm":
        return norm, 2 * io, 8 * rows * d
    if c["layer"] == "head":
        return norm + c["vocab"] * d, rows * (d + c["vocab"]), 2 * rows * d * c["vocab"]
    # embeddings: the vocabulary table is read whole by the tied projection
    return (c["layers"] * (att_w + mlp_w) + norm + c["vocab"] * d + (c["seq"] * d if bias else 0),
            rows * (2 + c["vocab"]), c["layers"] * (att_f + mlp_f) + 2 * rows * d * c["vocab"])


def work(case):
    weights, io, flops = _sizes(case)
    return {"bytes": 4 * (weights + io), "flops": flops}


# ---------------------------------------------------------------- a state

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rope(case):
    """Rotary tables of the case's positions, [1, 1, seq, head_dim]."""
    if case["style"] != "qwen" or not case["heads"]:
        return {}
    freq = 1.0 / THETA ** (torch.arange(0, case["head_dim"], 2, dtype=torch.float64) / case["head_dim"])
    angle = torch.arange(case["seq"], dtype=torch.float64)[:, None] * freq[None]
    angle = torch.cat((angle, angle), dim=-1)[None, None]
    return {"cos": angle.cos().float(), "sin": angle.sin().float()}


def _make(case, seed):
    """The case's model (fp32, on the host) and its inputs, from the seed alone."""
    dev = _device()
    gen = torch.Generator(dev).manual_seed(seed * 7919 + 13)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    with torch.device("meta"):
        model = MODELS[case["layer"]](case)
    rope, params = _rope(case), {}
    for name, p in model.named_parameters():
        scale = p.dim() < 2 and not name.endswith("bias")   # a norm's scale is near one
        params[name] = (1.0 + 0.1 * randn(*p.shape) if scale else 0.02 * randn(*p.shape)).cpu()
    for name, _ in model.named_buffers():
        params[name] = rope[name.rsplit(".", 1)[-1]]
    model.load_state_dict(params, strict=True, assign=True)
    model = model.eval().requires_grad_(False)
    b, s, d = case["batch"], case["seq"], case["width"]
    if case["layer"] == "lm":
        inputs = [torch.randint(0, case["vocab"], (b, s), generator=gen, device=dev)]
    else:
        inputs = [randn(b, s, d)]
    if case["layer"] == "norm":
        inputs.append(randn(b, s, d))
    if case["mask"]:
        # causal, and each sequence ends in some padding that no row looks at
        keep = torch.randint(max(1, s // 2), s + 1, (b,), generator=gen, device=dev)
        at = torch.arange(s, device=dev)
        off = (at[None, :] > at[:, None])[None] | (at[None, None, :] >= keep[:, None, None])
        m = torch.zeros(b, s, s, device=dev).masked_fill(off, -1e9)
        inputs.append(m[:, None].expand(b, case["heads"], s, s).contiguous())
    return model, [t.cpu() for t in inputs]


class _Resident:
    """A device buffer of a session's plan, for torch to look at without a copy."""

    def __init__(self, session, address, shape):
        self.session = session   # frees the buffer when it goes
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 2}


def prepare(case, seed):
    model, inputs = _make(case, seed)
    graph = export_model(model, tuple(inputs))
    session = Session(graph)
    session.create()
    feed = {name: t.numpy() for name, t in zip(graph.inputs, inputs)}
    state = {"session": session, "feed": feed, "call": case["call"]}
    if case["call"] == "resident":
        ex = session.executor
        ex.upload_inputs(feed)
        state["outputs"] = []
        for n in graph.outputs:
            t = torch.as_tensor(_Resident(session, ex.device_address(n), tuple(graph.tensors[n].shape)), device="cuda")
            t.session = session   # an output may outlive the state: its buffer has to, too
            state["outputs"].append(t)
    return state


def run(state):
    if state["call"] == "session":
        return list(state["session"].run(state["feed"]).values())
    state["session"].executor.launch()
    return state["outputs"]


def exact(case, seed):
    model, inputs = _make(case, seed)
    dev = _device()
    model = model.to(dev).double()
    with torch.no_grad():
        y = model(*[t.to(dev).double() if t.is_floating_point() else t.to(dev) for t in inputs])
    return list(y) if isinstance(y, tuple) else [y]


def tolerance(case):
    """About four times the distance from 64 bits that fp32 kernels were measured at: 7e-8 for
    the norms, 6e-7 for attention layers, 2.4e-6 where sums run over a feed-forward width."""
    rel = {"norm": 4e-7, "attention": 2.5e-6}.get(case["layer"], 1e-5)
    return {"rel": rel, "max": 20 * rel}
