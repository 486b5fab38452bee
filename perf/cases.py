"""Performance cases of the framework's public entry points, for timing and comparing outputs.

Every case is a dict of plain values; ``kind`` names the entry point that a pass calls:

* ``train``    -- ``flash_attn`` forward and backward through autograd (bf16 or fp32)
* ``prefill``  -- ``flash_attn`` forward alone, as when a prompt is read
* ``varlen``   -- ``flash_attn_varlen`` forward and backward over packed sequences
* ``decode``   -- ``flash_attn_decode``: new query rows against a KV cache
* ``prologue`` -- ``qk_norm_rope`` forward and backward through autograd
* ``layer``    -- the ``Attention`` block with ``attn_impl="hip"`` and the fused prologue,
  forward and backward under bf16 autocast

Inputs follow the distributions of ``tinytrain_amd.workloads``: q and k unit-RMS per head
(what the q/k norms produce), v ~ N(0, 1), the upstream gradient N(0, 1) * 1e-2 in bf16
and N(0, 1) in fp32.
"""

from __future__ import annotations

import math
import random

import torch

from tinytrain_amd.attention import Attention, precompute_rope
from tinytrain_amd.kernels.decode import flash_attn_decode
from tinytrain_amd.kernels.flash_attn import flash_attn, flash_attn_varlen
from tinytrain_amd.kernels.qk_prologue import qk_norm_rope

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
_HIDDEN = 768          # hidden size of the 112M model's layer
_ROPE_BASE = 1e6
_EPS = 1e-6


# ------------------------------------------------------------------------------- cases

def _attn(name, kind, B, Hq, Hkv, T, D, dtype="bf16"):
    return {"name": name, "kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "T": T, "D": D, "dtype": dtype}


def listed():
    return [
        # The tiny fp32 model that checks a training set-up: every launch counts.
        _attn("train_fp32_tiny", "train", 2, 4, 4, 256, 64, "fp32"),
        # fp32 attention of a debugging run at the 112M model's head shape, ragged length.
        _attn("train_fp32_gqa", "train", 2, 8, 2, 500, 128, "fp32"),
        # Fine-tuning on a small batch of short examples padded to an odd length.
        _attn("train_small_ragged", "train", 3, 8, 2, 333, 128),
        # 112M pretraining, multi-head.
        _attn("train_112m_mha", "train", 16, 12, 12, 1024, 64),
        # The reference model's own shape and batch, GQA 4.
        _attn("train_112m_gqa", "train", 32, 8, 2, 512, 128),
        # Long-context training, one sequence (the largest case).
        _attn("train_long", "train", 1, 16, 8, 16384, 128),
        # Reading one user's prompt before generating.
        _attn("prefill_prompt", "prefill", 1, 16, 8, 777, 128),
        # Packed pretraining documents of mixed lengths.
        {"name": "varlen_packed", "kind": "varlen", "tokens": 16384, "longest": 2048, "mix": 1,
         "Hq": 12, "Hkv": 12, "D": 64},
        # A serving batch: caches of one capacity, every request at its own position.
        {"name": "decode_batch", "kind": "decode", "B": 32, "Hq": 16, "Hkv": 8, "Tq": 1,
         "L": 4096, "D": 128, "least": 0.1, "mix": 1},
        # Interactive generation with the 112M model: one short cache.
        {"name": "decode_single", "kind": "decode", "B": 1, "Hq": 8, "Hkv": 2, "Tq": 1,
         "L": 512, "D": 128, "least": 0.5, "mix": 2},
        # The step between projections and attention at the 112M model's training shape.
        {"name": "prologue_112m", "kind": "prologue", "B": 32, "Hq": 8, "Hkv": 2, "T": 512,
         "D": 128},
        # A whole attention block of the 112M model in training.
        {"name": "layer_112m", "kind": "layer", "B": 16, "Hq": 8, "Hkv": 2, "T": 512, "D": 128},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of lo..hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_HEADS = {64: [(12, 12), (12, 4), (4, 4), (8, 2)], 128: [(16, 8), (8, 2), (8, 8), (6, 2)]}


def draw(rng: random.Random):
    kind = rng.choice(["train", "train", "train", "train", "prefill", "varlen", "decode", "decode",
                       "prologue", "layer"])
    D = rng.choice([64, 128])
    Hq, Hkv = rng.choice(_HEADS[D])
    if kind == "decode":
        B = _log(rng, 1, 64)
        L = min(_log(rng, 200, 16384), 262144 // B)  # the caches of a batch share the memory
        Tq = rng.choice([1, 1, 1, 2, 4])
        return {"kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "Tq": Tq, "L": L, "D": D,
                "least": rng.choice([0.1, 0.5, 1.0]), "mix": rng.randrange(1 << 20)}
    if kind == "varlen":
        tokens = _log(rng, 1000, 32768)
        return {"kind": kind, "tokens": tokens, "longest": min(tokens, _log(rng, 200, 4096)),
                "mix": rng.randrange(1 << 20), "Hq": Hq, "Hkv": Hkv, "D": D}
    if kind == "train" and rng.random() < 0.25:
        T = _log(rng, 32, 1024)
        return {"kind": kind, "B": max(1, _log(rng, T, 2048) // T), "Hq": Hq, "Hkv": Hkv, "T": T,
                "D": D, "dtype": "fp32"}
    if kind == "train":
        T = _log(rng, 64, 8192)
        return {"kind": kind, "B": max(1, _log(rng, T, 32768) // T), "Hq": Hq, "Hkv": Hkv, "T": T,
                "D": D, "dtype": "bf16"}
    if kind == "prefill":
        T = _log(rng, 32, 8192)
        return {"kind": kind, "B": max(1, _log(rng, T, 16384) // T), "Hq": Hq, "Hkv": Hkv, "T": T,
                "D": D, "dtype": "bf16"}
    T = _log(rng, 64, 2048)
    return {"kind": kind, "B": max(1, _log(rng, T, 16384) // T), "Hq": Hq, "Hkv": Hkv, "T": T,
            "D": D}


# ------------------------------------------------------------------------------ inputs

def _lengths(case):
    """Lengths of the packed sequences, or of the caches in use, from the case alone."""
    r = random.Random(case["mix"])
    if case["kind"] == "decode":
        lo = max(case["Tq"], int(case["least"] * case["L"]))
        return [r.randint(lo, case["L"]) for _ in range(case["B"])]
    lens, left = [], case["tokens"]
    while left > 0:
        n = min(left, r.randint(max(1, case["longest"] // 32), case["longest"]))
        lens.append(n)
        left -= n
    return lens


def _unit_rms(x):
    return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + _EPS)


class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator("cuda").manual_seed(seed)

    def __call__(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda")


def _leaf(x, dtype):
    return x.to(dtype).contiguous().requires_grad_()


def prepare(case, seed):
    rand, kind = _Draw(seed), case["kind"]
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    if kind in ("train", "prefill"):
        B, T, dt = case["B"], case["T"], _DTYPES[case["dtype"]]
        q, k, v = _unit_rms(rand(B, Hq, T, D)), _unit_rms(rand(B, Hkv, T, D)), rand(B, Hkv, T, D)
        if kind == "prefill":
            return {"kind": kind, "q": q.to(dt), "k": k.to(dt), "v": v.to(dt)}
        do = rand(B, Hq, T, D) * (1e-2 if dt == torch.bfloat16 else 1.0)
        return {"kind": kind, "q": _leaf(q, dt), "k": _leaf(k, dt), "v": _leaf(v, dt), "do": do.to(dt)}
    if kind == "varlen":
        lens, n, dt = _lengths(case), case["tokens"], torch.bfloat16
        cu = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
        return {"kind": kind, "q": _leaf(_unit_rms(rand(Hq, n, D)), dt),
                "k": _leaf(_unit_rms(rand(Hkv, n, D)), dt), "v": _leaf(rand(Hkv, n, D), dt),
                "do": (rand(Hq, n, D) * 1e-2).to(dt), "cu": cu, "longest": max(lens)}
    if kind == "decode":
        B, L, dt = case["B"], case["L"], torch.bfloat16
        return {"kind": kind, "q": _unit_rms(rand(B, Hq, case["Tq"], D)).to(dt),
                "k": _unit_rms(rand(B, Hkv, L, D)).to(dt), "v": rand(B, Hkv, L, D).to(dt),
                "lens": torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")}
    B, T, dt = case["B"], case["T"], torch.bfloat16
    cos, sin = (t.cuda() for t in precompute_rope(D, T, _ROPE_BASE))
    if kind == "prologue":
        s = {"kind": kind, "q": _leaf(rand(B, T, Hq, D), dt), "k": _leaf(rand(B, T, Hkv, D), dt),
             "v": _leaf(rand(B, T, Hkv, D), dt), "cos": cos, "sin": sin}
        for name in ("wq", "wk"):
            s[name] = _leaf(1.0 + 0.1 * rand(D), torch.float32)
        s["grads"] = [(rand(B, h, T, D) * 1e-2).to(dt) for h in (Hq, Hkv, Hkv)]
        return s
    layer = Attention(_HIDDEN, Hq, Hkv, D).cuda()
    layer.attn_impl, layer.fused_prologue = "hip", True
    with torch.no_grad():
        for w in layer.parameters():
            w.copy_(rand(*w.shape) * 0.02 if w.dim() == 2 else 1.0 + 0.1 * rand(*w.shape))
    return {"kind": kind, "layer": layer, "x": _leaf(rand(B, T, _HIDDEN), dt), "cos": cos, "sin": sin,
            "dy": (rand(B, T, _HIDDEN) * 1e-2).to(dt)}


# -------------------------------------------------------------------------------- pass

def run(state):
    s, kind = state, state["kind"]
    if kind == "train":
        o = flash_attn(s["q"], s["k"], s["v"])
        return (o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"]))
    if kind == "prefill":
        with torch.no_grad():
            return flash_attn(s["q"], s["k"], s["v"])
    if kind == "varlen":
        o = flash_attn_varlen(s["q"], s["k"], s["v"], s["cu"], s["longest"])
        return (o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"]))
    if kind == "decode":
        return flash_attn_decode(s["q"], s["k"], s["v"], s["lens"])
    if kind == "prologue":
        out = qk_norm_rope(s["q"], s["k"], s["v"], s["wq"], s["wk"], s["cos"], s["sin"], _EPS)
        ins = (s["q"], s["k"], s["v"], s["wq"], s["wk"])
        return (*out, *torch.autograd.grad(out, ins, s["grads"]))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = s["layer"](s["x"], s["cos"], s["sin"])
    return (y, *torch.autograd.grad(y, (s["x"], *s["layer"].parameters()), s["dy"]))


# -------------------------------------------------------------------------------- work

def _causal_work(pairs, rows, Hq, Hkv, D, size, backward):
    """Bytes and flops of causal attention over `pairs` visible (row, key) pairs a head."""
    row = D * size
    fwd = rows * (2 * Hq + 2 * Hkv) * row + rows * Hq * 4            # q, k, v -> o, lse
    bwd = rows * (2 * Hq + 2 * Hkv) * row if backward else 0         # do -> dq, dk, dv
    return {"bytes": fwd + bwd, "flops": (14 if backward else 4) * D * Hq * pairs}


def work(case):
    kind, Hq, Hkv, D = case["kind"], case["Hq"], case["Hkv"], case["D"]
    if kind == "varlen":
        lens = _lengths(case)
        return _causal_work(sum(n * (n + 1) // 2 for n in lens), sum(lens), Hq, Hkv, D, 2, True)
    if kind == "decode":
        lens, rows = _lengths(case), case["B"] * Hq * case["Tq"]
        return {"bytes": sum(lens) * Hkv * D * 4 + rows * (D * 4 + 4),
                "flops": 4 * D * Hq * case["Tq"] * sum(lens)}
    B, T = case["B"], case["T"]
    if kind in ("train", "prefill"):
        return _causal_work(B * T * (T + 1) // 2, B * T, Hq, Hkv, D, 2 if case["dtype"] == "bf16" else 4,
                            kind == "train")
    heads = Hq + 2 * Hkv
    if kind == "prologue":  # forward reads and writes every head; so does the backward, which
        return {"bytes": B * T * D * 2 * (4 * heads + Hq + Hkv) + 8 * T * D,  # re-reads q, k raw
                "flops": 40 * B * T * (Hq + Hkv) * D}
    weights = _HIDDEN * D * (heads + Hq)
    a = _causal_work(B * T * (T + 1) // 2, B * T, Hq, Hkv, D, 2, True)
    return {"bytes": B * T * _HIDDEN * 2 * 4 + weights * 8, "flops": 6 * B * T * weights + a["flops"]}


def tolerance(case):
    """About four times the error against exact(): fp32 6e-7, bf16 ops 2.5e-3, the block 8e-3."""
    if case.get("dtype") == "fp32":
        return {"rel": 2.5e-6}
    if case["kind"] == "layer":
        return {"rel": 3e-2}
    return {"rel": 1e-2}


# ------------------------------------------------------------------------ 64-bit results

def _attn_exact(q, k, v, do=None):
    """Causal attention of [T, D] rows of one head group: q/do [G, T, D], k/v [T, D] fp64."""
    T, D = k.shape
    scale = 1.0 / math.sqrt(D)
    mask = torch.ones(T, T, dtype=torch.bool, device=k.device).triu(1)
    o, dq, dk, dv = [], [], torch.zeros_like(k), torch.zeros_like(v)
    for g in range(q.shape[0]):
        p = torch.softmax((q[g] @ k.t() * scale).masked_fill_(mask, -math.inf), dim=-1)
        o.append(p @ v)
        if do is not None:
            dv += p.t() @ do[g]
            ds = do[g] @ v.t()
            ds.sub_((do[g] * o[-1]).sum(-1, keepdim=True)).mul_(p).mul_(scale)
            dq.append(ds @ k)
            dk += ds.t() @ q[g]
    return torch.stack(o), (torch.stack(dq), dk, dv) if do is not None else None


def _batch_exact(q, k, v, do=None):
    """_attn_exact over [B, H, T, D] tensors, in fp64."""
    q, k, v = (t.detach().double() for t in (q, k, v))
    do = do.double() if do is not None else None
    o, G = torch.empty_like(q), q.shape[1] // k.shape[1]
    grads = [torch.empty_like(t) for t in (q, k, v)] if do is not None else []
    for b in range(q.shape[0]):
        for h in range(k.shape[1]):
            s = slice(h * G, h * G + G)
            ob, gr = _attn_exact(q[b, s], k[b, h], v[b, h], None if do is None else do[b, s])
            o[b, s] = ob
            if gr is not None:
                grads[0][b, s], grads[1][b, h], grads[2][b, h] = gr
    return (o, *grads)


def _decode_exact(s, case):
    q, k, v = (s[n].double() for n in ("q", "k", "v"))
    B, Hq, Tq, D = q.shape
    G = Hq // k.shape[1]
    o, lse = torch.zeros_like(q), torch.zeros(B, Hq, Tq, dtype=torch.float64, device=q.device)
    for b, n in enumerate(_lengths(case)):
        pos = torch.arange(n, device=q.device)
        last = n - Tq + torch.arange(Tq, device=q.device)
        for h in range(Hq):
            x = q[b, h] @ k[b, h // G, :n].t() / math.sqrt(D)
            x = x.masked_fill(pos[None, :] > last[:, None], -math.inf)
            lse[b, h] = torch.logsumexp(x, -1)
            o[b, h] = torch.softmax(x, -1) @ v[b, h // G, :n]
    return o, lse


def _norm_rope_exact(q, k, v, wq, wk, cos, sin):
    def one(x, w):
        x = w * x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + _EPS)
        x = x.transpose(1, 2)
        a, b = x.chunk(2, dim=-1)
        return x * cos + torch.cat([-b, a], dim=-1) * sin
    return one(q, wq), one(k, wk), v.transpose(1, 2)


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind in ("train", "prefill"):
        out = _batch_exact(s["q"], s["k"], s["v"], s.get("do"))
        return out if kind == "train" else out[0]
    if kind == "varlen":
        outs, at = [], 0
        for n in _lengths(case):
            part = [s[x].detach()[None, :, at:at + n] for x in ("q", "k", "v", "do")]
            outs.append(_batch_exact(*part))
            at += n
        return tuple(torch.cat([o[i][0] for o in outs], dim=1) for i in range(4))
    if kind == "decode":
        return _decode_exact(s, case)
    # the tables as the bf16 model uses them
    cos, sin = (s[n].to(torch.bfloat16).double() for n in ("cos", "sin"))
    if kind == "prologue":
        ins = [s[n].detach().double().requires_grad_() for n in ("q", "k", "v", "wq", "wk")]
        out = _norm_rope_exact(*ins, cos, sin)
        return tuple(t.detach() for t in out) + torch.autograd.grad(out, ins, [g.double() for g in s["grads"]])
    B, T, Hq, Hkv, D = case["B"], case["T"], case["Hq"], case["Hkv"], case["D"]
    layer = s["layer"].double()
    x = s["x"].detach().double().requires_grad_()
    raw = [p(x).view(B, T, h, D) for p, h in ((layer.q_proj, Hq), (layer.k_proj, Hkv), (layer.v_proj, Hkv))]
    q, k, v = _norm_rope_exact(*raw, layer.q_norm.weight, layer.k_norm.weight, cos, sin)
    dy = s["dy"].double()
    flat = lambda t: t.transpose(1, 2).reshape(B, T, Hq * D)  # noqa: E731
    do = (dy @ layer.o_proj.weight.detach()).view(B, T, Hq, D).transpose(1, 2)
    o, dq, dk, dv = _batch_exact(q, k, v, do)
    names = [(n, p) for n, p in layer.named_parameters()]
    front = [p for n, p in names if n != "o_proj.weight"]
    got = iter(torch.autograd.grad((q, k, v), (x, *front), (dq, dk, dv)))
    dx = next(got)
    d_o = dy.reshape(-1, _HIDDEN).t() @ flat(o).reshape(-1, Hq * D)
    grads = [d_o if n == "o_proj.weight" else next(got) for n, _ in names]
    y = flat(o) @ layer.o_proj.weight.detach().t()
    return (y, dx, *grads)
