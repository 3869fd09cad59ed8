"""The work that users of this package have it do, as measurable cases.

Every case is one call (or forward + backward) through the public entry points of ``pope_amd``.  Its kinds:

  train    ``flash_attn_with_pope`` forward + backward: a training step of one attention layer
  forward  the same without gradients: encoding a prompt or evaluating
  chunk    a block of query rows against a longer key / value cache, without gradients: a prompt that is
           encoded piece by piece, several proposed tokens checked at once
  decode   one query row per sequence against a key / value cache: generating a token
  sim      ``compute_attn_similarity`` forward + backward, with either product arithmetic
  polar    ``apply_pope_to_qk`` forward + backward: the transform alone, for attention code of the user's own

``pos_emb`` comes from ``PoPE`` / ``AxialPoPE`` once, outside the call, as a model shares it between its layers; its
clamped bias is a leaf that receives a gradient.  Inputs are N(0, 1), biases uniform in [-2 pi, 0], key-padding
masks cut a random number of keys off each sequence's end.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.abspath("pope-pytorch_amd"))

import pope_amd  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

_DEFAULTS = dict(kind="train", B=1, Hq=8, Hk=8, Nq=0, Nk=0, D=64, R=64, dtype="bf16", causal=False, pad=0, head_first=True,
                 axial=False, tf32=True)


def _case(name=None, **kw):
    c = dict(_DEFAULTS, **kw)
    c["Nq"] = c["Nq"] or c["Nk"]
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # causal language-model training on a padded batch, half of each head rotated
        _case("train_causal", kind="train", B=2, Nk=4096, D=64, R=32, causal=True, pad=512),
        # video / volume training: three-axis positions on an (8, 16, 16) grid, a head dim that is no power of two
        _case("train_axial", kind="train", B=4, Nk=2048, D=96, R=96, axial=True),
        # grouped-query training with 128-wide heads at a ragged length
        _case("train_gqa_d128", kind="train", B=1, Hq=16, Hk=4, Nk=2999, D=128, R=64, causal=True),
        # training with 256-wide heads, fully rotated
        _case("train_wide_d256", kind="train", B=2, Nk=2048, D=256, R=256, causal=True),
        # a small training call, where launches and host time count
        _case("train_small", kind="train", B=1, Hq=4, Hk=4, Nk=257, D=64, R=64, dtype="fp16", causal=True, pad=64),
        # inference on fp32 tensors, the (1, 8, 1024, 64) shape of the plain reference computation
        _case("forward_fp32", kind="forward", B=1, Nk=1024, D=64, R=64, dtype="fp32"),
        # a block of a prompt against what is cached already
        _case("chunk_cache", kind="chunk", B=1, Nq=130, Nk=16000, D=64, R=64, pad=2000),
        # generation for eight sequences of 4096 to 32768 cached tokens
        _case("decode_batch", kind="decode", B=8, Hq=16, Hk=16, Nq=1, Nk=32768, D=64, R=64, pad=32768 - 4096),
        # generation for one sequence, grouped heads
        _case("decode_single", kind="decode", B=1, Hq=32, Hk=8, Nq=1, Nk=4001, D=128, R=64, pad=1000),
        # the similarity alone, the default product arithmetic
        _case("sim_train", kind="sim", B=2, Nk=2048, D=64, R=64, dtype="fp32"),
        # the same with full fp32 products, as parity checks ask for it
        _case("sim_fp32", kind="sim", B=1, Nk=1024, D=64, R=64, dtype="fp32", tf32=False),
        # the transform alone, both directions
        _case("polar_train", kind="polar", B=2, Nk=2048, D=64, R=64, dtype="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng, most):
    Hk = rng.choice([h for h in (1, 2, 4, 8, 16) if h <= most])
    return Hk * rng.choice([g for g in (1, 1, 1, 2, 4, 8) if Hk * g <= most]), Hk


def _rotate(rng, D):
    """All of the head, half or a quarter of it, or another number of its dims (odd ones among them)."""
    u = rng.random()
    if u < 0.45:
        return D
    if u < 0.75:
        return max(1, D // rng.choice([2, 4]))
    return rng.randint(1, D)


_FLOP_CAP = 1.5e11    # of one drawn case; train_causal has 1.5e11, train_wide_d256 1.9e11, train_axial 2.8e11


def _draw(rng):
    kind = rng.choice(["train", "train", "train", "wide", "forward", "chunk", "decode", "decode", "sim", "sim", "polar"])
    Hq, Hk = _heads(rng, 16)
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"])
    hf = rng.random() < 0.6
    if kind in ("train", "wide", "forward"):
        D = rng.choice([32, 48, 64, 64, 64, 72, 80, 96, 100, 112, 128, 128]) if kind != "wide" else \
            rng.choice([144, 160, 192, 192, 224, 250, 256, 256])
        Nk = _log_int(rng, 16, 4096 if kind != "wide" else 2048)
        return _case(kind="train" if kind == "wide" else kind, B=rng.choice([1, 1, 2, 4]), Hq=Hq, Hk=Hk, Nk=Nk, D=D,
                     R=_rotate(rng, D), dtype=dtype, causal=rng.random() < 0.6,
                     pad=rng.choice([0, Nk // 8, Nk // 3]), head_first=hf)
    if kind == "chunk":
        Nk = _log_int(rng, 512, 32768)
        D = rng.choice([32, 64, 64, 96, 128, 128])
        return _case(kind="chunk", B=rng.choice([1, 1, 2, 4]), Hq=Hq, Hk=Hk, Nq=_log_int(rng, 2, 512), Nk=Nk, D=D,
                     R=_rotate(rng, D), dtype=rng.choice(["bf16", "bf16", "fp16"]), pad=rng.choice([0, Nk // 4]), head_first=hf)
    if kind == "decode":
        Nk = _log_int(rng, 128, 32768)
        D = rng.choice([32, 64, 64, 64, 96, 128, 128])
        Hq, Hk = _heads(rng, 32)
        return _case(kind="decode", B=rng.choice([1, 1, 2, 4, 8]), Hq=Hq, Hk=Hk, Nq=1, Nk=Nk, D=D, R=rng.choice([D, D, D // 2]),
                     dtype=rng.choice(["bf16", "bf16", "fp16"]), pad=rng.choice([0, Nk // 4, Nk * 7 // 8]), head_first=hf)
    if kind == "sim":
        D = rng.choice([32, 48, 64, 64, 128, 128, 256])
        Nk = _log_int(rng, 32, 2048)
        return _case(kind="sim", B=rng.choice([1, 1, 2]), Hq=min(Hq, 8), Hk=min(Hk, 8), Nq=Nk if rng.random() < 0.7 else
                     rng.randint(1, Nk), Nk=Nk, D=D, R=_rotate(rng, D), dtype=rng.choice(["fp32", "fp32", "fp32", "bf16"]),
                     tf32=rng.random() < 0.7, head_first=hf)
    Nk = _log_int(rng, 16, 8192)
    D = rng.choice([32, 48, 64, 64, 96, 128, 256])
    return _case(kind="polar", B=rng.choice([1, 2, 4]), Hq=Hq, Hk=Hk, Nk=Nk, D=D, R=_rotate(rng, D), dtype=rng.choice(["fp32", "fp32", "bf16", "fp16"]))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= _FLOP_CAP and w["bytes"] <= 6e8 and not (c["kind"] == "sim" and not c["tf32"] and w["flops"] > 5e10):
            return c


def _visible(c):
    """Expected number of visible (query, key) pairs per (batch, query head)."""
    Nq, Nk = c["Nq"], c["Nk"]
    L = Nk - c["pad"] / 2
    if c["causal"]:
        return Nq * L - L * L / 2 if Nq >= L else Nq * Nq / 2
    return Nq * L


def work(case):
    c, eb = case, _BYTES[case["dtype"]]
    B, Hq, Hk, Nq, Nk, D, R = (c[n] for n in ("B", "Hq", "Hk", "Nq", "Nk", "D", "R"))
    E = D + R      # a rotated dim's term a c cos(phi - psi) is two products
    nq, nk, table = B * Hq * Nq * D, B * Hk * Nk * D, 4 * Nk * R + 4 * Hk * R
    if c["kind"] == "sim":
        pairs = B * Hq * Nq * Nk
        return {"bytes": 2 * eb * pairs + 2 * eb * (nq + nk) + table, "flops": 6 * E * pairs}
    if c["kind"] == "polar":
        # q, k read in both directions, q_hat and k_hat and their gradients, dq and dk
        rows = B * (Hq * Nq + Hk * Nk)
        return {"bytes": rows * (2 * 4 * E + 3 * eb * D) + 2 * table, "flops": 10 * rows * E}
    pairs = B * Hq * _visible(c)
    live = 1 - c["pad"] / 2 / Nk
    fwd_bytes = 2 * eb * nq + 2 * eb * nk * live + table
    if c["kind"] != "train":
        return {"bytes": fwd_bytes, "flops": 2 * (E + D) * pairs}
    # backward: the scores again, dP, dV, dQ_hat, dK_hat; q, k, v, o, do read, dq, dk, dv written
    return {"bytes": fwd_bytes + eb * (4 * nq + 4 * nk) + table, "flops": 2 * (E + D) * pairs + (6 * E + 4 * D) * pairs}


def tolerance(case):
    """About four times the largest error against 64 bits that 80 cases of these ranges show (2-norm; "max": the largest
    element, over the rms or the element itself).  dbias sums signed products over all keys and comes off worst."""
    if case["kind"] == "sim":
        # fp32: 16-bit halves of the operands, or (tf32 False) the fp32 rounding of phases up to 2048
        if case["dtype"] == "fp32":
            return {"rel": 4e-5, "max": 1.2e-3} if case["tf32"] else {"rel": 1.5e-5, "max": 1.2e-3}
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["kind"] == "polar":
        # fp32: the rounding of the key phase fl(F + bias) at phases up to 8192
        return {"fp32": {"rel": 5e-5, "max": 1.7e-3}, "fp16": {"rel": 1e-3, "max": 6e-3}, "bf16": {"rel": 8e-3, "max": 3e-2}}[case["dtype"]]
    if case["dtype"] == "bf16":
        return {"rel": 2e-2, "max": 0.6} if case["kind"] == "train" else {"rel": 1.2e-2, "max": 0.2}
    return {"rel": 3e-3, "max": 0.1} if case["kind"] == "train" else {"rel": 2e-3, "max": 0.03}    # fp16 operands


def _pos_emb(c):
    if c["axial"]:
        pope = pope_amd.AxialPoPE(c["R"], heads=c["Hk"], axial_dims=(c["R"] // 3,) * 3).cuda()
        freqs, _ = pope((c["Nk"] // 256, 16, 16))
    else:
        pope = pope_amd.PoPE(c["R"], heads=c["Hk"]).cuda()
        freqs, _ = pope(c["Nk"])
    return freqs.detach()


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[c["dtype"]]
    grad = c["kind"] in ("train", "sim", "polar")
    B, Hq, Hk, Nq, Nk, D, R = (c[n] for n in ("B", "Hq", "Hk", "Nq", "Nk", "D", "R"))

    def rows(H, N):
        shape = (B, H, N, D) if c["head_first"] else (B, N, H, D)
        return torch.randn(shape, generator=g, device="cuda").to(dt).requires_grad_(grad)

    s = {"case": c, "q": rows(Hq, Nq), "k": rows(Hk, Nk)}
    if c["kind"] not in ("sim", "polar"):
        s["v"] = rows(Hk, Nk)
    s["freqs"] = _pos_emb(c)
    s["bias"] = (torch.rand(Hk, R, generator=g, device="cuda") * (-2 * math.pi)).requires_grad_(grad)
    if c["pad"]:
        lens = Nk - torch.randint(0, c["pad"] + 1, (B,), generator=g, device="cuda")
        s["mask"] = torch.arange(Nk, device="cuda")[None, :] < lens[:, None]
    if c["kind"] == "train":
        s["do"] = torch.randn(s["q"].shape, generator=g, device="cuda").to(dt)
    elif c["kind"] == "sim":
        s["do"] = torch.randn((B, Hq, Nq, Nk), generator=g, device="cuda").to(dt)
    elif c["kind"] == "polar":
        s["do"] = tuple(torch.randn((B, H, N, D + R), generator=g, device="cuda") for H, N in ((Hq, Nq), (Hk, Nk)))
    return s


def run(state):
    s, c = state, state["case"]
    pos_emb = (s["freqs"], s["bias"])
    if c["kind"] == "sim":
        out = pope_amd.compute_attn_similarity(s["q"], s["k"], pos_emb, allow_tf32=c["tf32"], head_dimension_at_first=c["head_first"])
        dq, dk, dbias = torch.autograd.grad(out, (s["q"], s["k"], s["bias"]), s["do"])
        return {"sim": out.detach(), "dq": dq, "dk": dk, "dbias": dbias}
    if c["kind"] == "polar":
        q, k = (s["q"], s["k"]) if c["head_first"] else (s["q"].transpose(1, 2), s["k"].transpose(1, 2))
        qh, kh = pope_amd.apply_pope_to_qk(pope_amd.PolarEmbedReturn(*pos_emb), q, k)
        dq, dk, dbias = torch.autograd.grad((qh, kh), (s["q"], s["k"], s["bias"]), s["do"])
        return {"q_hat": qh.detach(), "k_hat": kh.detach(), "dq": dq, "dk": dk, "dbias": dbias}
    attend = lambda: pope_amd.flash_attn_with_pope(s["q"], s["k"], s["v"], pos_emb=pos_emb, mask=s.get("mask"),
                                                   causal=c["causal"], head_dimension_at_first=c["head_first"])
    if c["kind"] != "train":
        with torch.no_grad():
            return {"o": attend()}
    o = attend()
    dq, dk, dv, dbias = torch.autograd.grad(o, (s["q"], s["k"], s["v"], s["bias"]), s["do"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv, "dbias": dbias}


# ---------------------------------------------------------------- the same in 64 bits, plain torch

def _expand(x, phase, R):
    """(.., N, D) rows -> interleaved (a cos, a sin) pairs of the R rotated dims, then the others as they are."""
    a = F.softplus(x[..., :R])
    pairs = torch.stack((a * phase.cos(), a * phase.sin()), dim=-1).flatten(-2)
    return torch.cat((pairs, x[..., R:]), dim=-1)


def exact(case, seed):
    c, s = case, prepare(case, seed)
    B, Hq, Hk, Nq, Nk, D, R = (c[n] for n in ("B", "Hq", "Hk", "Nq", "Nk", "D", "R"))
    grad = c["kind"] in ("train", "sim", "polar")
    head_first = lambda t: t if c["head_first"] else t.transpose(1, 2)
    leaf = {n: s[n].detach().double().requires_grad_(grad) for n in ("q", "k", "v", "bias") if n in s}
    freqs = s["freqs"].double()
    q_phase = freqs[Nk - Nq:]
    wide = {n: torch.zeros_like(leaf[n]) for n in leaf}            # gradients
    if c["kind"] == "sim":
        out = torch.empty(B, Hq, Nq, Nk, dtype=torch.float64, device="cuda")
    elif c["kind"] == "polar":
        out = [torch.empty(B, H, N, D + R, dtype=torch.float64, device="cuda") for H, N in ((Hq, Nq), (Hk, Nk))]
    else:
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    visible = torch.ones(Nq, Nk, dtype=torch.bool, device="cuda")
    if c["causal"]:
        visible = visible.tril()
    names = [n for n in ("q", "k", "v", "bias") if n in leaf]
    # one (batch, query head) at a time; query head h reads key head h % Hk
    for b in range(B):
        for h in range(Hq):
            hk = h % Hk
            part = {n: (leaf[n][hk] if n == "bias" else head_first(leaf[n])[b, h if n == "q" else hk]).detach().requires_grad_(grad)
                    for n in names}
            qh = _expand(part["q"], q_phase, R)
            kh = _expand(part["k"], freqs + part["bias"], R)
            if c["kind"] == "polar":
                y = (qh, kh) if h < Hk else (qh,)
                out[0][b, h] = qh.detach()
                if h < Hk:
                    out[1][b, h] = kh.detach()
                up = (s["do"][0][b, h].double(),) + ((s["do"][1][b, h].double(),) if h < Hk else ())
            else:
                S = torch.mm(qh, kh.t().contiguous())
                if c["kind"] == "sim":
                    y, up = (S,), (s["do"][b, h].double(),)
                    out[b, h] = S.detach()
                else:
                    keep = visible & s["mask"][b] if "mask" in s else visible
                    P = torch.softmax((S * D ** -0.5).masked_fill(~keep, float("-inf")), dim=-1)
                    y = (torch.mm(P, part["v"]),)
                    head_first(out)[b, h] = y[0].detach()
                    up = (head_first(s["do"])[b, h].double(),) if grad else None
            if grad:
                for n, d in zip(names, torch.autograd.grad(y, [part[n] for n in names], up, allow_unused=True)):
                    if d is not None:
                        (wide[n][hk] if n == "bias" else head_first(wide[n])[b, h if n == "q" else hk]).add_(d)
    if c["kind"] == "sim":
        return {"sim": out, "dq": wide["q"], "dk": wide["k"], "dbias": wide["bias"]}
    if c["kind"] == "polar":
        return {"q_hat": out[0], "k_hat": out[1], "dq": wide["q"], "dk": wide["k"], "dbias": wide["bias"]}
    if not grad:
        return {"o": out}
    return {"o": out, "dq": wide["q"], "dk": wide["k"], "dv": wide["v"], "dbias": wide["bias"]}
