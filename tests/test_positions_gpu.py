"""Per-sample positions and position offsets through the fused kernels vs the oracle.

The phase table can be 2-D (N, R) -- shared by every batch and head --, 3-D (B, N, R) from a
(B, N) positions tensor (``PoPE(pos)``, pope.py:131-141, and ``b n d -> b 1 n d`` in
apply_pope_to_qk, pope.py:53-54), offset by ``pope(n, offset)`` (pope.py:135-137), or 4-D
(B, N, H, R) in the reference's (batch, seq, heads) operator layout
(triton_pope_flash_attn.py:237-245; one table per head, so query and kv heads coincide there).
Each layout runs through the flash attention (forward and backward, dfreqs included), the
decode kernel and the similarity, against the oracle on the same inputs.
Tolerances: 2e-2 absolute (beyond the bf16 rounding of the exact value) for bf16 flash and decode
outputs and per-element gradients,
2e-2 * max(1, ||ref||_inf) for the summed dbias / dfreqs; 1e-4 relative for the fp32 similarity.
"""
import math

import pytest
import torch

from gpu_common import excess_over, make_pope_inputs, max_abs, oracle_attention
from oracle import pope_oracle as orc

pytestmark = pytest.mark.gpu

TOL = 2e-2
SUMMED = ("dbias", "dfreqs")


def _check(got, ref, names):
    """Per-element bf16 outputs: 2e-2 beyond the bf16 rounding of the exact value (half a bf16 ulp
    alone is 1.6e-2 at |x| >= 4; gpu_common.excess_over).  Summed gradients: 2e-2 * max(1, ||ref||)."""
    for n in names:
        e = max_abs(got[n], ref[n])
        if n in SUMMED:
            ex = e - TOL * max(1.0, ref[n].abs().max().item())
        else:
            ex = excess_over(got[n], ref[n], TOL)
        print(f"{n}={e:.2e}", end=" ")
        assert ex <= 0, f"{n}: {e:.3e}, {ex:.3e} over the bound"
    print()


def _batch_positions(B, N, seed):
    """(B, N) positions: per-batch starts and uneven gaps (not an arange)."""
    g = torch.Generator().manual_seed(seed)
    steps = torch.randint(1, 4, (B, N), generator=g).float()
    return steps.cumsum(-1) + 100.0 * torch.arange(B).float()[:, None]


def _flash(inp, causal, layout="head_first"):
    import pope_amd
    from pope_amd.hip_pope_flash_attn import flash_attn
    t = [inp[n].detach().clone().requires_grad_(True) for n in ("q", "k", "v", "freqs", "bias")]
    if layout == "head_first":
        o = pope_amd.flash_attn_with_pope(t[0], t[1], t[2], pos_emb=(t[3], t[4]), mask=inp["mask"], causal=causal)
        o.backward(inp["do"])
        return dict(o=o, dq=t[0].grad, dk=t[1].grad, dv=t[2].grad, dfreqs=t[3].grad, dbias=t[4].grad)
    # the reference's operator layout: (B, N, H, D) tensors and (B, N, H, R) freqs
    tr = lambda x: x.detach().transpose(1, 2).contiguous().requires_grad_(True)
    qb, kb, vb, fb = tr(inp["q"]), tr(inp["k"]), tr(inp["v"]), tr(inp["freqs"])
    bias = inp["bias"].detach().clone().requires_grad_(True)
    o = flash_attn(qb, kb, vb, fb, bias, inp["mask"], causal)
    o.backward(inp["do"].transpose(1, 2))
    back = lambda x: x.transpose(1, 2)
    return dict(o=back(o), dq=back(qb.grad), dk=back(kb.grad), dv=back(vb.grad), dfreqs=back(fb.grad), dbias=bias.grad)


@pytest.mark.parametrize("causal", [True, False])
def test_flash_per_batch_positions(cuda, causal):
    B, H, N, D, R = 2, 4, 320, 64, 32
    inp = make_pope_inputs(61, B, H, H, N, N, D, R, torch.bfloat16, "prefix")
    inp["freqs"] = orc.pope_freqs(_batch_positions(B, N, 62), orc.inv_freqs(R)).cuda()   # (B, N, R)
    assert inp["freqs"].shape == (B, N, R)
    _check(_flash(inp, causal), oracle_attention(inp, causal), ["o", "dq", "dk", "dv", "dfreqs", "dbias"])


def test_flash_position_offset_matches_shifted_positions(cuda):
    """pope(n, offset): the rows of a longer table starting at `offset` (pope.py:135-137); with 2-D
    freqs the attention depends on position differences only, so the output matches offset 0."""
    import pope_amd
    B, H, N, D, R = 1, 4, 256, 64, 32
    inp = make_pope_inputs(63, B, H, H, N, N, D, R, torch.bfloat16, "none")
    pope = pope_amd.PoPE(R, heads=H).cuda()
    with torch.no_grad():
        pope.bias.copy_(inp["bias"])
    f_off, bias = pope(N, offset=1000)
    torch.testing.assert_close(f_off.cpu(), orc.pope_freqs(N, orc.inv_freqs(R), offset=1000), rtol=0, atol=0)
    inp_off = dict(inp, freqs=f_off.detach(), bias=bias.detach())
    got = _flash(inp_off, True)
    _check(got, oracle_attention(inp_off, True), ["o", "dq", "dk", "dv", "dfreqs", "dbias"])
    base = _flash(dict(inp, freqs=pope(N)[0].detach(), bias=bias.detach()), True)
    assert max_abs(got["o"], base["o"]) <= TOL


def test_flash_attn_per_head_tables_in_reference_layout(cuda):
    B, H, N, D, R = 2, 4, 192, 64, 32
    inp = make_pope_inputs(64, B, H, H, N, N, D, R, torch.bfloat16, "prefix")
    pos = _batch_positions(B * H, N, 65).view(B, H, N)
    inp["freqs"] = orc.pope_freqs(pos, orc.inv_freqs(R)).cuda()            # (B, H, N, R) head-first
    _check(_flash(inp, True, layout="bnhd"), oracle_attention(inp, True), ["o", "dq", "dk", "dv", "dfreqs", "dbias"])


def test_decode_per_batch_positions(cuda):
    import pope_amd
    from pope_amd import _lib
    B, H, N, D, R = 3, 4, 2048, 64, 64
    inp = make_pope_inputs(66, B, H, H, 1, N, D, R, torch.bfloat16, "prefix")
    inp["freqs"] = orc.pope_freqs(_batch_positions(B, N, 67), orc.inv_freqs(R)).cuda()
    _lib.profile_reset()
    _lib.profile_enable(True)
    o = pope_amd.flash_attn_with_pope(inp["q"], inp["k"], inp["v"], pos_emb=(inp["freqs"], inp["bias"]),
                                      mask=inp["mask"])
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    assert "flash_decode_split" in _lib.profile_read()
    _check(dict(o=o), oracle_attention(inp, False, grads=False), ["o"])


@pytest.mark.parametrize("allow_tf32", [True, False], ids=["split_bf16", "fp32"])
def test_similarity_per_batch_positions_and_offset(cuda, allow_tf32):
    import pope_amd
    g = torch.Generator().manual_seed(68)
    B, H, Nq, Nk, D, R = 2, 4, 100, 160, 64, 32
    q = torch.randn(B, H, Nq, D, generator=g)
    k = torch.randn(B, H, Nk, D, generator=g)
    bias = torch.rand(H, R, generator=g) * (-2 * math.pi)
    G = torch.randn(B, H, Nq, Nk, generator=g)
    for freqs in (orc.pope_freqs(_batch_positions(B, Nk, 69), orc.inv_freqs(R)),
                  orc.pope_freqs(Nk, orc.inv_freqs(R), offset=3000)):
        t = [x.clone().cuda().requires_grad_(True) for x in (q, k, freqs, bias)]
        S = pope_amd.compute_attn_similarity(t[0], t[1], (t[2], t[3]), allow_tf32=allow_tf32)
        S.backward(G.cuda())
        r = [x.clone().requires_grad_(True) for x in (q, k, freqs, bias)]
        S_ref = orc.sim_nonfused(*r)
        (S_ref * G).sum().backward()
        for a, b in zip([S] + [x.grad for x in t], [S_ref] + [x.grad for x in r]):
            rel = ((a.detach().double().cpu() - b.detach().double()).abs().max() / b.abs().max()).item()
            assert rel <= 1e-4, rel


@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("shape", ["batches", "heads", "longer"])
@pytest.mark.parametrize("path", ["native", "op"])
def test_gradient_of_broadcast_freqs(cuda, path, shape, deterministic):
    """A table expanded over batches or heads, in a view longer than the keys or not, gets the gradient of the table
    itself (fp32 sums in another order), with more query heads than the table has entries."""
    import pope_amd
    from pope_amd.hip_pope import sim_fwd_op
    from pope_amd.hip_pope_flash_attn import flash_fwd_op
    B, Hq, Hk, N, D, R = 3, 4, 2, 40, 64, 32
    inp = make_pope_inputs(97, B, Hq, Hk, N, N, D, R, torch.bfloat16)
    q, k, v, b, do = (inp[n] for n in ("q", "k", "v", "bias", "do"))
    up = torch.randn(B, Hq, N, N, device="cuda")
    view = {"batches": lambda t: t.expand(B, N, R), "heads": lambda t: t.expand(B, Hk, N, R),
            "longer": lambda t: torch.cat([t, t]).expand(B, Hk, 2 * N, R)}[shape]
    flash = (lambda f: pope_amd.flash_attn_with_pope(q, k, v, pos_emb=(f, b), causal=True)) if path == "native" else \
        (lambda f: flash_fwd_op(q, k, v, f, b, None, True, D ** -0.5)[0])
    sim = (lambda f: pope_amd.compute_attn_similarity(q.float(), k.float(), (f, b))) if path == "native" else \
        (lambda f: sim_fwd_op(q.float(), k.float(), f, b, True))
    torch.use_deterministic_algorithms(deterministic)
    try:
        for fn, grad in ((flash, do), (sim, up)):
            base = inp["freqs"].detach().requires_grad_(True)
            (want,) = torch.autograd.grad(fn(base), base, grad)
            torch.empty(1 << 20, device="cuda").fill_(1e9)   # what an allocation may find
            (got,) = torch.autograd.grad(fn(view(base)), base, grad)
            torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-5 * want.abs().max().item())
    finally:
        torch.use_deterministic_algorithms(False)


@pytest.mark.parametrize("R", [32, 20])   # 20: padded operands
def test_tables_and_keys_with_too_few_entries_are_refused(cuda, R):
    """They would be read past their end.  More entries than the call has are accepted, as before."""
    import pope_amd
    from pope_amd.hip_pope_flash_attn import flash_fwd_op
    B, H, N, D = 3, 4, 16, 64
    inp = make_pope_inputs(98, B, H, H, N, N, D, R, torch.bfloat16)
    q, k, v, f, b = (inp[n] for n in ("q", "k", "v", "freqs", "bias"))
    flash = lambda f: pope_amd.flash_attn_with_pope(q, k, v, pos_emb=(f, b))
    sim = lambda f, k=k: pope_amd.compute_attn_similarity(q.float(), k.float(), (f, b))
    for bad in (f.repeat(B - 1, 1, 1), f.repeat(B - 1, H, 1, 1), f.repeat(B, H - 1, 1, 1)):
        for fn in (flash, sim):
            with pytest.raises(ValueError):
                fn(bad)
    if R % 8 == 0:
        with pytest.raises(ValueError):
            flash_fwd_op(q, k, v, f.repeat(B - 1, 1, 1), b, None, False, 0.125)
    for bad in (k[:1], k[:2], k[..., :32]):
        with pytest.raises(ValueError):
            sim(f, bad)
    for fn in (flash, sim):
        want = fn(f)
        for good in (f[None], f.repeat(B + 1, 1, 1), f.expand(B, H, N, R), f.repeat(B, H, 1, 1)):
            assert torch.equal(fn(good), want)
    with pytest.raises(RuntimeError, match="per-head freqs"):   # grouped heads
        pope_amd.flash_attn_with_pope(q, k[:, :2], v[:, :2], pos_emb=(f.repeat(B, 2, 1, 1), b[:2]))
