"""Key splits of the flash forward: few query rows against many keys run as splits of the key axis and a
log-sum-exp merge.  Against the float64 oracle at the sizes where the splits end unevenly: lengths around tile
and split edges, splits without a visible key (masks, causal), one row and a partial second query block, every
step size of the kernels (128 keys: narrow rows; 64: D 96 and 128; 32: heads above 128).

The tolerance is the flash tests' own (2e-2 absolute beyond the rounding of the output format); lse 2e-2.
"""
import pytest
import torch

from gpu_common import excess_over, make_pope_inputs, oracle_attention
from oracle import pope_oracle as orc

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hk, Nq, Nk, D, R, mask, causal, dtype
    (1, 2, 2, 3, 2048, 64, 64, "none", False, torch.bfloat16),
    (1, 2, 1, 129, 2049, 64, 32, "prefix", False, torch.float16),
    (1, 1, 1, 2000, 2000, 64, 64, "none", True, torch.bfloat16),
    (2, 2, 2, 17, 4097, 32, 32, "half", False, torch.bfloat16),
    (2, 2, 2, 5, 1983, 64, 16, "dead_row", False, torch.float16),
    (1, 4, 2, 130, 3001, 96, 96, "random", False, torch.bfloat16),
    (1, 2, 2, 1, 1100, 128, 128, "half", False, torch.float16),
    (1, 1, 1, 1500, 1500, 128, 64, "prefix", True, torch.bfloat16),
    (1, 2, 1, 7, 999, 160, 32, "prefix", False, torch.bfloat16),
    (1, 1, 1, 257, 1025, 256, 256, "half", False, torch.bfloat16),
    (1, 2, 2, 500, 500, 192, 192, "none", True, torch.float16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_split_forward_against_the_oracle(cuda, case):
    from pope_amd import _lib
    from pope_amd.hip_pope_flash_attn import flash_attn_head_first, flash_fwd_op
    B, Hq, Hk, Nq, Nk, D, R, mask, causal, dtype = case
    inp = make_pope_inputs(8300 + Nk, B, Hq, Hk, Nq, Nk, D, R, dtype, mask)
    ref = oracle_attention(inp, causal, grads=False)
    if Nq > 1:   # one non-causal row takes the decode kernel through the public entry point
        _lib.profile_reset()
        _lib.profile_enable(True)
        o, lse, _ = flash_fwd_op(inp["q"], inp["k"], inp["v"], inp["freqs"], inp["bias"], inp["mask"], causal, D ** -0.5)
        torch.cuda.synchronize()
        _lib.profile_enable(False)
        assert "flash_merge" in _lib.profile_read()
        assert torch.equal(torch.isinf(lse).cpu(), torch.isinf(ref["lse"]))
        fin = torch.isfinite(ref["lse"])
        assert (lse.cpu().double()[fin] - ref["lse"][fin]).abs().max().item() <= 2e-2
    else:
        o = flash_attn_head_first(inp["q"], inp["k"], inp["v"], inp["freqs"], inp["bias"], mask=inp["mask"], causal=causal)
    assert excess_over(o, ref["o"], 2e-2) <= 0


def test_split_forward_feeds_the_backward(cuda):
    """Gradients through a split forward (its lse and o are the backward's inputs)."""
    import pope_amd
    inp = make_pope_inputs(8400, 1, 2, 1, 70, 3000, 64, 32, torch.bfloat16, "prefix")
    ref = oracle_attention(inp, False)
    q, k, v = (inp[n].requires_grad_(True) for n in ("q", "k", "v"))
    o = pope_amd.flash_attn_with_pope(q, k, v, pos_emb=(inp["freqs"], inp["bias"]), mask=inp["mask"])
    grads = torch.autograd.grad(o, (q, k, v), inp["do"])
    for got, name in zip(grads, ("dq", "dk", "dv")):
        assert excess_over(got, ref[name], 2e-2) <= 0, name


def test_partials_are_sized_and_optional(cuda):
    """pope_flash_fwd (no partials) gives the same result within fp32 merge rounding, and a short buffer is refused."""
    import ctypes

    from pope_amd import _lib
    from pope_amd.hip_pope_flash_attn import _desc
    inp = make_pope_inputs(8500, 1, 2, 2, 40, 2500, 64, 64, torch.bfloat16)
    q, k, v = inp["q"], inp["k"], inp["v"]
    d = _desc(q, k, inp["freqs"], inp["bias"], False, 0.125)
    o = torch.empty_like(q)
    d.q_s[:], d.k_s[:], d.v_s[:], d.o_s[:] = (_lib.strides3(t) for t in (q, k, v, o))
    lse = torch.empty(q.shape[:3], device="cuda")
    nb, pb = _lib.workspace_bytes(_lib.OP_FLASH_FWD, d), _lib.workspace_bytes(_lib.OP_FLASH_FWD_PARTIALS, d)
    assert pb > 0
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    pt = torch.full((pb,), 0xff, dtype=torch.uint8, device="cuda")   # NaN patterns: nothing unwritten is read
    args = [t.data_ptr() for t in (q, k, v, inp["freqs"], inp["bias"])] + [None, o.data_ptr(), lse.data_ptr(), ws.data_ptr(), nb]
    L, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    assert L.pope_flash_fwd(ctypes.byref(d), *args, s) == 0
    torch.cuda.synchronize()
    o1, lse1 = o.clone(), lse.clone()
    assert L.pope_flash_fwd_split(ctypes.byref(d), *args, pt.data_ptr(), pb - 256, s) == 3
    assert L.pope_flash_fwd_split(ctypes.byref(d), *args, pt.data_ptr(), pb, s) == 0
    torch.cuda.synchronize()
    # the unsplit kernel rounds P against one reference max, the splits against their own: bf16 P, fp32 sums
    assert (o1.float() - o.float()).abs().max().item() <= 1e-2
    assert (lse1 - lse).abs().max().item() <= 1e-3


@pytest.mark.parametrize("Hq,Hk,D,Nk", [(8, 8, 64, 1025), (12, 4, 128, 1100), (24, 8, 64, 1024), (32, 8, 128, 1333),
                                        (6, 2, 96, 2000), (64, 8, 128, 1024), (40, 40, 32, 1281)])
def test_decode_head_groups(cuda, Hq, Hk, D, Nk):
    """Few batch rows x splits: the decode's workgroups take groups of the query heads (4 to 10 heads per group
    here, group sizes that are no multiple of the four waves among them)."""
    import pope_amd
    inp = make_pope_inputs(8600 + Hq, 1, Hq, Hk, 1, Nk, D, D, torch.bfloat16, "prefix")
    ref = oracle_attention(inp, False, grads=False)
    o = pope_amd.flash_attn_with_pope(inp["q"], inp["k"], inp["v"], pos_emb=(inp["freqs"], inp["bias"]), mask=inp["mask"])
    assert excess_over(o, ref["o"], 2e-2) <= 0


BWD_CASES = [
    # B, Hq, Hk, Nq, Nk, D, R, mask, causal, dtype: split dK/dV and dQ jobs, or (R % 32 != 0) raw rows alone
    (1, 8, 1, 700, 700, 64, 64, "prefix", True, torch.bfloat16),
    (1, 1, 1, 1500, 1500, 64, 32, "half", True, torch.float16),
    (1, 2, 2, 1300, 1300, 32, 32, "none", False, torch.bfloat16),
    (1, 4, 1, 641, 900, 128, 64, "random", False, torch.bfloat16),
    (1, 2, 1, 1025, 1025, 128, 128, "none", True, torch.float16),
    (1, 4, 2, 33, 1200, 96, 96, "prefix", False, torch.bfloat16),
    (2, 2, 2, 70, 129, 64, 24, "dead_row", True, torch.bfloat16),
    (1, 2, 2, 257, 257, 80, 40, "prefix", True, torch.float16),
]


@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("case", BWD_CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_split_backward_against_the_oracle(cuda, case, deterministic):
    """dq, dk, dv within the flash tests' bound, dbias and dfreqs within 2e-2 max(1, ||ref||_inf), through the
    partial rows and their merge."""
    import pope_amd
    from pope_amd import _lib
    B, Hq, Hk, Nq, Nk, D, R, mask, causal, dtype = case
    inp = make_pope_inputs(8700 + Nk, B, Hq, Hk, Nq, Nk, D, R, dtype, mask)
    ref = oracle_attention(inp, causal)
    leaves = [inp[n].detach().requires_grad_(True) for n in ("q", "k", "v", "freqs", "bias")]
    torch.use_deterministic_algorithms(deterministic)
    try:
        o = pope_amd.flash_attn_with_pope(*leaves[:3], pos_emb=tuple(leaves[3:]), mask=inp["mask"], causal=causal)
        _lib.profile_reset()
        _lib.profile_enable(True)
        grads = torch.autograd.grad(o, leaves, inp["do"])
        torch.cuda.synchronize()
        _lib.profile_enable(False)
    finally:
        torch.use_deterministic_algorithms(False)
    assert "flash_chain" in _lib.profile_read()
    for got, name in zip(grads, ("dq", "dk", "dv", "dfreqs", "dbias")):
        if name in ("dfreqs", "dbias"):
            assert (got.double().cpu() - ref[name]).abs().max().item() <= 2e-2 * max(1.0, ref[name].abs().max().item()), name
        else:
            assert excess_over(got, ref[name], 2e-2) <= 0, name


@pytest.mark.parametrize("B,Hq,Hk,Nq,Nk,D,R", [(1, 1, 1, 512, 512, 64, 64), (1, 4, 1, 257, 300, 32, 16), (1, 2, 2, 1000, 1023, 64, 32),
                                               (1, 2, 1, 64, 1025, 128, 128), (2, 1, 1, 700, 701, 48, 8)])
def test_fp32_backward_with_split_reductions(cuda, B, Hq, Hk, Nq, Nk, D, R):
    """allow_tf32=False with few heads: U and W reduced in up to four parts, whose last ones are shorter and, for
    grouped heads, end inside a head.  Tolerance of the fp32 similarity: 1e-4 of ||ref||_inf."""
    import pope_amd
    inp = make_pope_inputs(8900 + Nk, B, Hq, Hk, Nq, Nk, D, R, torch.float32)
    leaves = [inp[n].detach().requires_grad_(True) for n in ("q", "k", "freqs", "bias")]
    sim = pope_amd.compute_attn_similarity(leaves[0], leaves[1], tuple(leaves[2:]), allow_tf32=False)
    G = torch.randn(sim.shape, generator=torch.Generator().manual_seed(1))
    got = [sim.detach()] + list(torch.autograd.grad(sim, leaves, G.to(sim.device)))
    refs = [t.detach().double().cpu().requires_grad_(True) for t in leaves]
    S = orc.sim_nonfused(*refs)
    want = [S.detach()] + list(torch.autograd.grad(S, refs, G.double()))
    for a, r in zip(got, want):
        assert (a.double().cpu() - r).abs().max().item() <= 1e-4 * r.abs().max().item()


@pytest.mark.parametrize("D,R,Nk", [(64, 32, 2048), (128, 128, 1100), (160, 32, 999), (256, 256, 1025)])
def test_split_forward_of_one_row(cuda, D, R, Nk):
    """One query row through the split forward itself: head dims above 128, and per-head tables, which the decode
    kernel does not take."""
    from pope_amd import _lib
    from pope_amd.hip_pope_flash_attn import flash_attn_head_first
    inp = make_pope_inputs(8600 + D, 2, 2, 2, 1, Nk, D, R, torch.bfloat16, "dead_row")
    ref = oracle_attention(inp, False, grads=False)
    _lib.profile_reset()
    _lib.profile_enable(True)
    o = flash_attn_head_first(inp["q"], inp["k"], inp["v"], inp["freqs"].repeat(2, 2, 1, 1), inp["bias"], mask=inp["mask"])
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    assert "flash_merge" in _lib.profile_read()
    assert excess_over(o, ref["o"], 2e-2) <= 0
