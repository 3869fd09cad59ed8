"""Wide heads (head dims above 128) where their kernels' jobs and tiles end unevenly: head counts that divide over the
eight dies and ones that do not, lengths around the 32-row tiles and the 64- and 128-row jobs, columns past the head
dim, every expanded width (256, 384, 512).  Against the float64 oracle with the flash tests' tolerance (2e-2 absolute
beyond the rounding of the output format); dk and dv sum the independent 16-bit operand roundings of their group's G
query heads, which grow as sqrt(G)."""
import math

import pytest
import torch

from gpu_common import excess_over, make_pope_inputs, oracle_attention

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hk, Nq, Nk, D, R, mask, causal, dtype
    (1, 8, 8, 65, 65, 256, 256, "none", True, torch.bfloat16),
    (2, 8, 4, 33, 97, 136, 104, "prefix", False, torch.float16),
    (1, 3, 3, 159, 159, 144, 144, "half", True, torch.bfloat16),
    (1, 16, 2, 31, 129, 200, 200, "random", True, torch.bfloat16),
    (4, 2, 2, 1, 63, 256, 64, "dead_row", False, torch.float16),
    (1, 5, 1, 96, 225, 192, 64, "none", False, torch.bfloat16),
    (2, 4, 4, 128, 128, 160, 96, "prefix", True, torch.float16),
    (1, 1, 1, 257, 289, 248, 136, "none", True, torch.bfloat16),
    # job splits in the backward: ragged shares, grouped heads, splits without a visible row
    (1, 1, 1, 700, 700, 160, 32, "none", False, torch.bfloat16),
    (2, 4, 1, 301, 333, 256, 256, "prefix", True, torch.float16),
    (1, 2, 2, 513, 900, 144, 144, "half", True, torch.bfloat16),
    (1, 8, 1, 130, 130, 192, 64, "dead_row", False, torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_wide_jobs_against_the_oracle(cuda, case):
    import pope_amd
    B, Hq, Hk, Nq, Nk, D, R, mask, causal, dtype = case
    inp = make_pope_inputs(8800 + Nk, B, Hq, Hk, Nq, Nk, D, R, dtype, mask)
    ref = oracle_attention(inp, causal)
    q, k, v = (inp[n].requires_grad_(True) for n in ("q", "k", "v"))
    o = pope_amd.flash_attn_with_pope(q, k, v, pos_emb=(inp["freqs"], inp["bias"]), mask=inp["mask"], causal=causal)
    assert excess_over(o.detach(), ref["o"], 2e-2) <= 0
    grads = torch.autograd.grad(o, (q, k, v), inp["do"])
    from pope_amd import hip_pope_flash_attn
    assert hip_pope_flash_attn._LAST_BWD_PREPARED   # the forward's preparation, reused
    for got, name in zip(grads, ("dq", "dk", "dv")):
        tol = 2e-2 if name == "dq" else 2e-2 * (Hq / Hk) ** 0.5
        assert excess_over(got, ref[name], tol) <= 0, name


def test_wide_forward_at_512_features_keeps_the_exact_maximum(cuda):
    """The row's largest probability is exactly 1 there, so its 16-bit rounding adds nothing: the running maximum moves
    with every growth, however small.  A row whose first tile holds a score x below its maximum (x < 8), then two keys in
    the ratio 4 : 3 whose probabilities 2^x and 0.75 2^x round apart in bf16 (1 and 0.75 do not): o = (1 - 0.75) / sum,
    within the rounding of the output."""
    import pope_amd
    from pope_amd import _lib
    D, R, Nk = 256, 136, 64
    xs = torch.linspace(6.5, 7.9, 2000, dtype=torch.float64)
    err = lambda p: (p.to(torch.bfloat16).double() - p) / p
    x = xs[(err(2 ** xs) - err(0.75 * 2 ** xs)).abs().argmax()].item()
    s = torch.full((Nk,), -60.0, dtype=torch.float64)
    s[0], s[32], s[33] = 0.0, x, x + torch.tensor(0.75).log2().item()
    q = torch.full((1, 1, 1, D), -30.0)   # softplus of the rotated dims: 1e-13
    k = torch.full((1, 1, Nk, D), -30.0)
    q[..., R:], k[..., R:] = 0.0, 0.0
    left = s.clone()
    for i in range(3):                    # the score in three bf16 parts, times q = 1
        q[..., R + i] = 1.0
        k[0, 0, :, R + i] = left.float().to(torch.bfloat16).float()
        left -= k[0, 0, :, R + i].double()
    v = torch.zeros(1, 1, Nk, D)
    v[:, :, 32], v[:, :, 33] = 1.0, -1.0
    w = 2.0 ** (s - left)
    ref = (w[32] - w[33]) / w.sum()
    q, k, v = (t.to(torch.bfloat16).cuda() for t in (q, k, v))
    freqs, bias = torch.zeros(Nk, R, device="cuda"), torch.zeros(1, R, device="cuda")
    _lib.profile_reset()
    _lib.profile_enable(True)
    o = pope_amd.flash_attn_with_pope(q, k, v, pos_emb=(freqs, bias), softmax_scale=math.log(2.0))
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    assert "flash_wide_fwd" in _lib.profile_read()
    assert excess_over(o, ref.expand(o.shape), 1e-4) <= 0
