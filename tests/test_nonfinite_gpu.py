"""NaN and infinite operands in the split flash forward (workgroups over the key axis, then a log-sum-exp merge) and in
the decode kernel: a row that sees a NaN score is NaN, as in the unsplit kernels and in torch's softmax, and no other
row changes.  A split whose visible scores are all NaN has no finite maximum, like a split without a visible key; only
its row sum tells the two apart.  No tolerance: patterns of NaN are compared, and untouched rows bit for bit.
"""
import ctypes

import pytest
import torch

from gpu_common import make_pope_inputs

pytestmark = pytest.mark.gpu

NAN, NEG_NAN, INF = float("nan"), "negative NaN", float("inf")


def _put(t, index, value):
    if value == NEG_NAN:   # sign bit set, as x86 and the matrix units write the default NaN
        t.view(torch.int16)[index] = -64 if t.dtype == torch.bfloat16 else -512
        assert torch.isnan(t[index]).all()
    else:
        t[index] = value


def _split_and_unsplit(inp, causal, scale=0.125):
    """(o, lse) of the split forward and of the unsplit one on the same inputs; the partials start as NaN patterns."""
    from pope_amd import _lib
    from pope_amd.hip_pope_flash_attn import _desc
    q, k, v, mask = (inp[n] for n in ("q", "k", "v", "mask"))
    d = _desc(q, k, inp["freqs"], inp["bias"], causal, scale)
    L, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    res = []
    for split in (True, False):
        o, lse = torch.empty_like(q), torch.empty(q.shape[:3], device="cuda")
        d.q_s[:], d.k_s[:], d.v_s[:], d.o_s[:] = (_lib.strides3(t) for t in (q, k, v, o))
        if mask is not None:
            d.mask_sb = mask.stride(0)
        nb, pb = _lib.workspace_bytes(_lib.OP_FLASH_FWD, d), _lib.workspace_bytes(_lib.OP_FLASH_FWD_PARTIALS, d)
        assert pb > 0   # the call splits
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        pt = torch.full((pb,), 0xff, dtype=torch.uint8, device="cuda") if split else None
        rc = L.pope_flash_fwd_split(ctypes.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), inp["freqs"].data_ptr(),
                                    inp["bias"].data_ptr(), _lib.ptr(mask), o.data_ptr(), lse.data_ptr(), ws.data_ptr(), nb,
                                    pt.data_ptr() if split else None, pb if split else 0, s)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        res.append((o, lse))
    return res


SPLIT = [   # Hq, Hk, Nq, Nk, D, R, causal, dtype: tiles of 64 and 32 keys, wide heads of 256 and 512 features
    (2, 2, 3, 2048, 64, 32, False, torch.bfloat16),
    (2, 1, 130, 3000, 96, 96, False, torch.float16),
    (1, 1, 1500, 1500, 128, 64, True, torch.bfloat16),
    (2, 1, 7, 999, 160, 32, False, torch.bfloat16),
    (1, 1, 2, 1025, 256, 256, False, torch.float16),
]


@pytest.mark.parametrize("case", SPLIT, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
@pytest.mark.parametrize("what", ["query_row", "lone_key", "negative_lone_key", "one_of_many_keys", "infinite_query",
                                  "infinite_key", "value"])
def test_split_forward_keeps_nan(cuda, case, what):
    Hq, Hk, Nq, Nk, D, R, causal, dtype = case
    inp = make_pope_inputs(77, 1, Hq, Hk, Nq, Nk, D, R, dtype)
    row, key = Nq - 1, Nk - 1
    if what in ("lone_key", "negative_lone_key"):   # the only visible key of the last split
        inp["mask"] = torch.ones(1, Nk, dtype=torch.bool, device="cuda")
        inp["mask"][:, Nk // 4:] = False
        inp["mask"][:, key] = True
    clean = _split_and_unsplit(inp, causal)[0][0].clone()
    if what == "query_row":
        _put(inp["q"], (0, 0, row), NAN)
    elif what == "infinite_query":
        _put(inp["q"], (0, 0, row), INF)
    elif what == "value":
        _put(inp["v"], (0, 0, key, 5), NAN)
    elif what == "infinite_key":
        _put(inp["k"], (0, 0, key), INF)
    else:
        _put(inp["k"], (0, 0, key), NEG_NAN if what == "negative_lone_key" else NAN)
    (o, lse), (ou, lu) = _split_and_unsplit(inp, causal)
    assert torch.equal(torch.isnan(o), torch.isnan(ou))
    assert torch.equal(torch.isnan(lse), torch.isnan(lu)) and torch.equal(torch.isinf(lse), torch.isinf(lu))
    bad = torch.zeros(1, Hq, Nq, dtype=torch.bool, device="cuda")   # rows that see the value
    if what in ("query_row", "infinite_query"):
        bad[:, 0, row] = True
    else:
        bad[:, ::Hk, (key if causal else 0):] = True
    if what != "value":
        assert torch.isnan(o[bad]).all()
    else:
        assert torch.isnan(o[bad][:, 5]).all()
    if what != "value" or not causal:   # a masked key's zero probability times a NaN value is NaN in its tile
        assert torch.equal(o[~bad], clean[~bad])


@pytest.mark.parametrize("Hq,Hk,D,R,Nk,dtype", [(2, 2, 64, 64, 576, torch.bfloat16), (4, 2, 128, 64, 300, torch.float16),
                                                (2, 1, 96, 96, 1500, torch.bfloat16), (8, 8, 64, 32, 2048, torch.bfloat16)])
@pytest.mark.parametrize("what", ["query", "key", "negative_key", "lone_key", "negative_lone_key", "value"])
def test_decode_keeps_nan(cuda, Hq, Hk, D, R, Nk, dtype, what):
    import pope_amd
    from pope_amd import _lib
    inp = make_pope_inputs(78, 1, Hq, Hk, 1, Nk, D, R, dtype)
    mask = torch.ones(1, Nk, dtype=torch.bool, device="cuda")
    if "lone" in what:   # the only visible key of its split
        mask[:, Nk // 4:] = False
        mask[:, Nk - 1] = True
    elif what == "query":   # masked keys beside the NaN scores
        mask[:, ::3] = False
    run = lambda: pope_amd.flash_attn_with_pope(inp["q"], inp["k"], inp["v"], pos_emb=(inp["freqs"], inp["bias"]), mask=mask)
    clean = run()
    if what == "query":
        _put(inp["q"], (0, 0, 0), NAN)
    elif what == "value":
        _put(inp["v"], (0, 0, Nk - 1, 5), NAN)
    else:
        _put(inp["k"], (0, 0, Nk - 1), NEG_NAN if "negative" in what else NAN)
    _lib.profile_reset()
    _lib.profile_enable(True)
    o = run()
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    assert "flash_decode_split" in _lib.profile_read()
    heads = torch.arange(Hq, device="cuda")
    bad = heads == 0 if what == "query" else heads % Hk == 0
    assert torch.isnan(o[0, bad, 0, 5] if what == "value" else o[0, bad]).all()
    assert torch.equal(o[:, ~bad], clean[:, ~bad])
