"""Head and rotate dims that are not multiples of 8 through the pad kernel, against the torch padding of pope_amd._pad:
the same padded operands run through the same kernels, so the same bits in every output and gradient (dbias and
dfreqs, summed by atomics, within fp32 rounding)."""
import pytest
import torch

from gpu_common import make_pope_inputs
from pope_amd._pad import pad_last, pad_plan, pad_qk

pytestmark = pytest.mark.gpu


def _run(fn, leaves, ups):
    out = fn(*leaves)
    outs = out if isinstance(out, tuple) else (out,)
    return [o.detach() for o in outs], torch.autograd.grad(outs, leaves, ups)


def _same(a, b):
    for x, y in zip([*a[0], *a[1]], [*b[0], *b[1]]):
        assert x.shape == y.shape and x.dtype == y.dtype
        assert torch.equal(x, y) or (x.dtype == torch.float32
                                     and torch.allclose(x, y, rtol=1e-5, atol=1e-5 * y.abs().max().item()))


@pytest.mark.parametrize("D,R", [(100, 100), (64, 20), (33, 1), (7, 7), (250, 96), (61, 40), (36, 0)])
@pytest.mark.parametrize("layout", ["dense", "seq_first", "feature_strided", "batch_freqs", "one_bias_row"])
def test_padded_flash_matches_the_torch_padding(cuda, D, R, layout):
    import pope_amd
    from pope_amd import _lib
    inp = make_pope_inputs(900 + D, 2, 4, 2, 37, 51, D, R, torch.bfloat16, "prefix")
    q, k, v, f, b, do = (inp[n] for n in ("q", "k", "v", "freqs", "bias", "do"))
    if layout == "seq_first":
        q, k, v, do = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v, do))
    if layout == "feature_strided":
        q, k, v, do = (t.transpose(2, 3).contiguous().transpose(2, 3) for t in (q, k, v, do))
    if layout == "batch_freqs" and R:
        f = torch.stack([f, f * 0.5])
    if layout == "one_bias_row" and R:
        b = b[:1]
    plan = pad_plan(D, R)
    leaves = [t.detach().requires_grad_(True) for t in ([q, k, v, f, b] if R else [q, k, v])]

    def torch_padding(q, k, v, f=None, b=None):
        o = _lib.host().flash(pad_qk(q, plan), pad_qk(k, plan), pad_last(v, plan.Dp), pad_last(f, plan.R8),
                              pad_last(b, plan.R8), inp["mask"], True, D ** -0.5, 1024, True)
        return o[..., :D]

    def api(q, k, v, f=None, b=None):
        return pope_amd.flash_attn_with_pope(q, k, v, pos_emb=None if f is None else (f, b), mask=inp["mask"], causal=True)

    _lib.profile_reset()
    _lib.profile_enable(True)
    got = _run(api, leaves, do)
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    assert "pad_rows" in _lib.profile_read()
    _same(got, _run(torch_padding, leaves, do))
    with torch.no_grad():
        assert torch.equal(api(*leaves), got[0][0])


@pytest.mark.parametrize("D,R", [(64, 20), (48, 31), (128, 1), (32, 9)])
def test_padded_similarity_and_polar_match_the_torch_padding(cuda, D, R):
    import pope_amd
    from pope_amd import _lib
    from pope_amd.hip_polar import polar
    inp = make_pope_inputs(950 + R, 2, 4, 2, 23, 40, D, R, torch.float32)
    plan = pad_plan(D, R)
    leaves = [inp[n].detach().requires_grad_(True) for n in ("q", "k", "freqs", "bias")]
    pads = lambda q, k, f, b: (pad_qk(q, plan), pad_qk(k, plan), pad_last(f, plan.R8), pad_last(b, plan.R8))
    up = torch.randn(2, 4, 23, 40, device="cuda")
    _same(_run(lambda q, k, f, b: pope_amd.compute_attn_similarity(q, k, (f, b)), leaves, up),
          _run(lambda *t: _lib.host().sim(*pads(*t), True), leaves, up))

    def torch_padding(*t):
        keep = lambda x: torch.cat([x[..., :2 * R], x[..., 2 * plan.R8:2 * plan.R8 + D - R]], -1)
        qh, kh = _lib.host().polar(*pads(*t), False)
        return keep(qh), keep(kh)

    ups = (torch.randn(2, 4, 23, D + R, device="cuda"), torch.randn(2, 2, 40, D + R, device="cuda"))
    _same(_run(polar, leaves, ups), _run(torch_padding, leaves, ups))


def test_in_place_change_of_a_padded_output_is_seen(cuda):
    import pope_amd
    inp = make_pope_inputs(990, 1, 1, 1, 9, 9, 20, 12, torch.float16)
    q = inp["q"].requires_grad_(True)
    o = pope_amd.flash_attn_with_pope(q, inp["k"], inp["v"], pos_emb=(inp["freqs"], inp["bias"]))
    o.mul_(2.0)
    with pytest.raises(RuntimeError, match="inplace"):
        o.sum().backward()


def test_pad_arguments_are_checked(cuda):
    from pope_amd import _lib
    q = torch.zeros(1, 1, 4, 12, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="does not have rows of 12"):
        _lib.host().flash_padded(q, q[..., :8], q, None, None, None, False, 1.0, 1024, True, 0, 0, 16)
