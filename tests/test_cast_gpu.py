"""The fp32 operands' fp16 conversion (pope_cast_f16) against Tensor.to, bit for bit, over layouts the kernel takes
by 4 elements and one by one, and its range flag."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _flag():
    f = torch.empty(1, dtype=torch.int32, pin_memory=True)
    f[0] = 0
    return f


@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (2, 3, 5, 8), (1, 2, 129, 64), (2, 1, 3, 7), (1, 1, 1, 1), (0, 2, 3, 8)])
@pytest.mark.parametrize("view", ["dense", "seq_first", "sliced", "offset", "expanded", "feature_stride"])
def test_cast_matches_to(cuda, shape, view):
    from pope_amd.hip_pope_flash_attn import _launch_half
    B, H, N, D = shape
    g = torch.Generator(device="cuda").manual_seed(5)
    base = torch.randn(max(B, 1) * (H + 1) * (N + 1) * (2 * D + 4) + 1, generator=g, device="cuda") * 100
    base[::7] = 0.0
    base[1::11] = 1e-6        # fp16 subnormals
    dense = base[:B * H * N * D].view(shape)
    x = {"dense": dense,
         "seq_first": base[:B * H * N * D].view(B, N, H, D).transpose(1, 2),
         "sliced": base[:B * H * N * (D + 4)].view(B, H, N, D + 4)[..., :D],
         "offset": base[1:1 + B * H * N * D].view(shape),
         "expanded": base[:H * N * D].view(1, H, N, D).expand(shape),
         "feature_stride": base[:B * H * N * 2 * D].view(B, H, N, 2 * D)[..., ::2]}[view]
    y = torch.randn(2, 2, 3, 8, generator=g, device="cuda")
    flag = _flag()
    a, b = _launch_half((x, y), flag)
    torch.cuda.synchronize()
    assert torch.equal(a, x.to(torch.float16)) and a.stride() == x.to(torch.float16).stride()
    assert torch.equal(b, y.to(torch.float16))
    assert int(flag[0]) == 0


@pytest.mark.parametrize("value,flagged", [(65504.0, 0), (65505.0, 1), (-7e4, 1), (3e38, 1), (float("inf"), 0), (float("-inf"), 0),
                                           (float("nan"), 0)])
@pytest.mark.parametrize("D", [8, 7])
def test_cast_flag(cuda, value, flagged, D):
    from pope_amd.hip_pope_flash_attn import _launch_half
    x = torch.ones(1, 2, 300, D, device="cuda")
    x[0, 1, 299, D - 1] = value
    flag = _flag()
    (h,) = _launch_half((x,), flag)
    torch.cuda.synchronize()
    assert int(flag[0]) == flagged
    assert torch.equal(h, x.to(torch.float16)) or value != value


def test_fp32_call_raises_after_a_good_one_and_keeps_gradients(cuda):
    import pope_amd
    q, k, v = (torch.randn(1, 2, 40, 64, device="cuda", requires_grad=True) for _ in range(3))
    o = pope_amd.flash_attn_with_pope(q, k, v)
    assert o.dtype == torch.float32
    grads = torch.autograd.grad(o.sum(), (q, v))
    assert all(t.dtype == torch.float32 for t in grads)
    with pytest.raises(ValueError, match="fp16's range"):
        pope_amd.flash_attn_with_pope(q * 1e6, k, v)
    with pytest.raises(ValueError, match="must match k"):
        pope_amd.flash_attn_with_pope(q, k[..., :32], v)
