"""Which calls may take the native call layer: its launches are invisible to tracers and modes, which work on the
torch.library ops."""
import torch


def test_tracing_and_modes_take_the_ops():
    """Every tracer sees the ops; plain eager calls, with or without a function mode, take the native call layer."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from pope_amd import _lib
    seen = []

    def fn(x):
        seen.append(_lib.eager(x))
        return x + 1

    x = torch.zeros(3)
    fn(x)
    with torch.device("cpu"):
        fn(x)
    assert seen == [True, True]
    seen.clear()
    torch.jit.trace(fn, (x,), check_trace=False)
    make_fx(fn)(x)
    make_fx(fn, pre_dispatch=True)(x)
    torch.vmap(fn)(x)
    torch.func.grad(lambda t: fn(t).sum())(x)
    torch.func.jvp(fn, (x,), (x,))
    with FakeTensorMode() as mode:
        fn(mode.from_tensor(x))
    assert seen == [False] * 7
