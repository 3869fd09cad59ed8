"""Eager calls through the native call layer against the torch.library ops they stand beside: the same kernels on
the same inputs, so the same bits (dbias, summed by atomics, within fp32 rounding); and the tracing and transform
machinery that works on the ops still sees them."""
import pytest
import torch

from gpu_common import make_pope_inputs

pytestmark = pytest.mark.gpu


def _grads(fn, leaves, up):
    out = fn(*leaves)
    outs = out if isinstance(out, tuple) else (out,)
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, up))


def _same(a, b):
    for x, y in zip(a, b):
        assert torch.equal(x, y) or torch.allclose(x, y, rtol=1e-5, atol=1e-5 * y.abs().max().item())


@pytest.mark.parametrize("layout", ["dense", "seq_first", "offset_freqs", "batch_freqs", "one_bias_row", "no_pope", "decode"])
def test_flash_matches_the_op(cuda, layout):
    from pope_amd import _lib
    from pope_amd.hip_pope_flash_attn import flash_fwd_op
    B, Hq, Hk, Nq, Nk, R = 2, 4, 2, 70, 90, 32
    if layout == "decode":
        Nq, Nk = 1, 1500
    inp = make_pope_inputs(61, B, Hq, Hk, Nq, Nk, 64, R, torch.bfloat16, "prefix")
    q, k, v, f, b = (inp[n] for n in ("q", "k", "v", "freqs", "bias"))
    if layout == "seq_first":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    if layout == "offset_freqs":   # a table longer than the cache, viewed at an offset that keeps its alignment
        f = torch.cat([f, f])[4:]
    if layout == "batch_freqs":
        f = torch.stack([f, f * 0.5])
    if layout == "one_bias_row":
        b = b[:1]
    names = [q, k, v] if layout == "no_pope" else [q, k, v, f, b]
    leaves = [t.detach().requires_grad_(True) for t in names]
    pad = [None] * (5 - len(leaves))
    scale = 0.125
    native = _grads(lambda *t: _lib.host().flash(*t, *pad, inp["mask"], False, scale, 1024, True), leaves, inp["do"])
    ops = _grads(lambda *t: flash_fwd_op(*t, *pad, inp["mask"], False, scale)[0], leaves, inp["do"])
    _same(native, ops)


@pytest.mark.parametrize("split", [False, True])
def test_similarity_and_polar_match_the_ops(cuda, split):
    from pope_amd import _lib
    from pope_amd.hip_polar import polar_fwd_op
    from pope_amd.hip_pope import sim_fwd_op
    inp = make_pope_inputs(62, 2, 4, 2, 40, 75, 64, 24, torch.float32)
    leaves = [inp[n].detach().requires_grad_(True) for n in ("q", "k", "freqs", "bias")]
    leaves[0] = inp["q"].transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(True)
    up = torch.randn(2, 4, 40, 75, device="cuda")
    _same(_grads(lambda *t: _lib.host().sim(*t, split), leaves, up), _grads(lambda *t: sim_fwd_op(*t, split), leaves, up))
    E = 128 if split else 64 + 24
    ups = (torch.randn(2, 4, 40, E, device="cuda"), torch.randn(2, 2, 75, E, device="cuda"))
    _same(_grads(lambda *t: _lib.host().polar(*t, split), leaves, ups), _grads(lambda *t: polar_fwd_op(*t, split), leaves, ups))


def test_transforms_and_modes_still_work_on_the_ops(cuda):
    import pope_amd
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    inp = make_pope_inputs(63, 1, 2, 2, 16, 16, 32, 16, torch.float32)
    q, k, f, b = (inp[n] for n in ("q", "k", "freqs", "bias"))
    sim = lambda q, k: pope_amd.compute_attn_similarity(q, k, (f, b))
    want = sim(q, k)
    assert torch.equal(make_fx(sim)(q, k)(q, k), want)
    leaf = q.detach().requires_grad_(True)
    flash = lambda q: pope_amd.flash_attn_with_pope(q, k.bfloat16(), k.bfloat16(), pos_emb=(f, b))
    for fn in (lambda t: sim(t, k).sum(), lambda t: flash(t.bfloat16()).float().sum()):
        with pytest.raises(RuntimeError):   # functorch transforms: refused, by the ops' autograd functions
            torch.func.grad(fn)(q)
    traced = make_fx(flash)(q.bfloat16())
    assert torch.equal(traced(q.bfloat16()), flash(q.bfloat16()))
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        fq, fk = mode.from_tensor(q), mode.from_tensor(k)
        assert sim(fq, fk).shape == want.shape
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t)[1], lambda t: t):
        s = sim(leaf, k)
        o = flash(leaf.bfloat16())
    assert len(packed) >= 8
    (s.sum() + o.float().sum()).backward()


def test_second_derivative_of_the_similarity_raises(cuda):
    import pope_amd
    inp = make_pope_inputs(64, 1, 1, 1, 8, 8, 32, 16, torch.float32)
    q = inp["q"].detach().requires_grad_(True)
    s = pope_amd.compute_attn_similarity(q, inp["k"], (inp["freqs"], inp["bias"]))
    (g,) = torch.autograd.grad(s.square().sum(), q, create_graph=True)
    with pytest.raises(RuntimeError):
        g.sum().backward()


def test_operands_on_another_device_are_refused(cuda):
    import pope_amd
    inp = make_pope_inputs(65, 1, 1, 1, 8, 8, 32, 16, torch.bfloat16)
    with pytest.raises(RuntimeError):
        pope_amd.flash_attn_with_pope(inp["q"], inp["k"], inp["v"], pos_emb=(inp["freqs"].cpu(), inp["bias"]))


def _flash(dtype):
    import pope_amd
    return lambda q, k, f, b: pope_amd.flash_attn_with_pope(q.to(dtype), k.to(dtype), k.to(dtype), pos_emb=(f, b), causal=True)


def _sim(q, k, f, b):
    from pope_amd.hip_pope import hip_compute_qk_similarity
    return hip_compute_qk_similarity(q, k, f, b)


def _polar(q, k, f, b):
    import pope_amd
    return pope_amd.apply_pope_to_qk(pope_amd.PolarEmbedReturn(f, b), q, k)


@pytest.mark.parametrize("R", [16, 12])   # 12: padded operands
@pytest.mark.parametrize("name", ["sim", "polar", "flash_bf16", "flash_fp32"])
@pytest.mark.parametrize("tracer", ["torch.jit.trace", "make_fx", "make_fx_pre_dispatch"])
def test_traced_calls_replay_on_other_inputs(cuda, name, R, tracer):
    """Tracers that are neither torch.compile nor a dispatch mode record the ops as well: a trace on one input gives the
    eager result on another.  (fp32 flash reads its range check back, which make_fx cannot record: it refuses.)"""
    from torch.fx.experimental.proxy_tensor import make_fx
    fn = {"sim": _sim, "polar": _polar, "flash_bf16": _flash(torch.bfloat16), "flash_fp32": _flash(torch.float32)}[name]
    a, b = (tuple(make_pope_inputs(s, 1, 2, 1, 16, 16, 32, R, torch.float32)[n] for n in ("q", "k", "freqs", "bias")) for s in (66, 67))
    if tracer == "torch.jit.trace":
        traced = torch.jit.trace(fn, a, check_trace=False)
    elif name == "flash_fp32":
        with pytest.raises(RuntimeError):
            make_fx(fn, pre_dispatch=tracer != "make_fx")(*a)
        return
    else:
        traced = make_fx(fn, pre_dispatch=tracer != "make_fx")(*a)
    got, want = traced(*b), fn(*b)
    for x, y in zip(*((t if isinstance(t, tuple) else (t,)) for t in (got, want))):
        assert torch.equal(x, y)


def test_fp32_flash_refuses_fake_tensors_and_runs_under_modes(cuda):
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Count(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops += "pope_amd" in str(func) or "_to_copy" in str(func)
            return func(*args, **(kwargs or {}))

    inp = make_pope_inputs(68, 1, 2, 1, 16, 16, 32, 16, torch.float32)
    q, k, f, b = (inp[n] for n in ("q", "k", "freqs", "bias"))
    want = _flash(torch.float32)(q, k, f, b)
    with Count() as mode:
        assert torch.equal(_flash(torch.float32)(q, k, f, b), want)
    assert mode.ops >= 5   # q, k, v and o converted where the mode sees it, and the op
    with FakeTensorMode(allow_non_fake_inputs=True) as mode, pytest.raises(RuntimeError):
        _flash(torch.float32)(mode.from_tensor(q), mode.from_tensor(k), f, b)


@pytest.mark.parametrize("R", [16, 12])   # 12: padded operands
@pytest.mark.parametrize("fn", [_sim, _polar])
def test_a_gradient_penalty_raises_instead_of_counting_as_constant(cuda, fn, R):
    inp = make_pope_inputs(69, 1, 1, 1, 8, 8, 32, R, torch.float32)
    q = inp["q"].detach().requires_grad_(True)
    out = fn(q, inp["k"], inp["freqs"], inp["bias"])
    loss = (out[0] if isinstance(out, tuple) else out).square().sum()
    (g,) = torch.autograd.grad(loss, q, create_graph=True)
    with pytest.raises(RuntimeError, match="second time|not differentiable"):
        (loss + g.square().sum()).backward()


@pytest.mark.parametrize("R", [16, 12])   # 12: padded operands
@pytest.mark.parametrize("name", ["sim", "polar", "flash_bf16", "flash_fp32"])
def test_compiled_autograd_takes_the_nodes(cuda, name, R):
    """A backward under compiled autograd (eager backend) gives the eager gradients."""
    from torch._dynamo import compiled_autograd
    fn = {"sim": _sim, "polar": _polar, "flash_bf16": _flash(torch.bfloat16), "flash_fp32": _flash(torch.float32)}[name]
    inp = make_pope_inputs(70, 1, 2, 1, 16, 16, 32, R, torch.float32)
    grads = []
    for compiled in (False, True):
        leaves = [inp["q"].clone().requires_grad_(True), inp["k"], inp["freqs"], inp["bias"].clone().requires_grad_(True)]
        out = fn(*leaves)
        loss = sum(t.float().square().sum() for t in (out if isinstance(out, tuple) else (out,)))
        if compiled:
            with compiled_autograd._enable(torch.compile(backend="eager")):
                loss.backward()
            torch._dynamo.reset()
        else:
            loss.backward()
        grads.append((leaves[0].grad, leaves[3].grad))
    _same(grads[1], grads[0])


@pytest.mark.parametrize("wanted", [(), ("bias",), ("freqs",), ("freqs", "bias")])
def test_the_ops_give_only_the_wanted_gradients(cuda, wanted):
    from pope_amd import _lib
    from pope_amd.hip_polar import polar_fwd_op
    from pope_amd.hip_pope import sim_fwd_op
    inp = make_pope_inputs(71, 1, 2, 2, 8, 12, 32, 16, torch.float32)
    leaves = [inp[n].detach().requires_grad_(n in ("q", "k", *wanted)) for n in ("q", "k", "freqs", "bias")]
    for op, native in ((polar_fwd_op, _lib.host().polar), (sim_fwd_op, _lib.host().sim)):
        grads = []
        for fn in (op, native):
            out = fn(*leaves, False)
            loss = sum(t.square().sum() for t in (out if isinstance(out, tuple) else (out,)))
            grads.append(torch.autograd.grad(loss, [t for t in leaves if t.requires_grad]))
        _same(*grads)


@pytest.mark.filterwarnings("ignore")   # vmap's per-sample fallback of the ops
@pytest.mark.parametrize("R", [16, 12])   # 12: padded operands
@pytest.mark.parametrize("name", ["sim", "polar", "flash_bf16", "flash_fp32"])
def test_transformed_backwards_run_on_the_ops(cuda, name, R):
    """The backward of an eager call under batched gradients (what a vectorised Jacobian does) and under make_fx: the
    node goes through the torch.library op, which those work on, and gives the same gradients."""
    from torch.fx.experimental.proxy_tensor import make_fx
    fn = {"sim": _sim, "polar": lambda *t: _polar(*t)[1], "flash_bf16": _flash(torch.bfloat16), "flash_fp32": _flash(torch.float32)}[name]
    inp = make_pope_inputs(72, 1, 2, 1, 16, 16, 32, R, torch.float32)
    leaves = [inp[n].detach().requires_grad_(True) for n in ("q", "k", "freqs", "bias")]
    out = fn(*leaves)
    wanted = leaves if name != "polar" else leaves[1:]
    G = torch.randn(3, *out.shape, device="cuda").to(out.dtype)
    back = lambda g, **kw: torch.autograd.grad(out, wanted, g, retain_graph=True, **kw)
    want = [back(g) for g in G]
    batched = back(G, is_grads_batched=True)
    traced = make_fx(back)(G[0])
    for i in range(3):
        _same([t[i] for t in batched], want[i])
        _same(traced(G[i]), want[i])
