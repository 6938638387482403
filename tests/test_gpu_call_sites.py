"""The functional and module forms run as native autograd nodes where every operand is ready, and through the Python
autograd functions otherwise.  The two must agree bit for bit in outputs and gradients and in what they do under hooks,
partial gradients, repeated backward, checkpointing, transforms and tangents."""
import threading

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.checkpoint import checkpoint

pytestmark = pytest.mark.gpu
EPS = 1e-6
KINDS = ["adaln", "module", "seq_first", "stream", "gated", "rms", "view", "view3", "qkv", "qkv_rope"]


@pytest.fixture(scope="module")
def FL(gpu_device):
    from teletron_amd import fusedlayers
    return fusedlayers


@pytest.fixture(autouse=True)
def fused(monkeypatch):
    monkeypatch.setenv("FUSED_KERNELS", "1")


def _case(FL, kind, dtype, dev):
    """leaves, gradients, the call under test, the same through the Python function"""
    gen = torch.Generator(device=dev).manual_seed(11)
    rnd = lambda *s, k=1.0: (k * torch.randn(*s, device=dev, generator=gen)).to(dtype)
    x, mods = rnd(2, 9, 3072), [rnd(2, 3072, k=0.2) for _ in range(2)]
    if kind in ("adaln", "module"):
        site = (lambda a, b, c: FL.modulated_layer_norm(a, b, c, eps=EPS)) if kind == "adaln" else FL.AdaLNCustom(3072, EPS)
        return [x, *mods], [rnd(2, 9, 3072)], site, lambda a, b, c: FL.AdaLNModelFunction.apply(a, b, c, EPS, 3072)
    if kind == "seq_first":
        return ([rnd(9, 2, 1536), *(rnd(2, 1536, k=0.2) for _ in range(2))], [rnd(9, 2, 1536)],
                lambda a, b, c: FL.modulated_layer_norm(a, b, c, eps=EPS, seq_first=True),
                lambda a, b, c: FL.AdaLNModelFunction.apply(a, b, c, EPS, 1536, True))
    if kind == "stream":
        return ([x, *mods], [rnd(2, 9, 3072) for _ in range(2)],
                lambda a, b, c: FL.modulated_layer_norm_keeping_stream(a, b, c, eps=EPS),
                lambda a, b, c: FL.AdaLNResidualFunction.apply(a, b, c, EPS))
    if kind == "gated":
        return ([x, rnd(2, 9, 3072), rnd(2, 3072, k=0.3), *mods], [rnd(2, 9, 3072) for _ in range(2)],
                lambda *a: FL.gated_residual_layer_norm(*a, eps=EPS), lambda *a: FL.GatedResidualAdaLNFunction.apply(*a, EPS))

    def norm(cols):
        return FL.RMSNorm(cols, eps=EPS).to(device=dev, dtype=dtype)

    def with_weight(module, w, call):
        """the module's parameter replaced by the leaf w, so that its gradient can be asked for"""
        del module.weight
        module.weight = w
        return call()

    if kind == "rms":
        m = norm(3072)
        return ([rnd(2, 9, 3072), rnd(3072)], [rnd(2, 9, 3072)],
                lambda a, w: with_weight(m, w, lambda: m(a)), lambda a, w: FL.RMSNormModelFunction.apply(a, w, EPS, 3072))
    if kind in ("view", "view3"):
        if kind == "view":
            base, cut, shape = rnd(2, 21, 3, 240), lambda t: t[..., 80:160].transpose(1, 2), (2, 3, 21, 80)
        else:
            base, cut, shape = rnd(2, 21, 240), lambda t: t[..., 80:160], (2, 21, 80)
        m = norm(80)
        return ([base, rnd(80)], [rnd(*shape)], lambda a, w: with_weight(m, w, lambda: m(cut(a))),
                lambda a, w: FL.RMSNormModelFunction.apply(cut(a), w, EPS, 80))
    tables = None
    if kind == "qkv_rope":
        angle = torch.arange(30 * 128, device=dev, dtype=torch.float32).view(30, 128) * 1e-3
        tables = (angle.cos(), angle.sin())

    nq, nk = norm(128), norm(128)

    def joint(a, wq, wk):
        return with_weight(nq, wq, lambda: with_weight(nk, wk, lambda: FL.split_qkv_and_norm(a, nq, nk, rotary=tables)))
    return ([rnd(2, 37, 3, 384), rnd(128), rnd(128)], [rnd(2, 3, 37, 128) for _ in range(3)], joint,
            lambda a, wq, wk: FL.QKVSplitNormFunction.apply(a, wq, wk, EPS, *(tables or ())))


def _tuple(outs):
    return outs if isinstance(outs, tuple) else (outs,)


def _leaves(args):
    # parameters, so that a module accepts them as its weight
    return [torch.nn.Parameter(a.detach().clone()) if a.dim() == 1 else a.detach().clone().requires_grad_(True) for a in args]


def _both(call, args, grads, use=None):
    leaves = _leaves(args)
    outs = _tuple(call(*leaves))
    picked = [(o, g) for i, (o, g) in enumerate(zip(outs, grads)) if use is None or i in use]
    got = torch.autograd.grad([o for o, _ in picked], leaves, [g for _, g in picked], allow_unused=True)
    return outs, [o.detach() for o in outs] + list(got)


def _same(a, b):
    return all((x is None and y is None) or (x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)) for x, y in zip(a, b))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", KINDS)
def test_native_node_equals_the_python_function(FL, gpu_device, kind, dtype):
    args, grads, site, function = _case(FL, kind, dtype, gpu_device)
    outs, got = _both(site, args, grads)
    ref, want = _both(function, args, grads)
    assert all("Site" in o.grad_fn.name() for o in outs if o.grad_fn.name().find("View") < 0)
    assert all(type(a) is type(b) and a.is_contiguous() == b.is_contiguous() and a.stride() == b.stride() for a, b in zip(outs, ref))
    assert _same(got, want)
    # gradients in another layout, off the alignment, of another dtype
    flat = torch.empty(grads[0].numel() + 1, dtype=dtype, device=gpu_device)
    shifted = [flat[1:].view(grads[0].shape).copy_(grads[0])] + grads[1:]
    assert _same(_both(site, args, shifted)[1], want)
    assert _same(_both(site, args, [g.transpose(-1, -2).contiguous().transpose(-1, -2) for g in grads])[1], want)
    # outputs that were not used
    for use in ([0], [len(grads) - 1]):
        assert _same(_both(site, args, grads, use)[1], _both(function, args, grads, use)[1])
    with torch.no_grad():
        assert _same(_tuple(site(*_leaves(args))), want) and not _tuple(site(*_leaves(args)))[0].requires_grad
    with torch.inference_mode():
        assert _same(_tuple(site(*[a.clone() if a.dim() > 1 else torch.nn.Parameter(a.clone()) for a in args])), want)


@pytest.mark.parametrize("kind", KINDS)
def test_hooks_repeats_and_checkpoints(FL, gpu_device, kind):
    args, grads, site, function = _case(FL, kind, torch.bfloat16, gpu_device)
    want = _both(function, args, grads)[1]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(gpu_device)):
        got = _both(site, args, grads)[1]
    if kind in ("view", "view3"):
        # the view comes back dense, its rows in another order: each sum of n terms is off by at most n 2^-24 of their
        # magnitudes (|xhat| <= sqrt(80)), and is rounded to bf16 once
        per_column = grads[0].float().abs().sum(tuple(range(grads[0].dim() - 1)))
        slack = 2 * (grads[0].numel() // 80) * 2.0 ** -24 * per_column * 80 ** 0.5
        apart = (got[2].float() - want[2].float()).abs()
        assert bool((apart <= slack + 2.0 ** -7 * want[2].float().abs()).all())
        got, want = got[:2], want[:2] + want[3:]
    assert packed and len(got) == len(want) and _same(got, want)
    want = _both(function, args, grads)[1]
    leaves = _leaves(args)
    outs = _tuple(site(*leaves))
    first = torch.autograd.grad(outs, leaves, grads, retain_graph=True)
    assert _same(torch.autograd.grad(outs, leaves, grads), first) and _same(first, want[len(outs):])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(outs, leaves, grads)
    for reentrant in (False, True):
        leaves = _leaves(args)
        outs = _tuple(checkpoint(site, *leaves, use_reentrant=reentrant))
        torch.autograd.backward(outs, grads)
        assert _same([p.grad for p in leaves], want[len(outs):])
    if kind != "gated":   # which keeps the sum it writes itself
        leaves = _leaves(args)   # what was saved may not be written over
        rows = leaves[0] * 1
        outs = _tuple(site(rows, *leaves[1:]))
        rows.detach().add_(1.0)
        with pytest.raises(RuntimeError, match="inplace"):
            torch.autograd.grad(outs, leaves, grads)


@pytest.mark.parametrize("kind", ["adaln", "stream", "gated", "rms", "qkv"])
def test_transforms_and_tangents_do_what_the_python_function_does(FL, gpu_device, kind):
    """Refused or handled alike: the call leaves the native path wherever one of them is active."""
    args, grads, site, function = _case(FL, kind, torch.bfloat16, gpu_device)
    rest = _leaves(args[1:])   # the row tensor alone is transformed: a module's parameter cannot be a wrapped tensor

    def tangent(call):
        with torch.autograd.forward_ad.dual_level():
            return call(torch.autograd.forward_ad.make_dual(args[0], torch.ones_like(args[0])))

    def outcome(run, call):
        try:
            return "ran", _tuple(run(lambda t: call(t, *rest)))
        except Exception as exc:
            return type(exc).__name__, str(exc)[:60]

    def batched(call):
        leaf = args[0].clone().requires_grad_(True)
        outs = _tuple(call(leaf))
        return torch.autograd.grad(outs, leaf, [torch.stack([g, g]) for g in grads], is_grads_batched=True)

    fixed = [torch.nn.Parameter(a.clone(), requires_grad=False) if a.dim() == 1 else a.clone() for a in args[1:]]

    def traced(call):   # operands that need a gradient cannot become constants of a trace
        rest[:] = fixed
        return torch.jit.trace(lambda t: call(t), (args[0],), check_trace=False)(args[0])

    def recorded(call):
        rest[:] = fixed
        return make_fx(lambda t: call(t))(args[0])(args[0])

    for run in (lambda c: torch.func.vmap(c)(args[0].unsqueeze(0)), lambda c: torch.func.vjp(c, args[0])[0], tangent, batched,
                traced, recorded):
        a, b = outcome(run, site), outcome(run, function)
        assert a[0] == b[0], (a, b)
        assert _same(a[1], b[1]) if a[0] == "ran" else a[1] == b[1], (a, b)


class _Tagged(torch.Tensor):
    pass


@pytest.mark.parametrize("kind", KINDS)
def test_subclasses_keep_what_the_python_function_gives_them(FL, gpu_device, kind):
    """The stream handed back is the caller's class, not a plain view of it."""
    args, grads, site, function = _case(FL, kind, torch.bfloat16, gpu_device)

    def run(call):
        leaves = _leaves(args)
        leaves[0] = leaves[0].detach().as_subclass(_Tagged).requires_grad_(True)
        outs = _tuple(call(*leaves))
        return [type(o) for o in outs], [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, grads))

    (a, got), (b, want) = run(site), run(function)
    assert a == b and _same(got, want)
    assert kind != "stream" or a[0] is _Tagged


@pytest.mark.parametrize("kind,scale,shift", [
    (kind, *shapes) for kind in ("adaln", "stream") for shapes in (
        ((2, 1, 3072), (2, 3072)), ((2, 3072), (2, 1, 3072)), ((3072,), (1, 3072)), ((1, 3072), (3072,)), ((1, 1, 3072), (3072,)))
] + [("seq_first", (2, 1, 1536), (2, 1536)), ("seq_first", (2, 1536), (2, 1, 1536))])
@pytest.mark.parametrize("how", ["ready", "gradient to prepare", "rows to prepare", "other dtypes"])
def test_scale_and_shift_of_unlike_shapes(FL, gpu_device, kind, scale, shift, how):
    """Each gets its gradient in its own shape and dtype, with the values that equal shapes get."""
    args, grads, site, function = _case(FL, kind, torch.bfloat16, gpu_device)
    if scale[0] != 2:   # one modulation row
        args, grads = [a[:1].contiguous() for a in args], [g[:1].contiguous() for g in grads]
    want = _both(function, args, grads)[1]
    shaped = [args[0], args[1].reshape(scale), args[2].reshape(shift)]
    if how == "gradient to prepare":
        grads = [g.transpose(-1, -2).contiguous().transpose(-1, -2) for g in grads]
    if how == "rows to prepare":
        shaped[0] = torch.empty(args[0].numel() + 1, dtype=args[0].dtype, device=gpu_device)[1:].view(args[0].shape).copy_(args[0])
    if how == "other dtypes":
        shaped[1] = shaped[1].float()
    for call in (site, function):
        leaves = [t.detach().requires_grad_(True) for t in shaped]
        outs = _tuple(call(*leaves))
        got = [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, grads))
        assert [(g.shape, g.dtype) for g in got[-2:]] == [(t.shape, t.dtype) for t in shaped[1:]]
        assert all(torch.equal(g.reshape(w.shape).to(w.dtype), w) for g, w in zip(got, want))


@pytest.mark.parametrize("kind", KINDS)
def test_a_second_derivative_is_refused(FL, gpu_device, kind):
    """Under create_graph the gradients are the same; a loss that mixes them with other terms is not differentiated without
    them in silence."""
    args, grads, site, function = _case(FL, kind, torch.bfloat16, gpu_device)
    want = _both(function, args, grads)[1]
    for call in (site, function):
        leaves = _leaves(args)
        outs = _tuple(call(*leaves))
        got = torch.autograd.grad(outs, leaves, grads, create_graph=True)
        assert _same([g.detach() for g in got], want[len(outs):]) and all(g.requires_grad for g in got)
        assert [g.stride() for g in got] == [g.stride() for g in want[len(outs):]]
        for g in got:
            with pytest.raises(RuntimeError, match="no second derivative"):
                torch.autograd.grad(g.float().sum() + leaves[0].float().pow(2).sum(), leaves[0], retain_graph=True)
        for i in range(len(grads) if len(grads) > 1 else 0):   # one output used, the others' gradients missing
            if kind == "stream" and i == 0:
                continue
            leaves = _leaves(args)
            some = torch.autograd.grad(_tuple(call(*leaves))[i], leaves, grads[i], create_graph=True, allow_unused=True)
            assert _same([g if g is None else g.detach() for g in some], _both(function, args, grads, [i])[1][len(outs):])
            with pytest.raises(RuntimeError, match="no second derivative"):
                torch.autograd.grad(some[0].float().sum() + leaves[0].float().pow(2).sum(), leaves[0])
        # operands that were copied first have no path to the copy; backward() refuses all the same
        leaves = _leaves(args)
        rows = torch.empty(args[0].numel() + 1, dtype=args[0].dtype, device=gpu_device)[1:].view(args[0].shape).copy_(leaves[0])
        got = torch.autograd.grad(_tuple(call(rows, *leaves[1:])), leaves, grads, create_graph=True)
        with pytest.raises(RuntimeError, match="no second derivative"):
            (got[0].float().sum() + leaves[0].float().pow(2).sum()).backward()
        if kind == "stream":   # the stream alone is an identity, differentiable as often as one likes
            leaves = _leaves(args)
            out = call(*leaves)[0]
            first, = torch.autograd.grad(out.float().pow(3).sum(), leaves[0], create_graph=True)
            second, = torch.autograd.grad(first.float().sum(), leaves[0])
            torch.testing.assert_close(second.float(), 6 * args[0].float(), rtol=2.0 ** -6, atol=0)


def test_another_stream_and_several_threads(FL, gpu_device):
    args, grads, site, function = _case(FL, "gated", torch.bfloat16, gpu_device)
    want = _both(function, args, grads)[1]
    torch.cuda.synchronize()
    results = [None] * 4

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(5):
                results[i] = _both(site, args, grads)[1]
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert all(r is not None and _same(r, want) for r in results)
