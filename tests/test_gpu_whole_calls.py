"""The autograd functions run as one native call where every operand is ready as it is (dense, 16-byte aligned, one
dtype) and through their Python preparation otherwise: the same values either way, in outputs and gradients,
also when saved tensors or incoming gradients pass through a hook or arrive in another layout."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 1e-6


def _shifted(t):
    """The same values one element off the 16-byte alignment."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


def _operands(kind, dtype, dev):
    gen = torch.Generator(device=dev).manual_seed(7)
    rnd = lambda *s, k=1.0: (k * torch.randn(*s, device=dev, generator=gen)).to(dtype)
    if kind in ("qkv", "qkv_rope"):
        return [rnd(2, 37, 3, 3 * 128), rnd(128, k=0.1), rnd(128, k=0.1)], [rnd(2, 3, 37, 128) for _ in range(3)]
    if kind == "rms":
        return [rnd(2, 9, 3072), rnd(3072)], [rnd(2, 9, 3072)]
    if kind == "view":
        return [rnd(2, 21, 3, 192), rnd(64)], [rnd(2, 3, 21, 64)]
    if kind == "seq_first":
        return [rnd(9, 2, 1536), rnd(2, 1536, k=0.1), rnd(2, 1536, k=0.1)], [rnd(9, 2, 1536)]
    x = [rnd(2, 9, 3072), rnd(2, 3072, k=0.1), rnd(2, 3072, k=0.1)]
    if kind == "gated":
        x = [x[0], rnd(2, 9, 3072), rnd(2, 3072, k=0.3), x[1], x[2]]
    return x, [rnd(2, 9, 3072) for _ in range(2 if kind in ("gated", "stream") else 1)]


def _run(kind, args, grads):
    from teletron_amd import fusedlayers as FL
    leaves = [a.detach().requires_grad_(True) for a in args]
    if kind == "adaln":
        outs = [FL.modulated_layer_norm(*leaves, eps=EPS)]
    elif kind == "seq_first":
        outs = [FL.modulated_layer_norm(*leaves, eps=EPS, seq_first=True)]
    elif kind == "stream":
        outs = list(FL.modulated_layer_norm_keeping_stream(*leaves, eps=EPS))
    elif kind == "gated":
        outs = list(FL.gated_residual_layer_norm(*leaves, eps=EPS))
    elif kind == "rms":
        outs = [FL.RMSNormModelFunction.apply(*leaves, EPS, 3072)]
    elif kind == "view":
        outs = [FL.RMSNormModelFunction.apply(leaves[0][..., 64:128].transpose(1, 2), leaves[1], EPS, 64)]
    else:
        angle = torch.arange(30 * 128, device=args[0].device, dtype=torch.float32).view(30, 128) * 1e-3
        tables = (angle.cos(), angle.sin()) if kind == "qkv_rope" else ()
        outs = list(FL.QKVSplitNormFunction.apply(*leaves, EPS, *tables))
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, grads))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["adaln", "seq_first", "stream", "gated", "rms", "view", "qkv", "qkv_rope"])
def test_ready_and_prepared_operands_agree(gpu_device, kind, dtype):
    args, grads = _operands(kind, dtype, gpu_device)
    want = _run(kind, args, grads)
    others = [
        ([_shifted(a) if a.dim() > 2 else a for a in args], grads),
        (args, [_shifted(g) for g in grads]),
        (args, [g.transpose(-1, -2).contiguous().transpose(-1, -2) for g in grads]),
        ([a if a.dim() > 2 else torch.stack([a, a], -1)[..., 0] for a in args], grads),
    ]
    if kind == "view":   # a misaligned view is copied and its rows walked in another order: another order of sums
        others = others[1:]
    for a, g in others:
        got = _run(kind, a, g)
        assert all(x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y) for x, y in zip(got, want))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.clone(), lambda t: t.clone()):
        got = _run(kind, args, grads)
    assert all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("kind", ["adaln", "stream", "gated", "rms", "qkv"])
def test_parameters_of_another_dtype_get_gradients_of_their_own(gpu_device, kind):
    args, grads = _operands(kind, torch.bfloat16, gpu_device)
    want = _run(kind, args, grads)
    wide = [a.float() if a.dim() < 3 else a for a in args]
    got = _run(kind, wide, grads)
    for a, x, y in zip(wide, got[-len(args):], want[-len(args):]):
        assert x.dtype == a.dtype and torch.equal(x, y.to(a.dtype))


# shapes of gate, scale and shift; [B, 1, C] is gate.unsqueeze(1), as a block that broadcasts it over the tokens holds it
@pytest.mark.parametrize("batch,gate,scale,shift", [
    (2, (2, 1, 3072), (2, 3072), (2, 3072)), (2, (2, 3072), (2, 1, 3072), (2, 1, 3072)),
    (2, (2, 3072), (2, 3072), (2, 1, 3072)), (1, (1, 1, 3072), (3072,), (3072,)), (1, (3072,), (1, 3072), (3072,))])
@pytest.mark.parametrize("dense_grad", [True, False])
def test_gated_modulation_rows_of_unlike_shapes(gpu_device, batch, gate, scale, shift, dense_grad):
    """Every modulation row gets its gradient in its own shape, with the values that equal shapes get."""
    args, grads = _operands("gated", torch.bfloat16, gpu_device)
    args = [a[:batch] for a in args]
    grads = [g[:batch] for g in grads]
    want = _run("gated", args, grads)
    shaped = args[:2] + [a.reshape(s) for a, s in zip(args[2:], (gate, scale, shift))]
    got = _run("gated", shaped, grads if dense_grad else [_shifted(g) for g in grads])
    for x, y, a in zip(got[2:], want[2:], shaped):
        assert x.shape == a.shape and torch.equal(x, y.reshape(a.shape))
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_projections_of_too_many_rows_take_one_norm_per_tensor(gpu_device, monkeypatch):
    """Past the joint kernels' row count (lowered here) the call runs one strided norm per tensor: the same values."""
    from teletron_amd import fusedlayers as FL
    args, grads = _operands("qkv", torch.bfloat16, gpu_device)
    args[0] = _shifted(args[0])   # prepared in Python, where the route is chosen
    want = _run("qkv", args, grads)
    monkeypatch.setattr(FL, "_MAX_JOINT_ROWS", args[0].numel() // 384 - 1)
    got = _run("qkv", args, grads)
    assert all(torch.equal(x, y) for x, y in zip(got[:4], want[:4]))
    # dweights: 222 terms near 1 in another order, at most 222 * 222 * 2^-24 = 3e-3 apart in fp32, then one bf16 rounding each
    for x, y in zip(got[4:], want[4:]):
        torch.testing.assert_close(x.float(), y.float(), rtol=2.0 ** -7, atol=3e-3)
