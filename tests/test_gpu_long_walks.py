"""Persistent backward grids walk a row at a time; from some length of the walk on a row's requests wait for the stores of the
row before it.  Rows do not depend on each other, so a long call must equal its halves, each of them below that length."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 1e-6
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def capi(gpu_device):
    from teletron_amd import capi as c
    c.lib()
    return c


def _sums_agree(whole, parts, terms, dtype):
    """Column sums of `terms` positive-variance terms of size about one: fp32 partial sums differ by their order (at most
    terms * 2^-24 of the sum of magnitudes, which is below 2 * terms), and each result is rounded once to the element type.
    The bound is wide beside a single row: that every row is counted is what the next test asks."""
    total = sum(p.float() for p in parts)
    slack = 2.0 * terms * terms ** 0.5 * 2.0 ** -24
    ulp = {BF: 2.0 ** -8, HF: 2.0 ** -11, F32: 2.0 ** -24}[dtype]
    size = torch.stack([whole.float().abs(), *(p.float().abs() for p in parts)]).sum(0)
    return bool(((whole.float() - total).abs() <= slack + ulp * size).all())


# 24 steps of 2048 wavefronts begin at 49 152 groups of heads and tokens
LONG = [
    (1, 8240, 24, 128, 0, BF), (1, 8241, 24, 128, 8200, BF), (2, 10925, 9, 80, 0, HF), (1, 6149, 16, 96, 0, F32), (1, 12000, 34, 64, 0, BF),
    (1, 4103, 24, 128, 4103, F32), (1, 8243, 24, 128, 0, HF), (1, 16390, 12, 128, 16001, HF)]


def _waits_for_stores(B, S, H, D, dtype, device):
    """Whether the call's walk is past the line: wavefronts take 64 / lanes tokens of a head at a time, two workgroups of
    four of them per compute unit."""
    pieces = D * torch.empty(0, dtype=dtype).element_size() // 16
    tokens = 64 // next(n for n in (8, 16, 32, 64) if pieces <= n)
    return B * -(-S // tokens) * H >= 24 * 8 * torch.cuda.get_device_properties(device).multi_processor_count


@pytest.mark.parametrize("B,S,H,D,rotated,dtype", LONG)
def test_joint_backward_equals_its_halves(capi, gpu_device, B, S, H, D, rotated, dtype):
    gen = torch.Generator(device=gpu_device).manual_seed(S + D)
    rnd = lambda *s: torch.randn(*s, device=gpu_device, generator=gen).to(dtype)
    mixed, w, grads = rnd(B, S, H, 3 * D), [rnd(D) for _ in range(2)], [rnd(B, H, S, D) for _ in range(3)]
    cos, sin = (torch.randn(rotated, D, device=gpu_device, generator=gen) for _ in range(2)) if rotated else (None, None)
    whole = capi.qkv_rmsnorm_backward(*grads, mixed, *w, EPS, cos, sin)
    half = S // 2 // 8 * 8
    assert _waits_for_stores(B, S, H, D, dtype, gpu_device)
    assert not any(_waits_for_stores(B, n, H, D, dtype, gpu_device) for n in (half, S - half))
    parts = []
    for cut in (slice(0, half), slice(half, S)):
        t = (None, None) if not rotated else tuple(a[cut].contiguous() for a in (cos, sin))
        parts.append(capi.qkv_rmsnorm_backward(*(g[:, :, cut].contiguous() for g in grads), mixed[:, cut].contiguous(), *w, EPS, *t))
    assert torch.equal(whole[0], torch.cat([p[0] for p in parts], 1))
    for i in (1, 2):
        assert _sums_agree(whole[i], [p[i] for p in parts], B * S * H, dtype)
    again = capi.qkv_rmsnorm_backward(*grads, mixed, *w, EPS, cos, sin)
    assert all(torch.equal(a, b) for a, b in zip(whole, again))


@pytest.mark.parametrize("B,S,H,D,rotated,dtype", LONG)
def test_joint_backward_counts_every_row(capi, gpu_device, B, S, H, D, rotated, dtype):
    """Rows of +-1 (their own norm at an epsilon that 32 bits lose beside 1), gradients of +-1 and rotations by quarter turns: every
    term of a column sum is +-1 and every order of fp32 additions exact, so the sums are whole numbers, rounded once."""
    gen = torch.Generator(device=gpu_device).manual_seed(S)
    signs = lambda *s: (2 * torch.randint(0, 2, s, device=gpu_device, generator=gen) - 1).to(dtype)
    mixed, grads, w = signs(B, S, H, 3 * D), [signs(B, H, S, D) for _ in range(3)], torch.ones(D, device=gpu_device, dtype=dtype)
    cos = sin = None
    turned = [g.double() for g in grads[:2]]
    if rotated:
        quarter = torch.randint(0, 2, (rotated, D // 2), device=gpu_device, generator=gen).repeat_interleave(2, 1).float()
        cos, sin = (1 - quarter).contiguous(), quarter
        # out = (cos x_even - sin x_odd, cos x_odd + sin x_even): its gradient turns the other way
        for g in turned:
            even, odd = g[:, :, :rotated, 0::2].clone(), g[:, :, :rotated, 1::2].clone()
            c, s = cos[:, 0::2].double(), sin[:, 0::2].double()
            g[:, :, :rotated, 0::2], g[:, :, :rotated, 1::2] = c * even + s * odd, c * odd - s * even
    _, dwq, dwk = capi.qkv_rmsnorm_backward(*grads, mixed, w, w, 1e-30, cos, sin)
    for i, dw in enumerate((dwq, dwk)):
        x = mixed[..., i * D:(i + 1) * D].transpose(1, 2).double()
        assert torch.equal(dw, (turned[i] * x).sum((0, 1, 2)).to(dtype))


@pytest.mark.parametrize("batch,rows,cols,dtype", [
    (1, 4099, 4096, BF), (2, 2051, 3072, F32), (1, 4095, 5128, HF), (1, 1031, 1152, BF), (3, 700, 2048, BF), (1, 2049, 1536, F32),
    (1, 2050, 3072, BF)])
def test_residual_backward_equals_the_plain_one_plus_the_other_gradient(capi, gpu_device, batch, rows, cols, dtype):
    gen = torch.Generator(device=gpu_device).manual_seed(rows + cols)
    rnd = lambda *s: torch.randn(*s, device=gpu_device, generator=gen).to(dtype)
    x, g, other, scale, shift = rnd(batch, rows, cols), rnd(batch, rows, cols), rnd(batch, rows, cols), rnd(batch, cols), rnd(batch, cols)
    _, mean, rstd = capi.adaln_forward(x, scale, shift, EPS)
    dx, dscale, dshift = capi.adaln_backward(g, x, scale, mean, rstd)
    got = capi.adaln_backward_residual(g, other, x, scale, mean, rstd)
    assert torch.equal(got[0], dx + other) and torch.equal(got[1], dscale) and torch.equal(got[2], dshift)


# wide rows: one, two and four rows per workgroup of the forward, each side of the lines (four and ten workgroups of one row per
# compute unit), rows that do not fill the last workgroup
@pytest.mark.parametrize("batch,rows,cols,dtype", [
    (1, 1, 4096, BF), (1, 1024, 4096, BF), (1, 1027, 4096, HF), (3, 853, 5128, BF), (1, 2563, 4096, BF), (2, 1283, 5120, BF),
    (1, 1023, 2048, F32), (5, 207, 3072, F32), (1, 2575, 2048, F32)])
def test_wide_forward_does_not_depend_on_its_grid(capi, gpu_device, batch, rows, cols, dtype):
    gen = torch.Generator(device=gpu_device).manual_seed(rows + cols)
    rnd = lambda *s: torch.randn(*s, device=gpu_device, generator=gen).to(dtype)
    x, attn, gate, scale, shift = rnd(batch, rows, cols), rnd(batch, rows, cols), rnd(batch, cols), rnd(batch, cols), rnd(batch, cols)

    def one_sample(b, cut):
        return (capi.adaln_forward(x[b:b + 1, cut].contiguous(), scale[b:b + 1].contiguous(), shift[b:b + 1].contiguous(), EPS),
                capi.gated_residual_adaln_forward(x[b:b + 1, cut].contiguous(), attn[b:b + 1, cut].contiguous(), gate[b:b + 1].contiguous(),
                                                  scale[b:b + 1].contiguous(), shift[b:b + 1].contiguous(), EPS))

    plain, gated = capi.adaln_forward(x, scale, shift, EPS), capi.gated_residual_adaln_forward(x, attn, gate, scale, shift, EPS)
    for b in range(batch):
        for start in range(0, rows, 400):
            cut = slice(start, min(start + 400, rows))
            a, g = one_sample(b, cut)
            for whole, part in zip((*plain, *gated), (*a, *g)):
                assert torch.equal(whole.view(batch, rows, -1)[b, cut], part.view(cut.stop - cut.start, -1))
    assert torch.isfinite(plain[0].float()).all()
