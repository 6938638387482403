"""The joint QK-norm kernels (qkv.hip): the sizes where a row's lanes, a wavefront's tokens, a workgroup's heads or the
persistent grid are partly empty, in every lane geometry, against the eager oracle on the CPU and, bit for bit where
the arithmetic is the same, the strided kernels one tensor at a time."""
import pytest
import torch

from oracle import norm_oracle as O

pytestmark = pytest.mark.gpu
EPS = 1e-6
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def capi(gpu_device):
    from teletron_amd import capi as c
    c.lib()
    return c


# B, S, H, D, rotated tokens.  D in 16-byte pieces of two-byte rows: 1, 8, 9, 16, 32, 63, 64 -> 8, 8, 16, 16, 32, 64, 64 lanes
CASES = [
    (1, 1, 1, 128, 0), (2, 3, 5, 8, 0), (3, 17, 2, 64, 0), (1, 33, 7, 72, 0), (2, 15, 3, 256, 0), (1, 9, 4, 504, 0),
    (2, 5, 3, 512, 0), (1, 1501, 24, 128, 0), (2, 61, 5, 128, 61), (1, 67, 9, 128, 40), (1, 5, 1, 128, 1),
    # few token groups or few heads: wavefronts of the forward workgroup on other samples or more tokens
    (5, 6, 3, 128, 0), (9, 1, 1, 64, 0), (7, 1, 3, 128, 1), (1, 300, 1, 128, 290), (3, 21, 3, 128, 21),
    # several runs of neighbouring heads per wavefront in the rotated backward, runs that straddle token groups and samples
    (2, 1501, 24, 128, 1501), (1, 2999, 11, 128, 2950), (3, 1000, 9, 128, 990),
]


@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("B,S,H,D,rotated", CASES)
def test_joint_kernels_match_the_oracle(capi, gpu_device, B, S, H, D, rotated, dtype):
    if dtype == F32 and D > 256:
        assert capi.lib().tt_qkv_rmsnorm_supported(D, capi.F32) == 0      # more than 64 pieces
        return
    gen = torch.Generator().manual_seed(S * 31 + D)
    mixed = torch.randn(B, S, H, 3 * D, generator=gen).to(dtype)
    w = [(1 + 0.02 * torch.randn(D, generator=gen)).to(dtype) for _ in range(2)]
    grads = [torch.randn(B, H, S, D, generator=gen).to(dtype) for _ in range(3)]
    tables = O.make_rope_tables(rotated, D, seed=5) if rotated else (None, None)
    dev = lambda t: None if t is None else t.to(gpu_device)
    cos, sin = dev(tables[0]), dev(tables[1])
    m_d, w_d, g_d = dev(mixed), [dev(t) for t in w], [dev(t) for t in grads]

    # outputs between margins that must stay as they are
    def guarded(*shape):
        buf = torch.full((2048 + torch.Size(shape).numel() + 2048,), 7.0, dtype=dtype, device=gpu_device)
        return buf, buf[2048:-2048].view(shape)

    buf, dmixed = guarded(B, S, H, 3 * D)
    q, k = capi.qkv_rmsnorm_forward(m_d, *w_d, EPS, cos, sin)
    _, dwq, dwk = capi.qkv_rmsnorm_backward(*g_d, m_d, *w_d, EPS, cos, sin, dmixed=dmixed)
    assert bool((buf[:2048] == 7.0).all()) and bool((buf[-2048:] == 7.0).all())
    assert torch.equal(dmixed[..., 2 * D:].transpose(1, 2), g_d[2])

    # 16-bit bars as for the per-tensor kernels; fp32 leaves room for the order of the sums only
    rtol, atol = (1e-4, 1e-5) if dtype == F32 else (1e-2, 1e-3)
    for t, (out, dw) in enumerate(((q, dwq), (k, dwk))):
        x = m_d[..., t * D:(t + 1) * D].transpose(1, 2)
        if rotated:
            want = capi.rmsnorm_rope_forward_strided(x, w_d[t], cos, sin, EPS)[0]
            e_out, e_dx, e_dw = O.eager_qk_norm_rope_fwd_bwd(x.cpu(), w[t], *tables, grads[t])
        else:
            want = capi.rmsnorm_forward_strided(x, w_d[t], EPS)[0]
            e_out, e_dx, e_dw = O.eager_rmsnorm_fwd_bwd(x.cpu(), w[t], grads[t])
        assert torch.equal(out, want)
        assert O.frac_outside(out.cpu(), e_out, 2.0 ** -6 if dtype != F32 else 1e-5, 2.0 ** -7 if dtype != F32 else 1e-6) == 0.0
        dx = dmixed[..., t * D:(t + 1) * D].transpose(1, 2)
        # short rows: the two terms of dx cancel, and a one-ulp disagreement has the size of the terms
        terms = e_dx.float().abs() + x.cpu().float().abs() + grads[t].float().abs()
        assert O.frac_outside(dx.cpu(), e_dx, rtol, atol, magnitude=terms) == 0.0
        y = torch.nn.functional.normalize(x.cpu().float(), dim=-1) * D ** 0.5
        assert O.colsum_outside(dw.cpu(), e_dw, (grads[t].float() * y).reshape(-1, D), dim=0, rtol=rtol,
                                ulp=2.0 ** -6 if dtype != F32 else 1e-5) == 0


@pytest.mark.parametrize("missing", [(0,), (1,), (2,), (0, 2)])
def test_outputs_that_were_not_used(capi, gpu_device, missing):
    """A missing gradient leaves zeros in its slice and its dweight and does not touch the others; a row of infinities
    under it leaves zeros too."""
    gen = torch.Generator(device=gpu_device).manual_seed(3)
    mixed = torch.randn(1, 21, 3, 384, device=gpu_device, generator=gen).to(BF)
    w = [torch.ones(128, device=gpu_device, dtype=BF) for _ in range(2)]
    grads = [torch.randn(1, 3, 21, 128, device=gpu_device, generator=gen).to(BF) for _ in range(3)]
    full = capi.qkv_rmsnorm_backward(*grads, mixed, *w, EPS)
    if 0 in missing:
        mixed[..., :128] = float("inf")
    got = capi.qkv_rmsnorm_backward(*[None if i in missing else g for i, g in enumerate(grads)], mixed, *w, EPS)
    for i in range(3):
        part, whole = (t[0][..., i * 128:(i + 1) * 128] for t in (got, full))
        assert (not part.any()) if i in missing else torch.equal(part, whole)
        if i < 2:
            assert (not got[1 + i].any()) if i in missing else torch.equal(got[1 + i], full[1 + i])


def test_empty_projection_and_refusals(capi, gpu_device):
    w = [torch.ones(64, device=gpu_device, dtype=BF) for _ in range(2)]
    mixed = torch.empty(2, 0, 4, 192, device=gpu_device, dtype=BF)
    none = torch.empty(2, 4, 0, 64, device=gpu_device, dtype=BF)
    assert capi.qkv_rmsnorm_forward(mixed, *w, EPS)[0].numel() == 0
    _, dwq, dwk = capi.qkv_rmsnorm_backward(none, none, none, mixed, *w, EPS)
    assert not dwq.any() and not dwk.any()
    wide = torch.empty(1, 2, 1, 3 * 520, device=gpu_device, dtype=BF)
    with pytest.raises(capi.NormError, match="64 whole 16-byte pieces"):
        capi.qkv_rmsnorm_forward(wide, *[torch.ones(520, device=gpu_device, dtype=BF)] * 2, EPS)


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("dtype", [BF, HF, F32])
def test_an_infinite_gradient_stays_in_its_column(capi, gpu_device, D, dtype):
    gen = torch.Generator(device=gpu_device).manual_seed(D)
    rnd = lambda *s: torch.randn(*s, device=gpu_device, generator=gen).to(dtype)
    mixed, w, grads = rnd(1, 19, 2, 3 * D), rnd(D), [rnd(1, 2, 19, D) for _ in range(3)]
    bad = [g.clone() for g in grads]
    bad[0][0, 1, 7, 20] = float("inf")
    others = torch.arange(D, device=gpu_device) != 20
    a, b = (capi.qkv_rmsnorm_backward(*g, mixed, w, w, EPS) for g in (grads, bad))
    assert torch.equal(a[1][others], b[1][others]) and not bool(torch.isfinite(b[1][20]))
    assert torch.equal(a[2], b[2])


# Both sides of the forward's rules: one head / two heads per wavefront (four workgroups of one head per compute unit; whole
# rows back to one from 32 on; odd heads, a single head), heads by pieces of 2048 tokens where tokens lie whole 4 KiB apart
# (three pieces and a ragged last one, and too few), and the throttled grid with tables.
SPLITS = [
    (1, 677, 24, 128, 0, BF), (1, 681, 24, 128, 0, BF), (3, 913, 5, 64, 0, HF), (1, 5463, 24, 128, 0, BF), (1, 20000, 1, 128, 0, BF),
    (1, 4099, 5, 80, 0, BF), (2, 9001, 7, 96, 0, F32), (1, 6143, 16, 128, 0, BF), (1, 6151, 16, 128, 0, BF), (2, 6149, 8, 128, 0, F32),
    (1, 8201, 32, 64, 0, HF), (1, 6147, 16, 128, 6100, BF), (1, 6147, 16, 128, 6147, F32), (1, 3417, 24, 128, 3400, BF),
]


@pytest.mark.parametrize("B,S,H,D,rotated,dtype", SPLITS)
def test_forward_splits_equal_one_norm_per_tensor(capi, gpu_device, B, S, H, D, rotated, dtype):
    gen = torch.Generator(device=gpu_device).manual_seed(S + D)
    mixed = torch.randn(B, S, H, 3 * D, device=gpu_device, generator=gen).to(dtype)
    w = [(1 + 0.02 * torch.randn(D, device=gpu_device, generator=gen)).to(dtype) for _ in range(2)]
    cos, sin = (t.to(gpu_device) for t in O.make_rope_tables(rotated, D, seed=5)) if rotated else (None, None)
    n = B * H * S * D
    buf = torch.full((2, 4096 + n + 4096), 7.0, dtype=dtype, device=gpu_device)
    q, k = (b[4096:-4096].view(B, H, S, D) for b in buf)
    p = capi._p
    capi._check(capi.lib().tt_qkv_rmsnorm_forward(p(q), p(k), p(mixed), p(w[0]), p(w[1]), p(cos), p(sin), rotated, B, S, H, D, EPS,
                                                  capi._dt(mixed), capi._stream(mixed)), "tt_qkv_rmsnorm_forward")
    for t, out in enumerate((q, k)):
        x = mixed[..., t * D:(t + 1) * D].transpose(1, 2)
        want = (capi.rmsnorm_rope_forward_strided(x, w[t], cos, sin, EPS) if rotated else
                capi.rmsnorm_forward_strided(x, w[t], EPS))[0]
        assert torch.equal(out, want)
    assert bool((buf[:, :4096] == 7.0).all()) and bool((buf[:, -4096:] == 7.0).all())
