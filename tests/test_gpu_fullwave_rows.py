"""Rows of 33 to 383 16-byte pieces (a full wavefront per row, anywidth.hip) where their kernels have edges: accesses
that end inside the row's last 1 KiB, the five-access geometry, fewer rows than wavefronts, and enough rows that the
forward kernel gives a wavefront two of them with a remainder.  Bars as in test_gpu_anywidth.py."""
import pytest
import torch

from oracle import norm_oracle as O
from tests.test_gpu_anywidth import colsum_ok, fwd_16bit_ok, grad_ok

pytestmark = pytest.mark.gpu
EPS = 1e-6
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32
# batch, rows per sample, pieces per row
CASES = [(1, 1, 33), (2, 4101, 65), (3, 7, 129), (1, 1025, 193), (2, 515, 257), (1, 4099, 289),
         (1, 5131, 257), (1, 3, 320), (2, 67, 321), (1, 130, 383)]


@pytest.fixture(scope="module")
def capi(gpu_device):
    from teletron_amd import capi as c
    c.lib()
    return c


def _margins(like):
    """A tensor like `like` inside a buffer whose margins must stay as they are."""
    buf = torch.full((4096 + like.numel() + 4096,), 7.0, dtype=like.dtype, device=like.device)
    return buf, buf[4096:-4096].view(like.shape)


@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("batch,seq,pieces", CASES)
def test_full_wavefront_rows_match_the_oracle(capi, gpu_device, batch, seq, pieces, dtype):
    cols = pieces * (4 if dtype == F32 else 8)
    d = O.make_adaln_inputs(batch, seq, cols, dtype, seed=pieces + seq, sigma=1.5)
    want_out, want_dx, want_ds, want_dh = O.eager_adaln_fwd_bwd(d["x"], d["scale"], d["shift"], d["grad"])
    x, sc, sh, g = (d[k].to(gpu_device) for k in ("x", "scale", "shift", "grad"))
    out, mean, rstd = capi.adaln_forward(x, sc, sh, EPS)
    dx, ds, dh = capi.adaln_backward(g, x, sc, mean, rstd)
    if dtype == F32:
        torch.testing.assert_close(out.cpu(), want_out, rtol=1e-5, atol=1e-5)
        grad_ok(dx, want_dx, "dx")
    else:
        fwd_16bit_ok(out, want_out, O.adaln_excuse(d["x"], d["scale"], d["shift"], want_out), "out")
        terms = O.adaln_dx_terms(d["x"], d["scale"], d["grad"])
        assert O.frac_outside(dx.cpu(), want_dx, 1e-2, 1e-3, magnitude=terms) <= 1e-4
    xn = torch.nn.functional.layer_norm(d["x"].float(), (cols,), None, None, EPS)
    colsum_ok(ds, want_ds, d["grad"].float() * xn, 1, "dscale")
    colsum_ok(dh, want_dh, d["grad"].float(), 1, "dshift")

    r = O.make_rmsnorm_inputs((batch * seq,), cols, dtype, seed=pieces)
    want_out, want_dx, want_dw = O.eager_rmsnorm_fwd_bwd(r["x"], r["weight"], r["grad"])
    x, w, g = (r[k].to(gpu_device) for k in ("x", "weight", "grad"))
    buf_o, out = _margins(x)
    buf_d, dx = _margins(x)
    _, rstd = capi.rmsnorm_forward(x, w, EPS, out=out)
    _, dw = capi.rmsnorm_backward(g, x, w, rstd, dx=dx)
    for buf in (buf_o, buf_d):
        assert bool((buf[:4096] == 7.0).all()) and bool((buf[-4096:] == 7.0).all())
    if dtype == F32:
        torch.testing.assert_close(out.cpu(), want_out, rtol=1e-5, atol=1e-6)
    else:
        fwd_16bit_ok(out, want_out, O.rmsnorm_excuse(want_out), "out")
    grad_ok(dx, want_dx, "dx", allow=1e-5)
    colsum_ok(dw, want_dw, r["grad"].float() * want_out.float(), 0, "dweight")


@pytest.mark.parametrize("dtype", [BF, HF, F32])
def test_an_infinite_gradient_stays_in_its_column(capi, gpu_device, dtype):
    """The column sums of the other columns are what they are without it."""
    d = O.make_adaln_inputs(1, 9, 1544, dtype, seed=3)
    x, sc, sh, g = (d[k].to(gpu_device) for k in ("x", "scale", "shift", "grad"))
    bad = g.clone()
    bad[0, 4, 100] = float("inf")
    others = torch.arange(1544, device=gpu_device) != 100
    _, mean, rstd = capi.adaln_forward(x, sc, sh, EPS)
    for a, b in zip(capi.adaln_backward(g, x, sc, mean, rstd)[1:], capi.adaln_backward(bad, x, sc, mean, rstd)[1:]):
        assert torch.equal(a[:, others], b[:, others]) and not bool(torch.isfinite(b[0, 100]))
    w = torch.ones(1544, dtype=dtype, device=gpu_device)
    _, rstd = capi.rmsnorm_forward(x[0], w, EPS)
    a, b = (capi.rmsnorm_backward(t[0], x[0], w, rstd)[1] for t in (g, bad))
    assert torch.equal(a[others], b[others]) and not bool(torch.isfinite(b[100]))
