"""The tile adjoints and the fused smoothing layer.

* wh_modwt_fwd_adj over one to several level groups, short and long signals,
  against the same sums in torch (64 bits; FP32 to its rounding);
* wh_modwt_fwd_details_adj equals it with zeros in the S_j slots, bit for bit;
* wh_modwt_inv_adj as tiles equals its sliding-window form bit for bit;
* wh_modwt_thresh_inv_adj against wh_modwt_inv_adj then wh_thresh_grad: the
  cotangent bit for bit, the per-level sums to the rounding of their order;
* smooth_levels' output and signal gradient equal the composite's bit for bit;
* wh_mse_grad against torch's mean of a square.
"""
import ctypes as C

import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import autograd as A
from wavecuda_amd import device as D

pytestmark = pytest.mark.gpu
SHAPES = [(3, 16, 2, "D4"), (1, 1024, 6, "LA8"), (5, 256, 7, "Haar"), (2, 1 << 12, 8, "LA8"),
          (3, 1 << 13, 10, "C6"), (2, 1 << 14, 13, "D4"), (70, 1 << 12, 8, "LA8"),
          (130, 1 << 12, 8, "LA8"), (260, 1 << 12, 4, "Haar"), (520, 1 << 12, 6, "D4")]


def _p(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _code(dt):
    return W.WH_F64 if dt == torch.float64 else W.WH_F32


def _rand(dtype, *shape):
    return torch.randn(*shape, dtype=dtype, device="cuda",
                       generator=torch.Generator(device="cuda").manual_seed(sum(shape)))


def _taps(filt):
    """(scaling, wavelet) filters read off the library's one-level transform."""
    L = W.FILTER_LENGTHS[filt]
    x = torch.zeros(64, dtype=torch.float64, device="cuda")
    x[0] = 1.0
    w = D.modwt_fwd(x, 1, filt).view(2, 64)
    k = [(-i) % 64 for i in range(L)]
    return w[0, k].tolist(), w[1, k].tolist()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,n,J,name", SHAPES)
def test_forward_adjoint(dtype, B, n, J, name):
    f = D.filter_code(name)
    g = _rand(dtype, B, 2 * n * J)
    gx, gd = torch.empty(B, n, dtype=dtype, device="cuda"), torch.empty(B, n, dtype=dtype, device="cuda")
    W.check(W.lib().wh_modwt_fwd_adj(_p(g), _p(gx), n, B, J, f, _code(dtype), None))
    c, d = _taps(f)
    v = g.double().view(B, J, 2, n)
    u = v[:, J - 1, 0]
    for j in range(J, 0, -1):
        s = 1 << (j - 1)
        up = v[:, j - 2, 0].clone() if j > 1 else torch.zeros(B, n, dtype=torch.float64, device="cuda")
        for k in range(len(c)):
            up += c[k] * torch.roll(u, k * s, -1) + d[k] * torch.roll(v[:, j - 1, 1], k * s, -1)
        u = up
    # each level adds 2 L products of relative rounding eps to sums of this size
    eps = 2.0 ** (-52 if dtype == torch.float64 else -23)
    assert (gx.double() - u).norm() <= 4 * len(c) * J * eps * u.norm()
    z = g.view(B, J, 2, n).clone()
    z[:, : J - 1, 0] = 0
    W.check(W.lib().wh_modwt_fwd_adj(_p(z), _p(gx), n, B, J, f, _code(dtype), None))
    W.check(W.lib().wh_modwt_fwd_details_adj(_p(g), _p(gd), n, B, J, f, _code(dtype), None))
    assert torch.equal(gx, gd)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,n,J,name", SHAPES)
def test_inverse_adjoint_and_threshold(dtype, B, n, J, name):
    f = D.filter_code(name)
    gy, c = _rand(dtype, B, n), _rand(dtype, B, 2 * n * J)
    lam = torch.linspace(0.9, 0.1, J, dtype=torch.float64, device="cuda")
    # the plain adjoint is the forward with level l scaled by 2^-l, S_j (j < J) zero
    full = torch.empty(B, 2 * n * J, dtype=dtype, device="cuda")
    for b in range(B):
        D.modwt_fwd(gy[b], J, f, out=full[b])
    v = full.view(B, J, 2, n)
    v *= torch.tensor([2.0 ** -l for l in range(1, J + 1)], dtype=dtype, device="cuda").view(J, 1, 1)
    v[:, : J - 1, 0] = 0
    gw = torch.full((B, 2 * n * J), 7.0, dtype=dtype, device="cuda")
    W.check(W.lib().wh_modwt_inv_adj(_p(gy), _p(gw), n, B, J, f, _code(dtype), None))
    assert torch.equal(gw, full)
    for hard, lo, hi in ((W.SOFT, 0, J - 1), (W.HARD, 0, J - 1), (W.SOFT, 1, max(1, J - 2))):
        thr = W.make_thresh(True, hard, lo, hi, 0.0, lam.data_ptr())
        want, wl = torch.empty_like(gw), torch.zeros(J, dtype=torch.float64, device="cuda")
        W.check(W.lib().wh_thresh_grad(_p(c), _p(gw), _p(want), _p(wl), n, B, J, W.MODWT, f,
                                       _code(dtype), C.byref(thr), None))
        got, gl = torch.full_like(gw, 7.0), torch.full_like(wl, 7.0)
        W.check(W.lib().wh_modwt_thresh_inv_adj(_p(gy), _p(c), _p(got), 0, _p(gl), n, B, J, f,
                                                _code(dtype), C.byref(thr), None))
        assert torch.equal(got, want)
        # sums of B n terms in 64 bits: rounding of the order, on their own size
        bound = B * n * 2.0 ** -52 * gw.double().abs().sum()
        assert torch.all((gl - wl).abs() <= bound)
        only = torch.full_like(wl, 7.0)
        W.check(W.lib().wh_modwt_thresh_inv_adj(_p(gy), _p(c), None, 1, _p(only), n, B, J, f,
                                                _code(dtype), C.byref(thr), None))
        assert torch.equal(only, gl)
        part = torch.full_like(gw, 7.0)
        W.check(W.lib().wh_modwt_thresh_inv_adj(_p(gy), _p(c), _p(part), 1, None, n, B, J, f,
                                                _code(dtype), C.byref(thr), None))
        pv = part.view(B, J, 2, n)
        assert torch.all(pv[:, : J - 1, 0] == 7.0)
        assert torch.equal(pv[:, :, 1], want.view(B, J, 2, n)[:, :, 1])
        assert torch.equal(pv[:, J - 1, 0], want.view(B, J, 2, n)[:, J - 1, 0])


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,n,J,name", [(3, 1 << 10, 6, "LA8"), (300, 1 << 13, 8, "D4")])
def test_layer_equals_composite(dtype, B, n, J, name):
    f = D.filter_code(name)
    lam0 = torch.linspace(0.5, 0.1, J, dtype=torch.float64, device="cuda")
    gy = _rand(dtype, B, n)
    outs = []
    for fused in (False, True):
        x = _rand(dtype, B, n).requires_grad_(True)
        lam = lam0.clone().requires_grad_(True)
        y = (A.smooth_levels(x, lam, J, f) if fused else
             A.ThresholdInverseFn.apply(A.ModwtFn.apply(x, J, f), lam, n, J, f, W.SOFT, 0, J - 1))
        gx, gl = torch.autograd.grad(y, (x, lam), gy)
        outs.append((y.detach(), gx, gl))
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1], outs[1][1])
    assert torch.allclose(outs[0][2], outs[1][2], rtol=1e-11, atol=1e-11 * float(outs[0][2].abs().max()))
    x = _rand(dtype, B, n)
    lam = lam0.clone().requires_grad_(True)
    (gl,) = torch.autograd.grad(A.smooth_levels(x, lam, J, f), (lam,), gy)
    assert torch.equal(gl, outs[1][2])


@pytest.mark.parametrize("total", [1, 255, 2049, (1 << 20) + 7])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_mse_grad(dtype, total):
    y, ref = _rand(dtype, total), _rand(dtype, total + 1)[1:].clone()
    want = torch.mean((y.double() - ref.double()) ** 2)
    yv = y.clone().requires_grad_(True)
    torch.mean((yv - ref) ** 2).backward()
    out = torch.empty(1, dtype=torch.float64, device="cuda")
    W.check(W.lib().wh_mse_grad(_p(y), _p(ref), _p(y), total, _code(dtype), _p(out), None))
    eps = 2.0 ** (-52 if dtype == torch.float64 else -23)
    assert abs(out.item() - want.item()) <= 4 * eps * want.item()
    assert torch.allclose(y, yv.grad, rtol=2 * eps, atol=0)


def test_fit_paths_agree():
    """Equal shapes and types take the direct step; a float64 target of float32
    signals keeps torch's promotion."""
    x = _rand(torch.float32, 6, 1 << 10)
    clean = _rand(torch.float32, 7, 1 << 10)[1:].contiguous()
    lam0 = torch.full((5,), 0.3, dtype=torch.float64)
    lam, losses = A.fit_level_thresholds(x, clean, 5, "LA8", lam0=lam0, steps=5)
    lam2, losses2 = A.fit_level_thresholds(x, clean.double(), 5, "LA8", lam0=lam0, steps=5)
    assert len(losses) == len(losses2) == 6
    assert torch.allclose(lam, lam2, rtol=1e-5)
    assert max(abs(a - b) for a, b in zip(losses, losses2)) <= 1e-6 * losses2[0]
