"""wh_dwt_fwd_many / wh_dwt_inv_many: every signal of a launch equals the
single-signal call bit for bit (the tile size follows the whole launch's
values, so several are covered: n count from 2^11 to 2^21), out of place and
in place, with and without a threshold; rows beyond one launch's limit."""
import ctypes as C

import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import autograd as A
from wavecuda_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,count,J,filt", [
    (8, 3, 0, W.HAAR), (2048, 1, 5, W.LA8), (2048, 65, 0, W.C6), (4096, 3, 6, W.LA8),
    (4096, 17, 1, W.D4), (1 << 14, 5, 0, W.LA8), (1 << 16, 31, 0, W.D4), (1 << 18, 5, 3, W.C6)])
def test_many_equals_single(dtype, n, count, J, filt):
    g = torch.Generator(device="cuda").manual_seed(n + count)
    x = torch.randn(count, n, dtype=dtype, device="cuda", generator=g)
    code, esz = (W.WH_F64, 16) if dtype == torch.float64 else (W.WH_F32, 8)
    thr = W.make_thresh(True, W.SOFT, 0, 0, 0.5)
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    y, z, xr, inp = (torch.empty_like(x) for _ in range(4))
    W.check(W.lib().wh_dwt_fwd_many(p(x), p(y), n, count, J, filt, code, None))
    W.check(W.lib().wh_dwt_inv_many(p(y), p(xr), n, count, J, filt, code, None, None))
    W.check(W.lib().wh_dwt_inv_many(p(y), p(z), n, count, J, filt, code, C.byref(thr), None))
    inp.copy_(x)
    W.check(W.lib().wh_dwt_fwd_many(p(inp), p(inp), n, count, J, filt, code, None))
    assert torch.equal(inp, y)
    W.check(W.lib().wh_dwt_inv_many(p(inp), p(inp), n, count, J, filt, code, None, None))
    assert torch.equal(inp, xr)
    for b in range(count):
        yb = D.dwt_fwd(x[b], J, filt)
        assert torch.equal(y[b], yb), f"signal {b}"
        assert torch.equal(xr[b], D.dwt_inv(yb, J, filt)), f"signal {b}"
        assert torch.equal(z[b], D.dwt_inv(yb, J, filt, dict(value=0.5, hardness=W.SOFT))), b
    assert W.lib().wh_dwt_fwd_many(p(x), p(y), n, 65536, J, filt, code, None) == W.WH_ERR_ARG


def test_more_rows_than_one_launch():
    x = torch.randn(70001, 4, dtype=torch.float32, device="cuda")
    y = A.dwt(x, 0, W.HAAR)
    for b in (0, 65534, 65535, 70000):
        assert torch.equal(y[b], D.dwt_fwd(x[b], 0, W.HAAR))
    assert torch.equal(A.idwt(y, 0, W.HAAR)[65535], D.dwt_inv(y[65535], 0, W.HAAR))
    assert A.dwt(x[:0], 0, W.HAAR).shape == (0, 4)
