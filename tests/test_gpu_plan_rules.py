"""Which launches run as tiles: not those whose deeper tiles would be mostly
padding, nor forwards that the sliding windows do in one group of two chunks;
and whichever form a launch takes, its values are the other form's, bit for
bit."""
import ctypes as C

import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import device as D

pytestmark = pytest.mark.gpu

RULES = [  # inverse, n, J, filter, dtype, count, tiles
    (False, 1 << 8, 7, "Haar", torch.float32, 1, False),
    (False, 1 << 10, 10, "Haar", torch.float64, 256, False),
    (False, 1 << 10, 8, "D4", torch.float64, 16, False),
    (False, 1 << 10, 6, "Haar", torch.float32, 4, True),
    (False, 1 << 10, 8, "LA8", torch.float64, 64, True),
    (False, 1 << 13, 12, "Haar", torch.float32, 64, False),
    (False, 1 << 18, 10, "LA8", torch.float64, 1, True),
    (True, 1 << 12, 12, "Haar", torch.float64, 256, False),
    (True, 1 << 13, 12, "D4", torch.float32, 256, False),
    (True, 1 << 8, 8, "Haar", torch.float32, 1024, False),
    (True, 1 << 8, 8, "Haar", torch.float32, 16, True),
    (True, 1 << 12, 12, "Haar", torch.float32, 64, True),
    (True, 1 << 13, 8, "D4", torch.float64, 256, True),
]


@pytest.mark.parametrize("inverse,n,J,filt,dtype,count,tiles", RULES)
def test_form(inverse, n, J, filt, dtype, count, tiles):
    plan = D.modwt_plan(inverse, n, J, filt, dtype, count=count)
    print(plan, flush=True)
    assert ("tile" in plan) == tiles


@pytest.mark.parametrize("inverse,n,J,filt,dtype,count,tiles", RULES)
def test_values(inverse, n, J, filt, dtype, count, tiles):
    """Against the same signals one by one as tiles, whatever the rule says."""
    f, code = D.filter_code(filt), W.WH_F64 if dtype == torch.float64 else W.WH_F32
    count = min(count, 256)
    g = torch.Generator(device="cuda").manual_seed(n + J)
    src = torch.randn(count, 2 * n * J if inverse else n, dtype=dtype, device="cuda", generator=g)
    out = torch.empty(count, n if inverse else 2 * n * J, dtype=dtype, device="cuda")
    call = W.lib().wh_modwt_inv_many if inverse else W.lib().wh_modwt_fwd_many
    args = [C.c_void_p(src.data_ptr()), C.c_void_p(out.data_ptr()), n, count, J, f, code]
    W.check(call(*args, *([None, None] if inverse else [None])))
    D.modwt_set_plan(inverse, n, J, f, dtype, (6, 1, 1, -512))
    try:
        for i in range(0, count, max(1, count // 4)):
            one = D.modwt_inv(src[i], n, J, f) if inverse else D.modwt_fwd(src[i], J, f)
            assert torch.equal(one, out[i]), i
    finally:
        D.modwt_set_plan(inverse, n, J, f, dtype, None)
    if not inverse:
        w = torch.empty_like(out)
        W.check(W.lib().wh_modwt_inv_adj(args[0], C.c_void_p(w.data_ptr()), n, count, J, f, code, None))
        v = out.view(count, J, 2, n)
        v *= torch.tensor([2.0 ** -l for l in range(1, J + 1)], dtype=dtype, device="cuda").view(J, 1, 1)
        v[:, : J - 1, 0] = 0
        assert torch.equal(w, out)


@pytest.mark.parametrize("details", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,J,count", [(1 << 12, 12, 64), (1 << 8, 8, 1024), (1 << 10, 10, 1024)])
def test_adjoint_by_level(n, J, count, dtype, details):
    """The forward's adjoint whose deepest levels run one by one, against
    launches of fewer signals, which run as tiles."""
    code = W.WH_F64 if dtype == torch.float64 else W.WH_F32
    g = torch.Generator(device="cuda").manual_seed(J)
    w = torch.randn(count, 2 * n * J, dtype=dtype, device="cuda", generator=g)
    out, one = (torch.empty(count, n, dtype=dtype, device="cuda") for _ in range(2))
    call = W.lib().wh_modwt_fwd_details_adj if details else W.lib().wh_modwt_fwd_adj
    W.check(call(C.c_void_p(w.data_ptr()), C.c_void_p(out.data_ptr()), n, count, J, W.HAAR, code, None))
    for i in range(0, count, 16):
        W.check(call(C.c_void_p(w[i].data_ptr()), C.c_void_p(one[i].data_ptr()), n, 16, J, W.HAAR,
                     code, None))
    assert torch.equal(out, one)
