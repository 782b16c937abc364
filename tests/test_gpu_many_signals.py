"""Launches over many short signals beside one long signal of as many samples:
the tiles' layout over the XCDs must not depend on where signals end.  Timed
(each side the best of several runs); 256 signals of eight tiles each once took
twice the long signal's time."""
import ctypes as C

import pytest
import torch

from wavecuda_amd import _lib as W

pytestmark = pytest.mark.gpu


def best_us(fn):
    out = float("inf")
    for _ in range(8):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(20):
            fn()
        b.record()
        b.synchronize()
        out = min(out, a.elapsed_time(b) * 50)
    return out


@pytest.mark.parametrize("call,J,filt,dtype", [("wh_modwt_inv_many", 8, W.HAAR, torch.float64),
                                               ("wh_modwt_fwd_adj", 7, W.D4, torch.float64)])
def test_many_as_one(call, J, filt, dtype):
    total = 1 << 21
    w = torch.randn(2 * total * J, dtype=dtype, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(1))
    x = torch.empty(total, dtype=dtype, device="cuda")
    p = [C.c_void_p(t.data_ptr()) for t in (w, x)]
    code = W.WH_F64 if dtype == torch.float64 else W.WH_F32
    last = [None, None] if call.endswith("many") else [None]
    us = {n: best_us(lambda: W.check(getattr(W.lib(), call)(*p, n, total // n, J, filt, code, *last)))
          for n in (total, 1 << 13)}
    print(call, us, flush=True)
    assert us[1 << 13] < 1.4 * us[total]
