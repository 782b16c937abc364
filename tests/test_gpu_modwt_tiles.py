"""The MODWT as tiles (modwt_tile.h) against the sliding windows: every
coefficient is computed with the same operations, so the two are equal bit
for bit, whatever the tile's threads and the depth of its groups -- signals
shorter than a tile and than the cascade's halo, one to four groups, one
signal and several, with per-level thresholds."""
import ctypes as C

import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import device as D

pytestmark = pytest.mark.gpu

SLIDING = (10, 1, 1, 512)
TILES = [(6, 1, 1, -512), (6, 1, 1, -256), (3, 1, 1, -256), (4, 1, 1, -512)]


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("filt,n,J", [
    ("Haar", 2, 1), ("Haar", 64, 6), ("Haar", 1 << 16, 16), ("D4", 16, 3), ("D4", 512, 5),
    ("D4", 1 << 14, 8), ("C6", 64, 4), ("C6", 1 << 12, 10), ("LA8", 8, 1), ("LA8", 1024, 6),
    ("LA8", 1024, 8), ("LA8", 1 << 13, 7), ("LA8", 1 << 16, 14)])
def test_tiles_equal_sliding(dtype, filt, n, J):
    f = D.filter_code(filt)
    x = torch.randn(n, dtype=dtype, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(n + J))
    thr = dict(hardness=W.SOFT, minlevel=0, maxlevel=J - 1,
               levels=torch.linspace(1.0, 0.1, J, dtype=torch.float64, device="cuda"))

    def both(knobs):
        for inverse in (False, True):
            D.modwt_set_plan(inverse, n, J, f, dtype, SLIDING if knobs is None else knobs)
        w = D.modwt_fwd(x, J, f)
        return w, D.modwt_inv(w, n, J, f), D.modwt_inv(w, n, J, f, thr)

    try:
        want = both(None)
        assert "tile" not in D.modwt_plan(True, n, J, f, dtype)
        for knobs in TILES:
            got = both(knobs)
            assert "tile" in D.modwt_plan(False, n, J, f, dtype)
            for a, b in zip(got, want):
                assert torch.equal(a, b), knobs
    finally:
        for inverse in (False, True):
            D.modwt_set_plan(inverse, n, J, f, dtype, None)


@pytest.mark.parametrize("n,count,J", [(256, 7, 5), (1 << 12, 5, 8), (1 << 16, 3, 10)])
def test_default_tiles_of_many_signals(n, count, J):
    """A many-signal launch within the tiles' range equals one call per signal."""
    assert "tile" in D.modwt_plan(True, n, J, W.LA8, count=count)
    x = torch.randn(count, n, dtype=torch.float64, device="cuda")
    w = torch.empty(count, 2 * n * J, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    W.check(W.lib().wh_modwt_fwd_many(_ptr(x), _ptr(w), n, count, J, W.LA8, W.WH_F64, None))
    W.check(W.lib().wh_modwt_inv_many(_ptr(w), _ptr(y), n, count, J, W.LA8, W.WH_F64, None, None))
    for b in range(count):
        assert torch.equal(w[b], D.modwt_fwd(x[b], J, W.LA8))
        assert torch.equal(y[b], D.modwt_inv(w[b], n, J, W.LA8))


WIDE = (8, 1, 1, -256)


@pytest.mark.parametrize("filt,n,J", [("Haar", 2048, 3), ("D4", 4096, 5), ("C6", 2048, 6),
                                      ("LA8", 2048, 8), ("LA8", 1 << 15, 7), ("Haar", 1 << 13, 8)])
def test_wide_tiles_equal_sliding(filt, n, J):
    """FP32 inverse as one wide tile: one tile per signal (the halo wraps) and
    many, with and without thresholds."""
    f, dtype = D.filter_code(filt), torch.float32
    w = torch.randn(2 * n * J, dtype=dtype, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(n + J))
    lam = torch.linspace(1.0, 0.1, J, dtype=torch.float64, device="cuda")
    thrs = [None] + [dict(hardness=h, minlevel=lo, maxlevel=J - 1, levels=lam)
                     for h, lo in ((W.SOFT, 0), (W.HARD, 1))]
    try:
        outs = []
        for knobs in (SLIDING, WIDE):
            D.modwt_set_plan(True, n, J, f, dtype, knobs)
            outs.append([D.modwt_inv(w, n, J, f, t) for t in thrs])
        plan = D.modwt_plan(True, n, J, f, dtype)
        assert "tile" in plan and f" g={J} " in plan
        for a, b in zip(*outs):
            assert torch.equal(a, b)
        with pytest.raises(W.WaveHipError):
            D.modwt_set_plan(True, n, J, f, torch.float64, WIDE)
    finally:
        for dt in (torch.float32, torch.float64):
            D.modwt_set_plan(True, n, J, f, dt, None)
