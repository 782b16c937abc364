"""The batch's tiles against the single-signal path.

Every signal must equal wh_smooth's result bit for bit (the same terms in the
same order, the same exact order statistics), whatever the tile does at its
edges: signals shorter than, equal to and longer than a tile, residue
sequences on both sides of a tile's length, every depth and filter, batches
smoothed in place, and batches split because their workspace is too large.
"""
import numpy as np
import pytest
import torch

import oracle_bind as O
from wavecuda_amd import _lib as W
from wavecuda_amd import device as D
from wavecuda_amd.batch import BatchPlan

pytestmark = pytest.mark.gpu
DTYPES = (torch.float64, torch.float32)


def check(lens, filters, ttypes, levels, dtype, hardness=W.SOFT, in_place=False, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    plan = BatchPlan(lens, filters, ttypes, levels, dtype=dtype, hardness=hardness)
    x = torch.randn(plan.total, dtype=torch.float64, device="cuda", generator=g).to(dtype)
    src = x.clone()
    y, t = plan.smooth(x, y=x if in_place else None)
    if not in_place:
        assert torch.equal(x, src)
    tc = t.cpu().numpy()
    o = plan.offsets
    for i in range(len(lens)):
        yi, ti = D.smooth(src[o[i]:o[i + 1]].clone(), int(levels[i]), int(ttypes[i]),
                          int(filters[i]), W.UNIV, hardness=hardness)
        case = f"signal {i}: n={lens[i]} filter={filters[i]} J={levels[i]}"
        assert ti == tc[i], case
        assert torch.equal(yi, y[o[i]:o[i + 1]]), case


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("filt", [W.HAAR, W.D4, W.C6, W.LA8])
def test_every_length_and_depth(filt, dtype):
    lens, levels = [], []
    for k in range(1, 18):
        n = 1 << k
        if n < W.FILTER_LENGTHS[filt]:
            continue
        for J in range(1, min(8, O.levels(n, 0, filt)) + 1):
            lens.append(n)
            levels.append(J)
    count = len(lens)
    check(lens, [filt] * count, [W.MODWT] * count, levels, dtype, seed=filt)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("filt", [W.HAAR, W.D4, W.C6, W.LA8])
def test_dwt_every_length(filt, dtype):
    """Whole signals (up to 4096 samples, or up to four levels) and tiles."""
    lens, levels = [], []
    for k in range(1, 18):
        n = 1 << k
        if n < W.FILTER_LENGTHS[filt]:
            continue
        jmax = O.levels(n, 0, filt)
        for J in sorted({1, 4, 5, 6, 9, jmax} & set(range(1, jmax + 1))):
            lens.append(n)
            levels.append(J)
    count = len(lens)
    check(lens, [filt] * count, [W.DWT] * count, levels, dtype, seed=10 + filt)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hardness", [W.SOFT, W.HARD])
def test_in_place(hardness, dtype):
    rng = np.random.Generator(np.random.PCG64(4))
    lens = [1 << int(k) for k in rng.integers(8, 17, size=40)]
    filters = [1 + i % 4 for i in range(40)]
    ttypes = [(i // 4) % 2 for i in range(40)]
    levels = [4 + i % 3 if t else 0 for i, t in enumerate(ttypes)]
    check(lens, filters, ttypes, levels, dtype, hardness, in_place=True, seed=5)


@pytest.mark.parametrize("dtype", DTYPES)
def test_split_workspace(dtype):
    # each long signal needs more than half of the tiles' workspace
    k = 27 if dtype == torch.float64 else 28
    lens = [1 << k, 1 << 12, 1 << k, 1 << 9]
    check(lens, [W.LA8, W.D4, W.HAAR, W.C6], [W.MODWT, W.DWT, W.MODWT, W.MODWT], [6, 0, 3, 5],
          dtype, seed=9)
