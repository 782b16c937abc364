"""Batches whose signals hold NaN or infinities, against the single-signal
path: the same thresholds (NaN deviations rank above every number, whatever
route the selection takes) and the same outputs, NaN where it has NaN.
Lengths whose details the selection holds in registers, brackets by a sample,
and reads in whole; a few bad samples, enough to crowd the selection's bins,
and so many that the threshold itself is a NaN."""
import numpy as np
import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import device as D
from wavecuda_amd.batch import BatchPlan

pytestmark = pytest.mark.gpu


def same(a, b):
    return bool(torch.all((a == b) | (a.isnan() & b.isnan())))


@pytest.mark.parametrize("hardness", [W.SOFT, W.HARD])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("bad", [float("nan"), -float("nan"), float("inf"), -float("inf")])
def test_matches_single(bad, dtype, hardness):
    lens, filters, ttypes, levels, share = [], [], [], [], []
    for k in (6, 9, 11, 13, 14, 15, 16, 17):
        for s, (f, tt, J) in enumerate([(W.HAAR, 0, 1), (W.LA8, 1, 2), (W.D4, 0, 3), (W.C6, 1, 5),
                                        (W.HAAR, 0, 5), (W.D4, 1, 1)]):
            if J > k - 3:
                continue
            for part in (0, 1 / 64, 1 / 10, 1 / 2):
                lens.append(1 << k)
                filters.append(f)
                ttypes.append(tt)
                levels.append(J)
                share.append(part)
    plan = BatchPlan(lens, filters, ttypes, levels, dtype=dtype, hardness=hardness)
    g = torch.Generator().manual_seed(17)
    x = torch.randn(plan.total, generator=g, dtype=torch.float64).to(dtype)
    o = plan.offsets
    for i, n in enumerate(lens):
        at = torch.randperm(n, generator=g)[:max(2, int(share[i] * n))]
        x[int(o[i]) + at] = bad
        if i % 3 == 0:  # beside one of the other sign
            x[int(o[i]) + int(at[0])] = -bad
    xg = x.cuda()
    y, t = plan.smooth(xg)
    wrong = []
    for i in range(len(lens)):
        yi, ti = D.smooth(xg[o[i]:o[i + 1]].clone(), levels[i], ttypes[i], filters[i], W.UNIV,
                          hardness=hardness)
        if not (ti == t[i].item() or (np.isnan(ti) and np.isnan(t[i].item()))):
            wrong.append((lens[i], filters[i], ttypes[i], levels[i], share[i], ti, t[i].item()))
        elif not same(yi, y[o[i]:o[i + 1]]):
            wrong.append((lens[i], filters[i], ttypes[i], levels[i], share[i], "output"))
    assert not wrong, f"{len(wrong)} of {len(lens)}: {wrong[:12]}"
