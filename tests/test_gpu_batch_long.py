"""Batches of long signals: details on both sides of the sampled selection's
range for every thread count, first digits counted by the forward (DWT signals
without tiles beyond it), and the shape an untuned plan of such signals takes."""
import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import device as D
from wavecuda_amd.batch import BatchPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [128, 256, 512])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_matches_single(dtype, threads):
    lens = [1 << k for k in (17, 18, 19, 17, 18, 19, 20, 20, 20, 21)]
    ttypes = [1, 1, 1, 0, 0, 0, 0, 0, 0, 0]
    levels = [2, 1, 3, 3, 4, 2, 3, 1, 4, 2]
    filters = [W.LA8, W.HAAR, W.D4, W.C6, W.LA8, W.HAAR, W.D4, W.HAAR, W.LA8, W.C6]
    plan = BatchPlan(lens, filters, ttypes, levels, dtype=dtype)
    plan.set_shape(threads, len(lens))
    g = torch.Generator(device="cuda").manual_seed(threads)
    x = torch.randn(plan.total, dtype=torch.float64, device="cuda", generator=g).to(dtype)
    o = plan.offsets
    x[int(o[6]):int(o[6]) + 4096] = 0.25  # ties
    x[int(o[9]) + 5] = float("inf")
    y, t = plan.smooth(x)
    for i in range(len(lens)):
        yi, ti = D.smooth(x[o[i]:o[i + 1]].clone(), levels[i], ttypes[i], filters[i], W.UNIV)
        case = f"signal {i}: n={lens[i]} ttype={ttypes[i]} J={levels[i]}"
        assert ti == t[i].item(), case
        a, b = yi, y[o[i]:o[i + 1]]
        assert torch.all((a == b) | (a.isnan() & b.isnan())), case


@pytest.mark.parametrize("count,n,J,threads", [(1024, 1 << 16, 3, 512), (768, 1 << 17, 2, 512),
                                               (4096, 1 << 13, 3, 256), (1024, 1 << 16, 0, 256)])
def test_untuned_threads(count, n, J, threads):
    plan = BatchPlan([n] * count, [W.LA8] * count, [W.DWT] * count, [J] * count,
                     dtype=torch.float32)
    assert plan.info()["threads"] == threads
