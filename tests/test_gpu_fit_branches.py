"""fit_level_thresholds beside its direct step: thresholds of another shape and a
fit without gradients are refused, whatever the target is."""
import pytest
import torch

from wavecuda_amd.autograd import fit_level_thresholds

pytestmark = pytest.mark.gpu
N, J, STEPS = 1 << 11, 6, 4


def signals(dtype, *shape, seed=1):
    return torch.randn(*shape, dtype=dtype, device="cuda",
                       generator=torch.Generator(device="cuda").manual_seed(seed))


def lam0():
    return torch.full((J,), 0.4, dtype=torch.float64)


@pytest.mark.parametrize("branch", ["same", "broadcast"])
def test_refused(branch):
    x = signals(torch.float64, 3, N)
    clean = signals(torch.float64, 3, N, seed=2)[: 1 if branch == "broadcast" else 3]
    with pytest.raises(RuntimeError):
        fit_level_thresholds(x, clean, J, "LA8", lam0=lam0().view(1, J), steps=STEPS)
    with torch.no_grad(), pytest.raises(RuntimeError):
        fit_level_thresholds(x, clean, J, "LA8", lam0=lam0(), steps=STEPS)
