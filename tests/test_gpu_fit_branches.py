"""fit_level_thresholds beside its direct step: targets that broadcast, promote or
ask for gradients transform the (unchanging) signals once, too, and fit the same
thresholds; thresholds of another shape and a fit without gradients are refused,
whatever the target is."""
import pytest
import torch

from wavecuda_amd import _lib as W
from wavecuda_amd import autograd as A
from wavecuda_amd.autograd import fit_level_thresholds

pytestmark = pytest.mark.gpu
N, J, STEPS = 1 << 11, 6, 4


class Counting:
    """The library with the calls of every name counted."""

    def __init__(self, lib):
        self.lib, self.calls = lib, {}

    def __getattr__(self, name):
        self.calls[name] = self.calls.get(name, 0) + 1
        return getattr(self.lib, name)


def signals(dtype, *shape, seed=1):
    return torch.randn(*shape, dtype=dtype, device="cuda",
                       generator=torch.Generator(device="cuda").manual_seed(seed))


def lam0():
    return torch.full((J,), 0.4, dtype=torch.float64)


@pytest.mark.parametrize("branch", ["same", "broadcast", "promoted", "requires_grad"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_one_transform(branch, dtype, monkeypatch):
    x = signals(dtype, 5, N)
    clean = signals(dtype, 1, N, seed=2).expand(5, N)
    ref, losses0 = fit_level_thresholds(x, clean.contiguous(), J, "LA8", lam0=lam0(), steps=STEPS)
    other = torch.float32 if dtype == torch.float64 else torch.float64
    target = {"same": clean, "broadcast": clean[:1], "promoted": clean.to(other),
              "requires_grad": clean.contiguous().requires_grad_(True)}[branch]
    counting = Counting(W.lib())
    monkeypatch.setattr(A.W, "lib", lambda: counting)
    lam, losses = fit_level_thresholds(x, target, J, "LA8", lam0=lam0(), steps=STEPS)
    forwards = sum(v for k, v in counting.calls.items() if k.startswith("wh_modwt_fwd"))
    assert forwards == 1
    # the losses' rounding is x's type's; Adam's first steps follow the gradients' signs
    tol = 1e-4 if torch.float32 in (dtype, target.dtype) else 1e-9
    assert torch.allclose(lam, ref, rtol=tol)
    assert len(losses) == STEPS + 1
    assert max(abs(a - b) for a, b in zip(losses, losses0)) <= tol * losses0[0]


@pytest.mark.parametrize("branch", ["same", "broadcast"])
def test_refused(branch):
    x = signals(torch.float64, 3, N)
    clean = signals(torch.float64, 3, N, seed=2)[: 1 if branch == "broadcast" else 3]
    with pytest.raises(RuntimeError):
        fit_level_thresholds(x, clean, J, "LA8", lam0=lam0().view(1, J), steps=STEPS)
    with torch.no_grad(), pytest.raises(RuntimeError):
        fit_level_thresholds(x, clean, J, "LA8", lam0=lam0(), steps=STEPS)


def test_thresholds_alone():
    """ThresholdInverseFn's gradient of the thresholds alone against both."""
    for dtype, eps in ((torch.float64, 2.0 ** -52), (torch.float32, 2.0 ** -23)):
        w, gy = signals(dtype, 3, 2 * N * J), signals(dtype, 3, N, seed=4)
        for lo, hi in ((0, J - 1), (1, 3)):
            lam = lam0().cuda().requires_grad_(True)
            wg = w.clone().requires_grad_(True)
            y = A.ThresholdInverseFn.apply(wg, lam, N, J, W.LA8, W.SOFT, lo, hi)
            gw, both = torch.autograd.grad(y, (wg, lam), gy)
            y = A.ThresholdInverseFn.apply(w, lam, N, J, W.LA8, W.SOFT, lo, hi)
            (alone,) = torch.autograd.grad(y, (lam,), gy)
            # sums in 64 bits of the same terms, in another order
            assert (alone - both).abs().max() <= 3 * N * 2.0 ** -52 * gw.double().abs().sum()
