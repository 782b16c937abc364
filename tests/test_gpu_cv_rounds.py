"""Cross-validated smoothing with three candidates a round and with one, at
the lengths where the rule changes (2^18 / 2^19 MODWT, 2^20 / 2^21 DWT): the
chosen threshold and the smoothed signal against the oracle's sequential
search, and tolerances that stop it at once, on a certain and on an uncertain
step."""
import numpy as np
import pytest
import torch

import oracle_bind as O
from wavecuda_amd import device as D
from wavecuda_amd.signals import noisy_doppler

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ttype,filt,J,tol", [
    (1 << 18, 1, 2, 3, 0.01), (1 << 19, 1, 2, 3, 0.01), (1 << 20, 0, 4, 6, 0.01),
    (1 << 21, 0, 4, 6, 0.01), (1 << 12, 1, 4, 6, 1.0), (1 << 12, 1, 4, 6, 0.3),
    (1 << 12, 0, 1, 6, 0.12), (1 << 12, 0, 1, 6, 0.05), (1 << 12, 1, 3, 6, 1e-4)])
def test_rounds_follow_the_search(n, ttype, filt, J, tol):
    x, _ = noisy_doppler(n, 3.0, seed=J)
    want, t_want, _ = O.smooth(x, J, ttype, filt, 2, None, 1, 0, J - 1, tol)
    y, t = D.smooth(torch.tensor(x, device="cuda"), J, ttype, filt, 2, None, 1, 0, J - 1, tol)
    assert abs(t - t_want) <= 1e-12 * t_want
    assert O.relerr(y.cpu().numpy(), want) <= 1e-12


def test_constant_signal():
    """Every coefficient and the bracket are zero: the search stops at once."""
    x = torch.zeros(1 << 10, dtype=torch.float64, device="cuda")
    y, t = D.smooth(x, 5, 1, 4, 2, None, 1, 0, 4)
    assert t == 0.0 and torch.equal(y, x)
