"""Cross-validated smoothing on both sides of the lengths up to which a round has
three candidates (2^19 MODWT, 2^21 DWT), against the oracle's sequential search."""
import pytest
import torch

import oracle_bind as O
from wavecuda_amd import device as D
from wavecuda_amd.signals import noisy_doppler

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ttype,filt,J", [(1 << 19, 1, 1, 2), (1 << 20, 1, 1, 2),
                                            (1 << 21, 0, 2, 5), (1 << 22, 0, 2, 5)])
def test_line(n, ttype, filt, J):
    x, _ = noisy_doppler(n, 3.0, seed=J)
    want, t_want, _ = O.smooth(x, J, ttype, filt, 2, None, 1, 0, J - 1, 0.01)
    y, t = D.smooth(torch.tensor(x, device="cuda"), J, ttype, filt, 2, None, 1, 0, J - 1, 0.01)
    assert abs(t - t_want) <= 1e-12 * t_want
    assert O.relerr(y.cpu().numpy(), want) <= 1e-12
