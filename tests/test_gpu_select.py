"""Exact median and MAD (select.hip) at the edges of its paths -- one
workgroup (the sample is every value; sampled) and the grid, with and without
the refining pass -- over distributions that crowd, tie, straddle scales or
hide from the sample; the result must equal sorting, bit for bit."""
import numpy as np
import pytest
import torch

import oracle_bind as O
from wavecuda_amd import device as D

pytestmark = pytest.mark.gpu

ONE, SAMPLE = 8192, 512


def sample_positions(count):
    """The positions the selection samples."""
    m = SAMPLE
    out = []
    for i in range(m):
        lo, hi = i * count // m, (i + 1) * count // m
        h = ((i + 1) * 0x9E3779B97F4A7C15) & (2**64 - 1)
        h ^= h >> 29
        h = (h * 0xBF58476D1CE4E5B9) & (2**64 - 1)
        out.append(lo + (((h >> 32) * (hi - lo)) >> 32))
    return np.array(out)


def make(kind, n):
    rng = np.random.Generator(np.random.PCG64(n))
    x = rng.standard_normal(n)
    if kind == "ties":
        x = np.round(x * 4) / 4
    elif kind == "constant":
        x = np.full(n, -0.75)
    elif kind == "two_scales":  # half rounding noise, half signal
        x = np.where(rng.random(n) < 0.5, x * 1e-17, x)
    elif kind == "crowded":
        x = 1.0 + rng.integers(0, 1 << 20, n) * 2.0 ** -40
    elif kind == "ramp":
        x = np.arange(n, dtype=np.float64)
    elif kind == "infinite":
        x = np.where(rng.random(n) < 0.3, np.inf * np.sign(x), x)
    elif kind == "hidden" and n > SAMPLE:  # the sample sees the tail only
        x[sample_positions(n)] = 1e6
    return x


def check(x, dtype):
    g = torch.tensor(x, dtype=dtype, device="cuda")
    med, mad = D.median(g).item(), D.mad(g).item()
    s = np.sort(g.cpu().numpy())
    n = len(s)
    m = 0.5 * (float(s[(n - 1) // 2]) + float(s[n // 2]))
    with np.errstate(invalid="ignore"):
        d = np.sort(np.abs(g.cpu().numpy() - s.dtype.type(m)))
    assert med == m
    want = 1.4826 * (0.5 * (float(d[(n - 1) // 2]) + float(d[n // 2])))
    assert np.array_equal(mad, want, equal_nan=True)  # inf - inf where the median is infinite


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 2, 511, 512, 513, 5000, ONE - 1, ONE, ONE + 1, 300007])
@pytest.mark.parametrize("kind", ["noise", "ties", "constant", "two_scales", "crowded", "ramp",
                                  "infinite", "hidden"])
def test_equals_sorting(kind, n, dtype):
    check(make(kind, n), dtype)


@pytest.mark.parametrize("kind", ["noise", "two_scales", "hidden"])
def test_refining_pass(kind):
    check(make(kind, (1 << 24) + 3), torch.float64)


@pytest.mark.parametrize("lo,hi", [(0, 0), (0, 5), (2, 4), (9, 12), (15, 17)])
@pytest.mark.parametrize("n", [1 << 16, 1 << 18])
def test_dwt_level_ranges(n, lo, hi):
    """Levels picked out of the interleaved layout, from one value up."""
    J = O.levels(n, 0, 1)
    if hi >= J:
        pytest.skip("level range beyond this length's depth")
    y = np.random.Generator(np.random.PCG64(n)).standard_normal(n)
    got = D.univ_thresh(torch.tensor(y, device="cuda"), n, J, 0, "Haar", lo, hi).item()
    assert got == O.univ_thresh(y, n, J, 0, lo, hi)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [ONE, 1 << 17])
@pytest.mark.parametrize("which", [0, 1])
def test_one_middle_rank_is_an_edge(which, n, dtype):
    """A sampled value at one middle rank and a thousand values, the other
    middle rank among them, to the next sampled one: more than are ranked by
    counting."""
    k = n // 2 - 1 + which
    sampled = np.concatenate([np.linspace(10, k - 1000, 255), [k],
                              np.linspace(k + 1000, n - 10, 256)]).astype(np.int64)
    x = np.empty(n)
    pos = sample_positions(n)
    x[pos] = sampled
    rest = np.setdiff1d(np.arange(n), pos)
    x[rest] = np.random.Generator(np.random.PCG64(which)).permutation(
        np.setdiff1d(np.arange(n), sampled))
    check(x, dtype)
