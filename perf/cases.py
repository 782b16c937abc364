"""The measured workloads of wavecuda_amd: its transforms, smoothers, the
batched pipeline and the differentiable layer, through the public Python
entry points, over the sizes its tests and benchmark use.

A case is a dict of plain values; `kind` says which entry points it runs:

  dwt     device.dwt_fwd then device.dwt_inv of one signal in HBM
  modwt   device.modwt_fwd then device.modwt_inv (with a hard threshold
          fused into the inverse's reads where `thresh` is set)
  smooth  device.smooth: forward, universal or cross-validated threshold,
          inverse, of one signal in HBM
  host    rsurface.GPUSmooth on a host vector, as the R package calls it
  batch   BatchPlan.smooth over many signals of mixed length, filter and
          transform
  layer   autograd.smooth_levels forward and backward over a batch of
          equal-length signals, gradients to the signals and the thresholds
  fit     autograd.fit_level_thresholds: a few Adam steps

Signals are Donoho-Johnstone doppler plus Gaussian noise, made on the GPU
from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from wavecuda_amd import autograd as A
from wavecuda_amd import device as D
from wavecuda_amd import rsurface as R
from wavecuda_amd.batch import BatchPlan

FILTERS = ("Haar", "D4", "C6", "LA8")
TAPS = {"Haar": 2, "D4": 4, "C6": 6, "LA8": 8}
DTYPES = {"f64": torch.float64, "f32": torch.float32}
SIZES = {"f64": 8, "f32": 4}
UNIV, CV = 1, 2
HARD, SOFT = 0, 1

# scaling filters (the wavelet filter is g_k = (-1)^k c_{L-1-k})
SCALING = {
    "Haar": (0.70710678118654752440, 0.70710678118654752440),
    "D4": (0.4829629131445341, 0.8365163037378079, 0.2241438680420134, -0.1294095225512604),
    "C6": (-7.273261951252645e-2, 3.378976624574818e-1, 8.525720202116004e-1,
           3.848648468648577e-1, -7.273261951252645e-2, -1.565572813579199e-2),
    "LA8": (-7.576571478950221e-2, -2.963552764600249e-2, 4.976186676327750e-1,
            8.037387518051321e-1, 2.978577956053061e-1, -9.921954357663353e-2,
            -1.260396726203130e-2, 3.222310060405147e-2),
}


def max_levels(n: int, filt: str) -> int:
    return int(math.log2(n)) - math.ceil(math.log2(TAPS[filt])) + 1


def listed():
    return [
        # the smallest call: one short signal, bound by launches and the host
        {"name": "dwt_small", "kind": "dwt", "n": 1 << 10, "levels": 0, "filter": "D4",
         "dtype": "f64"},
        # the largest single DWT of the benchmark, full depth
        {"name": "dwt_large", "kind": "dwt", "n": 1 << 24, "levels": 0, "filter": "LA8",
         "dtype": "f64"},
        # the benchmark's headline transform pair
        {"name": "modwt_large", "kind": "modwt", "n": 1 << 24, "levels": 10, "filter": "LA8",
         "dtype": "f64", "thresh": 0.0},
        # an ordinary single-precision analysis with a given threshold
        {"name": "modwt_mid_f32", "kind": "modwt", "n": 1 << 20, "levels": 8, "filter": "D4",
         "dtype": "f32", "thresh": 0.25},
        # universal smoothing of one signal, the benchmark's size
        {"name": "smooth_univ", "kind": "smooth", "n": 1 << 18, "levels": 10, "filter": "LA8",
         "dtype": "f64", "ttype": 1, "rule": UNIV, "hardness": SOFT},
        # cross-validated smoothing of one signal, the benchmark's size
        {"name": "smooth_cv", "kind": "smooth", "n": 1 << 18, "levels": 10, "filter": "LA8",
         "dtype": "f64", "ttype": 1, "rule": CV, "hardness": SOFT},
        # what an R user calls: a host vector in, the smoothed vector back
        {"name": "host_smooth", "kind": "host", "n": 1 << 16, "levels": 8, "filter": "D4",
         "ttype": 0, "rule": CV, "hardness": SOFT},
        # the benchmark's batch: 8192 mixed signals of 2^8..2^16 samples
        {"name": "batch_f64", "kind": "batch", "count": 8192, "kmin": 8, "kmax": 16,
         "table": 2024, "dtype": "f64"},
        # a smaller single-precision batch with an odd number of signals
        {"name": "batch_f32", "kind": "batch", "count": 3001, "kmin": 8, "kmax": 16,
         "table": 7, "dtype": "f32"},
        # thresholds fitted to 512 signals, the benchmark's fit (a few steps)
        {"name": "fit", "kind": "fit", "rows": 512, "n": 1 << 14, "levels": 8, "filter": "LA8",
         "dtype": "f32", "steps": 4},
        # the smoother as a layer of a model: forward, and gradients to the
        # signals and the thresholds
        {"name": "layer_modwt", "kind": "layer", "rows": 257, "n": 1 << 13, "levels": 8,
         "filter": "LA8", "dtype": "f32", "ttype": 1},
        {"name": "layer_dwt", "kind": "layer", "rows": 63, "n": 1 << 12, "levels": 6,
         "filter": "LA8", "dtype": "f32", "ttype": 0},
    ]


def draw(rng):
    kind = rng.choice(("dwt", "dwt", "modwt", "modwt", "smooth", "smooth", "host", "batch",
                       "layer", "layer", "fit"))
    filt = rng.choice(FILTERS)
    dtype = rng.choice(("f64", "f32"))
    if kind == "dwt":
        n = 1 << rng.randint(10, 24)
        return {"kind": kind, "n": n, "levels": rng.choice((0, rng.randint(1, max_levels(n, filt)))),
                "filter": filt, "dtype": dtype}
    if kind == "modwt":
        n = 1 << rng.randint(10, 23)
        return {"kind": kind, "n": n, "levels": rng.randint(1, min(10, max_levels(n, filt))),
                "filter": filt, "dtype": dtype, "thresh": rng.choice((0.0, 0.25))}
    if kind == "smooth":
        n = 1 << rng.randint(12, 20)
        return {"kind": kind, "n": n, "levels": rng.randint(3, min(10, max_levels(n, filt))),
                "filter": filt, "dtype": dtype, "ttype": rng.randint(0, 1),
                "rule": rng.choice((UNIV, CV)), "hardness": SOFT}
    if kind == "host":
        n = 1 << rng.randint(10, 18)
        return {"kind": kind, "n": n, "levels": rng.randint(3, min(10, max_levels(n, filt))),
                "filter": filt, "ttype": rng.randint(0, 1), "rule": rng.choice((UNIV, CV)),
                "hardness": SOFT}
    if kind == "batch":
        return {"kind": kind, "count": int(math.exp(rng.uniform(math.log(100), math.log(8192)))),
                "kmin": 8, "kmax": rng.randint(12, 16), "table": rng.randint(1, 1 << 20),
                "dtype": dtype}
    n = 1 << rng.randint(10, 14)
    rows = int(math.exp(rng.uniform(math.log(4), math.log(512))))
    levels = rng.randint(3, min(8, max_levels(n, filt)))
    if kind == "fit":
        return {"kind": kind, "rows": rows, "n": n, "levels": levels, "filter": filt,
                "dtype": dtype, "steps": rng.randint(2, 4)}
    ttype = rng.randint(0, 1)
    if ttype == 0:
        rows = min(rows, 128)
    return {"kind": kind, "rows": rows, "n": n, "levels": levels, "filter": filt, "dtype": dtype,
            "ttype": ttype}


# ------------------------------------------------------------------- inputs

def device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def generator(seed: int):
    return torch.Generator(device=device()).manual_seed(int(seed))


def clean_sd(n: int) -> float:
    t = np.arange(1, n + 1) / n
    return float(np.std(np.sqrt(t * (1 - t)) * np.sin(2 * np.pi * 1.05 / (t + 0.05)), ddof=1))


def doppler(t):
    return torch.sqrt(t * (1.0 - t)) * torch.sin(2.0 * math.pi * 1.05 / (t + 0.05))


def signals(rows: int, n: int, seed: int):
    """(noisy, clean) float64 of shape (rows, n), SNR uniform in [1, 10]."""
    g = generator(seed)
    clean = doppler(torch.arange(1, n + 1, dtype=torch.float64, device=device()) / n)
    snr = 1.0 + 9.0 * torch.rand(rows, 1, dtype=torch.float64, device=device(), generator=g)
    noise = torch.randn(rows, n, dtype=torch.float64, device=device(), generator=g)
    return clean + noise * (clean_sd(min(n, 1 << 16)) / snr), clean.expand(rows, n)


def batch_table(case):
    """Lengths, filters, transforms and levels of a batch's signals: k
    uniform in kmin..kmax (n = 2^k), filter and transform uniform, the DWT at
    full depth, the MODWT at min(8, k - 2) levels."""
    rng = np.random.default_rng(case["table"])
    k = rng.integers(case["kmin"], case["kmax"] + 1, size=case["count"])
    filters = rng.integers(1, 5, size=case["count"]).astype(np.int32)
    ttypes = rng.integers(0, 2, size=case["count"]).astype(np.int32)
    levels = np.where(ttypes == 1, np.minimum(8, k - 2), 0).astype(np.int32)
    return (1 << k).astype(np.int32), filters, ttypes, levels


def batch_signals(lens, seed: int):
    """The packed noisy signals, float64."""
    g = generator(seed)
    total, count = int(lens.sum()), len(lens)
    dev = device()
    n = torch.as_tensor(lens.astype(np.int64), device=dev)
    off = torch.cumsum(n, 0) - n
    sd = torch.as_tensor(np.array([clean_sd(int(v)) for v in np.unique(lens)]), device=dev)
    which = torch.as_tensor(np.searchsorted(np.unique(lens), lens), device=dev)
    snr = 1.0 + 9.0 * torch.rand(count, dtype=torch.float64, device=dev, generator=g)
    sig = torch.repeat_interleave(torch.arange(count, device=dev), n)
    t = (torch.arange(total, device=dev) - off[sig] + 1).double() / n[sig]
    return doppler(t) + torch.randn(total, dtype=torch.float64, device=dev,
                                    generator=g) * (sd[which] / snr)[sig]


def inputs(case, seed: int):
    kind = case["kind"]
    if kind == "batch":
        return batch_signals(batch_table(case)[0], seed).to(DTYPES[case["dtype"]])
    if kind in ("layer", "fit"):
        x, clean = signals(case["rows"], case["n"], seed)
        dt = DTYPES[case["dtype"]]
        lam = torch.linspace(0.3, 0.05, case["levels"], dtype=torch.float64, device=device())
        return x.to(dt), clean.to(dt).contiguous(), lam
    x = signals(1, case["n"], seed)[0][0]
    if kind == "host":
        return x.cpu().numpy()
    return x.to(DTYPES[case["dtype"]]).contiguous()


def prepare(case, seed):
    state = {"case": dict(case), "x": inputs(case, seed)}
    if case["kind"] == "batch":
        state["plan"] = BatchPlan(*batch_table(case), dtype=DTYPES[case["dtype"]])
    elif case["kind"] == "layer":
        x, clean, lam = state["x"]
        state["x"] = (x.requires_grad_(True), clean, lam.requires_grad_(True))
    return state


# --------------------------------------------------------------------- pass

def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "dwt":
        y = D.dwt_fwd(x, case["levels"], case["filter"])
        return [y, D.dwt_inv(y, case["levels"], case["filter"])]
    if kind == "modwt":
        w = D.modwt_fwd(x, case["levels"], case["filter"])
        thr = None
        if case["thresh"] > 0:
            thr = dict(value=case["thresh"], hardness=HARD, minlevel=0,
                       maxlevel=case["levels"] - 1)
        return [w, D.modwt_inv(w, case["n"], case["levels"], case["filter"], thr)]
    if kind == "smooth":
        y, t = D.smooth(x, case["levels"], case["ttype"], case["filter"], case["rule"],
                        hardness=case["hardness"])
        return [y, t]
    if kind == "host":
        return R.GPUSmooth(x, case["levels"], "MODWT" if case["ttype"] else "DWT",
                           case["filter"], "cv" if case["rule"] == CV else "univ",
                           hard_soft="soft" if case["hardness"] == SOFT else "hard")
    if kind == "batch":
        y, t = state["plan"].smooth(x)
        return [y, t]
    xs, clean, lam = x
    if kind == "layer":
        y = A.smooth_levels(xs, lam, case["levels"], case["filter"], case["ttype"])
        loss = torch.mean((y - clean) ** 2)
        gx, glam = torch.autograd.grad(loss, (xs, lam))
        return [y.detach(), loss.detach(), gx, glam]
    lam, losses = A.fit_level_thresholds(xs, clean, case["levels"], case["filter"], lam0=lam,
                                         steps=case["steps"])
    return [lam, losses]


# --------------------------------------------------------------------- work

def transform_flops(n: float, levels: int, filt: str, modwt: bool) -> float:
    """Multiply-adds of one direction, two operations each."""
    outs = 2.0 * n * levels if modwt else 2.0 * n * (1.0 - 0.5 ** levels)
    return 2.0 * TAPS[filt] * outs


def work(case):
    kind = case["kind"]
    if kind == "batch":
        lens, filters, ttypes, levels = batch_table(case)
        flops = 0.0
        for n, f, tt, j in zip(lens.tolist(), filters.tolist(), ttypes.tolist(), levels.tolist()):
            filt = FILTERS[f - 1]
            flops += 2 * transform_flops(n, j or max_levels(n, filt), filt, tt == 1)
        return {"bytes": 2.0 * int(lens.sum()) * SIZES[case["dtype"]] + 8.0 * len(lens),
                "flops": flops}
    n, filt = case["n"], case["filter"]
    J = case["levels"] or max_levels(n, filt)
    esz = SIZES[case.get("dtype", "f64")]
    if kind == "dwt":  # x -> y, y -> x
        return {"bytes": 4.0 * n * esz, "flops": 2 * transform_flops(n, J, filt, False)}
    if kind == "modwt":  # x -> S_j, D_j of every level; D_j and S_J -> x
        return {"bytes": float(n) * esz * ((1 + 2 * J) + (J + 2)),
                "flops": 2 * transform_flops(n, J, filt, True)}
    if kind in ("smooth", "host"):
        modwt = case["ttype"] == 1
        one = transform_flops(n, J, filt, modwt)
        # cross validation: both halves forward, and an inverse per
        # candidate (at least ten at the default tolerance)
        return {"bytes": 2.0 * n * esz, "flops": 2 * one + (11 * one if case["rule"] == CV else 0)}
    rows = case["rows"]
    one = transform_flops(float(rows) * n, J, filt, case.get("ttype", 1) == 1)
    if kind == "layer":  # x, clean -> y, gx
        return {"bytes": 4.0 * rows * n * esz, "flops": 4 * one}
    # x, clean read; every step reads the coefficients for y and for the
    # gradient, and the last loss reads them again
    return {"bytes": float(rows) * n * esz * (2 + (J + 1) * (2 * case["steps"] + 1)),
            "flops": one * (2 + 2 * case["steps"])}


# ---------------------------------------------- the same in plain torch, 64 bits

def taps(filt: str):
    c = SCALING[filt]
    return c, [(-1) ** k * c[len(c) - 1 - k] for k in range(len(c))]


def modwt_ref(x, J, filt):
    c, g = taps(filt)
    S, D_, s = [], [], x
    for j in range(1, J + 1):
        h = 1 << (j - 1)
        r = [torch.roll(s, -k * h, -1) for k in range(len(c))]
        S.append(sum(a * v for a, v in zip(c, r)))
        D_.append(sum(a * v for a, v in zip(g, r)))
        s = S[-1]
    return S, D_


def imodwt_ref(s, details, filt):
    c, g = taps(filt)
    for j in range(len(details), 0, -1):
        h, d = 1 << (j - 1), details[j - 1]
        s = 0.5 * sum(c[k] * torch.roll(s, k * h, -1) + g[k] * torch.roll(d, k * h, -1)
                      for k in range(len(c)))
    return s


def dwt_ref(x, J, filt):
    c, g = taps(filt)
    D_, s = [], x
    for _ in range(J):
        r = [torch.roll(s, -k, -1)[..., ::2] for k in range(len(c))]
        D_.append(sum(a * v for a, v in zip(g, r)))
        s = sum(a * v for a, v in zip(c, r))
    return s, D_


def idwt_ref(s, details, filt):
    c, g = taps(filt)
    for d in reversed(details):
        out = []
        for par in (0, 1):
            out.append(sum(c[2 * q + par] * torch.roll(s, q, -1)
                           + g[2 * q + par] * torch.roll(d, q, -1) for q in range(len(c) // 2)))
        s = torch.stack(out, -1).flatten(-2)
    return s


def interleave(s, details, n):
    y = torch.empty(n, dtype=s.dtype, device=s.device)
    for j, d in enumerate(details, 1):
        y[(1 << (j - 1))::(1 << j)] = d
    y[::(1 << len(details))] = s
    return y


def forward_ref(x, J, filt, ttype):
    """(coarsest scaling coefficients, details by level)."""
    if ttype == 0:
        return dwt_ref(x, J, filt)
    S, D_ = modwt_ref(x, J, filt)
    return S[-1], D_


def inverse_ref(s, details, filt, ttype):
    return idwt_ref(s, details, filt) if ttype == 0 else imodwt_ref(s, details, filt)


def cut(c, t, hardness):
    if hardness == HARD:
        return torch.where(c.abs() < t, torch.zeros_like(c), c)
    return torch.sign(c) * torch.relu(c.abs() - t)


def median_ref(v):
    v = torch.sort(v, -1).values
    m = v.shape[-1]
    return 0.5 * (v[..., (m - 1) // 2] + v[..., m // 2])


def mad_ref(v):
    return 1.4826 * median_ref((v - median_ref(v).unsqueeze(-1)).abs())


def cv_threshold_ref(x, s, details, case):
    n, J, filt, ttype = case["n"], case["levels"], case["filter"], case["ttype"]
    if ttype == 0:
        t3 = mad_ref(torch.cat([interleave(s, details, n)[1:]])) * math.sqrt(2 * math.log(n - 1))
    else:
        t3 = mad_ref(torch.cat(details)) * math.sqrt(2 * math.log(n))
    t3 = float(t3)
    half = [forward_ref(x[p::2].contiguous(), J - 1, filt, ttype) for p in (0, 1)]

    def err(t):
        ye, yo = (inverse_ref(hs, [cut(d, t, case["hardness"]) for d in hd], filt, ttype)
                  for hs, hd in half)
        ie = 0.5 * (yo + torch.cat([yo[:1], yo[:-1]]))
        io = 0.5 * (ye + torch.cat([ye[1:], ye[-1:]]))
        return float(((ie - x[::2]) ** 2 + (io - x[1::2]) ** 2).sum())

    r = 0.61803399
    t0, t2 = 0.0, t3 / 2
    t1 = t2 - (1 - r) * t2
    m1, m2 = err(t1), err(t2)
    it = 0
    while abs(t3 - t0) > 0.01 * (t1 + t2) and it <= 50:
        if m2 < m1:
            t0, t1, t2 = t1, t2, r * t2 + (1 - r) * t3
            m1, m2 = m2, err(t2)
        else:
            t3, t2, t1 = t2, t1, r * t1 + (1 - r) * t0
            m2, m1 = m1, err(t1)
        it += 1
    return (t1 if m1 < m2 else t2) / math.sqrt(1 - math.log(2) / math.log(n))


def exact(case, seed):
    kind, x = case["kind"], inputs(case, seed)
    if kind == "batch":
        return exact_batch(case, x.double())
    filt = case["filter"]
    if kind in ("layer", "fit"):
        return exact_layer(case, *(v.double() for v in x))
    x = torch.as_tensor(x, device=device()).double()
    J = case["levels"] or max_levels(case["n"], filt)
    if kind == "dwt":
        s, d = dwt_ref(x, J, filt)
        return [interleave(s, d, case["n"]), idwt_ref(s, d, filt)]
    if kind == "modwt":
        S, d = modwt_ref(x, J, filt)
        w = torch.cat([v for pair in zip(S, d) for v in pair])
        if case["thresh"] > 0:
            d = [cut(v, case["thresh"], HARD) for v in d]
        return [w, imodwt_ref(S[-1], d, filt)]
    s, d = forward_ref(x, J, filt, case["ttype"])
    if case["rule"] == UNIV:
        t = float(mad_ref(d[0])) * math.sqrt(2 * math.log(case["n"]))
    else:
        t = cv_threshold_ref(x, s, d, case)
    y = inverse_ref(s, [cut(v, t, case["hardness"]) for v in d], filt, case["ttype"])
    return y.cpu().numpy() if kind == "host" else [y, t]


def exact_batch(case, x):
    lens, filters, ttypes, levels = batch_table(case)
    off = np.cumsum(lens.astype(np.int64)) - lens
    y, t = torch.empty_like(x), torch.empty(len(lens), dtype=torch.float64, device=x.device)
    for key in sorted(set(zip(lens.tolist(), filters.tolist(), ttypes.tolist()))):
        n, f, tt = key
        filt = FILTERS[f - 1]
        sel = np.nonzero((lens == n) & (filters == f) & (ttypes == tt))[0]
        J = int(levels[sel[0]]) or max_levels(n, filt)
        at = torch.as_tensor(off[sel], device=x.device).unsqueeze(1) + torch.arange(n, device=x.device)
        s, d = forward_ref(x[at], J, filt, tt)
        lam = mad_ref(d[0]) * math.sqrt(2 * math.log(n))
        y[at] = inverse_ref(s, [cut(v, lam.unsqueeze(-1), SOFT) for v in d], filt, tt)
        t[torch.as_tensor(sel, device=x.device)] = lam
    return [y, t]


def exact_layer(case, x, clean, lam):
    J, filt, tt = case["levels"], case["filter"], case.get("ttype", 1)

    def smooth(s, d, lv):
        return inverse_ref(s, [cut(d[j], lv[j], SOFT) for j in range(J)], filt, tt)

    if case["kind"] == "layer":
        x, lam = x.requires_grad_(True), lam.requires_grad_(True)
        y = smooth(*forward_ref(x, J, filt, tt), lam)
        loss = torch.mean((y - clean) ** 2)
        gx, glam = torch.autograd.grad(loss, (x, lam))
        return [y.detach(), loss.detach(), gx, glam]
    s, d = forward_ref(x, J, filt, tt)
    lam = lam.requires_grad_(True)
    opt = torch.optim.Adam([lam], lr=1e-2)
    losses = []
    for _ in range(case["steps"]):
        opt.zero_grad()
        loss = torch.mean((smooth(s, d, lam) - clean) ** 2)
        loss.backward()
        opt.step()
        losses.append(float(loss))
    with torch.no_grad():
        losses.append(float(torch.mean((smooth(s, d, lam) - clean) ** 2)))
    return [lam.detach(), losses]
