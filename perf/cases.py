"""Timed cases of galario_amd: the calls that a fit of interferometric visibilities makes, through the
public entry points, over the sizes, types and directions in use.

``listed()`` names them, ``draw(rng)`` gives one more of the same ranges, ``prepare(case, seed)`` makes what a
program holds before the call (data sets on the GPU, plans, parameters; host arrays for the host-array
functions), ``run(state)`` is one call, ``work(case)`` the bytes and operations that the call cannot do
without, and ``exact(case, seed)`` its result in 64 bits from plain torch.

Fields of a case
  kind     chi2_host      galario_amd.<double|single>.chi2Profile on numpy arrays (galario's own interface)
           image_chi2     chi2Image on numpy arrays
           image_sample   sampleImage on numpy arrays
           chi2           Dataset.chi2_profile (the observation stays on the GPU between calls)
           sample         Dataset.sample_profile (visibilities out, in the caller's order)
           grad           Dataset.chi2_profile_grad (chi2, d/dprofile, d/d(inc, PA, dRA, dDec))
           autograd       chi2_profile_autograd and its backward (parameters and loss in the case's type)
           batch          BatchedChi2Profile call: many walkers' chi2 over several data sets
           batch_grad     BatchedChi2Profile.grad
           batch_autograd BatchedChi2Profile.autograd and its backward
  dtype    f64, f32, or mixed (float32 data and parameters with FP64 geometry and phase: batched forms)
  nxy      image size; pixels of DXY
  nvis     number of (u, v) points
  nr, bins profile bins, and bins per pixel: the model disc ends nr / bins pixels from its centre
  near     shortest baseline in cells of the Fourier grid, reach: longest as a fraction of half the grid
           (galario's get_image_size gives 3 cells and 0.4; a grid at its Nyquist limit 1 cell and 0.97)
  walkers, sets  batched forms: parameter sets, and the data sets as "nxy:nvis ..." on one pixel size
"""
import math

import numpy as np
import torch

import galario_amd.double as g_double
import galario_amd.single as g_single
from galario_amd import torch_api

ARCSEC = 4.84813681109536e-06
DXY = 0.01 * ARCSEC
RMIN = 1e-4 * ARCSEC
HOST = ("chi2_host", "image_chi2", "image_sample")


def listed():
    return [
        # galario's quickstart as its users have it: one walker of an emcee ensemble, host arrays in, a number
        # out, a small observation: latency counts
        {"name": "quickstart_f64", "kind": "chi2_host", "dtype": "f64", "nxy": 512, "nvis": 2013, "nr": 600,
         "bins": 12.0, "near": 3.0, "reach": 0.4},
        # the same call on an ordinary ALMA observation
        {"name": "fit_host_f64", "kind": "chi2_host", "dtype": "f64", "nxy": 1024, "nvis": 200000, "nr": 1500,
         "bins": 12.0, "near": 3.0, "reach": 0.4},
        # a fit with model images (a ring on 1024 x 1024 pixels against 1e5 visibilities)
        {"name": "image_chi2_f64", "kind": "image_chi2", "dtype": "f64", "nxy": 1024, "nvis": 100000,
         "near": 1.5, "reach": 0.3},
        # visibilities of an image from a radiative-transfer code, whose sizes are round decimal numbers
        {"name": "image_sample_f32", "kind": "image_sample", "dtype": "f32", "nxy": 1000, "nvis": 20011,
         "near": 3.0, "reach": 0.4},
        # the benchmark's profile fit: the observation resident on the GPU, 4096 x 4096 pixels, 1e6 points
        {"name": "chi2_f64", "kind": "chi2", "dtype": "f64", "nxy": 4096, "nvis": 1000000, "nr": 1000,
         "bins": 5.0, "near": 1.0, "reach": 0.97},
        # model visibilities for plots and residual maps, single precision
        {"name": "sample_f32", "kind": "sample", "dtype": "f32", "nxy": 4096, "nvis": 1000000, "nr": 1000,
         "bins": 5.0, "near": 1.0, "reach": 0.97},
        # an extended disc: the profile reaches far out in the image, finely binned
        {"name": "wide_chi2_f64", "kind": "chi2", "dtype": "f64", "nxy": 4096, "nvis": 300001, "nr": 9600,
         "bins": 12.0, "near": 3.0, "reach": 0.4},
        # gradient of a small problem (an optimiser's step on one execution block)
        {"name": "grad_small_f64", "kind": "grad", "dtype": "f64", "nxy": 512, "nvis": 5003, "nr": 500,
         "bins": 12.0, "near": 3.0, "reach": 0.4},
        # gradient at the benchmark's size
        {"name": "grad_f64", "kind": "grad", "dtype": "f64", "nxy": 4096, "nvis": 1000000, "nr": 1000,
         "bins": 5.0, "near": 1.0, "reach": 0.97},
        # a single-precision training step on 2e6 points: loss and gradients through torch.autograd
        {"name": "autograd_f32", "kind": "autograd", "dtype": "f32", "nxy": 2048, "nvis": 2000000, "nr": 500,
         "bins": 2.5, "near": 1.0, "reach": 0.97},
        # an ensemble sampler's step: 256 walkers, three data sets of uneven size
        {"name": "batch_f64", "kind": "batch", "dtype": "f64", "walkers": 256,
         "sets": "512:10000 1024:200000 2048:1000000", "nr": 300, "bins": 4.5, "near": 2.2, "reach": 0.87},
        # a gradient sampler's step: 64 parameter sets, three data sets (5e6 points) on one 4096 grid; the largest
        {"name": "batch_grad_f64", "kind": "batch_grad", "dtype": "f64", "walkers": 64,
         "sets": "4096:500000 4096:1500000 4096:3000000", "nr": 500, "bins": 2.5, "near": 1.0, "reach": 0.97},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _set_list(case):
    return [tuple(int(x) for x in s.split(":")) for s in case["sets"].split()]


def _cost(case):
    """Walker-points plus walker-cells of a batched case, against the largest listed one."""
    return case["walkers"] * sum(nvis + nxy * nxy / 8 for nxy, nvis in _set_list(case))


def draw(rng):
    kind = rng.choice(["chi2_host", "image_chi2", "image_sample", "chi2", "sample", "grad", "autograd", "batch",
                       "batch_grad", "batch_autograd"])
    near, reach = rng.choice([(3.0, 0.4), (3.0, 0.4), (1.0, 0.97), (1.5, 0.7)])
    case = {"kind": kind, "dtype": rng.choice(["f64", "f64", "f32"]), "near": near, "reach": reach}
    if kind.startswith("image"):
        nxy = 2 * _log_int(rng, 100, 1024)
        if rng.random() < 0.6:
            nxy = 1 << (nxy - 1).bit_length()
        case.update(nxy=min(nxy, 2048), nvis=_log_int(rng, 1000, 200000))
        return case
    if kind == "batch_autograd":
        case["dtype"] = rng.choice(["f64", "mixed", "f32"])
    elif case["dtype"] == "f32":   # a single-precision program takes its results in single precision
        kind = case["kind"] = {"chi2": "sample", "grad": "autograd", "batch": "batch_autograd",
                               "batch_grad": "batch_autograd"}.get(kind, kind)
    grad = "grad" in kind
    if kind.startswith("batch"):
        size = 1 << rng.randint(9, 12)
        sets = []
        for _ in range(rng.randint(1, 3)):
            n = size if grad else max(256, size >> rng.randint(0, 2))
            sets.append("%d:%d" % (n, _log_int(rng, 5000, 1000000)))
        case.update(walkers=_log_int(rng, 2, 256), sets=" ".join(sets))
        while case["walkers"] > 2 and _cost(case) > 2e8:
            case["walkers"] //= 2
        small = min(n for n, _ in _set_list(case))
    else:
        top = 11 if kind == "chi2_host" else 12
        small = 1 << rng.randint(8, top)
        case.update(nxy=small, nvis=_log_int(rng, 500, 200000 if kind == "chi2_host" else 1500000))
    # the disc ends between an eighth and eight tenths of the way to the image's edge
    radius = max(8.0, small / 2 * math.exp(rng.uniform(math.log(0.06), math.log(0.8))))
    case["bins"] = rng.choice([2.5, 5.0, 12.0, 15.0])
    case["nr"] = int(radius * case["bins"]) + rng.randint(0, 30)
    if grad:
        case["nr"] = min(case["nr"], 2048)
    return case


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------
def _profile(rng, nr, dR, walkers=None):
    """Two Gaussian rings and a power-law envelope (Jy/sr), sized by the disc, with 10% lognormal jitter per bin."""
    R = RMIN + dR * np.arange(nr)
    a = (RMIN + nr * dR) / 2.0
    base = 1e10 * (np.exp(-((R - 0.4 * a) ** 2) / (2 * (0.05 * a) ** 2))
                   + 0.5 * np.exp(-((R - 0.9 * a) ** 2) / (2 * (0.08 * a) ** 2))
                   + 0.3 * (R / a) ** -0.8 * np.exp(-R / (1.2 * a)))
    shape = (nr,) if walkers is None else (walkers, nr)
    return base * np.exp(0.1 * rng.standard_normal(shape))


def _geometry(rng, walkers=None):
    """(inc, PA, dRA, dDec): around 40 deg, 120 deg, 0.02" and 0.02"."""
    z = rng.standard_normal((1 if walkers is None else walkers, 4))
    g = np.stack([0.70 + 0.05 * z[:, 0], 2.09 + 0.2 * z[:, 1], (0.02 + 0.005 * z[:, 2]) * ARCSEC,
                  (0.02 + 0.005 * z[:, 3]) * ARCSEC], axis=1)
    return g[0] if walkers is None else g


def _observation(rng, nxy, nvis, near, reach, size, flux):
    """Log-uniform baselines at random angles; the visibilities of a Gaussian source of this size (rad) and flux
    (Jy) with noise, sigma log-uniform in [0.5, 2] x the median amplitude."""
    duv = 1.0 / (nxy * DXY)
    b = np.exp(rng.uniform(math.log(near * duv), math.log(reach * nxy / 2 * duv), nvis))
    th = rng.uniform(0.0, 2.0 * np.pi, nvis)
    u, v = b * np.cos(th), b * np.sin(th)
    amp = flux * (0.02 + np.exp(-2.0 * (np.pi * size * b) ** 2))
    phase = 2.0 * np.pi * 0.02 * ARCSEC * (u + v)
    sigma = float(np.median(amp)) * np.exp(rng.uniform(math.log(0.5), math.log(2.0), nvis))
    re = amp * np.cos(phase) + sigma * rng.standard_normal(nvis)
    im = amp * np.sin(phase) + sigma * rng.standard_normal(nvis)
    return u, v, re, im, 1.0 / sigma ** 2


def _image(rng, nxy):
    """A Gaussian ring of radius nxy / 10 pixels on a noisy background (Jy / pixel)."""
    c = (nxy // 2 - np.arange(nxy)) / nxy
    r = np.hypot(c[None, :], c[:, None])
    return np.exp(-((r - 0.1) ** 2) / (2 * 0.02 ** 2)) + rng.uniform(0.0, 1e-3, (nxy, nxy))


def _inputs(case, seed):
    """All inputs of a case as numpy arrays in its type, from the seed alone."""
    rng = np.random.default_rng(seed)
    real = np.float64 if case["dtype"] == "f64" else np.float32
    to = lambda a: np.ascontiguousarray(a, dtype=real)  # noqa: E731
    d = {}
    if case["kind"].startswith("image"):
        img = _image(rng, case["nxy"])
        d["image"] = to(img)
        size, flux = 0.1 * case["nxy"] * DXY, float(img.sum())
    else:
        d["dR"] = DXY / case["bins"]
        W = case.get("walkers")
        I = _profile(rng, case["nr"], d["dR"], W)
        d["I"] = to(I)
        out = case["nr"] * d["dR"]
        size, flux = 0.3 * out, 0.2 * 1e10 * math.pi * out * out
    g = _geometry(rng, case.get("walkers"))
    d["geom"] = g.astype(real)
    sets = _set_list(case) if "sets" in case else [(case["nxy"], case["nvis"])]
    d["sets"] = [(n,) + tuple(to(a) for a in _observation(rng, n, m, case["near"], case["reach"], size, flux))
                 for n, m in sets]
    return d


def _guard(case):
    """galario's central-pixel check wants at least five bins in half a pixel; coarser profiles switch it off."""
    return case["bins"] >= 11.0


def prepare(case, seed):
    d = _inputs(case, seed)
    kind, f64 = case["kind"], case["dtype"] == "f64"
    s = {"kind": kind}
    if kind in HOST:
        s["mod"] = g_double if f64 else g_single
        inc, PA, dRA, dDec = (float(x) for x in d["geom"])
        n, u, v, re, im, w = d["sets"][0]
        if kind == "chi2_host":
            s["args"] = (d["I"], RMIN, d["dR"], n, DXY, u, v, re, im, w)
            s["kw"] = dict(dRA=dRA, dDec=dDec, PA=PA, inc=inc, check_central_pixel=_guard(case))
        else:
            s["args"] = (d["image"], DXY, u, v) + ((re, im, w) if kind == "image_chi2" else ())
            s["kw"] = dict(dRA=dRA, dDec=dDec, PA=PA)
        return s
    dt = torch.float64 if f64 else torch.float32
    data = [(torch_api.Dataset(u, v, re, im, w, device="cuda:0", dtype=dt), n) for n, u, v, re, im, w in d["sets"]]
    s["I"] = torch.from_numpy(d["I"]).to("cuda:0")
    if kind.startswith("batch"):
        s["plan"] = torch_api.BatchedChi2Profile([(ds, n, DXY) for ds, n in data], case["nr"], RMIN, d["dR"],
                                                 case["walkers"], check_central_pixel=_guard(case),
                                                 phase_f64=case["dtype"] == "mixed")
        s["geom"] = torch.from_numpy(d["geom"]).to("cuda:0")
        if kind == "batch_autograd":
            s["I"].requires_grad_(True)
            s["geom"].requires_grad_(True)
        return s
    s["ds"], n = data[0]
    s["grid"] = (RMIN, d["dR"], n, DXY)
    if kind == "autograd":
        s["I"].requires_grad_(True)
        s["geom"] = torch.from_numpy(d["geom"]).requires_grad_(True)   # read on the host: kept there
        s["guard"] = _guard(case)
    else:
        inc, PA, dRA, dDec = (float(x) for x in d["geom"])
        s["kw"] = dict(dRA=dRA, dDec=dDec, PA=PA, inc=inc, check_central_pixel=_guard(case))
    return s


def run(s):
    kind = s["kind"]
    if kind == "chi2_host":
        return s["mod"].chi2Profile(*s["args"], **s["kw"])
    if kind == "image_chi2":
        return s["mod"].chi2Image(*s["args"], **s["kw"])
    if kind == "image_sample":
        return s["mod"].sampleImage(*s["args"], **s["kw"])
    if kind == "chi2":
        return s["ds"].chi2_profile(s["I"], *s["grid"], **s["kw"])
    if kind == "sample":
        return s["ds"].sample_profile(s["I"], *s["grid"], **s["kw"])
    if kind == "grad":
        return s["ds"].chi2_profile_grad(s["I"], *s["grid"], **s["kw"])
    if kind == "autograd":
        chi2 = torch_api.chi2_profile_autograd(s["ds"], s["I"], s["geom"], *s["grid"],
                                               check_central_pixel=s["guard"])
        loss = (0.5 * chi2).to(s["I"].dtype)
        return (loss.detach(),) + torch.autograd.grad(loss, (s["I"], s["geom"]))
    if kind == "batch":
        return s["plan"](s["I"], s["geom"])
    if kind == "batch_grad":
        return s["plan"].grad(s["I"], s["geom"])
    chi2 = s["plan"].autograd(s["I"], s["geom"])
    logp = (-0.5 * chi2).to(s["I"].dtype)
    return (logp.detach(),) + torch.autograd.grad(logp.sum(), (s["I"], s["geom"]))


def work(case):
    """Inputs read once and outputs written once; operations: the swept box, a real transform of the image (a
    quarter of it for a profile, whose image is even in both axes), and about 80 per point, three times as many
    with the gradient."""
    kind, b = case["kind"], 8 if case["dtype"] == "f64" else 4
    W = case.get("walkers", 1)
    sets = _set_list(case) if "sets" in case else [(case["nxy"], case["nvis"])]
    grad = 3.0 if "grad" in kind else 1.0
    nbytes = flops = 0.0
    for k, (n, m) in enumerate(sets):
        nbytes += m * b * (4 if "sample" in kind else 5)
        fft = 2.5 * n * n * math.log2(n * n)
        if kind.startswith("image"):
            nbytes += n * n * b
            flops += fft
        elif n not in [x for x, _ in sets[:k]]:
            r = min(case["nr"] / case["bins"], n / 2)
            flops += W * grad * (30 * r * r + fft / 4)
        flops += W * grad * 80 * m
    if not kind.startswith("image"):
        nbytes += W * (case["nr"] + 4) * (b + (8 if grad > 1 else 0))
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------------------------------------------
# the same results in 64 bits from plain torch
# ---------------------------------------------------------------------------------------------------------------
def _swept(I, inc, dR, n):
    """n x n image of a profile: linear interpolation in radius, the central pixel by the trapezoid rule."""
    nr, dev = I.shape[0], I.device
    half = min(int(math.ceil((RMIN + nr * dR) / DXY)), n // 2)
    k = torch.arange(half, -half, -1, dtype=torch.float64, device=dev) * DXY
    xs = k[None, :] / torch.cos(inc)
    r = torch.sqrt(torch.clamp(xs ** 2 + (k ** 2)[:, None], min=1e-300))
    bin_ = torch.clamp(torch.floor((r.detach() - RMIN) / dR), min=0.0)
    at = (bin_ <= nr - 2).reshape(-1).nonzero().reshape(-1)
    r, i = r.reshape(-1).index_select(0, at), bin_.reshape(-1).index_select(0, at)
    lo, hi = I.index_select(0, i.long()), I.index_select(0, i.long() + 1)
    val = DXY * DXY * (lo + (r - i * dR - RMIN) * (hi - lo) / dR)
    box = torch.zeros(4 * half * half, dtype=torch.float64, device=dev).index_copy(0, at, val)
    m = int(math.floor((DXY / 2 - RMIN) / dR))
    Ri = RMIN + dR * torch.arange(m + 2, dtype=torch.float64, device=dev)
    h = DXY / 2
    edge = (I[m + 1] - I[m]) / dR * (h - Ri[m]) + I[m]
    flux = dR * (RMIN * I[0] + 2 * (Ri[1:m] * I[1:m]).sum() + Ri[m] * I[m])
    flux = flux + (Ri[m] * I[m] + h * edge) * (h - Ri[m])
    centre = DXY * DXY * flux / (h * h - RMIN * RMIN)
    box = box.index_copy(0, torch.tensor([half * 2 * half + half], device=dev), centre.reshape(1))
    p = n // 2 - half
    return torch.nn.functional.pad(box.reshape(2 * half, 2 * half), (p, p, p, p))


def _spectrum(img):
    return torch.fft.fftshift(torch.fft.rfft2(torch.fft.fftshift(img)), dim=0)


def _visibilities(S, u, v, PA, dRA, dDec):
    """Amplitude and phase of the spectrum interpolated at the rotated points, shifted by the offsets."""
    n, ncol = S.shape
    c, s = torch.cos(PA), torch.sin(PA)
    ur, vr = u * c - v * s, u * s + v * c
    duv = 1.0 / (n * DXY)
    sg = torch.where(ur.detach() < 0, -1.0, 1.0).double()
    x, y = torch.abs(ur) / duv, n // 2 + sg * vr / duv
    i, j = torch.floor(x.detach()), torch.floor(y.detach())
    q, t = x - i, y - j
    at = (j * ncol + i).long()
    R = torch.view_as_real(S).reshape(-1, 2)
    y0, y1, y2, y3 = (R.index_select(0, at + o) for o in (0, ncol, ncol + 1, 1))
    b0, b1, b2, b3 = (1 - t) * (1 - q), t * (1 - q), t * q, (1 - t) * q
    Z = y0 * b0[:, None] + y1 * b1[:, None] + y2 * b2[:, None] + y3 * b3[:, None]
    A = sum(torch.sqrt((k * k).sum(dim=1)) * b for k, b in ((y0, b0), (y1, b1), (y2, b2), (y3, b3)))
    ph = sg * torch.atan2(Z[:, 1], Z[:, 0]) + 2 * math.pi * (u * dRA + v * dDec)
    return A * torch.cos(ph), A * torch.sin(ph)


def _chi2(V, re, im, w):
    return (((V[0] - re) ** 2 + (V[1] - im) ** 2) * w).sum()


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    dev = "cuda:0" if torch.cuda.is_available() else "cpu"
    put = lambda a: torch.from_numpy(np.asarray(a, dtype=np.float64)).to(dev)  # noqa: E731
    sets = [(s[0],) + tuple(put(a) for a in s[1:]) for s in d["sets"]]
    geom = put(d["geom"])
    with torch.set_grad_enabled("grad" in kind):
        if kind.startswith("image"):
            n, u, v, re, im, w = sets[0]
            V = _visibilities(_spectrum(put(d["image"])), u, v, geom[1], geom[2], geom[3])
            return float(_chi2(V, re, im, w)) if kind == "image_chi2" else torch.complex(*V).cpu().numpy()
        if kind == "sample":
            n, u, v = sets[0][:3]
            S = _spectrum(_swept(put(d["I"]), geom[0], d["dR"], n))
            return torch.complex(*_visibilities(S, u, v, geom[1], geom[2], geom[3]))
        Is, gs = put(np.atleast_2d(d["I"])), geom.reshape(-1, 4)
        per, gI, gg = [], [], []
        for I, g in zip(Is, gs):
            if "grad" in kind:
                I, g = I.clone().requires_grad_(True), g.clone().requires_grad_(True)
            spectra, each = {}, []
            for n, u, v, re, im, w in sets:
                if n not in spectra:
                    spectra[n] = _spectrum(_swept(I, g[0], d["dR"], n))
                each.append(_chi2(_visibilities(spectra[n], u, v, g[1], g[2], g[3]), re, im, w))
            per.append(torch.stack(each))
            if "grad" in kind:
                a, b = torch.autograd.grad(per[-1].sum(), (I, g))
                per[-1] = per[-1].detach()
                gI.append(a)
                gg.append(b)
        per = torch.stack(per)
        tot = per.sum(dim=1)
        if kind == "chi2_host":
            return float(tot[0])
        if kind in ("chi2", "batch"):
            return tot
        gI, gg = torch.stack(gI), torch.stack(gg)
        if kind == "grad":
            return tot, gI[0], gg[0]
        if kind == "autograd":
            return 0.5 * tot[0], 0.5 * gI[0], 0.5 * gg[0]
        if kind == "batch_grad":
            return tot, per, gI, gg
        return -0.5 * tot, -0.5 * gI, -0.5 * gg
