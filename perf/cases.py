"""Timed cases of the pair-counting estimator, through its Python entry points.

The path's users estimate the Lyman-alpha forest correlation function of a
catalogue (one pass over every candidate pixel pair), of its sky-bin
subsamples with their covariance, of batches of mock catalogues, or of plain
3D points.  Catalogues are drawn like the package's generator does it:
quasars uniform in area, pixels on one wavelength grid for the whole survey
(3e-4 in log10 lambda), delta ~ N(0, 0.2), weights 1 / (0.04 + sigma^2),
distances from flat LCDM; `masked` is the fraction of pixels a survey's
quality cuts take out of the sightlines.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "turbo-octo-spice_amd"))

import tos_amd  # noqa: E402
from tos_amd import GridSpec, synth  # noqa: E402

LYA = 1216.0
DEG = math.pi / 180.0
DLOG = 3e-4
_PRECISION = {"fp64": tos_amd.FP64, "fp32c": tos_amd.FP32C}
_GRIDS = {
    # (axis 0, axis 1) of the package's defaults and of its tests
    "cartesian": ("[0:200]*50", "[0:200]*50"),
    "polar": ("[0:200]*50", "[0:1]*20"),
    "observing": ("[0:0.02]*20", "[0:0.06]*6"),
}


# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------
def _xi(name, n_qso, area, grid, precision, accum="core", nz=1, masked=0.0):
    return {"name": name, "kind": "xi", "n_qso": n_qso, "area": area, "grid": grid, "precision": precision,
            "accum": accum, "nz": nz, "masked": masked}


def listed():
    return [
        # a test patch: launches, copies and set-up are all there is
        _xi("xi_patch_cart_fp32c", 120, 40.0, "cartesian", "fp32c"),
        # a survey field at the default precision
        _xi("xi_field_cart_fp64", 10000, 1000.0, "cartesian", "fp64"),
        # the same field in (r, mu), a few percent of its pixels masked
        _xi("xi_field_polar_fp32c", 9973, 1000.0, "polar", "fp32c", masked=0.04),
        # a smaller, denser field in observed coordinates
        _xi("xi_field_observing_fp32c", 5003, 300.0, "observing", "fp32c"),
        # every XiBin sum over three z bins, masked pixels
        _xi("xi_sums_cart_fp64", 2003, 400.0, "cartesian", "fp64", accum="all", nz=3, masked=0.04),
        # a survey at the full density and area: the benchmark's workload
        _xi("xi_survey_cart_fp32c", 160000, 10000.0, "cartesian", "fp32c"),
        # from host arrays to the histogram: upload, candidate search on the
        # device, one pass (what a user with a new catalogue runs)
        {"name": "estimate_cart_fp32c", "kind": "estimate", "n_qso": 40001, "area": 2500.0, "grid": "cartesian",
         "precision": "fp32c", "nz": 1, "masked": 0.04},
        # the pass with one histogram per sky bin, for the covariance
        {"name": "skybins_cart_fp32c", "kind": "skybins", "n_qso": 10000, "area": 1000.0, "grid": "cartesian",
         "precision": "fp32c", "nz": 1, "masked": 0.0},
        # mock catalogues of mixed sizes in one batched launch
        {"name": "batch_mocks_cart_fp32c", "kind": "batch", "n_jobs": 12, "n_lo": 2000, "n_hi": 12000,
         "area": 2000.0, "grid": "cartesian", "precision": "fp32c", "nz": 1, "masked": 0.0},
        # 10,000 points in 3D (the brute-force benchmark)
        {"name": "brute_fp64", "kind": "brute", "n": 10000, "mode": "fp64", "nbins": 50},
        # covariance of a survey's sky-bin subsamples on a 50 x 50 grid
        {"name": "covariance_survey", "kind": "covariance", "samples": 1900, "nbins": 2500},
        # distance transform of a field's pixels
        {"name": "distances_field", "kind": "distances", "n": 1500007},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["xi", "xi", "xi", "xi", "estimate", "skybins", "batch", "brute", "covariance", "distances"])
    grid = rng.choice(["cartesian", "cartesian", "polar", "observing"])
    precision = rng.choice(["fp32c", "fp64"])
    masked = rng.choice([0.0, 0.0, 0.02, 0.08])
    if kind in ("xi", "estimate", "skybins"):
        n = _logint(rng, 100, 40000 if kind != "skybins" else 20000)
        density = math.exp(rng.uniform(math.log(3.0), math.log(20.0)))   # quasars per square degree
        case = {"kind": kind, "n_qso": n, "area": round(n / density, 3), "grid": grid, "precision": precision,
                "nz": rng.choice([1, 1, 2, 3]), "masked": masked}
        if kind == "xi":
            case["accum"] = rng.choice(["core", "core", "core", "all"]) if n <= 10000 else "core"
        return case
    if kind == "batch":
        lo = _logint(rng, 200, 4000)
        return {"kind": "batch", "n_jobs": rng.randint(2, 24), "n_lo": lo, "n_hi": lo * rng.randint(1, 4),
                "area": round(rng.uniform(500.0, 4000.0), 3), "grid": grid, "precision": precision, "nz": 1,
                "masked": masked}
    if kind == "brute":
        return {"kind": "brute", "n": _logint(rng, 64, 200000), "mode": rng.choice(["fp64", "fp32"]),
                "nbins": rng.choice([20, 50, 50, 75, 200])}
    if kind == "covariance":
        return {"kind": "covariance", "samples": _logint(rng, 40, 2000), "nbins": rng.choice([120, 1000, 1001, 2500])}
    return {"kind": "distances", "n": _logint(rng, 1000, 12000000)}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _los_distance(z):
    """Flat LCDM (0.7, 0.3) comoving distance in Mpc/h: composite Simpson."""
    z = np.asarray(z, np.float64)
    n = 2048
    t = np.linspace(0.0, 1.0, n + 1)
    w = np.full(n + 1, 2.0)
    w[1::2] = 4.0
    w[0] = w[-1] = 1.0
    out = np.empty_like(z)
    for s in range(0, len(z), 2048):
        a = np.log1p(z[s:s + 2048])[:, None] * t[None, :]
        f = np.exp(a) / np.sqrt(0.3 * np.exp(3.0 * a) + 0.7)
        out[s:s + 2048] = 2997.92458 * (f @ w) * np.log1p(z[s:s + 2048]) / (3.0 * n)
    return out


def _catalog(n_qso, area, masked, seed):
    rng = np.random.default_rng(seed)
    # a patch of RA extent a and |sin dec| < s around the equator, 2 a s = area
    lo, hi = 0.0, 1.0
    for _ in range(100):
        s = 0.5 * (lo + hi)
        lo, hi = (s, hi) if 4.0 * s * math.asin(s) < area * DEG * DEG else (lo, s)
    a = area * DEG * DEG / (2.0 * s)
    ra = rng.uniform(0.0, a, n_qso)
    dec = np.arcsin(rng.uniform(-s, s, n_qso))
    zq = np.clip(rng.normal(2.4, 0.4, n_qso), 2.1, 3.5)
    logs = math.log10(3600.0) + DLOG * np.arange(1, 720)
    lam = 10.0 ** logs
    k_lo = np.searchsorted(lam, 1040.0 * (1.0 + zq), side="left")
    k_hi = np.searchsorted(lam, 1200.0 * (1.0 + zq), side="right")
    cnt = np.maximum(k_hi - k_lo, 0)
    off = np.zeros(n_qso + 1, np.int64)
    np.cumsum(cnt, out=off[1:])
    idx = np.repeat((k_lo - off[:-1]).astype(np.int32), cnt) + np.arange(off[-1], dtype=np.int32)
    if masked > 0:
        keep = rng.random(len(idx), dtype=np.float32) >= masked
        owner = np.repeat(np.arange(n_qso), cnt)[keep]
        off = np.zeros(n_qso + 1, np.int64)
        np.cumsum(np.bincount(owner, minlength=n_qso), out=off[1:])
        idx = idx[keep]
    loglam = logs.astype(np.float32)
    dist = _los_distance(10.0 ** (loglam.astype(np.float64) - math.log10(LYA)) - 1.0)
    value = rng.standard_normal(len(idx), dtype=np.float32) * np.float32(0.2)
    noise = rng.random(len(idx), dtype=np.float32) * np.float32(0.45) + np.float32(0.05)
    weight = np.float32(1.0) / (np.float32(0.04) + noise * noise)
    first = off[:-1][np.diff(off) > 0]
    return synth.Catalog(ra, dec, off, value, loglam[idx], weight, dist.astype(np.float32)[idx], zq,
                         float(dist[idx[first]].min()))


def _grid(case):
    a0, a1 = _GRIDS[case["grid"]]
    z = "[3.556:3.735]*%d" % case["nz"]
    return GridSpec.from_specs({"cartesian": tos_amd.CARTESIAN, "polar": tos_amd.POLAR,
                                "observing": tos_amd.OBSERVING}[case["grid"]], a0, a1, z)


def _points(case, seed):
    rng = np.random.default_rng(seed)
    xyz = rng.uniform(0.0, 100.0, (3, case["n"]))
    return [xyz[0].copy(), xyz[1].copy(), xyz[2].copy(), rng.normal(0.0, 1.0, case["n"]),
            rng.uniform(0.5, 1.5, case["n"])]


def _samples(case, seed):
    rng = np.random.default_rng(seed)
    k, n = case["samples"], case["nbins"]
    wgt = rng.gamma(4.0, 50.0, (k, n))
    wgt[rng.random((k, n), dtype=np.float32) < 0.02] = 0.0
    return wgt * rng.standard_normal((k, n)) * 1e-3, wgt


def _pixels(case, seed):
    rng = np.random.default_rng(seed)
    logs = (math.log10(3600.0) + DLOG * np.arange(1, 720)).astype(np.float32)
    return logs[rng.integers(0, len(logs), case["n"])]


def _batch_sizes(case, seed):
    return np.random.default_rng([seed, 1]).integers(case["n_lo"], case["n_hi"] + 1, case["n_jobs"])


_DEV = None


def _device():
    """The program's one device context."""
    global _DEV
    if _DEV is None:
        _DEV = tos_amd.Device(0)
    return _DEV


class _State:
    """Resident catalogues and pair lists, freed with the state."""

    def __init__(self, case):
        self.case, self.owned = case, []

    def resident(self, cat, grid):
        dcat = _device().upload(cat)
        pairs = dcat.pairs(grid.max_angular_scale(cat.scale), order=4, on_device=True)
        self.owned += [pairs, dcat]
        return pairs

    def __del__(self):
        for h in self.owned:
            h.free()


def prepare(case, seed):
    st = _State(case)
    kind = case["kind"]
    if kind in ("xi", "skybins"):
        st.grid = _grid(case)
        st.pairs = st.resident(_catalog(case["n_qso"], case["area"], case["masked"], seed), st.grid)
    elif kind == "estimate":
        st.grid = _grid(case)
        st.cat = _catalog(case["n_qso"], case["area"], case["masked"], seed)
    elif kind == "batch":
        st.grid = _grid(case)
        cats = [_catalog(int(n), case["area"], case["masked"], [seed, q])
                for q, n in enumerate(_batch_sizes(case, seed))]
        st.jobs = [(st.resident(c, st.grid), st.grid, _PRECISION[case["precision"]]) for c in cats]
    elif kind == "brute":
        st.points = _points(case, seed)
    elif kind == "covariance":
        st.samples = _samples(case, seed)
    else:
        st.loglam = _pixels(case, seed)
    _device()
    return st


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def _histogram(h):
    out = {"num_pairs": h.num_pairs, "didj": h.didj, "wgt": h.wgt}
    out.update(h.extra)
    return out


def run(st):
    case = st.case
    kind = case["kind"]
    if kind == "xi":
        accum = tos_amd.ACC_ALL if case["accum"] == "all" else tos_amd.ACC_CORE
        return _histogram(st.pairs.run(st.grid, precision=_PRECISION[case["precision"]], accum=accum))
    if kind == "estimate":
        dcat = _device().upload(st.cat)
        pairs = dcat.pairs(st.grid.max_angular_scale(st.cat.scale), order=4, on_device=True)
        out = _histogram(pairs.run(st.grid, precision=_PRECISION[case["precision"]]))
        stats = pairs.stats()
        out["sightline_pairs"] = stats["num_sightline_pairs_used"]
        out["pixel_pairs"] = stats["num_pixel_pairs"]
        pairs.free()
        dcat.free()
        return out
    if kind == "skybins":
        h, keys, sn, sd, sw = st.pairs.run_per_skybin(st.grid, precision=_PRECISION[case["precision"]])
        return {"total": _histogram(h), "keys": keys, "num_pairs": sn, "didj": sd, "wgt": sw}
    if kind == "batch":
        return [_histogram(h) for h in _device().batch_run(st.jobs)[0]]
    if kind == "brute":
        mode = tos_amd.BRUTE_FP64 if case["mode"] == "fp64" else tos_amd.BRUTE_FP32
        d, w, n, _ = _device().brute3d(*st.points, 0.0, 100.0, case["nbins"], mode=mode)
        return {"dsum": d, "wsum": w, "counts": n}
    if kind == "covariance":
        cov, mean, weight = _device().subsample_covariance(*st.samples)
        return {"cov": cov, "mean": mean, "weight": weight}
    return _device().pixel_distances(st.loglam)


# --------------------------------------------------------------------------
# Bytes and operations of a pass
# --------------------------------------------------------------------------
_MEAN_PIXELS = 146.0   # of a sightline drawn as above


def _xi_work(n, area, grid, nbins_total, masked):
    pix = _MEAN_PIXELS * (1.0 - masked)
    radius = 0.06 if grid == "observing" else 200.0 / 3500.0
    cap = min(1.0, 2.0 * math.pi * (1.0 - math.cos(radius)) / (area * DEG * DEG))
    pairs = 0.5 * n * n * cap
    # pixels of 2 Mpc/h (or 3e-4) along a partner inside the axis-0 range
    window = min(pix, 2 * 0.02 / DLOG if grid == "observing" else 200.0)
    flops = {"cartesian": 20, "polar": 18, "observing": 11}[grid] * pairs * pix * 0.6 * window
    return n * pix * 16.0 + pairs * 12.0 + nbins_total * 24.0, flops


def work(case):
    kind = case["kind"]
    if kind in ("xi", "estimate", "skybins"):
        nb = _grid(case).nbins_total
        b, f = _xi_work(case["n_qso"], case["area"], case["grid"], nb, case["masked"])
        if kind == "skybins":
            b += nb * 24.0 * (case["area"] / 13.4)
        return {"bytes": b, "flops": f}
    if kind == "batch":
        n = 0.5 * (case["n_lo"] + case["n_hi"])
        b, f = _xi_work(n, case["area"], case["grid"], _grid(case).nbins_total, case["masked"])
        return {"bytes": b * case["n_jobs"], "flops": f * case["n_jobs"]}
    if kind == "brute":
        n = case["n"]
        return {"bytes": n * 40.0 + case["nbins"] * 24.0, "flops": 16.0 * 0.5 * n * (n - 1)}
    if kind == "covariance":
        k, n = case["samples"], case["nbins"]
        return {"bytes": 16.0 * k * n + 8.0 * n * n, "flops": 2.0 * k * n * n}
    return {"bytes": 8.0 * case["n"], "flops": case["n"] * 512.0 * 10.0}


# --------------------------------------------------------------------------
# The same in 64 bits, plain torch and numpy
# --------------------------------------------------------------------------
def _exact_xi(cat, case, limit=4e9):
    """The estimator's definition: bins from the pixels' float distances and
    wavelengths (their differences, squares and sums are floats), sums of the
    products in 64 bits."""
    ra, dec, off = cat.ra, cat.dec, cat.offsets
    n = len(ra)
    if n > 12000:
        return None
    cnt = np.diff(off)
    grid = case["grid"]
    (n0, min0, w0, max0), (n1, min1, w1, max1) = [
        (int(s.split("*")[1]), float(s[1:].split(":")[0]), 0.0, float(s.split(":")[1].split("]")[0]))
        for s in _GRIDS[grid]]
    w0, w1 = (max0 - min0) / n0, (max1 - min1) / n1
    nz, minz = case["nz"], 3.556
    reach = max1 if grid == "observing" else (max0 if grid == "polar" else max1) / cat.scale
    sd, cd, sr, cr = np.sin(dec), np.cos(dec), np.sin(ra), np.cos(ra)
    pi, pj, pc = [], [], []
    for i in range(n):
        c = sd[i] * sd[i + 1:] + cd[i] * cd[i + 1:] * (sr[i] * sr[i + 1:] + cr[i] * cr[i + 1:])
        j = np.nonzero(c > math.cos(reach))[0]
        pi.append(np.full(len(j), i))
        pj.append(j + i + 1)
        pc.append(c[j])
    pi, pj, pc = np.concatenate(pi), np.concatenate(pj), np.concatenate(pc)
    if float((cnt[pi] * cnt[pj]).sum()) > limit:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    nb = n0 * n1 * nz
    width = int(cnt.max()) if n else 0
    pos = torch.arange(width, device=dev)
    toff, tcnt = torch.as_tensor(off[:-1], device=dev), torch.as_tensor(cnt, device=dev)
    pix = {k: torch.as_tensor(getattr(cat, k), device=dev) for k in ("value", "loglam", "weight", "distance")}
    last = max(0, cat.n_pix - 1)
    total = torch.zeros(nb, dtype=torch.int64, device=dev)
    keys = ["didj", "wgt"] + (["di", "dj", "wi", "wj", "z"] if case.get("accum") == "all" else [])
    sums = {k: torch.zeros(nb, dtype=torch.float64, device=dev) for k in keys}
    f64 = torch.float64
    for s in range(0, len(pi), 512):
        ti, tj = (torch.as_tensor(x[s:s + 512], device=dev) for x in (pi, pj))
        c = torch.as_tensor(pc[s:s + 512], device=dev)[:, None, None]
        ia, ja = (toff[t][:, None] + pos for t in (ti, tj))
        ok = (pos < tcnt[ti][:, None])[:, :, None] & (pos < tcnt[tj][:, None])[:, None, :]
        d1, l1, a1, v1 = (pix[k][ia.clamp(max=last)][:, :, None] for k in ("distance", "loglam", "weight", "value"))
        d2, l2, a2, v2 = (pix[k][ja.clamp(max=last)][:, None, :] for k in ("distance", "loglam", "weight", "value"))
        if grid == "observing":
            x0 = (l1 - l2).abs().to(f64)
            x1 = torch.arccos(c).expand_as(x0)
        else:
            r_par = (d1 - d2).abs().to(f64)
            r_sq = (d1 * d1).to(f64) + (d2.to(f64) - (2 * d1).to(f64) * c) * d2.to(f64)
            if grid == "cartesian":
                x0, x1 = r_par, torch.sqrt((r_sq - r_par * r_par).abs())
            else:
                x0 = torch.sqrt(r_sq)
                x1 = r_par / x0
                ok &= x0 != 0
                # r^2 < 0 counts in the first bin, like the C cast of a NaN
                x0, x1 = torch.nan_to_num(x0, 0.0), torch.nan_to_num(x1, 0.0)
        t0, t1 = (x0 - min0) * (1.0 / w0), (x1 - min1) * (1.0 / w1)
        tz = (0.5 * (l1 + l2).to(f64) - minz) * (1.0 / nz)
        ok &= (t0 > -1) & (t0 < n0) & (t1 > -1) & (t1 < n1) & (tz > -1)
        b = (tz.to(torch.int64) + (t1.to(torch.int64) + t0.to(torch.int64) * n1) * nz)[ok]
        total += torch.bincount(b, minlength=nb)[:nb]
        wa, wb = a1.to(f64), a2.to(f64)
        da, db = wa * v1.to(f64), wb * v2.to(f64)
        full = ok.shape
        terms = {"didj": da * db, "wgt": wa * wb}
        if len(keys) > 2:
            terms.update(di=da.expand(full), dj=db.expand(full), wi=wa.expand(full), wj=wb.expand(full),
                         z=0.5 * (l1.to(f64) + l2.to(f64)))
        for k in keys:
            sums[k] += torch.bincount(b, weights=terms[k][ok], minlength=nb)[:nb]
    out = {"num_pairs": total.cpu().numpy().astype(np.uint64)}
    out.update({k: v.cpu().numpy() for k, v in sums.items()})
    return out


def _exact_brute(case, seed):
    n, nb = case["n"], case["nbins"]
    if n > 20000:
        return None
    x, y, z, d, w = _points(case, seed)
    fp64 = case["mode"] == "fp64"
    slots = nb if fp64 else nb + 2
    counts, dsum, wsum = np.zeros(slots, np.uint64), np.zeros(slots), np.zeros(slots)
    t = np.float64 if fp64 else np.float32
    px, py, pz = x.astype(t), y.astype(t), z.astype(t)
    step = t(100.0) / t(nb)
    for i in range(n - 1):
        dx, dy, dz = px[i] - px[i + 1:], py[i] - py[i + 1:], pz[i] - pz[i + 1:]
        rsq = dx * dx + dy * dy + dz * dz
        ww = w[i] * w[i + 1:]
        wd = ww * d[i] * d[i + 1:]
        b = np.floor(np.sqrt(rsq) / step).astype(np.int64)
        if fp64:
            ok = (rsq < 10000.0) & (b < nb)
            b, ww, wd = b[ok], ww[ok], wd[ok]
        else:
            b = np.where(np.sqrt(rsq) >= t(100.0), nb + 1, np.minimum(b + 1, nb + 1))
        counts += np.bincount(b, minlength=slots).astype(np.uint64)
        wsum += np.bincount(b, weights=ww, minlength=slots)
        dsum += np.bincount(b, weights=wd, minlength=slots)
    return {"dsum": dsum, "wsum": wsum, "counts": counts}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("xi", "estimate"):
        if case["n_qso"] > 12000:
            return None
        cat = _catalog(case["n_qso"], case["area"], case["masked"], seed)
        out = _exact_xi(cat, case)
        if out is not None and kind == "estimate":
            out["sightline_pairs"] = out["pixel_pairs"] = None
        return out
    if kind == "brute":
        return _exact_brute(case, seed)
    if kind == "covariance":
        didj, wgt = _samples(case, seed)
        x = np.where(wgt > 0, didj / np.where(wgt > 0, wgt, 1.0), 0.0)
        w = np.where(wgt > 0, wgt, 0.0).sum(axis=1)
        mean = (w[:, None] * x).sum(axis=0) / w.sum()
        x -= mean
        return {"cov": (w[:, None] * x).T @ x / w.sum(), "mean": mean, "weight": float(w.sum())}
    if kind == "distances":
        loglam = _pixels(case, seed)
        uniq, inv = np.unique(loglam, return_inverse=True)
        return _los_distance(10.0 ** (uniq.astype(np.float64) - math.log10(LYA)) - 1.0)[inv]
    return None
