"""Performance cases of the pair counters: what a program that counts pairs asks of the library.

A case is one call of a public entry point on one synthetic catalog (or one batched call on many):
the Python functions of corrfunc_amd.theory and corrfunc_amd.mocks on the caller's numpy arrays
("place": "host"), the C entry points and the batched call on catalogs kept in GPU memory
("place": "device", the arrangement of a program that counts one catalog several times).

  kind     DD, DDrppi, DDsmu, xi, wp, batch (many DD), DDrppi_mocks, DDsmu_mocks (on-sky catalogs)
  n1, n2   points of the first / second catalog (n2 = 0: autocorrelation); ncat catalogs in a batch,
           their sizes log-uniform in [n1, n2]
  sample   uniform; clumps (Gaussian clumps, sigma 2 per axis, ~2000 points each); halos (60 % of the
           points in NFW-profile halos of log-normal occupancy, the rest uniform); sky (RA, DEC, cz)
  avg, weights   the averages of the separations, pair_product weights U(0.5, 1.5)
"""
import ctypes
import math
import os

import numpy as np
import torch

from corrfunc_amd import _abi, _lib, mocks, theory

SEED = 7919
THREADS = 16
SIGMA = 2.0          # clump size
PER_CLUMP = 2097     # points of a clump, on average
C_KM_S = 299800.0


def _case(name, kind, place, n1, n2, dtype, box, sample, rmin, rmax, nbins, log=True, avg=False, weights=False,
          periodic=True, pimax=0.0, nmu=0, ncat=1):
    c = dict(kind=kind, place=place, n1=n1, n2=n2, ncat=ncat, dtype=dtype, box=box, sample=sample, rmin=rmin,
             rmax=rmax, nbins=nbins, log=log, avg=avg, weights=weights, periodic=periodic, pimax=pimax, nmu=nmu)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's documentation example: ten thousand double points, counts only; a call this
        # small is what an MCMC or a notebook makes over and over, and latency is all of it
        _case("dd_10k", "DD", "host", 10000, 0, "f8", 420.0, "uniform", 0.1, 25.0, 20),
        # a small survey patch against its randoms: cross counts, open boundaries, float32, weights,
        # averages, sizes that fill no tile
        _case("dd_cross_60k", "DD", "host", 20011, 60007, "f4", 250.0, "uniform", 0.1, 12.0, 9, avg=True,
              weights=True, periodic=False),
        # DD(r) of a million double points in a periodic box (simulation snapshot), averages
        _case("dd_1M", "DD", "device", 1048576, 0, "f8", 420.0, "uniform", 0.1, 25.0, 20, avg=True),
        # DD(r) of a dense float32 box out to a tenth of its side, counts only (RR of a periodic box)
        _case("dd_counts_2M", "DD", "device", 2000003, 0, "f4", 500.0, "uniform", 0.5, 50.0, 18),
        # DD(rp, pi) of a clustered mock with weights and averages (redshift-space clustering)
        _case("rppi_4M", "DDrppi", "device", 4194304, 0, "f4", 1000.0, "clumps", 0.1, 30.0, 14, avg=True,
              weights=True, pimax=40.0),
        # w_p(rp) of a clustered double catalog through the Python function, counts only (its default)
        _case("wp_1M", "wp", "host", 1000003, 0, "f8", 1000.0, "clumps", 0.1, 30.0, 14, pimax=40.0),
        # xi(r) of the particles of a halo simulation, the largest catalog
        _case("xi_16M", "xi", "device", 16777216, 0, "f4", 1000.0, "halos", 0.1, 40.0, 25, avg=True),
        # DD(s, mu) of clustered data against ten times as many randoms out to the acoustic scale: the
        # largest call by pairs (BAO analyses)
        _case("smu_cross_10M", "DDsmu", "device", 1000000, 10000000, "f4", 1000.0, "clumps", 0.0, 150.0, 30,
              log=False, avg=True, weights=True, nmu=40),
        # DD(s, mu) autocorrelation of a double catalog through the Python function, counts only
        _case("smu_300k", "DDsmu", "host", 300007, 0, "f8", 500.0, "uniform", 1.0, 61.0, 12, log=False, nmu=20),
        # one batched call on many boxes of very different sizes (an ensemble of simulations)
        _case("batch_64", "batch", "device", 50000, 2000000, "f4", 500.0, "uniform", 0.5, 50.0, 18, avg=True,
              ncat=64),
        # one batched call on many small weighted catalogs (jackknife or bootstrap resamples)
        _case("batch_small_96", "batch", "device", 2000, 20000, "f4", 200.0, "uniform", 0.5, 20.0, 12, avg=True,
              weights=True, ncat=96),
        # DD(rp, pi) of a galaxy survey given as RA, DEC, cz, weights and averages, through the Python function
        _case("sky_rppi_1M", "DDrppi_mocks", "host", 1000000, 0, "f8", 0.0, "sky", 0.1, 25.0, 14, avg=True,
              weights=True, periodic=False, pimax=40.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: kind, sizes (log-uniform), box, bins and options at random."""
    kind = rng.choice(["DD", "DD", "DDrppi", "DDsmu", "xi", "wp", "batch", "DDrppi_mocks", "DDsmu_mocks"])
    dtype = rng.choice(["f4", "f8"])
    avg, weights = rng.random() < 0.5, rng.random() < 0.4
    box = rng.choice([250.0, 420.0, 500.0, 1000.0])
    rmax = round(box * math.exp(rng.uniform(math.log(0.015), math.log(0.09))), 2)
    nbins = rng.randint(6, 30)
    if kind == "batch":
        ncat = rng.randint(12, 128)
        lo = _log_int(rng, 1000, 60000)
        hi = min(2000000, _log_int(rng, 2 * lo, 40 * lo))
        # the whole call costs no more than the listed ensemble
        while ncat * hi * hi * (rmax / box) ** 3 > 64 * 4e12 * 1e-3 / 4:
            hi = max(lo + 1, hi // 2)
            ncat = max(8, ncat * 3 // 4)
        return _case(None, kind, "device", lo, hi, "f4", box, "uniform", 0.5, rmax, nbins, avg=avg, weights=weights,
                     ncat=ncat)
    if kind in ("DDrppi_mocks", "DDsmu_mocks"):
        n1 = _log_int(rng, 20000, 1000000)
        n2 = _log_int(rng, n1, 2 * n1) if rng.random() < 0.4 and n1 < 400000 else 0
        smu = kind == "DDsmu_mocks"
        return _case(None, kind, "host", n1, n2, "f8", 0.0, "sky", 0.5 if smu else 0.1,
                     round(rng.uniform(20.0, 40.0 if smu else 25.0), 1), nbins, log=not smu, avg=avg, weights=weights,
                     periodic=False, pimax=0.0 if smu else float(rng.randint(20, 40)), nmu=rng.randint(5, 50) if smu else 0)
    sample = rng.choice(["uniform", "clumps"] if kind != "xi" else ["uniform", "halos"])
    place = rng.choice(["host", "device"])
    n1 = _log_int(rng, 3000, 3000000)
    n2 = _log_int(rng, n1, 5 * n1) if kind in ("DD", "DDrppi", "DDsmu") and rng.random() < 0.35 else 0
    pimax = float(rng.randint(15, 40)) if kind in ("DDrppi", "wp") else 0.0
    # no dearer than the listed calls: expected pairs in range below 2e10
    while n1 * (n2 or n1) * (rmax / box) ** 2 * (max(rmax, pimax) / box) * 4.2 > 2e10:
        n1, n2 = max(2, n1 // 2), n2 // 2
    return _case(None, kind, place, n1, n2, dtype, box, sample, 0.1 if kind != "DDsmu" else 1.0, rmax, nbins,
                 log=kind != "DDsmu", avg=avg, weights=weights,
                 periodic=kind in ("xi", "wp") or rng.random() < 0.7, pimax=pimax,
                 nmu=rng.randint(5, 60) if kind == "DDsmu" else 0)


# ------------------------------------------------------------------ catalogs
def _fold(p, box, dtype):
    p = np.mod(p, box).astype(dtype)
    p[p >= dtype.type(box)] = 0
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


def _nfw_radius(u, conc):
    """r / r_scale with NFW enclosed mass fraction u, from a table of the mass profile."""
    x = np.linspace(0.0, 15.0, 4096)
    m = np.log1p(x) - x / (1.0 + x)
    return np.interp(u * np.interp(conc, x, m), m, x)


def _points(sample, n, box, dtype, rng):
    dtype = np.dtype(dtype)
    real = np.float32 if dtype.itemsize == 4 else np.float64
    if sample == "clumps":
        k = rng.integers(0, max(1, n // PER_CLUMP), n)
        parents = rng.uniform(0, box, (max(1, n // PER_CLUMP), 3)).astype(real)
        p = rng.standard_normal((n, 3), dtype=real)
        p *= real(SIGMA)
        p += parents[k]
        return _fold(p, box, dtype)
    if sample == "halos":
        nh, nhalo = int(0.6 * n), max(1, n // 839)
        occ = rng.lognormal(0.0, 1.0, nhalo)
        occ = rng.multinomial(nh, occ / occ.sum())
        conc = rng.uniform(5.0, 15.0, nhalo)
        size = np.cbrt(np.maximum(occ, 1) * nhalo / max(nh, 1)) / conc
        k = np.repeat(np.arange(nhalo), occ)
        r = _nfw_radius(rng.random(nh), conc[k]) * size[k]
        v = rng.standard_normal((nh, 3), dtype=np.float32)
        v *= (r / np.maximum(np.sqrt((v * v).sum(1)), 1e-20))[:, None].astype(np.float32)
        p = np.empty((n, 3), dtype=real)
        p[:nh] = rng.uniform(0, box, (nhalo, 3))[k]
        p[:nh] += v
        p[nh:] = box * rng.random((n - nh, 3), dtype=real)
        return _fold(p, box, dtype)
    p = rng.random((n, 3), dtype=real)
    p *= real(box)
    return _fold(p, box, dtype)


def _sky(n, rng):
    """RA, DEC (degrees) and cz (km/s): half uniform over a survey window and in volume, half in clumps."""
    def window(m):
        return (rng.uniform(120.0, 240.0, m), np.degrees(np.arcsin(rng.uniform(0.0, math.sin(math.pi / 3), m))),
                np.cbrt(rng.uniform(3000.0 ** 3, 30000.0 ** 3, m)))
    nc, nclump = n // 2, max(1, n // 333)
    ra, dec, cz = window(n)
    cra, cdec, ccz = window(nclump)
    k = rng.integers(0, nclump, nc)
    ra[:nc] = np.clip(cra[k] + rng.normal(0, 0.15, nc), 120.0, 240.0)
    dec[:nc] = np.clip(cdec[k] + rng.normal(0, 0.15, nc), 0.0, 60.0)
    cz[:nc] = np.clip(ccz[k] + rng.normal(0, 200.0, nc), 3000.0, 30000.0)
    return [ra, dec, cz]


def _catalogs(case, seed):
    """[(coordinates, weights or None), ...]: the one or two catalogs of a call, or those of a batch."""
    rng = np.random.default_rng([SEED, seed])
    real = np.float32 if case["dtype"] == "f4" else np.float64

    def one(n, sample):
        x = _sky(n, rng) if sample == "sky" else _points(sample, n, case["box"], case["dtype"], rng)
        return x, (rng.uniform(0.5, 1.5, n).astype(real) if case["weights"] else None)
    if case["kind"] == "batch":
        sizes = np.rint(np.exp(rng.uniform(math.log(case["n1"]), math.log(case["n2"]), case["ncat"]))).astype(int)
        # the sizes' mean square, which sets the pairs, does not depend on the seed
        lo, hi = case["n1"], case["n2"]
        want = (hi * hi - lo * lo) / (2 * math.log(hi / lo))
        sizes = np.clip(np.rint(sizes * math.sqrt(want / np.mean(sizes.astype(float) ** 2))).astype(int), 2, None)
        return [one(int(n), "uniform") for n in sizes]
    cats = [one(case["n1"], case["sample"])]
    if case["n2"]:
        # the second catalog of a box is its randoms; of the sky, a second survey
        cats.append(one(case["n2"], "sky" if case["sample"] == "sky" else "uniform"))
    return cats


def _edges(case):
    if case["log"]:
        return np.logspace(math.log10(case["rmin"]), math.log10(case["rmax"]), case["nbins"] + 1)
    return np.linspace(case["rmin"], case["rmax"], case["nbins"] + 1)


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    cats = _catalogs(case, seed)
    if case["place"] == "device":
        cats = [([_lib.DeviceArray(a) for a in x], _lib.DeviceArray(w) if w is not None else None) for x, w in cats]
    state = {"case": case, "cats": cats, "edges": _edges(case)}
    if case["place"] == "device" and case["kind"] != "batch":
        state["bins"] = _BinFile(state["edges"])
    return state


class _BinFile:
    """The bin file that a C caller names in each call."""

    def __init__(self, edges):
        self.path = _abi.write_bin_file(edges)[0]

    def __del__(self):
        try:
            os.remove(self.path)
        except Exception:
            pass


def _host_call(s):
    c, (x, w) = s["case"], s["cats"][0]
    y, v = s["cats"][1] if len(s["cats"]) > 1 else ([None] * 3, None)
    auto, kw = int(not c["n2"]), {}
    if c["weights"]:
        kw["weight_type"] = "pair_product"
    if c["kind"] in ("xi", "wp"):
        if c["weights"]:
            kw["weights"] = w
        if c["kind"] == "xi":
            r = theory.xi(c["box"], THREADS, s["edges"], *x, output_ravg=c["avg"], **kw)
            return {"xi": r["xi"], "avg": r["ravg"], "npairs": r["npairs"].astype(np.int64), "weightavg": r["weightavg"]}
        r = theory.wp(c["box"], c["pimax"], THREADS, s["edges"], *x, output_rpavg=c["avg"], **kw)
        return {"wp": r["wp"], "avg": r["rpavg"], "npairs": r["npairs"].astype(np.int64), "weightavg": r["weightavg"]}
    if c["weights"]:
        kw.update(weights1=w, weights2=v)
    if c["kind"] in ("DDrppi_mocks", "DDsmu_mocks"):
        kw.update(RA2=y[0], DEC2=y[1], CZ2=y[2])
        if c["kind"] == "DDrppi_mocks":
            r = mocks.DDrppi_mocks(auto, 1, THREADS, c["pimax"], s["edges"], *x, output_rpavg=c["avg"], **kw)
        else:
            r = mocks.DDsmu_mocks(auto, 1, THREADS, 1.0, c["nmu"], s["edges"], *x, output_savg=c["avg"], **kw)
    else:
        kw.update(X2=y[0], Y2=y[1], Z2=y[2], periodic=c["periodic"], boxsize=c["box"] if c["periodic"] else None)
        if c["kind"] == "DD":
            r = theory.DD(auto, THREADS, s["edges"], *x, output_ravg=c["avg"], **kw)
        elif c["kind"] == "DDrppi":
            r = theory.DDrppi(auto, THREADS, c["pimax"], s["edges"], *x, output_rpavg=c["avg"], **kw)
        else:
            r = theory.DDsmu(auto, THREADS, s["edges"], 1.0, c["nmu"], *x, output_savg=c["avg"], **kw)
    name = [n for n in r.dtype.names if n.endswith("avg") and n != "weightavg"][0]
    return {"avg": r[name], "npairs": r["npairs"].astype(np.int64), "weightavg": r["weightavg"]}


_ENTRY = {"DD": "countpairs", "DDrppi": "countpairs_rp_pi", "DDsmu": "countpairs_s_mu", "xi": "countpairs_xi",
          "wp": "countpairs_wp"}


def _options(c):
    return _abi.make_options(periodic=c["periodic"], boxsize=c["box"] if c["periodic"] else None,
                             need_avg_sep=c["avg"], float_type=4 if c["dtype"] == "f4" else 8)


def _device_call(s):
    c, (x, w) = s["case"], s["cats"][0]
    mode, lib = _ENTRY[c["kind"]], _lib.lib()
    o, e = _options(c), _abi.get_extra_options(_abi.WEIGHT_PAIR_PRODUCT if c["weights"] else _abi.WEIGHT_NONE)
    args = [c["n1"]] + [ctypes.c_void_p(a.ptr) for a in x]
    if w is not None:
        e.weights0.weights[0] = w.ptr
    if c["kind"] in ("xi", "wp"):
        args += [c["box"], THREADS, s["bins"].path.encode()]
    else:
        if c["n2"]:
            y, v = s["cats"][1]
            args += [c["n2"]] + [ctypes.c_void_p(a.ptr) for a in y] + [THREADS, 0]
            if v is not None:
                e.weights1.weights[0] = v.ptr
        else:
            args += [0, None, None, None, THREADS, 1]
        args += [s["bins"].path.encode()]
    if c["kind"] in ("DDrppi", "wp"):
        args += [c["pimax"]]
    if c["kind"] == "DDsmu":
        args += [1.0, c["nmu"]]
    res = _abi._RES[mode]()
    if getattr(lib, mode)(*args, ctypes.byref(res), ctypes.byref(o), ctypes.byref(e)) != 0:
        raise RuntimeError("%s failed" % mode)
    r = _abi._collect(mode, res)
    getattr(lib, _abi._FREE[mode])(ctypes.byref(res))
    out = {"avg": r["ravg"], "npairs": r["npairs"].astype(np.int64), "weightavg": r["weightavg"]}
    if c["kind"] in ("xi", "wp"):
        out[c["kind"]] = r[c["kind"]]
    n, m = r["nbin"], r.get("npibin", r.get("nmu_bins", 0))
    if m:
        return {k: np.ascontiguousarray(a.reshape(n + 1, m + 1)[1:n, :m]).reshape(-1) for k, a in out.items()}
    return {k: a[1:n] for k, a in out.items()}


def run(state):
    c = state["case"]
    if c["kind"] == "batch":
        cats = state["cats"]
        res = _lib.countpairs_batch([tuple(x) for x, _ in cats], state["edges"], options=_options(c),
                                    weights=[w for _, w in cats] if c["weights"] else None, nthreads=THREADS)
        return {"avg": np.stack([r["ravg"][1:] for r in res]), "weightavg": np.stack([r["weightavg"][1:] for r in res]),
                "npairs": np.stack([r["npairs"][1:].astype(np.int64) for r in res])}
    return _host_call(state) if c["place"] == "host" else _device_call(state)


# ------------------------------------------------------------------ what a pass cannot do without
def _pairs_in_range(case):
    """Expected pairs that are counted (each once)."""
    kind, reach = case["kind"], case["pimax"]
    if case["sample"] == "sky":
        volume = (math.pi / 180 * 120) * math.sin(math.pi / 3) / 3 * 280.0 ** 3
    else:
        volume = case["box"] ** 3
    r = case["rmax"]
    shell = 2 * math.pi * r * r * reach if reach else 4.0 / 3.0 * math.pi * r ** 3
    if kind == "batch":
        lo, hi = case["n1"], case["n2"]
        return case["ncat"] * (hi * hi - lo * lo) / (2 * math.log(hi / lo)) / 2 * min(1.0, shell / volume)
    n = float(case["n1"])
    if case["n2"]:
        return n * case["n2"] * min(1.0, shell / volume)
    own = {"clumps": PER_CLUMP, "halos": 503 * 0.36 * math.e, "sky": 166 * 0.25}.get(case["sample"], 0.0)
    return n / 2 * (n * min(1.0, shell / volume) + min(own, n))


def work(case):
    if case["kind"] == "batch":
        points = case["ncat"] * (case["n2"] - case["n1"]) / math.log(case["n2"] / case["n1"])
    else:
        points = case["n1"] + case["n2"]
    size = 4 if case["dtype"] == "f4" else 8
    slots = case["nbins"] * max(1, int(case["pimax"]) if case["kind"].startswith("DDrppi") else case["nmu"]) * case["ncat"]
    # a counted pair: the squared separation (8), the separation's root and sum (2), the weight's product and sum (2)
    flops = 8 + (2 if case["avg"] else 0) + (2 if case["weights"] else 0)
    return {"bytes": float(points * size * (4 if case["weights"] else 3) + 24 * slots),
            "flops": float(flops * _pairs_in_range(case))}


# ------------------------------------------------------------------ the same in plain torch, 64 bits
def _distances(cz):
    """Comoving distance (Mpc/h), flat with Omega_m = 0.25, linear between multiples of 1e-4 in z."""
    z = cz / C_KM_S
    n = int(z.max() * 10000) + 102
    t, wt = np.polynomial.legendre.leggauss(5)
    lo = np.arange(n) * 1e-4
    zz = lo[:, None] + 0.5e-4 * (t[None, :] + 1.0)
    seg = (wt[None, :] / np.sqrt(0.25 * (1 + zz) ** 3 + 0.75)).sum(1) * 0.5e-4
    d = np.concatenate([[0.0], np.cumsum(seg)]) * C_KM_S * 0.01
    return np.interp(z, np.arange(n + 1) * 1e-4, d)


def _xyz(case, x):
    if case["sample"] != "sky":
        return np.stack([a.astype(np.float64) for a in x], 1)
    ra, dec, d = np.radians(x[0]), np.radians(x[1]), _distances(x[2])
    return np.stack([d * np.cos(dec) * np.cos(ra), d * np.cos(dec) * np.sin(ra), d * np.sin(dec)], 1)


def _slots(case, p, q, d, e2):
    """(slot, squared separation to be averaged, kept) of pairs at p and q with separation d; slots 0.. as the results lie."""
    kind = case["kind"]
    r2 = (d * d).sum(1)
    key, col, m = r2, None, 1
    if kind in ("DDrppi", "wp"):
        key, par = d[:, 0] ** 2 + d[:, 1] ** 2, d[:, 2].abs()
        ok = par < case["pimax"]
        if kind == "DDrppi":
            m = int(case["pimax"])
            col = (par * (m / case["pimax"])).long()
    elif kind == "DDsmu":
        m = case["nmu"]
        mu = (d[:, 2] ** 2 / r2).sqrt()
        ok, col = mu < 1.0, (mu * m).long()
    elif kind in ("DDrppi_mocks", "DDsmu_mocks"):
        line = p + q
        dot2, l2 = (d * line).sum(1) ** 2, (line * line).sum(1)
        if kind == "DDrppi_mocks":
            par2 = dot2 / l2
            m = int(case["pimax"])
            ok, col, key = par2 < case["pimax"] ** 2, (par2.sqrt() * (m / case["pimax"])).long(), r2 - par2
        else:
            mu = (dot2 / (l2 * r2)).sqrt()
            m = case["nmu"]
            ok, col = mu < 1.0, (mu * m).long()
    else:
        ok = torch.ones_like(r2, dtype=torch.bool)
    k = torch.searchsorted(e2, key, right=True) - 1
    ok = ok & (key >= e2[0]) & (key < e2[-1])
    return (k if col is None else k * m + col.clamp(max=m - 1)), key, ok


def _sums(case, p1, w1, p2, w2, limit):
    """Counts, sums of separations and of weight products over all ordered pairs; None beyond `limit` candidates."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    auto = p2 is None
    a = torch.from_numpy(p1).to(dev)
    b = a if auto else torch.from_numpy(p2).to(dev)
    wa = torch.from_numpy(w1.astype(np.float64)).to(dev) if w1 is not None else None
    wb = wa if auto else (torch.from_numpy(w2.astype(np.float64)).to(dev) if w2 is not None else None)
    e2 = torch.from_numpy(_edges(case) ** 2).to(dev)
    box = case["box"] if case["periodic"] else 0.0
    rxy = case["rmax"] if case["sample"] != "sky" else math.hypot(case["rmax"], case["pimax"])
    rz = case["pimax"] if case["kind"] in ("DDrppi", "wp") else rxy
    lo = torch.minimum(a.amin(0), b.amin(0)) if not box else torch.zeros(3, dtype=torch.float64, device=dev)
    span = (torch.maximum(a.amax(0), b.amax(0)) - lo).tolist() if not box else [box] * 3
    nx, ny = [max(1, min(512, int(s / (rxy * (1 + 1e-9))))) for s in span[:2]]

    def column(t):
        ix = ((t[:, 0] - lo[0]) * (nx / span[0])).long().clamp(0, nx - 1)
        iy = ((t[:, 1] - lo[1]) * (ny / span[1])).long().clamp(0, ny - 1)
        return ix, iy
    big = 8.0 * (span[2] + rz)
    bx, by = column(b)
    kb, order = torch.sort((bx * ny + by) * big + (b[:, 2] - lo[2]) + rz)
    sb = b[order]
    ax, ay = column(a)
    m = {"DDrppi": int(case["pimax"]), "DDrppi_mocks": int(case["pimax"]), "DDsmu": case["nmu"],
         "DDsmu_mocks": case["nmu"]}.get(case["kind"], 1)
    n = case["nbins"] * m
    out = [torch.zeros(n, dtype=torch.float64, device=dev) for _ in range(3)]
    ranges, total = [], 0
    for ox in sorted({o % nx for o in (-1, 0, 1)} if box else {-1, 0, 1}):
        for oy in sorted({o % ny for o in (-1, 0, 1)} if box else {-1, 0, 1}):
            cx, cy = ax + ox, ay + oy
            if box:
                cx, cy = cx % nx, cy % ny
                live = torch.ones_like(cx, dtype=torch.bool)
            else:
                live = (cx >= 0) & (cx < nx) & (cy >= 0) & (cy < ny)
            base = (cx * ny + cy) * big + (a[:, 2] - lo[2]) + rz
            for shift in ((-box, 0.0, box) if box else (0.0,)):
                z = (a[:, 2] - lo[2]) + shift
                hit = live & (z > -rz * 1.001) & (z < span[2] + rz * 1.001)
                first = torch.searchsorted(kb, base + (shift - rz * (1 + 1e-9)))
                last = torch.searchsorted(kb, base + (shift + rz * (1 + 1e-9)))
                count = torch.where(hit, last - first, torch.zeros_like(first))
                total += int(count.sum())
                if total > limit:
                    return None
                ranges.append((first, count))
    for first, count in ranges:
        ends = torch.cumsum(count, 0)
        done, n_all = 0, int(ends[-1]) if len(ends) else 0
        while done < n_all:
            # primaries whose candidates fit one chunk
            i0 = int(torch.searchsorted(ends, done, right=True))
            i1 = max(i0 + 1, int(torch.searchsorted(ends, done + 40_000_000, right=True)))
            cnt = count[i0:i1]
            i = torch.repeat_interleave(torch.arange(i0, i1, device=dev), cnt)
            start = ends[i0:i1] - cnt - done
            j = first[i] + torch.arange(len(i), device=dev) - torch.repeat_interleave(start, cnt)
            done = int(ends[i1 - 1])
            d = sb[j] - a[i]
            if box:
                d -= box * torch.round(d / box)
            near = (d[:, 0].abs() < rxy) & (d[:, 1].abs() < rxy) & (d[:, 2].abs() < rz)
            if auto:
                near &= order[j] != i
            i, j, d = i[near], j[near], d[near]
            slot, key, ok = _slots(case, a[i], sb[j], d, e2)
            slot, key = slot[ok], key[ok]
            out[0] += torch.bincount(slot, minlength=n)
            out[1] += torch.bincount(slot, weights=key.sqrt(), minlength=n)
            if wa is not None:
                out[2] += torch.bincount(slot, weights=wa[i[ok]] * wb[order[j[ok]]], minlength=n)
    return [t.cpu().numpy() for t in out]


def exact(case, seed):
    if _pairs_in_range(case) > 3e9:
        return None
    cats, tables = _catalogs(case, seed), []
    pairs = [(c, None) for c in cats] if case["kind"] == "batch" else [(cats[0], cats[1] if len(cats) > 1 else None)]
    for one, two in pairs:
        s = _sums(case, _xyz(case, one[0]), one[1], _xyz(case, two[0]) if two else None, two[1] if two else None, 3e10)
        if s is None:
            return None
        count, sep, wgt = s
        some = np.maximum(count, 1)
        t = {"avg": sep / some if case["avg"] else 0 * sep, "npairs": count.astype(np.int64),
             "weightavg": wgt / some if case["weights"] else 0 * wgt}
        if case["kind"] in ("xi", "wp"):
            e, box, n = _edges(case), case["box"], case["n1"]
            tot = float(one[1].astype(np.float64).sum()) if case["weights"] else float(n)
            density = tot * (tot - tot / n) / box ** 3
            pairs_w = wgt if case["weights"] else count
            if case["kind"] == "xi":
                t["xi"] = pairs_w / (density * 4.0 / 3.0 * math.pi * (e[1:] ** 3 - e[:-1] ** 3)) - 1.0
            else:
                depth = 2.0 * case["pimax"]
                t["wp"] = (pairs_w / (density * math.pi * (e[1:] ** 2 - e[:-1] ** 2) * depth) - 1.0) * depth
        tables.append(t)
    if case["kind"] == "batch":
        return {k: np.stack([t[k] for t in tables]) for k in tables[0]}
    return tables[0]
