"""The pair-count work that users of fcfc_amd run, as cases that can be timed.

Each case is one pass through the public entry points (Engine.count_pairs,
Engine.count_batch, xi.WeightFitCounts with xi.xi_multipoles_torch) on seeded
synthetic catalogues of the kinds this repository measures itself on:
periodic boxes (uniform, or half uniform and half in Gaussian halos of 500
members) and survey caps (r in [1000, 2000) Mpc/h, |RA| and |Dec| <= 30 deg,
FKP weights).  Lengths are in Mpc/h.

Fields of a case
  kind    "count": one histogram; "mocks": a batch of DD, DR and RR of many
          boxes and their multipoles; "fit": one step of weight fitting,
          forward and backward
  geom    "box" (side L, periodic) or "survey"
  bins    "iso", "smu" (nmu mu bins) or "spi" (pi bins of 1/40 of pmax)
  edges   "lin": 40 equal bins in [0, smax); "log": 24 logarithmic bins in
          [smax / 400, smax), whose squared edges are no integers
  n1, n2  objects; n2 = 0: auto pairs of the first catalogue
  prec    the form of the count ("fp64" or "fp32")
  weighted, clustered, host: per-object weights; halos; catalogues in host
          memory, as read from a file, instead of on the GPU
"""
import math

import numpy as np
import torch

import fcfc_amd as F
from fcfc_amd.xi import WeightFitCounts, multipoles, xi_multipoles_torch

_NS = {"lin": 40, "log": 24}
_NP = 40
_BIN = {"iso": F.BIN_ISO, "smu": F.BIN_SMU, "spi": F.BIN_SPI}
_RMIN, _RMAX = 1000.0, 2000.0
# operations per pair: the separation (and mu or pi) arithmetic alone
_FLOPS = {("box", "iso"): 8, ("box", "smu"): 10, ("box", "spi"): 6,
          ("survey", "iso"): 8, ("survey", "smu"): 14, ("survey", "spi"): 13}


def _case(kind="count", geom="box", bins="smu", edges="lin", smax=200.0, pmax=0.0, nmu=1,
          L=1000.0, n1=0, n2=0, weighted=False, clustered=False, host=False, prec="fp64",
          nmock=0, name=None):
    c = dict(kind=kind, geom=geom, bins=bins, edges=edges, smax=smax, pmax=pmax, nmu=nmu, L=L,
             n1=n1, n2=n2, weighted=weighted, clustered=clustered, host=host, prec=prec,
             nmock=nmock)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one jackknife patch or halo sample, read from a file
        _case(name="patch_iso", bins="iso", n1=2000, host=True),
        # the 1e5-object box whose xi(s) is the usual first measurement, from host arrays
        _case(name="box_iso_1e5", bins="iso", n1=100000, host=True),
        # DD of a weighted galaxy sample for redshift-space multipoles
        _case(name="box_smu_dd", nmu=100, n1=500123, weighted=True, clustered=True),
        # the DR of such a sample against ten times as many randoms
        _case(name="box_smu_dr", nmu=100, n1=200000, n2=2000000, weighted=True, clustered=True),
        # RR of a large box, the largest single count of an analysis
        _case(name="box_smu_rr", nmu=100, n1=4000000),
        # the same at an odd size in the FP32 form with FP64 re-evaluation
        _case(name="box_smu_rr_fp32", nmu=100, n1=1500007, prec="fp32"),
        # projected clustering w_p: small scales, logarithmic s_perp bins, pi to 40
        _case(name="box_wp_log", bins="spi", edges="log", smax=40.0, pmax=40.0, n1=1000000,
              clustered=True),
        # small-scale cross-correlation of galaxies and matter particles, logarithmic bins
        _case(name="box_iso_log_cross", bins="iso", edges="log", smax=30.0, n1=300000, n2=1000003,
              weighted=True, clustered=True, prec="fp32"),
        # survey DR with FKP weights in (s_perp, pi)
        _case(name="survey_spi_dr", geom="survey", bins="spi", pmax=200.0, n1=30011, n2=1000000,
              weighted=True),
        # survey RR with FKP weights in (s, mu) for the multipoles
        _case(name="survey_smu_rr", geom="survey", nmu=100, n1=1200000, weighted=True, prec="fp32"),
        # covariance mocks: DD, DR, RR of 16 small boxes in one batched call
        _case(name="mocks_smu", kind="mocks", nmu=100, n1=2500, n2=25000, weighted=True,
              clustered=True, nmock=16),
        # one step of fitting object weights: counts by a prepared plan, and the gradient
        _case(name="fit_smu", kind="fit", nmu=100, n1=40000, n2=200000, weighted=True,
              clustered=True),
    ]


def draw(rng):
    """A case of the ranges above: sizes log-uniform, at most a few 1e10
    expected pairs (the largest listed case has 2.7e11)."""
    kind = rng.choice(["count"] * 8 + ["mocks", "fit"])
    if kind == "mocks":
        lo = int(math.exp(rng.uniform(math.log(1000), math.log(8000))))
        return _case(kind=kind, nmu=rng.choice([20, 100, 120]), n1=lo, n2=lo * rng.randint(2, 8),
                     weighted=True, clustered=True, nmock=rng.randint(4, 20),
                     prec=rng.choice(["fp64", "fp64", "fp32"]))
    if kind == "fit":
        n1 = int(math.exp(rng.uniform(math.log(5000), math.log(80000))))
        return _case(kind=kind, nmu=rng.choice([20, 100]), n1=n1, n2=n1 * rng.randint(2, 5),
                     weighted=True, clustered=True)
    geom = rng.choice(["box", "box", "survey"])
    bins = rng.choice(["iso", "smu", "smu", "spi"])
    edges = rng.choice(["lin", "lin", "log"])
    smax = float(rng.choice([80, 120, 160, 200])) if edges == "lin" else \
        round(rng.uniform(15.0, 60.0), 1)
    pmax = float(rng.choice([40, 80, 120, 200])) if bins == "spi" else 0.0
    c = _case(geom=geom, bins=bins, edges=edges, smax=smax, pmax=pmax,
              nmu=rng.choice([10, 60, 100, 120]) if bins == "smu" else 1,
              L=float(rng.choice([500, 1000, 1500])) if geom == "box" else 1000.0,
              weighted=rng.random() < 0.5 or geom == "survey",
              clustered=geom == "box" and rng.random() < 0.5, host=rng.random() < 0.2,
              prec=rng.choice(["fp64", "fp64", "fp32"]))
    cross = rng.random() < 0.5
    c["n1"] = int(math.exp(rng.uniform(math.log(2000), math.log(1000000))))
    c["n2"] = c["n1"] * rng.randint(2, 10) + rng.randint(0, 99) if cross else 0
    while _pairs(c) > 3e10 or c["n2"] > 4000000:
        c["n1"] = c["n1"] * 3 // 4
        c["n2"] = c["n2"] * 3 // 4
    return c


def _volume(c):
    if c["geom"] == "box":
        return c["L"] ** 3
    return (_RMAX ** 3 - _RMIN ** 3) / 3 * (math.pi / 3) * 1.0     # patch of 60 deg x 60 deg


def _pairs(c):
    """Pairs inside the binned range, as a uniform catalogue has them."""
    if c["bins"] == "spi":
        v = math.pi * c["smax"] ** 2 * 2 * c["pmax"]
    else:
        v = 4 / 3 * math.pi * c["smax"] ** 3
    f = min(v / _volume(c), 1.0)
    n1, n2 = c["n1"], c["n2"]
    return f * (0.5 * n1 * n1 if n2 == 0 else float(n1) * n2)


def _mock_sizes(c):
    """nmock sizes spread evenly over the logarithm of [n1, n2]."""
    m = c["nmock"]
    return [int(c["n1"] * (c["n2"] / c["n1"]) ** (k / max(1, m - 1))) for k in range(m)]


def work(c):
    fl = _FLOPS[c["geom"], c["bins"]] + (2 if c["weighted"] else 0)
    per = 32 if c["weighted"] else 24
    ntot = _NS[c["edges"]] * (c["nmu"] if c["bins"] == "smu" else _NP if c["bins"] == "spi" else 1)
    if c["kind"] == "count":
        return {"bytes": per * (c["n1"] + c["n2"]) + 8 * ntot, "flops": fl * _pairs(c)}
    if c["kind"] == "mocks":
        n, b = 0.0, 0.0
        for m in _mock_sizes(c):
            r = 5 * m
            n += sum(_pairs(dict(c, n1=x, n2=y)) for x, y in ((m, 0), (m, r), (r, 0)))
            b += 32 * m + 24 * r + 24 * ntot
        return {"bytes": b, "flops": fl * n}
    n = _pairs(dict(c, n2=0)) + _pairs(c)
    return {"bytes": 2 * (32 * c["n1"] + 32 * c["n2"]) + 12 * c["n1"], "flops": (2 * fl + 2) * n}


# ---- inputs -----------------------------------------------------------------
def _gen(seed, k):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + 7919 * k) % (1 << 62))
    return dict(generator=g, device="cuda", dtype=torch.float64)


def _points(c, seed, k, n, clustered):
    """(n, 3) positions in Mpc/h and n weights."""
    kw = _gen(seed, k)
    if c["geom"] == "survey":
        u = torch.rand((n, 3), **kw)
        r = (_RMIN ** 3 + (_RMAX ** 3 - _RMIN ** 3) * u[:, 0]) ** (1 / 3)
        ra, sd = (u[:, 1] - 0.5) * (math.pi / 3), u[:, 2] - 0.5
        cd = torch.sqrt(1 - sd * sd)
        p = torch.stack([r * cd * torch.cos(ra), r * cd * torch.sin(ra), r * sd], 1)
        nr = 3e-4 * torch.exp(-(r - 1500.0) ** 2 / (2 * 200.0 ** 2))
        return p, 1 / (1 + nr * 1e4)
    L = c["L"]
    if clustered:
        nh = max(1, n // 1000)
        nm = min(500, max(1, (n // 2) // nh))
        cen = torch.rand((nh, 1, 3), **kw) * L
        halo = (cen + 2.0 * torch.randn((nh, nm, 3), **kw)).reshape(-1, 3)
        p = torch.cat([torch.rand((n - nh * nm, 3), **kw) * L, halo])
        p = torch.remainder(p, L)
        p = torch.where(p >= L, p - L, p)
    else:
        p = torch.rand((n, 3), **kw) * L
    w = torch.exp(0.3 * torch.randn(n, **kw)).to(torch.float32).to(torch.float64)
    return p, w


def _log_edges(c):
    return np.geomspace(c["smax"] / 400, c["smax"], _NS["log"] + 1)


def _bins(c):
    geom = F.GEOM_BOX if c["geom"] == "box" else F.GEOM_SURVEY
    L = c["L"] if c["geom"] == "box" else None
    dpi = c["pmax"] / _NP if c["bins"] == "spi" else 1.0
    if c["edges"] == "lin":
        return F.Bins.linear(geom, _BIN[c["bins"]], 0.0, c["smax"], c["smax"] / _NS["lin"],
                             nmu=c["nmu"], pmin=0.0, pmax=c["pmax"], dpi=dpi, bsize=L)
    pe = np.arange(_NP + 1) * dpi if c["bins"] == "spi" else None
    return F.Bins.edges(geom, _BIN[c["bins"]], _log_edges(c), nmu=c["nmu"], pedges=pe, bsize=L)


def _catalog(b, p, w, host=False):
    if host:
        q = p.cpu().numpy()
        return F.Catalog(b, q[:, 0], q[:, 1], q[:, 2], None if w is None else w.cpu().numpy())
    q = p * b.rescale
    return F.Catalog(b, q[:, 0].contiguous(), q[:, 1].contiguous(), q[:, 2].contiguous(), w)


_ENG = []


def _engine():
    """The engine of the program: one for all its counts."""
    if not _ENG:
        _ENG.append(F.Engine())
    return _ENG[0]


def _mocks(c, seed):
    """(D positions, D weights, R positions) of every mock; R has five times
    as many objects and unit weights."""
    out = []
    for k, n in enumerate(_mock_sizes(c)):
        p, w = _points(c, seed, 2 * k, n, True)
        r, _ = _points(c, seed, 2 * k + 1, 5 * n, False)
        out.append((p, w, r))
    return out


def _target(seed):
    g = np.random.default_rng(int(seed) % (1 << 32))
    return torch.tensor(g.normal(0, 0.01, (2, _NS["lin"])), dtype=torch.float64, device="cuda")


def prepare(case, seed):
    c, eng, b = case, _engine(), _bins(case)
    if c["kind"] == "mocks":
        jobs, norm = [], []
        for p, w, r in _mocks(c, seed):
            D, R = _catalog(b, p, w), _catalog(b, r, None)
            jobs += [(D, None, True, True), (D, R, False, True), (R, None, True, False)]
            norm.append((D.sumw, R.n))
        return {"c": c, "eng": eng, "b": b, "jobs": jobs, "norm": norm}
    p, w = _points(c, seed, 0, c["n1"], c["clustered"])
    A = _catalog(b, p, w if c["weighted"] else None, c["host"])
    B = None
    if c["n2"]:
        q, v = _points(c, seed, 1, c["n2"], False)
        unit = c["geom"] == "box"              # box randoms carry no weights, survey ones FKP
        B = _catalog(b, q, v if c["weighted"] and not unit else None, c["host"])
    s = {"c": c, "eng": eng, "b": b, "A": A, "B": B}
    if c["kind"] == "fit":
        wd = w.to(torch.float32).requires_grad_(True)
        wr = torch.ones(c["n2"], dtype=torch.float64, device="cuda")
        D = F.Catalog(b, A.x, A.y, A.z)
        rr = eng.count_pairs(B, None, b, isauto=True).astype(np.float64)
        s.update(wd=wd, wr=wr, rr=torch.from_numpy(rr).cuda(), target=_target(seed),
                 fit=WeightFitCounts(eng, D, B, b))
        s["A"] = D
    return s


def run(s):
    c, eng, b = s["c"], s["eng"], s["b"]
    if c["kind"] == "count":
        return eng.count_pairs(s["A"], s["B"], b, isauto=s["B"] is None, withwt=c["weighted"],
                               precision=c["prec"])
    if c["kind"] == "mocks":
        res = eng.count_batch(s["jobs"], b, precision=c["prec"])
        dd, dr, rr = (np.stack(res[k::3]) for k in range(3))
        return {"dd": dd, "dr": dr, "rr": rr, "xi": _mock_poles(c, dd, dr, rr, s["norm"])}
    s["wd"].grad = None
    xi = xi_multipoles_torch(s["wd"], s["wr"], eng, s["A"], s["B"], b, rr_cnt=s["rr"],
                             poles=(0, 2), fit=s["fit"])
    ((xi - s["target"]) ** 2).sum().backward()
    return {"xi": xi.detach(), "grad": s["wd"].grad}


def _mock_poles(c, dd, dr, rr, norm):
    """Landy-Szalay xi_0,2,4 of every mock; bins without random pairs give 0."""
    sw = np.array([v[0] for v in norm])[:, None]
    nr = np.array([float(v[1]) for v in norm])[:, None]
    ddn, drn, rrn = dd * 2 / (sw * (sw - 1)), dr / (sw * nr), rr * 2 / (nr * (nr - 1))
    xi = np.where(rr > 0, (ddn - 2 * drn + rrn) / np.where(rr > 0, rrn, 1.0), 0.0)
    return multipoles(xi.reshape(len(norm), c["nmu"], _NS[c["edges"]]), c["nmu"], (0, 2, 4))


# ---- the same values by brute force in 64 bits ------------------------------
_MOST = 1.3e11        # pairs of objects that a brute-force value is computed for


def _each(c, p, q):
    """Yields (i, j, k, (i0, i1, j0)): pairs of p and q (of p with itself:
    each once) and their bin, for the pairs in range; i0 <= i < i1, j >= j0."""
    se = torch.arange(_NS["lin"] + 1, device="cuda", dtype=torch.float64) * (c["smax"] / _NS["lin"]) \
        if c["edges"] == "lin" else torch.from_numpy(_log_edges(c)).cuda()
    s2e, ns = se * se, _NS[c["edges"]]
    auto = q is None
    q = p if auto else q
    n, m = p.shape[0], q.shape[0]
    r2 = float(s2e[-1]) + (c["pmax"] ** 2 if c["bins"] == "spi" else 0.0)
    i0 = 0
    while i0 < n:
        j0 = i0 if auto else 0
        i1 = min(n, i0 + max(1, (1 << 25) // max(1, m - j0)))
        d2, dz = None, None
        for a in range(3):
            d = q[None, j0:, a] - p[i0:i1, a, None]
            if c["geom"] == "box":
                L = c["L"]
                d = torch.where(d > L / 2, d - L, torch.where(d < -L / 2, d + L, d))
            d2 = d * d if d2 is None else d2.addcmul_(d, d)
            dz = d if a == 2 and c["geom"] == "box" else None
        i, j = torch.nonzero(d2 < r2, as_tuple=True)
        s2 = d2[i, j]
        z2 = dz[i, j] ** 2 if dz is not None else None
        i, j = i + i0, j + j0
        if auto:
            keep = j > i
            i, j, s2 = i[keep], j[keep], s2[keep]
            z2 = z2[keep] if z2 is not None else None
        if z2 is None and c["bins"] != "iso":
            u, t = p[i], q[j]
            l = u + t
            z2 = ((u - t) * l).sum(1) ** 2 / (l * l).sum(1)
        t2 = s2 - z2 if c["bins"] == "spi" else s2
        k = torch.bucketize(t2, s2e, right=True) - 1
        if c["bins"] == "spi" and c["edges"] == "lin":
            k = torch.clamp(k, min=0)
        ok = (k >= 0) & (k < ns)
        if c["bins"] == "smu":
            mu = torch.floor(c["nmu"] * torch.sqrt(z2 / s2)).to(torch.int64)
            ok &= mu < c["nmu"]
            k = k + ns * mu
        elif c["bins"] == "spi":
            pe = torch.arange(_NP + 1, device="cuda", dtype=torch.float64) * (c["pmax"] / _NP)
            pk = torch.bucketize(torch.sqrt(z2), pe, right=True) - 1
            ok &= pk < _NP
            k = k + ns * pk
        yield i[ok], j[ok], k[ok], (i0, i1, j0)
        i0 = i1


def _count(c, p, q, w, v):
    """The histogram of the pairs; w, v: weights (None: whole counts)."""
    ntot = _NS[c["edges"]] * (c["nmu"] if c["bins"] == "smu" else _NP if c["bins"] == "spi" else 1)
    h = torch.zeros(ntot, device="cuda", dtype=torch.int64 if w is None else torch.float64)
    v = w if q is None else v
    for i, j, k, _ in _each(c, p, q):
        h += torch.bincount(k, minlength=ntot) if w is None else \
            torch.bincount(k, weights=w[i] * v[j], minlength=ntot)
    return h


def _grad(c, p, q, w, v, g):
    """d(sum_k g_k count_k)/dw of the first catalogue."""
    out = torch.zeros_like(w)
    auto = q is None
    v = w if auto else v
    for i, j, k, (i0, i1, j0) in _each(c, p, q):
        m = torch.zeros((i1 - i0, len(v) - j0), device="cuda", dtype=torch.float64)
        m[i - i0, j - j0] = g[k]
        out[i0:i1] += m @ v[j0:]
        if auto:
            out[j0:] += m.T @ w[i0:i1]
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "mocks":
        if sum(18.0 * m * m for m in _mock_sizes(c)) > _MOST:
            return None
        hs, norm = [], []
        for p, w, r in _mocks(c, seed):
            one = torch.ones(r.shape[0], device="cuda", dtype=torch.float64)
            hs.append([_count(c, p, None, w, None), _count(c, p, r, w, one),
                       _count(c, r, None, None, None)])
            norm.append((float(w.sum()), r.shape[0]))
        dd, dr, rr = (np.stack([h[k].cpu().numpy() for h in hs]) for k in range(3))
        sw = np.array([v[0] for v in norm])[:, None]
        nr = np.array([float(v[1]) for v in norm])[:, None]
        ddn, drn, rrn = dd * 2 / (sw * (sw - 1)), dr / (sw * nr), rr * 2 / (nr * (nr - 1))
        xi = np.where(rr > 0, (ddn - 2 * drn + rrn) / np.where(rr > 0, rrn, 1.0), 0.0)
        xi = xi.reshape(len(norm), c["nmu"], _NS[c["edges"]])
        mu = (np.arange(c["nmu"]) + 0.5) / c["nmu"]
        leg = [np.ones_like(mu), (3 * mu ** 2 - 1) / 2, (35 * mu ** 4 - 30 * mu ** 2 + 3) / 8]
        po = np.stack([(2 * l + 1) / c["nmu"] * (xi * q[None, :, None]).sum(1)
                       for l, q in zip((0, 2, 4), leg)], 1)
        return {"dd": dd, "dr": dr, "rr": rr, "xi": po}
    n1, n2 = float(c["n1"]), float(c["n2"])
    cost = n1 * n2 if n2 else 0.5 * n1 * n1
    if c["kind"] == "fit":
        cost = 2 * (n1 * n2 + 0.5 * n1 * n1) + 0.5 * n2 * n2
    if cost > _MOST:
        return None
    p, w = _points(c, seed, 0, c["n1"], c["clustered"])
    q = v = None
    if c["n2"]:
        q, v = _points(c, seed, 1, c["n2"], False)
        if c["geom"] == "box":
            v = torch.ones_like(v)
    if c["kind"] == "count":
        return _count(c, p, q, w if c["weighted"] else None, v).cpu().numpy()
    w = w.to(torch.float32).to(torch.float64)
    dd = _count(c, p, None, w, None).requires_grad_(True)
    dr = _count(c, p, q, w, v).requires_grad_(True)
    rr = _count(c, q, None, None, None).to(torch.float64)
    wl = w.clone().requires_grad_(True)
    sw, nr = wl.sum(), n2
    rrn = 2 * rr / (nr * (nr - 1))
    safe = torch.where(rr > 0, rrn, torch.ones_like(rrn))
    x = torch.where(rr > 0, (2 * dd / (sw * (sw - 1)) - 2 * dr / (sw * nr) + rrn) / safe,
                    torch.zeros_like(rrn)).reshape(c["nmu"], -1)
    mu = (torch.arange(c["nmu"], dtype=torch.float64, device="cuda") + 0.5) / c["nmu"]
    xi = torch.stack([(x * (1 / c["nmu"])).sum(0),
                      (x * (5 / c["nmu"] * (1.5 * mu * mu - 0.5))[:, None]).sum(0)])
    ((xi - _target(seed)) ** 2).sum().backward()
    g = wl.grad + _grad(c, p, None, w, None, dd.grad) + _grad(c, p, q, w, v, dr.grad)
    return {"xi": xi.detach(), "grad": g}
