"""The workloads this library is timed on, each through its public entry points.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw()`
more of the same ranges, `prepare()` what a program holds before the call,
`run()` one call, `work()` the operations and bytes the call cannot do without
and `exact()` its result in plain FP64 torch.

Kinds of call:
  loglik    one log-likelihood evaluation of a problem that stays on the GPU
            (a step of a maximum-likelihood fit)
  batch     one evaluation each of several small regions at once
  predict   kriging of new locations with the factor of the last evaluation
  generate  synthetic observations z = L(theta) e
  serve     a burst of requests (evaluations and kriging) to the server
"""
import math

import numpy as np
import torch

import exageostatcpp_amd as egs
from exageostatcpp_amd import capi

EARTH_KM = 6371.0
SERVE_DTS = 384        # the tile size the serving benchmark registers its regions with
PREDICT_POINTS = 100   # new locations of a served kriging request


def _loglik(name, n, dts, sigma2, rng, nu, plan="fp64", dim=2):
    return {"name": name, "kind": "loglik", "kernel": "univariate", "plan": plan, "dim": dim, "n": n, "dts": dts,
            "sigma2": sigma2, "range": rng, "nu": nu}


def listed():
    return [
        # the smallest regions users fit or serve: launches and latency
        _loglik("fp64_n400", 400, 320, 1.0, 0.1, 0.5),
        # the exponential field of the maximum-likelihood tests (40 x 40 grid, tiles of 320)
        _loglik("fp64_n1600", 1600, 320, 1.0, 0.1, 0.5),
        # a mid-size served region, ragged, at a smoothness a fit passes through (K_nu of general order)
        _loglik("fp64_n10007_nu0.83", 10007, 384, 1.3, 0.07, 0.83),
        # the size of the host comparison in the benchmark
        _loglik("fp64_n20000", 20000, 960, 1.0, 0.05, 0.5),
        # the smooth-field workflow (200 x 200 grid, K_1)
        _loglik("fp64_n40000_nu1", 40000, 960, 1.0, 0.1, 1.0),
        # the bivariate field on the sphere, great-circle distance, odd number of locations
        {"name": "bivariate_gcd_n9001", "kind": "loglik", "kernel": "bivariate", "plan": "fp64", "dim": 2, "n": 9001,
         "dts": 960, "sigma2": 1.0, "sigma2b": 1.0, "range": 637.1, "nu": 0.5, "nub": 1.0, "rho": 0.5},
        # mixed plan at a general smoothness, ragged, mid-size: a step of a mixed fit
        _loglik("mixed_n45001_nu0.55", 45001, 960, 1.2, 0.06, 0.55, plan="mixed"),
        # the headline evaluation: mixed plan at 100,000 locations
        _loglik("mixed_n100000", 100000, 960, 1.0, 0.05, 0.5, plan="mixed"),
        # many small regions evaluated together
        {"name": "batch_24", "kind": "batch", "regions": 24, "nmin": 500, "nmax": 3000, "dts": SERVE_DTS},
        # kriging of 1,000 held-out locations after a fit
        {"name": "predict_n20000", "kind": "predict", "n": 20000, "dts": 960, "targets": 1000, "sigma2": 1.0,
         "range": 0.1, "nu": 1.0},
        # synthetic data for a simulation study
        {"name": "generate_n6001", "kind": "generate", "n": 6001, "dts": 960, "sigma2": 1.0, "range": 0.1, "nu": 0.5,
         "e_seed": 3},
        # a burst of requests to the server: evaluations of uneven regions, kriging on their factors
        {"name": "serve_16", "kind": "serve", "regions": 16, "nmin": 500, "nmax": 6000, "dts": SERVE_DTS,
         "workers": 4},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: sizes log-uniform, mostly odd."""
    theta = {"sigma2": round(rng.uniform(0.5, 2.0), 4), "range": round(rng.uniform(0.03, 0.15), 4),
             "nu": rng.choice([0.5, 1.5, round(rng.uniform(0.3, 1.3), 4), round(rng.uniform(0.3, 1.3), 4)])}
    u = rng.random()
    if u < 0.45:
        n = _log_uniform(rng, 400, 40000)
        dim = 3 if rng.random() < 0.15 else 2
        return dict({"kind": "loglik", "kernel": "univariate", "plan": "fp64", "dim": dim, "n": n,
                     "dts": rng.choice([320, 384, 960])}, **theta)
    if u < 0.55:
        return {"kind": "loglik", "kernel": "bivariate", "plan": "fp64", "dim": 2, "n": _log_uniform(rng, 400, 20000),
                "dts": rng.choice([320, 384, 960]), "sigma2": theta["sigma2"],
                "sigma2b": round(rng.uniform(0.5, 2.0), 4), "range": round(rng.uniform(300.0, 900.0), 1),
                "nu": 0.5, "nub": round(rng.uniform(0.6, 1.2), 4), "rho": round(rng.uniform(-0.5, 0.6), 3)}
    if u < 0.65:
        return _unnamed(_loglik("", _log_uniform(rng, 30000, 90000), 960, theta["sigma2"],
                                round(rng.uniform(0.04, 0.08), 4), rng.choice([0.5, round(rng.uniform(0.45, 0.6), 4)]),
                                plan="mixed"))
    if u < 0.75:
        return {"kind": "batch", "regions": rng.randint(4, 32), "nmin": 500, "nmax": rng.randint(1000, 4000),
                "dts": SERVE_DTS}
    if u < 0.86:
        return dict({"kind": "predict", "n": _log_uniform(rng, 1000, 30000), "dts": rng.choice([320, 384, 960]),
                     "targets": _log_uniform(rng, 100, 2000)}, **theta)
    if u < 0.93:
        return dict({"kind": "generate", "n": _log_uniform(rng, 1000, 20000), "dts": rng.choice([320, 384, 960]),
                     "e_seed": rng.randint(0, 1000)}, **theta)
    return {"kind": "serve", "regions": rng.randint(8, 24), "nmin": 500, "nmax": rng.randint(2000, 9000),
            "dts": SERVE_DTS, "workers": rng.choice([2, 4, 8])}


def _unnamed(case):
    del case["name"]
    return case


# ---- inputs -------------------------------------------------------------------

def _morton(cols):
    """Order of points by the interleaved bits of their 16-bit coordinates."""
    step = np.uint64(len(cols))
    code = np.zeros(len(cols[0]), dtype=np.uint64)
    for axis, c in enumerate(cols):
        q = np.round(c * 65535.0).astype(np.uint64)
        for b in range(16):
            code |= ((q >> np.uint64(b)) & np.uint64(1)) << (np.uint64(b) * step + np.uint64(axis))
    return np.argsort(code, kind="stable")


def _jittered_grid(r, n, dim):
    """n points, one per cell of a regular grid in the unit square (cube),
    jittered by up to 0.4 cells and Morton-ordered."""
    root = math.ceil(round(n ** (1.0 / dim), 9))
    cells = np.arange(n)
    cols = []
    for axis in range(dim):
        cols.append((cells // root ** (dim - 1 - axis) % root + 0.5 + r.uniform(-0.4, 0.4, n)) / root)
    order = _morton(cols)
    return [np.ascontiguousarray(c[order]) for c in cols]


def _sphere(r, n):
    """n points uniform on the sphere, latitude and longitude in degrees, Morton-ordered."""
    lat = np.degrees(np.arcsin(2.0 * r.random_sample(n) - 1.0))
    lon = 360.0 * r.random_sample(n) - 180.0
    order = _morton([(lon + 180.0) / 360.0, (lat + 90.0) / 180.0])
    return [np.ascontiguousarray(lat[order]), np.ascontiguousarray(lon[order])]


def _field(r, cols, rng, nu, features=2048):
    """A Matern field at the points (spectral sampling: frequencies follow the
    covariance's spectral density, a multivariate t with 2 nu degrees)."""
    dim = len(cols)
    w = r.standard_normal((dim, features)) / np.sqrt(r.chisquare(2.0 * nu, features)) / rng
    phase, amp = r.uniform(0.0, 2.0 * math.pi, features), r.standard_normal(features) * math.sqrt(2.0 / features)
    x, w, phase, amp = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (np.stack(cols, 1), w, phase, amp))
    out = [torch.cos(x[i:i + 16384] @ w + phase) @ amp for i in range(0, len(x), 16384)]
    return torch.cat(out).cpu().numpy()


def _theta(case):
    if case.get("kernel") == "bivariate":
        return [case["sigma2"], case["sigma2b"], case["range"], case["nu"], case["nub"], case["rho"]]
    return [case["sigma2"], case["range"], case["nu"]]


def _region(case, seed):
    """Locations, theta and observations of one problem."""
    r = np.random.RandomState((int(seed) * 7919 + 13) % (1 << 31))
    if case.get("kernel") == "bivariate":
        loc = _sphere(r, case["n"])
        lat, lon = np.radians(loc[0]), np.radians(loc[1])
        xyz = [EARTH_KM * np.cos(lat) * np.cos(lon), EARTH_KM * np.cos(lat) * np.sin(lon), EARTH_KM * np.sin(lat)]
        f, g = _field(r, xyz, case["range"], case["nu"]), _field(r, xyz, case["range"], case["nub"])
        z = np.empty(2 * case["n"])
        z[0::2] = math.sqrt(case["sigma2"]) * f
        z[1::2] = math.sqrt(case["sigma2b"]) * g
    else:
        loc = _jittered_grid(r, case["n"], case.get("dim", 2))
        z = math.sqrt(case["sigma2"]) * _field(r, loc, case["range"], case["nu"])
    return {"loc": loc, "theta": _theta(case), "z": z, "kernel": case.get("kernel", "univariate"), "rand": r}


def _regions(case, seed):
    """The uneven regions of a batch or a serving burst, each with its own theta."""
    r = np.random.RandomState((int(seed) * 104729 + 7) % (1 << 31))
    out = []
    for k in range(case["regions"]):
        n = int(round(math.exp(r.uniform(math.log(case["nmin"]), math.log(case["nmax"])))))
        one = {"n": n, "sigma2": r.uniform(0.5, 2.0), "range": r.uniform(0.03, 0.15),
               "nu": 0.5 if k % 4 == 0 else r.uniform(0.3, 1.3)}
        out.append(_region(one, int(seed) * 64 + k))
    return out


def _targets(region, m):
    return [np.ascontiguousarray(c) for c in region["rand"].random_sample((2, m))]


def _problem(ctx, case, region):
    loc = region["loc"]
    name = "BivariateMaternParsimonious" if region["kernel"] == "bivariate" else "UnivariateMaternStationary"
    p = egs.Problem(ctx, name, loc[0], loc[1], loc[2] if len(loc) == 3 else None,
                    metric=1 if region["kernel"] == "bivariate" else 0, dts=case["dts"])
    if case.get("plan") == "mixed":
        p.set_precision(egs.PRECISION_MIXED)
    p.set_observations(region["z"])
    return p


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        regions = _regions(case, seed)
        if kind == "batch":
            ctx = egs.Context(0)
            return {"kind": kind, "ctx": ctx, "thetas": [g["theta"] for g in regions],
                    "problems": [_problem(ctx, case, g) for g in regions]}
        server = capi.Server(0, hbm_budget_bytes=32 << 30, workers=case["workers"])
        ids = [server.add_region("UnivariateMaternStationary", g["loc"][0], g["loc"][1], g["z"], dts=case["dts"])
               for g in regions]
        return {"kind": kind, "server": server, "ids": ids, "thetas": [g["theta"] for g in regions],
                "targets": [_targets(g, PREDICT_POINTS) for g in regions[::4]]}
    region = _region(case, seed)
    ctx = egs.Context(0)
    p = _problem(ctx, case, region)
    state = {"kind": kind, "ctx": ctx, "p": p, "theta": region["theta"], "plan": case.get("plan", "fp64"),
             "e_seed": case.get("e_seed", 0)}
    if kind == "predict":
        state["targets"] = _targets(region, case["targets"])
        p.loglik(region["theta"])   # the fit's last evaluation: its factor stays on the GPU
    return state


def run(s):
    kind = s["kind"]
    if kind == "loglik":
        llh, logdet, quad = s["p"].loglik(s["theta"])
        if s["plan"] == "mixed":
            # log|Sigma| comes off a factor updated in 16 and 32 bits and carries
            # single precision; the refined quadratic form carries double
            return {"loglik": np.float32(llh), "logdet": np.float32(logdet), "quad": np.float64(quad)}
        return {"loglik": np.float64(llh), "logdet": np.float64(logdet), "quad": np.float64(quad)}
    if kind == "batch":
        return {"values": np.array(capi.loglik_batch(s["problems"], s["thetas"]))}
    if kind == "predict":
        return {"zmiss": s["p"].predict(s["theta"], *s["targets"])[0]}
    if kind == "generate":
        return {"z": s["p"].generate_observations(s["theta"], seed=s["e_seed"])}
    srv = s["server"]
    tickets = [srv.submit_loglik(i, th) for i, th in zip(s["ids"], s["thetas"])]
    krige = [srv.submit_predict(s["ids"][4 * k], s["thetas"][4 * k], *t) for k, t in enumerate(s["targets"])]
    llh = [srv.wait(t)[0] for t in tickets]
    return {"loglik": np.array(llh), "zmiss": np.concatenate([srv.wait(t)[1] for t in krige])}


# ---- floors ---------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        # sizes log-uniform in [nmin, nmax]: their mean n, n^2 and n^3
        a, b, k = float(case["nmin"]), float(case["nmax"]), case["regions"]
        mean = [(b ** q - a ** q) / (q * math.log(b / a)) for q in (1, 2, 3)]
        extra = PREDICT_POINTS * mean[0] * 20.0 * (k // 4) if kind == "serve" else 0.0
        return {"bytes": k * (24.0 * mean[0] + 24.0), "flops": k * (mean[2] / 3.0 + mean[1]) + extra}
    n = float(case["n"]) * (2 if case.get("kernel") == "bivariate" else 1)
    inputs = 8.0 * case.get("dim", 2) * case["n"] + 8.0 * n
    if kind == "predict":
        # the factor read once; both triangular solves; a covariance entry per target and location
        return {"bytes": 4.0 * n * n + inputs + 24.0 * case["targets"], "flops": 2.0 * n * n + 20.0 * n * case["targets"]}
    return {"bytes": inputs + (8.0 * n if kind == "generate" else 24.0), "flops": n ** 3 / 3.0 + n * n}


# ---- the same results in plain FP64 torch -----------------------------------------

def _matern(d, sigma2, nu, con):
    """con d^nu K_nu(d), sigma2 at d = 0; K_nu by the trapezoidal rule on its
    integral exp(-d cosh t) cosh(nu t)."""
    if nu in (0.5, 1.5):
        return sigma2 * torch.exp(-d) * ((1.0 + d) if nu == 1.5 else 1.0)
    dd = torch.where(d > 0.0, d, torch.ones_like(d))
    h, t_max = 1.0 / 7.0, math.acosh(1.0 + 800.0 / max(float(dd.min()), 1e-9))
    out = 0.5 * torch.exp(-dd)
    for i in range(1, int(min(t_max, 60.0) / h) + 1):
        # exp(nu t - d cosh t): the other half of cosh(nu t) beside it
        t = i * h
        out += torch.exp(dd * -math.cosh(t) + nu * t) * (0.5 * (1.0 + math.exp(-2.0 * nu * t)))
    out *= h * con
    out *= dd ** nu
    return torch.where(d > 0.0, out, torch.full_like(out, sigma2))


def _covariance(a, b, theta, kernel):
    """Covariance of the variables at the points a (rows) with those at b."""
    if kernel == "bivariate":
        s1, s2, rng, nu1, nu2, corr = theta
        nu12, g = 0.5 * (nu1 + nu2), math.gamma
        rho = corr * math.sqrt(g(nu1 + 1) * g(nu2 + 1) / (g(nu1) * g(nu2))) * g(nu12) / g(nu12 + 1)
        s12 = rho * math.sqrt(s1 * s2)
        la, lb = torch.deg2rad(a[0])[:, None], torch.deg2rad(b[0])[None]
        u = torch.sin((lb - la) * 0.5)
        v = torch.sin((torch.deg2rad(b[1])[None] - torch.deg2rad(a[1])[:, None]) * 0.5)
        d = 2.0 * EARTH_KM * torch.asin(torch.sqrt(u * u + torch.cos(la) * torch.cos(lb) * v * v)) / rng
        out = torch.empty((2 * len(a[0]), 2 * len(b[0])), dtype=torch.float64, device=d.device)
        for i, j, s, nu in ((0, 0, s1, nu1), (0, 1, s12, nu12), (1, 0, s12, nu12), (1, 1, s2, nu2)):
            out[i::2, j::2] = _matern(d, s, nu, s / (2.0 ** (nu - 1.0) * math.gamma(nu)))
        return out
    d2 = sum((p[:, None] - q[None]) ** 2 for p, q in zip(a, b))
    s, rng, nu = theta
    return _matern(torch.sqrt(d2) / rng, s, nu, s / (2.0 ** (nu - 1.0) * math.gamma(nu)))


def _factor(region):
    """The lower Cholesky factor of the region's covariance, blocked so that
    every product is a plain matrix product (upper part: rubbish)."""
    loc = [torch.from_numpy(c).cuda() for c in region["loc"]]
    kernel, p = region["kernel"], 2 if region["kernel"] == "bivariate" else 1
    n = p * len(loc[0])
    s = torch.empty((n, n), dtype=torch.float64, device="cuda")
    rows = max(1, 20_000_000 // n)
    for i in range(0, len(loc[0]), rows):
        hi = min(i + rows, len(loc[0]))
        s[p * i:p * hi, :p * hi] = _covariance([c[i:hi] for c in loc], [c[:hi] for c in loc], region["theta"], kernel)
    nb = 2048
    for k in range(0, n, nb):
        e = min(k + nb, n)
        dia = torch.linalg.cholesky(torch.tril(s[k:e, k:e]) + torch.tril(s[k:e, k:e], -1).T)
        s[k:e, k:e] = dia
        if e < n:
            pan = torch.linalg.solve_triangular(dia, s[e:, k:e].T.contiguous(), upper=False).T.contiguous()
            s[e:, k:e] = pan
            for j in range(e, n, 2 * nb):
                f = min(j + 2 * nb, n)
                s[j:, j:f] -= pan[j - e:] @ pan[j - e:f - e].T
    return s


def _solve(low, b, trans):
    """L^{-1} b or L^{-T} b by blocks."""
    n, nb, x = len(low), 2048, b.clone()
    starts = list(range(0, n, nb))
    for k in reversed(starts) if trans else starts:
        e = min(k + nb, n)
        dia = torch.tril(low[k:e, k:e])
        x[k:e] = torch.linalg.solve_triangular(dia.T if trans else dia, x[k:e, None], upper=trans)[:, 0]
        if trans:
            x[:k] -= low[k:e, :k].T @ x[k:e]
        else:
            x[e:] -= low[e:, k:e] @ x[k:e]
    return x


def _exact_loglik(region):
    low = _factor(region)
    z = torch.from_numpy(region["z"]).cuda()
    w = _solve(low, z, False)
    quad, logdet = float(w @ w), 2.0 * float(torch.log(torch.diagonal(low)).sum())
    return low, z, [-0.5 * quad - 0.5 * logdet - 0.5 * len(z) * math.log(2.0 * math.pi), logdet, quad]


def _exact_predict(region, low, z, targets):
    x = _solve(low, _solve(low, z, False), True)
    loc = [torch.from_numpy(c).cuda() for c in region["loc"]]
    tgt = [torch.from_numpy(c).cuda() for c in targets]
    return torch.cat([_covariance([c[i:i + 64] for c in tgt], loc, region["theta"], region["kernel"]) @ x
                      for i in range(0, len(tgt[0]), 64)]).cpu().numpy()


def _dlarnv_normal(n, seed):
    """LAPACK's dlarnv(3, {seed, seed, seed, 1}): pairs of the 48-bit
    multiplicative congruential stream through Box-Muller."""
    mask, a = (1 << 48) - 1, 33952834046453
    state = (((seed * 4096 + seed) * 4096 + seed) * 4096 + 1) & mask
    u = np.empty(2 * n)
    for j in range(2 * n):
        state = (state * a) & mask
        u[j] = state * 2.0 ** -48
    return np.sqrt(-2.0 * np.log(u[0::2])) * np.cos(2.0 * math.pi * u[1::2])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        values, zmiss = [], []
        for k, region in enumerate(_regions(case, seed)):
            low, z, v = _exact_loglik(region)
            values.append(v)
            if kind == "serve" and k % 4 == 0:
                zmiss.append(_exact_predict(region, low, z, _targets(region, PREDICT_POINTS)))
        if kind == "batch":
            return {"values": np.array(values)}
        return {"loglik": np.array(values)[:, 0], "zmiss": np.concatenate(zmiss)}
    region = _region(case, seed)
    if kind == "generate":
        e = torch.from_numpy(_dlarnv_normal(case["n"], case["e_seed"])).cuda()
        return {"z": (torch.tril(_factor(region)) @ e).cpu().numpy()}
    targets = _targets(region, case["targets"]) if kind == "predict" else None
    low, z, (llh, logdet, quad) = _exact_loglik(region)
    if kind == "predict":
        return {"zmiss": _exact_predict(region, low, z, targets)}
    return {"loglik": np.float64(llh), "logdet": np.float64(logdet), "quad": np.float64(quad)}
