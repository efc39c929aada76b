"""Timing cases of the period scan: what a user of the framework has it do, through its Python entry points.

Four kinds of call, each over the sizes it is used at:
  eval   PeriodSearch.eval: model evaluations with their normal equations (and the raw Jacobian rows)
         for given parameter vectors -- shape work outside the scan, derivative checks, other optimisers;
  fit    PeriodSearch.fit_batch: Levenberg-Marquardt fits of given (period, pole) pairs -- one period
         looked at again, a round of the convexity-weight search (10 periods x 10 poles);
  scan   PeriodSearch.scan: the output lines of a range of trial periods -- the main work;
  batch  Batch.run: the fits of many asteroids of different sizes in one call.

The photometry is synthetic: a convex model with random log-area coefficients and pole, seen from Earth
on a 2.5 AU orbit, dense relative lightcurves and sparse calibrated points with Gaussian noise.  Fits run
6 LM iterations: every iteration of a fit is the same work (one damped solve, one evaluation), and after
6 two roundings of the same fit still agree to 1e-11, while over the 50 of a production scan about one
trajectory in a hundred turns a last-bit difference into a visible one.

exact() computes the same outputs in 64 bits with plain torch, without the package's code.
"""
import math

import numpy as np
import torch

import periodsearch_amd as pa

STOP = 6  # LM iterations per fit
PHASE = (0.5, 0.1, -0.5)
CL = 0.1
CONW = 0.1
LAMBDA0, LAMBDA_INCR = 0.1, 5.0
JD0 = 2455000.0
POLE_BETA = [0, 0, 0, 0, 60, 60, 60, -60, -60, -60]
POLE_LAMBDA = [0, 90, 180, 270, 60, 180, 300, 60, 180, 300]
FIT_FLOATS = ("dev", "prd", "dark", "totarea", "la", "be", "chisq")
FIT_INTS = ("niter", "nsolve_fail")
LINE_FIELDS = ("per", "dev", "chi2", "dark", "la", "be")


def _case(name, kind, **kw):
    c = dict(name=name, kind=kind, lmax=6, nrows=6, dense=40, pts_min=50, pts_max=50, sparse=400, years=15.0,
             cl_free=False, mixed=False, periods=0, vecs=0, raw=False, asteroids=0)
    c.update(kw)
    return c


def listed():
    return [
        # one evaluation of a small model: the call an interactive tool or an outside optimiser makes
        _case("eval_one", "eval", lmax=3, dense=10, pts_min=60, pts_max=60, sparse=0, years=2.0, vecs=1),
        # raw model and Jacobian rows at the production shape: plots, derivative checks
        _case("eval_raw", "eval", vecs=16, raw=True),
        # the differentiation workload: thousands of evaluations at the production shape
        _case("eval_many", "eval", vecs=4096),
        # one period looked at again: its ten poles at the production shape
        _case("fit_period", "fit", periods=1),
        # a round of the convexity-weight search (10 periods x 10 poles), plain Lmax 3 shape
        _case("prepass_small", "fit", lmax=3, dense=10, pts_min=60, pts_max=60, sparse=100, years=2.0, periods=10),
        # the same at the production shape
        _case("prepass", "fit", periods=10),
        # the main scan at the production shape: 40 lightcurves x 50 points + 400 sparse points
        _case("scan_production", "scan", periods=256),
        # a sparse survey: 5000 calibrated points, 512 facets
        _case("scan_survey", "scan", nrows=8, dense=0, sparse=5000, years=10.0, periods=64),
        # lightcurves of any length, odd sizes everywhere, the Lambert weight fitted too
        _case("scan_ragged", "scan", lmax=5, nrows=7, dense=37, pts_min=5, pts_max=120, sparse=611, cl_free=True,
              periods=53),
        # lightcurves of a whole long night or a space telescope: longer than 128 points
        _case("scan_long_curves", "scan", lmax=6, dense=9, pts_min=90, pts_max=400, sparse=150, periods=31),
        # the mixed-precision option
        _case("scan_mixed", "scan", mixed=True, periods=64),
        # asteroids of very different sizes in one call
        _case("batch_uneven", "batch", asteroids=12, periods=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["eval", "eval", "fit", "fit", "scan", "scan", "scan", "batch"])
        long_curves = kind != "batch" and rng.random() < 0.15
        lo, hi = (60, 400) if long_curves else sorted((rng.randint(5, 120), rng.randint(5, 120)))
        c = _case("", kind, lmax=rng.choice([2, 3, 4, 5, 6, 6, 6]), nrows=rng.randint(4, 8), dense=rng.randint(0, 60),
                  pts_min=lo, pts_max=hi, sparse=rng.choice([0, _log_int(rng, 150, 5000)]), years=rng.uniform(1.0, 15.0))
        del c["name"]
        if long_curves:
            c["dense"] = rng.randint(2, 12)
        if kind != "eval" and not c["sparse"]:  # the phase function and the size need calibrated points
            c["sparse"] = _log_int(rng, 150, 5000)
        if kind == "eval":
            c["vecs"] = _log_int(rng, 1, 4096)
            c["raw"] = c["vecs"] <= 64 and rng.random() < 0.4
        elif kind == "fit":
            c["periods"] = _log_int(rng, 1, 40)
        elif kind == "scan":
            c["periods"] = _log_int(rng, 4, 256)
        else:
            c["asteroids"] = rng.randint(3, 16)
            c["periods"] = rng.randint(1, 4)
            return c
        points = c["dense"] * (lo + hi) / 2 + c["sparse"]
        c["mixed"] = kind != "eval" and rng.random() < 0.15
        c["cl_free"] = not c["mixed"] and c["sparse"] >= 500 and rng.random() < 0.3
        evals = c["vecs"] + 10 * c["periods"] * (STOP + 1)
        cost = evals * points * 8 * c["nrows"] ** 2 * (c["lmax"] + 1) ** 2
        if points >= 200 and cost <= 6e14:
            return c


# ---------------------------------------------------------------------------------------------
# The synthetic asteroid and its input file.
# ---------------------------------------------------------------------------------------------
def _mesh(nrows):
    """Normals and areas of the facets of the triangulated sphere: ring i of an octant has i edges."""
    def vertex(i, j):  # ring i (0 = the pole), j-th of 4i vertices
        th, ph = i * math.pi / (2 * nrows), (j * math.pi / (2 * i) if i else 0.0)
        return [math.sin(th) * math.cos(ph), math.sin(th) * math.sin(ph), math.cos(th)]
    tri = []
    for i in range(1, nrows + 1):
        for q in range(4):
            for j in range(i):
                tri.append([vertex(i - 1, q * (i - 1) + j), vertex(i, q * i + j), vertex(i, q * i + j + 1)])
            for j in range(i - 1):
                tri.append([vertex(i - 1, q * (i - 1) + j), vertex(i, q * i + j + 1),
                            vertex(i - 1, q * (i - 1) + j + 1)])
    north = np.array(tri)
    south = (north * [1, 1, -1])[:, [0, 2, 1]]
    t = np.concatenate([north, south])
    cr = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    ln = np.linalg.norm(cr, axis=1)
    return cr / ln[:, None], ln / 2


def _basis(nor, lmax):
    """Unnormalised real spherical harmonics at the normals: for every m, l >= m: cos, then sin for m > 0."""
    x = nor[:, 2]
    st, ph = np.sqrt(1 - x * x), np.arctan2(nor[:, 1], nor[:, 0])
    cols = []
    for m in range(lmax + 1):
        p = {m: st ** m * math.prod(range(1, 2 * m, 2))}
        for l in range(m + 1, lmax + 1):
            p[l] = ((2 * l - 1) * x * p[l - 1] - (l + m - 1) * p.get(l - 2, 0.0)) / (l - m)
        for l in range(m, lmax + 1):
            cols.append(p[l] * np.cos(m * ph))
            if m:
                cols.append(p[l] * np.sin(m * ph))
    return np.stack(cols, 1)


def _orbits(jd):
    """Asteroid-centric Sun and Earth vectors [AU]."""
    t = jd - JD0
    te, ta, inc = 2 * np.pi * t / 365.25 + 0.3, 2 * np.pi * t / (365.25 * 2.5 ** 1.5) + 1.1, math.radians(8.0)
    earth = np.stack([np.cos(te), np.sin(te), 0 * t], -1)
    ast = 2.5 * np.stack([np.cos(ta), np.sin(ta) * math.cos(inc), np.sin(ta) * math.sin(inc)], -1)
    return -ast, earth - ast


def _unit(v):
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _nights(years):
    """Dates at which the asteroid is away from the Sun in the sky and not exactly at opposition."""
    jd = JD0 + np.arange(0, years * 365.25, 0.5)
    sun, earth = _orbits(jd)
    alpha = np.degrees(np.arccos(np.sum(_unit(sun) * _unit(earth), -1)))
    elong = np.degrees(np.arccos(np.clip(np.sum(_unit(sun - earth) * _unit(-earth), -1), -1, 1)))
    return jd[(alpha >= 2.0) & (elong >= 100.0)]


def _pole_matrix(beta, lam):
    cb, sb, cl, sl = math.cos(beta), math.sin(beta), math.cos(lam), math.sin(lam)
    return np.array([[cb * cl, cb * sl, -sb], [-sl, cl, 0.0], [sb * cl, sb * sl, cb]])


class _Asteroid:
    """The synthetic input file of a case and seed, and the numbers in it."""

    def __init__(self, case, seed):
        rng = np.random.default_rng([seed, 77])
        nor, darea = _mesh(8)
        lm = 3
        d = _basis(nor, lm)
        coef = rng.normal(0.0, 0.3, d.shape[1])
        coef[0] = 0.0
        area = darea * np.exp(d @ coef)
        lam, beta = rng.uniform(0, 2 * np.pi), np.arccos(rng.uniform(-1, 1))
        self.period = float(rng.uniform(2.5, 18.0))
        bl = _pole_matrix(beta, lam)
        nights = _nights(case["years"])

        def brightness(jd):
            sun, earth = _orbits(jd)
            e, e0 = _unit(earth), _unit(sun)
            f = 2 * np.pi * 24 / self.period * (jd - JD0)
            c, s = np.cos(f)[:, None], np.sin(f)[:, None]
            def body(v):
                p = v @ bl.T
                return np.concatenate([c * p[:, :1] + s * p[:, 1:2], -s * p[:, :1] + c * p[:, 1:2], p[:, 2:]], 1)
            mu, mu0 = body(e) @ nor.T, body(e0) @ nor.T
            vis = (mu > 0) & (mu0 > 0)
            al = np.arccos(np.sum(e * e0, -1))
            br = np.where(vis, mu * mu0 * (CL + 1 / np.where(vis, mu + mu0, 1.0)), 0.0) @ area
            return br * (1 + PHASE[0] * np.exp(-al / PHASE[1]) + PHASE[2] * al), sun, earth

        curves = []
        dense = case["dense"]
        if dense:
            first = np.sort(rng.choice(nights, size=dense, replace=dense > len(nights)))
            for k in range(dense):
                n = int(rng.integers(case["pts_min"], case["pts_max"] + 1))
                jd = first[k] + np.arange(n) * (6.0 / 24 / 50)  # a point every 7 minutes
                y, sun, earth = brightness(jd)
                y = y * (1 + 0.01 * rng.standard_normal(n))
                curves.append((0, jd, y / y.mean(), sun, earth))
        if case["sparse"]:
            jd = np.sort(rng.choice(nights, size=case["sparse"]) + rng.uniform(0, 0.5, case["sparse"]))
            y, sun, earth = brightness(jd)
            y = y * (1 + 0.02 * rng.standard_normal(len(jd)))
            for c0 in range(0, len(jd), 1000):
                sl = slice(c0, c0 + 1000)
                curves.append((1, jd[sl], y[sl], sun[sl], earth[sl]))
        # a scan window around the true period, wide enough for the case's trial periods
        alljd = np.concatenate([c[1] for c in curves])
        df = 0.5 / (alljd.max() - alljd.min()) / 24
        f = 1 / self.period
        half = (case["periods"] // 2 + 5) * df
        self.per = [float("%.9f" % (1 / (f + half))), float("%.9f" % (1 / max(f - 3 * half, 0.2 * f)))]
        out = ["%.9f 1 %.9f 1" % tuple(self.per), "0", "0", "%g" % CONW, "%d %d" % (case["lmax"], case["lmax"]),
               "%d" % case["nrows"]]
        out += ["%g 1" % p for p in PHASE]
        out += ["%g %d" % (CL, case["cl_free"]), "%d" % STOP, "10", "%g" % LAMBDA_INCR, "%g" % LAMBDA0,
                "%d" % len(curves)]
        rows = []
        self.curves = []  # (calibrated, number of points)
        for calib, jd, y, sun, earth in curves:
            self.curves.append((calib, len(jd)))
            out.append("%d %d" % (len(jd), calib))
            lines = ["%.6f %.6e %.6e %.6e %.6e %.6e %.6e %.6e" % (jd[i], y[i], *sun[i], *earth[i]) for i in range(len(jd))]
            out += lines
            rows += lines
        out.append("1 1")
        self.text = "\n".join(out) + "\n"
        self.rows = rows  # parsed by _Problem


def _vectors(case, seed, cg0):
    """Parameter vectors around and away from a model: shape coefficients scaled by their basis function's
    largest value, any pole, periods of 2-20 h."""
    rng = np.random.default_rng([seed, 78])
    span = np.abs(_basis(_mesh(case["nrows"])[0], case["lmax"])).max(0)
    nc, nv = len(span), case["vecs"]
    a = np.zeros((nv, nc + 8))
    a[:, 0] = cg0
    a[:, 1:nc] = rng.normal(0, 0.3, (nv, nc - 1)) / span[1:]
    a[:, nc] = np.arccos(rng.uniform(-1, 1, nv))
    a[:, nc + 1] = rng.uniform(0, 2 * np.pi, nv)
    a[:, nc + 2] = 24 * 2 * np.pi / rng.uniform(2, 20, nv)
    a[:, nc + 3:nc + 6] = PHASE
    a[:, nc + 6] = math.log(CL)
    a[:, nc + 7] = 1.0
    return a


def _asteroid_cases(case, seed):
    """The asteroids of a batch: 300 to 8000 points, Lmax 3, 4 or 6, 288 or 512 facets."""
    rng = np.random.default_rng([seed, 79])
    out = []
    for _ in range(case["asteroids"]):
        n = int(round(math.exp(rng.uniform(math.log(300), math.log(8000)))))
        dense = min(150, int(round(n * 5 / 6 / 50)))
        out.append(dict(case, lmax=int(rng.choice([3, 4, 6])), nrows=int(rng.choice([6, 8])), dense=dense, pts_min=50,
                        pts_max=50, sparse=max(100, n - 50 * dense), years=15.0))
    return out


def _first_period(nmax, periods):
    return max(1, min(4, nmax - periods + 1))


def prepare(case, seed):
    if case["kind"] == "batch":
        searches, prob, freq = [], [], []
        for i, c in enumerate(_asteroid_cases(case, seed)):
            ps = pa.PeriodSearch.from_text(_Asteroid(c, seed * 1000 + i).text).prepare(device=0)
            n = _first_period(ps.info()["nmax"], case["periods"]) + np.arange(case["periods"])
            freq.append(ps.freq(np.repeat(n, 10)))
            prob.append(np.full(len(freq[-1]), i))
            searches.append(ps)
        freq, prob = np.concatenate(freq), np.concatenate(prob)
        return {"case": case, "searches": searches, "batch": pa.Batch(searches), "prob": prob, "freq": freq,
                "pole": 1 + np.arange(len(freq)) % 10, "conw_r": np.array([s.info()["conw_r0"] for s in searches])}
    ps = pa.PeriodSearch.from_text(_Asteroid(case, seed).text)
    ps.prepare(device=0, precision=pa.PS_MIXED if case["mixed"] else pa.PS_FP64)
    info = ps.info()
    state = {"case": case, "ps": ps, "conw_r": info["conw_r0"]}
    if case["kind"] == "eval":
        state["a"] = _vectors(case, seed, ps.geometry()["cg_first"][0])
    else:
        state["n0"] = _first_period(info["nmax"], case["periods"])
        n = state["n0"] + np.arange(case["periods"])
        state["freq"], state["pole"] = ps.freq(np.repeat(n, 10)), 1 + np.arange(10 * len(n)) % 10
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "eval":
        return state["ps"].eval(state["a"], state["conw_r"], raw=case["raw"])
    if case["kind"] == "scan":
        out = state["ps"].scan(state["n0"], state["n0"] + case["periods"] - 1, state["conw_r"])
        return {k: out[k] for k in LINE_FIELDS}
    if case["kind"] == "fit":
        out = state["ps"].fit_batch(state["freq"], state["pole"], state["conw_r"])
    else:
        out = state["batch"].run(state["conw_r"], state["prob"], state["freq"], state["pole"])
    return {k: out[k] for k in FIT_FLOATS + FIT_INTS}


def _work_one(case, evals, solves, points):
    n, nf, nc = points + 3, 8 * case["nrows"] ** 2, (case["lmax"] + 1) ** 2
    mfit = nc - (0 if case["sparse"] else 1) + 6 + int(case["cl_free"])
    # the shape-Jacobian contraction, the normal equations, the damped solves; the points read once
    flops = evals * n * (2.0 * nf * nc + mfit * (mfit + 1) + 2 * mfit) + solves * mfit ** 3 / 3.0 * 2
    return 11 * 8.0 * n + nf * nc * 8.0, flops, mfit


def work(case):
    pts = case["dense"] * (case["pts_min"] + case["pts_max"]) // 2 + case["sparse"]
    if case["kind"] == "eval":
        b, f, mfit = _work_one(case, case["vecs"], 0, pts)
        ma = (case["lmax"] + 1) ** 2 + 8
        out = mfit * mfit + mfit + 1 + ((pts + 3) * (ma + 1) if case["raw"] else 0)
        return {"bytes": b + case["vecs"] * 8.0 * (ma + out), "flops": f}
    if case["kind"] == "batch":  # on average over the sizes an asteroid is drawn from
        fits = 10 * case["periods"] * case["asteroids"]
        c = dict(case, lmax=5, nrows=7, sparse=100)
        b, f, _ = _work_one(c, fits * (STOP + 1), fits * STOP, 1970)
        return {"bytes": b * case["asteroids"] + 84.0 * fits, "flops": f}
    fits = 10 * case["periods"]
    b, f, _ = _work_one(case, fits * (STOP + 1), fits * STOP, pts)
    return {"bytes": b + 84.0 * fits, "flops": f}


# ---------------------------------------------------------------------------------------------
# The same outputs in 64 bits, in plain torch.
# ---------------------------------------------------------------------------------------------
class _Problem:
    def __init__(self, case, seed):
        ast = _Asteroid(case, seed)
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        v = np.array([[float(x) for x in r.split()] for r in ast.rows])
        jd, y, sun, earth = v[:, 0], v[:, 1], v[:, 2:5], v[:, 5:8]
        e, e0 = _unit(earth), _unit(sun)
        self.ndata = len(jd)
        lc = np.repeat(np.arange(len(ast.curves)), [n for _, n in ast.curves])
        rel = np.array([c == 0 for c, _ in ast.curves])
        cnt = np.array([n for _, n in ast.curves])
        sig = (np.bincount(lc, y) / cnt)[lc]
        alpha = np.arccos(np.sum(e * e0, -1))
        # the initial ellipsoid's size from the first point of the curve seen nearest to opposition
        starts = np.concatenate([[0], np.cumsum(cnt)[:-1]])
        cand = starts if rel.all() else starts[~rel]
        k = cand[np.argmin(alpha[cand])]
        abc = np.array([1.05, 1.0, 0.95])
        escl = math.sqrt(2 * sig[k] / (0.5 * math.pi * (1 + math.cos(alpha[k])))) / math.sqrt(
            (abc[0] * abc[1] + abc[1] * abc[2] + abc[0] * abc[2]) / 3)
        escl *= 1.0 if rel.all() else 0.8
        self.escl, self.conw_r = escl, CONW / escl / escl
        nor, darea = _mesh(case["nrows"])
        d = _basis(nor, case["lmax"])
        self.nc = nc = d.shape[1]
        self.ma = nc + 8
        abc = abc * escl
        self.cg_first = np.linalg.lstsq(d, 2 * (math.log(abc.prod()) - np.log(np.sum((abc * nor) ** 2, 1))), rcond=None)[0]
        fit = np.ones(self.ma, bool)
        fit[0], fit[nc + 6], fit[nc + 7] = not rel.all(), case["cl_free"], False
        self.f0 = 1 / ast.per[0]
        self.df = 0.5 / (jd.max() - jd.min()) / 24
        self.nmax = int((self.f0 - 1 / ast.per[1]) / self.df) + 1
        T = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=dev)  # noqa: E731
        self.dev = dev
        self.t, self.y, self.sig, self.e, self.e0, self.alpha = (T(x) for x in (jd - int(jd.min()), y, sig, e, e0, alpha))
        self.lc, self.rel, self.cnt = T(lc), T(rel), T(cnt.astype(float))
        self.nor, self.darea, self.d = T(nor), T(darea), T(d)
        self.fit = T(np.flatnonzero(fit))
        w = 1 / sig ** 2
        self.w = T(np.concatenate([w, np.full(3, self.conw_r ** 2)]))

    def model(self, a):
        """Areas, model values and Jacobian rows (the three convexity rows last) of vectors a [V, ma]."""
        nc, V, N = self.nc, a.shape[0], self.ndata
        area = self.darea * torch.exp(a[:, :nc] @ self.d.T)
        cl, cls = torch.exp(a[:, nc + 6])[:, None, None], a[:, nc + 7][:, None, None]
        b, l, om = a[:, nc], a[:, nc + 1], a[:, nc + 2]
        cb, sb, c, s, z = torch.cos(b), torch.sin(b), torch.cos(l), torch.sin(l), torch.zeros_like(b)
        mat = lambda *r: torch.stack(r, -1).reshape(V, 3, 3)  # noqa: E731
        B = mat(cb * c, cb * s, -sb, -s, c, z, sb * c, sb * s, cb)
        dB = [mat(-sb * c, -sb * s, -cb, z, z, z, cb * c, cb * s, -sb), mat(-cb * s, cb * c, z, -c, -s, z, -sb * s, sb * c, z)]
        ph = torch.fmod(om[:, None] * self.t, 2 * math.pi)
        cf, sf = torch.cos(ph), torch.sin(ph)
        rz = lambda p: torch.stack([cf * p[..., 0] + sf * p[..., 1], cf * p[..., 1] - sf * p[..., 0], p[..., 2]], -1)  # noqa: E731
        drz = lambda p: torch.stack([cf * p[..., 1] - sf * p[..., 0], -cf * p[..., 0] - sf * p[..., 1], 0 * p[..., 2]], -1)  # noqa: E731
        def dirs(v):
            p = v @ B.transpose(1, 2)
            return rz(p), [rz(v @ dB[0].transpose(1, 2)), rz(v @ dB[1].transpose(1, 2)), self.t[:, None] * drz(p)]
        e, de = dirs(self.e.expand(V, N, 3))
        e0, de0 = dirs(self.e0.expand(V, N, 3))
        mu, mu0 = e @ self.nor.T, e0 @ self.nor.T
        vis = ((mu > 1e-8) & (mu0 > 1e-8)).to(mu.dtype)
        rd = 1 / torch.clamp(mu + mu0, min=1e-8)
        A = area[:, None, :] * vis
        Amm = A * mu * mu0
        X = Amm * (cl + cls * rd)
        S = (A * (cls * (mu0 * rd) ** 2 + cl * mu0)) @ self.nor
        U = (A * (cls * (mu * rd) ** 2 + cl * mu)) @ self.nor
        br = X.sum(-1)
        p1, p2, p3 = (a[:, nc + 3 + i][:, None] for i in range(3))
        ex = torch.exp(-self.alpha / p2)
        scale = 1 + p1 * ex + p3 * self.alpha
        cols = [scale[..., None] * (X @ self.d)]
        cols += [(scale * ((S * x).sum(-1) + (U * x0).sum(-1)))[..., None] for x, x0 in zip(de, de0)]
        cols += [(br * k)[..., None] for k in (ex, p1 * ex * self.alpha / p2 ** 2, self.alpha.expand(V, N))]
        cols += [(scale * Amm.sum(-1) * cl[..., 0])[..., None], (scale * (Amm * rd).sum(-1))[..., None]]
        J = torch.zeros(V, N + 3, self.ma, dtype=a.dtype, device=a.device)
        J[:, :N] = torch.cat(cols, -1)
        J[:, N:, :nc] = torch.einsum("vf,fc,fk->vck", area, self.nor, self.d)
        return area, torch.cat([br * scale, area @ self.nor], 1), J

    def normal(self, a):
        """alpha, beta, chi2, the areas and the raw rows of vectors a."""
        area, ymod, J = self.model(a)
        N, V, nlc = self.ndata, a.shape[0], len(self.rel)
        idx = self.lc.expand(V, N)
        ave = torch.zeros(V, nlc, dtype=a.dtype, device=a.device).scatter_add_(1, idx, ymod[:, :N])
        dave = torch.zeros(V, nlc, self.ma, dtype=a.dtype, device=a.device).index_add_(1, self.lc, J[:, :N])
        rel = self.rel[self.lc]
        av = ave[:, self.lc]
        coef = torch.where(rel, self.sig * self.cnt[self.lc] / av, torch.ones_like(av))
        Jn = J.clone()
        y = ymod[:, :N]
        norm = coef[..., None] * (J[:, :N] - y[..., None] * dave[:, self.lc] / av[..., None])
        norm[..., 0] = 0.0
        Jn[:, :N] = torch.where(rel[:, None], norm, J[:, :N])
        res = torch.cat([self.y - coef * y, -ymod[:, N:]], 1)
        Jf = Jn[..., self.fit]
        Jw = Jf * self.w[:, None]
        return Jw.transpose(1, 2) @ Jf, (Jw * res[..., None]).sum(1), (self.w * res * res).sum(1), area, ymod, J

    def step(self):
        return max(1, int(4e8 / (8 * (self.ndata + 3) * (len(self.darea) + 4 * self.ma))))

    def fits(self, freq, pole):
        """The fits of (freq, pole) pairs: the LM loop with its bookkeeping."""
        res = [self._fits(freq[i:i + self.step()], pole[i:i + self.step()]) for i in range(0, len(freq), self.step())]
        return {k: np.concatenate([r[k] for r in res]) for k in FIT_FLOATS}

    def _fits(self, freq, pole):
        nc, V = self.nc, len(freq)
        g = np.zeros((V, self.ma))
        g[:, :nc] = self.cg_first
        g[:, nc] = np.radians(90.0 - np.array(POLE_BETA)[pole - 1])
        g[:, nc + 1] = np.radians(np.array(POLE_LAMBDA)[pole - 1])
        g[:, nc + 2] = 24 * 2 * math.pi * freq
        g[:, nc + 3:nc + 6] = PHASE
        g[:, nc + 6], g[:, nc + 7] = math.log(CL), 1.0
        cg = torch.as_tensor(g, device=self.dev)
        alpha, beta, ochisq, area, _, _ = self.normal(cg)
        lam = torch.full((V,), LAMBDA0, dtype=cg.dtype, device=self.dev)
        chck = torch.zeros(V, dtype=cg.dtype, device=self.dev)
        rchisq = torch.full_like(chck, -1.0)
        best = area
        eye = torch.eye(len(self.fit), dtype=cg.dtype, device=self.dev)
        for it in range(STOP):
            da = torch.linalg.solve(alpha * (1 + eye * lam[:, None, None]), beta[..., None])[..., 0]
            tr = cg.clone()
            tr[:, self.fit] += da
            al, be, chi, area, _, _ = self.normal(tr)
            ok = chi < ochisq
            lam = torch.where(ok, lam / LAMBDA_INCR, lam * LAMBDA_INCR)
            cg = torch.where(ok[:, None], tr, cg)
            alpha, beta = torch.where(ok[:, None, None], al, alpha), torch.where(ok[:, None], be, beta)
            ochisq = torch.where(ok, chi, ochisq)
            best = torch.where(ok[:, None], area, best)
            new = ok | (it == 0)
            s2 = ((best @ self.nor) ** 2).sum(1)
            chck = torch.where(new, s2, chck)
            rchisq = torch.where(new, ochisq - s2 * self.conw_r ** 2, rchisq)
            last = best if it == 0 else area
        out = {"dev": torch.sqrt(rchisq / self.ndata), "prd": 2 * math.pi / cg[:, nc + 2], "dark": torch.sqrt(chck),
               "totarea": last.sum(1), "la": cg[:, nc + 1] * (180 / math.pi), "be": 90 - cg[:, nc] * (180 / math.pi),
               "chisq": ochisq}
        return {k: v.cpu().numpy() for k, v in out.items()}


def exact(case, seed):
    if case["kind"] == "batch":
        res = []
        for i, c in enumerate(_asteroid_cases(case, seed)):
            p = _Problem(c, seed * 1000 + i)
            n = _first_period(p.nmax, case["periods"]) + np.arange(case["periods"])
            res.append(p.fits(p.f0 - (np.repeat(n, 10) - 1) * p.df, 1 + np.arange(10 * len(n)) % 10))
        return {**{k: np.concatenate([r[k] for r in res]) for k in FIT_FLOATS}, **{k: None for k in FIT_INTS}}
    p = _Problem(case, seed)
    if case["kind"] == "eval":
        a = torch.as_tensor(_vectors(case, seed, p.cg_first[0]), device=p.dev)
        parts = [p.normal(a[i:i + p.step()]) for i in range(0, len(a), p.step())]
        out = {k: torch.cat([q[j] for q in parts]).cpu().numpy() for k, j in (("alpha", 0), ("beta", 1), ("chisq", 2))}
        if case["raw"]:
            out.update({k: torch.cat([q[j] for q in parts]).cpu().numpy() for k, j in (("ymod", 4), ("dyda", 5))})
        return out
    n = _first_period(p.nmax, case["periods"]) + np.arange(case["periods"])
    fits = p.fits(p.f0 - (np.repeat(n, 10) - 1) * p.df, 1 + np.arange(10 * len(n)) % 10)
    if case["kind"] == "fit":
        return {**fits, **{k: None for k in FIT_INTS}}
    f = {k: v.reshape(-1, 10) for k, v in fits.items()}
    i, r = np.argmin(f["dev"], 1), np.arange(len(n))
    dev, la = f["dev"][r, i], f["la"][r, i]
    dark = np.where(n == 1, p.conw_r * p.escl ** 2, f["dark"][r, i] / f["totarea"][r, i] * 100)
    return {"per": 24 * f["prd"][r, i], "dev": dev, "chi2": dev ** 2 * p.ndata, "dark": dark,
            "la": np.where(la < 0, la + 360, la), "be": f["be"][r, i]}
