"""What a user of this package has it do, as cases to time: resident runs of
the 2DDI step between two output times, single steps through the per-step
call sites, storm ensembles as one batch, and the drop-in JCG.

A case is a dict of plain values:

path     "run"    ``steps`` steps in one resident run (adcgpu_run), then the
                  fields an output file takes back to the host, as the
                  case-directory driver does between two output times;
         "step"   ``steps`` calls of adcgpu_timestep with the host's met
                  forcing (the Fortran timestep loop), then the same fields;
         "batch"  ``members`` storms on one mesh stepped together
                  (adcgpu_batch_run);
         "jcg" / "jcg_noalloc"
                  one solve of a GWCE system in the caller's host arrays
                  (CALL JCG), with and without device allocation.
mesh     "basin" (no wet/dry, tide only), "beach" (wet/dry under a small
         storm) or "coastal" (graded Delaunay shelf, wet/dry, M2 + K1 and a
         Holland storm), at about ``nodes`` nodes.
start    the JCG start: "previous" (the reference's), "extrapolated" or
         "learned".

The mesh's geometry depends on its kind and size only; bathymetry, friction,
the initial surge and the storm are drawn from the seed.  A pass continues
the run where the last one left it.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np

from adcirc_amd import _lib, meshgen, prep
from adcirc_amd.model import Batch, Model, cold_wetdry_state, jcg

SPIN_UP = 40         # steps that take the drawn surge into a moving wetting front
STORM_TIME = 10800.0  # s: runs start at hour 3 of the storm, as the benchmark's window


def listed():
    run = dict(path="run", precision="fp64", start="previous", lumped=False, tide=False)
    return [
        # the smallest calls: one step of a small wet/dry beach, host forcing
        # handed in and the fields taken back each step (a coupled host code)
        dict(name="beach_861_step", path="step", mesh="beach", nodes=861, steps=1),
        # the reference's own test basin between two hourly outputs
        dict(run, name="basin_5k_run", mesh="basin", nodes=5151, steps=100),
        # the drop-in solver on that basin's system, in a loop that cannot allocate
        dict(name="basin_5k_jcg_noalloc", path="jcg_noalloc", mesh="basin", nodes=5151),
        # the drop-in solver in a Fortran code on a regional mesh
        dict(name="coastal_20k_jcg", path="jcg", mesh="coastal", nodes=20000),
        # a regional storm run, and the same per step from the host
        dict(run, name="coastal_20k_run", mesh="coastal", nodes=20000, steps=50),
        dict(name="coastal_100k_step", path="step", mesh="coastal", nodes=100000, steps=4),
        # the explicit (lumped) form of the GWCE
        dict(run, name="coastal_100k_lumped", mesh="coastal", nodes=100000, steps=20, lumped=True),
        # the learned JCG start
        dict(run, name="coastal_50k_learned", mesh="coastal", nodes=50000, steps=20,
             start="learned"),
        # an ensemble of storms on one mesh
        dict(name="coastal_50k_batch8", path="batch", mesh="coastal", nodes=50000, steps=10,
             members=8),
        # a basin-scale mesh
        dict(run, name="coastal_250k_run", mesh="coastal", nodes=250000, steps=20),
        # the full-size mesh: plain, and in its fastest configuration
        dict(run, name="coastal_1m_run", mesh="coastal", nodes=1000000, steps=20),
        dict(run, name="coastal_1m_mixed_extrapolated", mesh="coastal", nodes=1000000, steps=20,
             precision="mixed", start="extrapolated"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["run", "run", "run", "step", "batch", "jcg", "jcg_noalloc"])
    if path == "jcg":
        return dict(path=path, mesh=rng.choice(["basin", "coastal"]), nodes=size(1500, 120000))
    if path == "jcg_noalloc":
        return dict(path=path, mesh=rng.choice(["basin", "coastal"]), nodes=size(1500, 30000))
    if path == "step":
        return dict(path=path, mesh=rng.choice(["beach", "coastal"]), nodes=size(1500, 150000),
                    steps=rng.randint(1, 4))
    if path == "batch":
        return dict(path=path, mesh="coastal", nodes=size(3000, 80000), steps=rng.randint(4, 12),
                    members=rng.randint(2, 8))
    mesh = rng.choice(["basin", "beach", "coastal", "coastal", "coastal"])
    lumped = mesh != "basin" and rng.random() < 0.2
    return dict(path=path, mesh=mesh, steps=rng.randint(10, 60),
                nodes=size(1500, 300000) if mesh == "coastal" else size(900, 60000),
                precision="mixed" if rng.random() < 0.3 else "fp64", lumped=lumped,
                start="previous" if lumped else rng.choice(
                    ["previous", "previous", "extrapolated", "learned"]),
                tide=mesh == "basin" and rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=6)
def _mesh(kind, nodes):
    if kind == "coastal":
        case = meshgen.coastal(nodes)
    else:  # 1 km cells in the basin, 200 m on the beach
        ny = max(4, int(round(math.sqrt(nodes / 2.0))))
        nx = max(4, nodes // ny)
        cell = 1000.0 if kind == "basin" else 200.0
        make = meshgen.basin if kind == "basin" else meshgen.beach
        case = make(nx=nx, ny=ny, lx=cell * (nx - 1), ly=cell * (ny - 1))
    return case, prep.build_tables(case.mesh, case.run.nolifa, case.run.h0, case.run.anginn)


def _inputs(case, seed, member=0):
    """(tables, run, emo, efa, fric, eta2): what the host program read from
    its files, and the surge it starts from."""
    rng = np.random.default_rng([seed, member, 29])
    base, tables = _mesh(case["mesh"], case["nodes"])
    t = dict(tables)
    x, y = t["x"], t["y"]
    lx, ly = x.max() - x.min(), y.max() - y.min()

    def waves(amp, n=4):
        f = np.zeros_like(x)
        for _ in range(n):
            kx, ky = rng.uniform(0.5, 4.0, 2) * 2.0 * math.pi
            f += np.cos(kx * x / lx + ky * y / ly + rng.uniform(0.0, 2.0 * math.pi))
        return amp / n * f

    t["dp"] = t["dp"] + waves(0.1)
    fric = base.run.cf * (1.0 + waves(0.3))
    over = {}
    if case.get("lumped"):
        over["ilump"] = 1
    if case.get("start") in ("extrapolated", "learned"):
        over["warm_start"] = 1 if case["start"] == "extrapolated" else 2
    if case.get("tide"):
        over.update(tipot=meshgen.TIPOT_M2S2K1O1, slam0=-75.0, sfea0=35.0)
    hol = None
    if case["mesh"] == "coastal":
        eta2 = rng.uniform(0.4, 0.8) * np.exp(-np.abs(x - meshgen.COAST_X) / 20.0e3) + waves(0.05)
        hol = list(meshgen.storm_ensemble(base, 1, seed=int(rng.integers(1 << 30)))[0])
    else:
        eta2 = waves(0.2)
        if base.run.holland is not None:
            hol = list(base.run.holland)
            hol[0] = float(rng.uniform(980.0, 995.0))
    if hol is not None:  # the vortex where it is at hour 3, at full strength
        hol[4] += hol[6] * STORM_TIME
        hol[5] += hol[7] * STORM_TIME
        hol[9] = 0.0
        over.update(holland=tuple(hol), statim=STORM_TIME / 86400.0)
    run = dataclasses.replace(base.run, **over)
    return t, run, base.emo, base.efa, fric, eta2


def _model(case, seed, member=0):
    t, run, emo, efa, fric, eta2 = _inputs(case, seed, member)
    m = Model(t, run, fric=fric, emo=emo, efa=Model.radians(efa),
              precision=_lib.MIXED if case.get("precision") == "mixed" else _lib.FP64)
    m.cold_start(*cold_wetdry_state(t, run, eta2))
    it = 1
    if run.warm_start == 2:  # the learned start, trained on the run's own solves
        m.ml_collect(4096)
    if run.holland is not None:
        m.holland(0.0, run.holland)
    if run.holland is not None or run.warm_start == 2:
        m.run_resident(it, SPIN_UP, holland=run.holland)
        it += SPIN_UP
    if run.warm_start == 2:
        m.ml_collect(0)
        m.ml_train(1, seed=seed + 1)
    return m, run, it


def _elements(t, run, dp, tau0):
    """The consistent GWCE matrix of every element, all wet: [ne, 3, 3]."""
    nm = t["nm"].reshape(-1, 3) - 1
    fx, fy = t["fdxe"].reshape(-1, 3), t["fdye"].reshape(-1, 3)
    area2 = t["areas"]
    ga = run.a00 * run.g * dp[nm].mean(1) / (2.0 * area2)
    ms = 0.5 * area2 * (1.0 / run.dtdp + tau0[nm].mean(1) / 2.0) / run.dtdp / 12.0
    k = ga[:, None, None] * (fx[:, :, None] * fx[:, None, :] + fy[:, :, None] * fy[:, None, :])
    return nm, k + ms[:, None, None] * (np.ones((3, 3)) + np.eye(3))


def _system(case, seed):
    """A GWCE system in CALL JCG's layout: JCOEF and COEF (NP, MNEI) with the
    diagonal first, the right-hand side and the start."""
    t, run, _, _, _, eta2 = _inputs(case, seed)
    n, w = t["np"], t["mnei"]
    dp = np.maximum(t["dp"], 1.0)  # wet everywhere
    nm, k = _elements(t, run, dp, prep.tau0_nodal(run.tau0, dp))
    coef = np.zeros(w * n)
    np.add.at(coef, nm.ravel(), np.einsum("eii->ei", k).ravel())
    csr = t["csr"].reshape(-1, 3, 2).astype(np.int64) - 1
    for a in range(3):
        for b, c in enumerate([c for c in range(3) if c != a]):
            np.add.at(coef, csr[:, a, b] * n + nm[:, a], k[:, a, c])
    rng = np.random.default_rng([seed, 31])
    jcoef = np.ascontiguousarray(t["neitab"], np.int32)
    want = 1.0e-3 * eta2
    cols = np.maximum(jcoef.reshape(w, n) - 1, 0)
    rhs = (coef.reshape(w, n) * want[cols]).sum(0)
    u = want * (1.0 + 0.1 * rng.standard_normal(n))
    return jcoef, coef, rhs, u, run


def prepare(case, seed):
    if case["path"] in ("jcg", "jcg_noalloc"):
        jcoef, coef, rhs, u, run = _system(case, seed)
        return dict(path=case["path"], jcoef=jcoef, coef=coef, rhs=rhs, u=u, itmax=run.itmax,
                    zeta=run.convcr)
    if case["path"] == "batch":
        got = [_model(case, seed, k) for k in range(case["members"])]
        models = [m for m, _, _ in got]
        return dict(path="batch", batch=Batch(models), models=models, it=got[0][2],
                    holland=[r.holland for _, r, _ in got], steps=case["steps"])
    m, run, it = _model(case, seed)
    s = dict(path=case["path"], model=m, holland=run.holland, it=it, steps=case["steps"])
    if case["path"] == "step":
        # the host's met forcing of the coming steps (WSX2, WSY2, PR2)
        s["forcing"] = []
        for k in range(8):
            m.holland((it + k) * run.dtdp, run.holland)
            s["forcing"].append(tuple(m.get(f) for f in ("wsx2", "wsy2", "pr2")))
    return s


def _fields(m):
    return {k: m.get(k) for k in ("eta2", "uu2", "vv2", "nodecode")}


def run(state):
    path = state["path"]
    if path in ("jcg", "jcg_noalloc"):
        # the caller's own arrays: the solve scales and unscales COEF and the
        # right-hand side in place and leaves the solution in u
        rhs, u = state["rhs"].copy(), state["u"].copy()
        iparm = np.array([state["itmax"], 0, 0, 16, 0, 1, 1, 0, -2, 0, 0, 3], np.int32)
        rparm = np.zeros(12)
        rparm[:5] = state["zeta"], 0.0, 0.0, 0.75, 1.0
        jcg(state["coef"], state["jcoef"], rhs, u, iparm, rparm, noalloc=path == "jcg_noalloc")
        return {"u": u, "rhs": rhs, "coef": state["coef"]}
    it, n = state["it"], state["steps"]
    state["it"] = it + n
    if path == "batch":
        state["batch"].run(it, n, holland=state["holland"])
        return [_fields(m) for m in state["models"]]
    m = state["model"]
    if path == "step":
        for k in range(n):
            m.timestep(it + k, state["forcing"][(it + k) % len(state["forcing"])])
    else:
        m.run_resident(it, n, holland=state["holland"])
    return _fields(m)


def work(case):
    """Per solve iteration the products and vector updates (2 operations per
    matrix entry, 20 per row); per step the element terms.  Bytes: the nodal
    state and forcing read and written once per step (20 and 14 doubles), the
    nodal and element tables read once per step, the matrix formed and read
    once per solve; a solve's iterations need no more than that."""
    np_ = case["nodes"]
    ne, z = 2 * np_, 6 * np_
    k = 15
    solve_flops = k * (2.0 * z + 20.0 * np_)
    if case["path"] in ("jcg", "jcg_noalloc"):  # the system read, and what is written back
        return {"bytes": 12.0 * (z + np_) + 16.0 * np_ + 8.0 * (z + np_) + 16.0 * np_,
                "flops": solve_flops}
    steps = case["steps"] * case.get("members", 1)
    word = 4 if case.get("precision") == "mixed" else 8
    solve = not case.get("lumped")
    step_bytes = 8.0 * (20 + 14) * np_ + 8.0 * 8 * np_ + (12 + 3 * word) * ne
    step_flops = 500.0 * ne + 100.0 * np_
    if solve:
        step_bytes += 12.0 * (z + np_) + 8.0 * 6 * np_
        step_flops += solve_flops
    out = 28.0 * np_ * case.get("members", 1)
    return {"bytes": steps * step_bytes + out, "flops": steps * step_flops}


# ------------------------------------------------------------------ 64 bits
def _cg(coef, cols, rhs, x):
    """Conjugate gradients with the diagonal as preconditioner, run until the
    residual is at rounding level: coef, cols [w, n], diagonal in row 0."""
    d = coef[0]
    r = rhs - (coef * x[cols]).sum(0)
    zv = r / d
    p, rz = zv.copy(), float(r @ zv)
    stop = 1.0e-30 * max(float(rhs @ (rhs / d)), 1.0e-300)
    for _ in range(2000):
        if rz <= stop:
            break
        q = (coef * p[cols]).sum(0)
        a = rz / float(p @ q)
        x = x + a * p
        r = r - a * q
        zv = r / d
        new = float(r @ zv)
        p = zv + new / rz * p
        rz = new
    return x


def exact(case, seed):
    if case["path"] in ("jcg", "jcg_noalloc"):
        jcoef, coef, rhs, u, _ = _system(case, seed)
        n = rhs.shape[0]
        cols = np.maximum(jcoef.reshape(-1, n) - 1, 0)
        return {"u": _cg(coef.reshape(-1, n), cols, rhs, u), "rhs": rhs, "coef": coef}
    if (case["path"] != "run" or case["mesh"] != "basin" or case["tide"] or case["lumped"]
            or case["start"] == "learned" or case["nodes"] * case["steps"] > 1200000):
        # wetting and drying decides by thresholds: no value to be near to
        return None
    return _basin(case, seed)


def _basin(case, seed):
    """The basin's steps without wet/dry and wind: the generalized wave
    continuity equation and the explicit momentum equation, FP64."""
    t, run, emo, efa, fric, eta2 = _inputs(case, seed)
    n, g, dt = t["np"], run.g, run.dtdp
    dp, tau0 = t["dp"], prep.tau0_nodal(run.tau0, t["dp"])
    nm, k = _elements(t, run, dp, tau0)
    fx, fy = t["fdxe"].reshape(-1, 3), t["fdye"].reshape(-1, 3)
    area2 = t["areas"]
    w = t["mnei"]
    cols = np.maximum(np.asarray(t["neitab"]).reshape(w, n).astype(np.int64) - 1, 0)
    coef = np.zeros((w, n))
    np.add.at(coef[0], nm.ravel(), np.einsum("eii->ei", k).ravel())
    csr = t["csr"].reshape(-1, 3, 2).astype(np.int64) - 1
    for a in range(3):
        for b, c in enumerate([c for c in range(3) if c != a]):
            np.add.at(coef, (csr[:, a, b], nm[:, a]), k[:, a, c])
    nbd = t["nbd"].astype(np.int64) - 1
    free = np.ones(n, bool)
    free[nbd] = False
    inner = coef * (free[None, :] & free[cols])
    inner[0][nbd] = 1.0
    total = np.bincount(nm.ravel(), np.repeat(area2 / 2.0, 3), n)
    dxy = lambda f: ((f[nm] * fx).sum(1), (f[nm] * fy).sum(1))  # noqa: E731
    avg = lambda f: f[nm].mean(1)  # noqa: E731
    scatter = lambda v: np.bincount(nm.ravel(), v.ravel(), n)  # noqa: E731
    e1 = e2 = eta2
    es = np.zeros(n)
    u = v = np.zeros(n)
    h = dp + e2
    qx = qy = np.zeros(n)
    evm = run.eslm
    lbc = t["lbcodei"][t["me2gw"] - 1]
    wall = t["nbv"][t["me2gw"] - 1].astype(np.int64) - 1
    cs, si = t["csii"][t["me2gw"] - 1], t["siii"][t["me2gw"] - 1]
    slip = (lbc >= 0) & (lbc <= 9)
    amig = run.amig
    for it in range(1, case["steps"] + 1):
        timeloc = it * dt + run.statim * 86400.0
        ramp = math.tanh((2.0 * timeloc / 86400.0) / run.drampelev) if run.nramp else 1.0
        bc = sum(emo[:, j] * run.ff[j] * ramp * np.cos(
            amig[j] * (it * dt) + math.radians(run.face[j]) - np.radians(efa[:, j]))
            for j in range(len(amig)))
        tk = np.minimum(fric * np.hypot(u, v) / (dp + e2), 2.0 / dt)
        # the load vector
        msr = 0.5 * area2 * (1.0 / dt - avg(tau0) / 2.0) / dt / 12.0
        jv = []
        sx, sy = dxy(es)
        sq = dxy(e2 * e2)
        for vel, q, grad, se in ((u, qx, dxy(u), sx), (v, qy, dxy(v), sy)):
            gsq = sq[len(jv)]
            jv.append(-g / (2.0 * area2) * gsq - avg(tk * q) - evm / dt * se / area2
                      + avg(tau0 * q) - (avg(qx) * grad[0] + avg(qy) * grad[1]) / area2
                      + avg(vel) * avg(es) / dt)
        gdp = g * avg(dp) / (2.0 * area2)
        g0, g1 = dxy(e1), dxy(e2)
        gt = dxy(tau0)
        spa = (avg(qx) * gt[0] + avg(qy) * gt[1]) / 6.0
        esn = es[nm]
        lv = ((esn + esn.sum(1)[:, None]) * msr[:, None]
              - gdp[:, None] * (run.c00 * (fx * g0[0][:, None] + fy * g0[1][:, None])
                                + (run.a00 + run.b00) * (fx * g1[0][:, None]
                                                         + fy * g1[1][:, None]))
              + (jv[0][:, None] * fx + jv[1][:, None] * fy) * 0.5 + spa[:, None])
        rhs = scatter(lv)
        known = np.zeros(n)
        known[nbd] = bc - e2[nbd]
        rhs = rhs - (coef * known[cols]).sum(0)
        rhs[nbd] = known[nbd]
        start = es.copy()
        start[nbd] = known[nbd]
        es = _cg(inner, cols, rhs, start)
        e1, e2 = e2, e2 + es
        h1, h = h, dp + e2
        # momentum
        ux, uy = dxy(u)
        vx, vy = dxy(v)
        bx, by = dxy(0.5 * (e1 + e2))
        mom = []
        for (dx, dy), press in (((ux, uy), bx), ((vx, vy), by)):
            adv = -0.5 * (avg(u) * dx + avg(v) * dy) - 0.5 * g * press
            lat = 1.5 * evm * (dx[:, None] * fx + dy[:, None] * fy) / area2[:, None]
            mom.append(scatter(dt * (adv[:, None] - lat)) / total)
        vxx = 0.5 * dt * tk
        cor = 0.5 * dt * run.cori
        mx = mom[0] + (1.0 - vxx) * u + cor * v
        my = mom[1] + (1.0 - vxx) * v - cor * u
        a0, a1, a2, a3 = 1.0 + vxx, 1.0 + vxx, np.full(n, -cor), np.full(n, cor)
        i, c, s = wall[slip], cs[slip], si[slip]
        mx[i], my[i] = s * mx[i] - c * my[i], 0.0
        a2[i], a3[i], a1[i] = -c * a0[i], c * a0[i], s * a0[i]
        a0[i] = s * a0[i]
        i = wall[(lbc >= 10) & (lbc <= 19)]
        mx[i] = my[i] = 0.0
        det = a0 * a1 - a2 * a3
        u, v = (mx * a1 - my * a2) / det, (my * a0 - mx * a3) / det
        qx, qy = u * h, v * h
    return {"eta2": e2, "uu2": u, "vv2": v, "nodecode": None}
