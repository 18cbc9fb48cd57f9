"""The workloads this framework's throughput is watched on: whole passes
through the public entry points of `walicxe2d_amd.capi` and
`walicxe2d_amd.surrogate`, as a program that runs the code calls them.

A pass of a single mesh (`kind` "mesh") is the inner part of a run: restart
from a saved state, `steps` iterations of the time loop (timestep, tstep,
admesh) on the GPU, and the dump of every leaf block.  A pass of an ensemble
(`kind` "ensemble") advances all instances by `steps` and dumps them (the jets
go on from where they are, the supernovae start at t = 0).  The
"host" pass is the loop of a Fortran host that keeps the tree itself
(timestep, tstep and criteria through their own entry points).  "pairs",
"infer" and "train" are the three device passes of the surrogate's training
program.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the pass
    run(state)          one pass
    work(case)          the bytes and operations it cannot do without
    exact(case, seed)   the pass in plain numpy, where that is feasible
"""
from __future__ import annotations

import ctypes
import math

import numpy as np

from walicxe2d_amd import params as P
from walicxe2d_amd import surrogate as S
from walicxe2d_amd.capi import Ensemble, Simulation


def _leaves(case):
    """Leaf blocks of a pass, about (as seen on the listed meshes); work() only."""
    roots, levels = case["rootx"] * case["rooty"], case["nlevs"] or 4.5   # 0: 3 to 6 levels
    more = {"explosion": 0., "supernova": 80. * (levels - 1), "jet": 50. * (levels - 1)}[case["problem"]]
    return (roots + more) * case.get("instances", 1)


def _mesh(name, problem, roots, nlevs, warm, steps, **kw):
    c = dict(name=name, kind="mesh", problem=problem, rootx=roots[0], rooty=roots[1], nlevs=nlevs, warm=warm,
             steps=steps, solver="HLLC", limiter=1, neq=5 if problem == "jet" else 4, cylindrical=False,
             surrogate=False)
    c.update(kw)
    return c


def _ens(name, problem, roots, nlevs, instances, warm, steps, **kw):
    c = _mesh(name, problem, roots, nlevs, warm, steps, instances=instances, groups=2)
    c.update(kind="ensemble", **kw)
    return c


def listed():
    return [
        # the point explosion on one level, 4x4 root blocks: its whole run of
        # 200 steps from t = 0; 16 workgroups a launch, so launches and
        # latency count
        _mesh("explosion_4x4", "explosion", (4, 4), 1, 0, 200),
        # the supernova with 5 levels of refinement and the tabulated cooling
        # (8x8 roots, a few hundred leaves), the mesh changing as the shell moves
        _mesh("supernova_5_levels", "supernova", (8, 8), 5, 200, 400),
        # the cooling jet (64x16 roots, 4 levels, reflective axis): the main
        # single-mesh workload
        _mesh("jet_64x16", "jet", (64, 16), 4, 200, 400),
        # the same jet on a mesh large enough for the device-built tables
        _mesh("jet_144x36", "jet", (144, 36), 4, 100, 300),
        # the options other than the default ones: hybrid solver, van Leer
        # limiter, axisymmetric sources and a passive scalar, on an odd layout
        _mesh("jet_cylindrical_hybrid", "jet", (37, 11), 3, 100, 400, solver="HLL_HLLC", limiter=2, neq=6,
              cylindrical=True),
        # the throughput workload: 16 jet variants in one ensemble, two groups
        _ens("jet_ensemble_16", "jet", (64, 16), 4, 16, 100, 400),
        # a parameter study of supernovae with 3 to 6 levels, many small meshes
        _ens("supernova_ensemble_48", "supernova", (4, 4), 0, 48, 100, 300),
        # jet variants with the learned cooling in place of coolingh
        _ens("jet_ensemble_surrogate", "jet", (32, 8), 4, 8, 100, 300, surrogate=True),
        # a host program that keeps the tree and calls the routines one by one
        dict(name="host_driven_supernova", kind="host", problem="supernova", rootx=16, rooty=16, nlevs=4, warm=60,
             steps=100, solver="HLLC", limiter=1, neq=4, cylindrical=False, surrogate=False),
        # training pairs and features of harvested cells, the surrogate's data
        dict(name="cooling_pairs_1m", kind="pairs", n=1_000_003),
        # evaluation of a trained network on held-out cells
        dict(name="surrogate_infer_2m", kind="infer", n=2_000_005),
        # training steps at the trainer's default batch
        dict(name="surrogate_train_16384", kind="train", n=200_000, batch=16384, steps=200),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mesh", "mesh", "mesh", "ensemble", "ensemble", "host", "pairs", "infer", "train"])
    if kind == "pairs":
        return dict(kind="pairs", n=_log_int(rng, 1000, 1_000_000))
    if kind == "infer":
        return dict(kind="infer", n=_log_int(rng, 1000, 2_000_000))
    if kind == "train":
        batch = _log_int(rng, 250, 16384)
        return dict(kind="train", n=_log_int(rng, batch, 200_000), batch=batch, steps=rng.randint(20, 200))
    problem = rng.choice(["explosion", "supernova", "jet"]) if kind == "mesh" else rng.choice(["supernova", "jet"])
    lim, solver = rng.choice([1, 1, 2]), rng.choice(["HLLC", "HLLC", "HLL", "HLL_HLLC"])
    if problem == "explosion":
        c = _mesh("", problem, (_log_int(rng, 3, 40), _log_int(rng, 3, 40)), 1, 0, rng.randint(100, 250))
    elif problem == "supernova":
        n = _log_int(rng, 4, 16)
        c = _mesh("", problem, (n, n), rng.randint(3, 5), rng.randint(30, 100), rng.randint(100, 300))
    else:
        ry = _log_int(rng, 6, 28)
        c = _mesh("", problem, (ry * rng.randint(2, 4) + rng.randint(0, 3), ry), rng.randint(2, 4),
                  rng.randint(30, 100), rng.randint(100, 300), neq=rng.choice([5, 5, 6]),
                  cylindrical=rng.random() < 0.3)
    c.update(solver=solver, limiter=lim)
    if kind == "host":
        c.update(kind="host", steps=rng.randint(50, 100))
    if kind == "ensemble":
        if problem == "supernova":
            c.update(rootx=4, rooty=4, nlevs=0)
        else:
            c.update(rootx=rng.randint(12, 32), rooty=rng.randint(4, 8), surrogate=rng.random() < 0.3)
        c.update(kind="ensemble", instances=rng.randint(2, 10), groups=rng.randint(1, 3))
    c.pop("name")
    return c


# --------------------------------------------------------------------------
def _config(case, seed, i=0):
    """The run's configuration; the seed draws the explosion's energy, place
    and medium, or the jet's speed and density."""
    rng = np.random.default_rng(seed)
    rx, ry, nl = case["rootx"], case["rooty"], case["nlevs"]
    opts = dict(solver=case["solver"], limiter=case["limiter"], neq=case["neq"], cylindrical=case["cylindrical"],
                nbrootx=rx, nbrooty=ry)
    if case["problem"] == "explosion":
        # the hazard-free boundary order, so that the run has a closed form on
        # the whole grid; the energy in a disc of about 1/50 of the box
        return P.config_c1(compat=P.COMPAT_HLLC_TYPO, xmax=rx / 4., ymax=ry / 4., nlevs=1,
                           nblocks=rx * ry + 8,
                           ic_args=dict(rho=1.0, p=1e-5, E=rng.uniform(0.5, 2.0), r=0.04,
                                        xc=rx / 4. * rng.uniform(0.4, 0.6), yc=ry / 4. * rng.uniform(0.4, 0.6)),
                           **opts)
    if case["problem"] == "supernova":
        if nl == 0:
            # energy, medium and place drawn; 3 to 6 levels
            nl = 3 + i % 4
            c = P.config_c4(int(rng.integers(0, 1 << 20)), nlevs=nl, nblocks={3: 600, 4: 1200, 5: 2400, 6: 4000}[nl])
            opts["nbrootx"] = opts["nbrooty"] = 4
        else:
            c = P.config_c2(nlevs=nl, nblocks=rx * ry * 16 + 1500)
            c.ic_args = dict(c.ic_args, n=10.0 ** rng.uniform(-0.5, 0.5), E=10.0 ** rng.uniform(50.7, 51.3),
                             xc=rng.uniform(0.3, 0.7), yc=rng.uniform(0.3, 0.7))
            # a wider initial ball on wide boxes, so that the root grid sees it
            c.ic_args["R"] = max(c.ic_args["R"], 40. * P.PC / (16 * rx) * 1.5)
        for k, v in opts.items():
            setattr(c, k, v)
        return c
    c = P.config_c5(int(rng.integers(0, 1 << 20)), xmax=4.0 * rx / 64, ymax=ry / 16., xphys=4.e17 * rx / 64,
                    nlevs=nl, nblocks=rx * ry * 2 + 2000, **opts)
    return c


def _start(cfg, warm):
    """A run developed by `warm` steps from its initial state."""
    sim = Simulation(cfg)
    sim.basegrid()
    if cfg.nlevs > 1:
        for _ in range(4):
            sim.admesh()
    if warm:
        sim.step(warm)
    return sim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mesh" or kind == "host":
        cfg = _config(case, seed)
        sim = _start(cfg, case["warm"])
        lp, leaf, ic, nbmax, nl = sim.tree()
        return dict(case=case, sim=sim, u=sim.download(), tree=(lp, leaf, ic, nbmax, nl), time=sim.time,
                    amr=cfg.nlevs > 1, leaf_rows=np.isin(np.arange(1, cfg.nblocks + 1), np.nonzero(leaf)[0]))
    if kind == "ensemble":
        cfgs = [_config(case, 1000 * seed + i, i) for i in range(case["instances"])]
        ens = Ensemble(cfgs, groups=min(case["groups"], len(cfgs)))
        ens.basegrid()
        for _ in range(4):
            ens.admesh()
        if case["surrogate"]:
            ens.set_surrogate(S.SurrogateModel.load())
        ens.step(case["warm"])
        ens.set_graph(True)
        return dict(case=case, ens=ens, roots=[np.ascontiguousarray(P.initial_state(c)[0]) for c in cfgs])
    if kind == "pairs":
        return dict(case=case, params=P.config_c5(0).params(), states=_cells(case["n"], seed))
    if kind == "infer":
        m = S.SurrogateModel.load()
        return dict(case=case, model=m, x=_features(case["n"], seed)[0])
    x, t = _features(case["n"], seed)
    return dict(case=case, x=x, t=t, seed=seed)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mesh":
        sim = state["sim"]
        sim.upload(state["u"], *state["tree"])
        sim.set_time(state["time"])
        t, dt, zones = sim.step(case["steps"], admesh=state["amr"])
        return dict(u=_leaf_cells(sim.download(), sim.tree(), sim.cap), time=t, dt=dt, zones=zones)
    if kind == "host":
        sim = state["sim"]
        sim.upload(state["u"], *state["tree"])
        sim.locatebounds()
        t, dts = state["time"], []
        for _ in range(case["steps"]):
            dt = sim.timestep()
            t += dt
            sim.tstep(t, dt)
            up, down = sim.criteria()
            dts.append(dt)
        # u(nb, ieq, i, j) with nb fastest, over the host's nblocks rows; its
        # leaf rows are what the run writes
        u = sim.download_fortran(sim.cap).reshape(P.NP, P.NP, case["neq"], sim.cap)[2:18, 2:18]
        u = np.where(state["leaf_rows"], u, 0.0)
        return dict(u=u, dt=np.array(dts), refine=up, coarsen=down)
    if kind == "ensemble":
        ens = state["ens"]
        if case["problem"] == "supernova":
            # a study of explosions starts each batch from t = 0; the jets run on
            for i, u in enumerate(state["roots"]):
                ens.L.wx_ens_basegrid(ens.h, i, u.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), u.shape[0] - 1)
            for _ in range(4):
                ens.admesh()
        zones = ens.step(case["steps"])
        out = [_leaf_cells(ens.download(i), ens.tree(i), c.nblocks) for i, c in enumerate(ens.cfgs)]
        return dict(u=out, zones=zones)
    if kind == "pairs":
        f, cedt = S.features(state["params"], state["states"])
        return dict(pairs=S.exact_pairs(state["params"], state["states"]), features=f, cedt=cedt)
    if kind == "infer":
        return S.infer(state["model"], state["x"])
    model = S.SurrogateModel(seed=state["seed"])
    hist = S.train_steps(model, state["x"], state["t"], case["batch"], case["steps"], 1e-3, 1e-4)
    return dict(theta=model.theta, loss=hist)


def _leaf_cells(u, tree, cap):
    """The interior cells of the leaf blocks, by block ID as a host's arrays
    of `cap` blocks hold them (zero where an ID is not a leaf)."""
    out = np.zeros((cap + 1, u.shape[1], 16, 16))
    ids = np.nonzero(tree[1])[0]
    out[ids] = u[ids, :, 2:18, 2:18]
    return out


# --------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("mesh", "host", "ensemble"):
        leaves = _leaves(case)
        zones = leaves * 256 * case["steps"]
        # two stages of five passes over the variables; per zone about 1300
        # operations of hydro, 700 more of coolingh
        state = leaves * case["neq"] * 400 * 8
        return dict(bytes=zones * 5 * case["neq"] * 8 + 2 * state,
                    flops=zones * (2000. if case["problem"] == "jet" else 1300.))
    n = case["n"]
    if kind == "pairs":
        return dict(bytes=n * (2 * 32 + 16 + 20), flops=n * 1000.)
    mac = 4 * 64 + 2 * 64 * 64 + 64 * 2
    if kind == "infer":
        return dict(bytes=n * 24 + S.NPARAM * 4, flops=n * 2. * mac)
    return dict(bytes=case["steps"] * (case["batch"] * 24 + S.NPARAM * 40), flops=case["steps"] * case["batch"] * 6. * mac)


# --------------------------------------------------------------------------
# inputs of the surrogate's passes
def _cells(n, seed):
    """Cell states (n, T, y0, dt[s]) as harvested from jets: the medium, the
    shocked gas between 1e4 and 1e6 K and the cooled shell."""
    rng = np.random.default_rng(seed)
    T = 10.0 ** np.where(rng.random(n) < 0.4, rng.normal(3.0, 0.05, n), rng.uniform(3.0, 5.8, n))
    hot = 1.0 / (1.0 + np.exp((np.log10(T) - 4.2) / 0.1))
    y0 = np.clip(hot * rng.uniform(0.9, 1.0, n), 1e-4, 1.0 - 1e-4)
    dens = 10.0 ** rng.uniform(1.0, 4.0, n)
    dt = 10.0 ** rng.uniform(5.0, 6.3, n)
    return np.stack([dens, T, y0, dt], axis=1)


def _features(n, seed):
    """Standardised features and smooth targets."""
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n, 4)).astype(np.float32)
    t = np.stack([np.sin(x[:, 0]) * x[:, 1] + 0.1 * x[:, 2], np.cos(x[:, 3]) - 0.5 * x[:, 0]], axis=1)
    return x, t.astype(np.float32)


# --------------------------------------------------------------------------
# the passes in plain numpy, 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind == "pairs":
        return _exact_pairs(case, seed)
    if kind == "infer":
        m = S.SurrogateModel.load()
        return _mlp(m.theta.astype(np.float64), _features(case["n"], seed)[0].astype(np.float64))
    if kind == "train":
        if case["steps"] * min(case["batch"], case["n"]) > 3_500_000:
            return None   # over 20 s
        return _exact_train(case, seed)
    if kind == "mesh" and case["problem"] == "explosion" and case["limiter"] in (1, 2) and case["solver"] != "HLL_HLLC":
        if case["steps"] * case["rootx"] * case["rooty"] > 20_000:
            return None
        return _exact_uniform(case, seed)
    return None   # an adaptive mesh of many blocks over hundreds of steps takes minutes


def _layers(theta):
    out, k = [], 0
    for o, i in ((64, 4), (64, 64), (64, 64), (2, 64)):
        out.append((theta[k:k + o * i].reshape(o, i), theta[k + o * i:k + o * i + o]))
        k += o * i + o
    return out


def _mlp(theta, x, keep=None):
    h = x
    for j, (w, b) in enumerate(_layers(theta)):
        z = h @ w.T + b
        if keep is not None:
            keep.append((h, z))
        h = z / (1.0 + np.exp(-z)) if j < 3 else z
    return h


def _exact_train(case, seed):
    x, t = (a.astype(np.float64) for a in _features(case["n"], seed))
    th = S.SurrogateModel(seed=seed).theta.astype(np.float64)
    m, v, hist = np.zeros_like(th), np.zeros_like(th), []
    n, steps, nb = case["n"], case["steps"], min(case["batch"], case["n"])
    for k in range(steps):
        idx = (k * nb % n + np.arange(nb)) % n
        keep = []
        y = _mlp(th, x[idx], keep)
        e = y - t[idx]
        hist.append(float((e * e).sum() / nb))
        d, g = 2.0 * e / nb, []
        for j in (3, 2, 1, 0):
            h, z = keep[j]
            if j < 3:
                s = 1.0 / (1.0 + np.exp(-z))
                d = d * (s * (1.0 + z * (1.0 - s)))
            g.insert(0, np.concatenate([(d.T @ h).ravel(), d.sum(axis=0)]))
            d = d @ _layers(th)[j][0]
        g = np.concatenate(g)
        lr = 1e-3 * (1e-4 / 1e-3) ** (k / (steps - 1) if steps > 1 else 0.0)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        th = th - lr * (m / (1 - 0.9 ** (k + 1))) / (np.sqrt(v / (1 - 0.999 ** (k + 1))) + 1e-8)
    return dict(theta=th, loss=np.array(hist))


def _aloss(y0, den, dh0, T):
    """Radiative losses of src/coolingh.f90:88-165."""
    te = np.maximum(T, 1000.)
    dhp = (1. - y0) * den
    de = dhp + 1e-4 * den
    lo = 0.5732 + te * (1.8288e-5 + te * (-1.15822e-10 + te * 9.4288e-16))
    hi = 0.5856 + te * (1.55083e-5 + te * (-9.669e-12 + te * 5.716e-19))
    fr = np.clip((te - 55000.) / 17000., 0., 1.)
    omega = (1. - fr) * lo + fr * hi
    ecoll = np.maximum(de * dh0 * 8.6287e-6 / (2. * np.sqrt(te)) * omega * np.exp(-118409. / te) * 1.634e-11, 0.)
    eion = de * dh0 * 5.834e-11 * np.sqrt(te) * np.exp(-1.579e5 / te) * 2.179e-11
    ex = np.exp(-2. * (np.clip(te, 44770., 54770.) - 49770.) / 500.)
    w = np.where(te <= 44770., 0., np.where(te >= 54770., 1., 0.5 * (1. + (1. - ex) / (1. + ex))))
    a = 157890. / te
    beta = 1.133e-24 / np.sqrt(a) * (-0.0713 + 0.5 * np.log(a) + 0.640 * a ** -0.33333)
    tm = 1. / te
    eoi = np.maximum(de * 1e-3 * dh0 * 10. ** (1381465. * tm * tm - 12328.69 * tm - 19.82621), 0.)
    eoii = np.maximum(de * 1e-3 * dhp * 10. ** (-2061075. * tm * tm - 14596.24 * tm - 19.01402), 0.)
    low = np.maximum(de * dhp * beta, 0.) + 7.033 * (eoi + eoii)
    high = 1.0455e-18 / te ** 0.63 * (1. - np.exp(-((te * 1e-5) ** 1.63))) * de * den + de * dhp * 1.3 * 1.42e-27 * te ** 0.5
    return ecoll + eion + low * (1. - w) + high * w


def _exact_pairs(case, seed):
    c = _cells(case["n"], seed)
    n, T0, y0, dt = c.T
    p = P.config_c5(0).params()
    uu4 = y0 * n
    T = np.maximum(1., T0)
    rec = 2.55e-13 * (1e4 / T) ** 0.79
    col = 5.83e-11 * np.sqrt(T) * np.exp(-157828. / T)
    xi = 1e-4
    a, b, cc = rec + col, -((2. + xi) * rec + (1. + xi) * col), (1. + xi) * rec
    d = np.sqrt(b * b - 4. * a * cc)
    g0 = (2. * a * y0 + b + d) / (2. * a * y0 + b - d)
    e = np.exp(-(d * n * dt))
    y1 = np.clip((-b - d * (1. + g0 * e) / (1. - g0 * e)) / (2. * a), 0.0001, 1.)
    dh0 = y1 * n
    ce = 2. * n * (_aloss(uu4 / n, n, dh0, T) / (n * n)) / (3. * 1.3807e-16 * T)
    t1 = np.maximum(np.minimum(np.maximum(10. + (T - 10.) * np.exp(-(ce * dt)), 0.1 * T), 10. * T), 10.)
    # features: ce from the bilinear table of log10 ALOSS/n^2
    nt, nx = 321, 81
    tg = 10.0 ** (1.0 + 0.025 * np.arange(nt))[:, None]
    rr = 10.0 ** (-4. + 8. * np.arange(nx) / (nx - 1))[None, :]
    xg = np.clip((rr * (1. + 1e-4) - 1e-4) / (1. + rr), 0., 1.)
    tab = np.log10(np.maximum(_aloss(1. - xg, 1., 1. - xg, tg + 0. * xg), 1e-300))
    x = 1. - y0
    ft = np.clip((np.log10(T0) - 1.0) / 0.025, 0., nt - 1 - 1e-3)
    fx = np.clip((np.log10((x + 1e-4) / (1. - x + 1e-4)) + 4.) * 0.125 * (nx - 1), 0., nx - 1 - 1e-3)
    it, ix = ft.astype(int), fx.astype(int)
    wt, wx = ft - it, fx - ix
    al = 10.0 ** ((1. - wt) * ((1. - wx) * tab[it, ix] + wx * tab[it, ix + 1])
                  + wt * ((1. - wx) * tab[it + 1, ix] + wx * tab[it + 1, ix + 1]))
    cedt = 2. * n * al / (3. * 1.3807e-16 * T0) * dt
    f = np.stack([np.log10(n), np.log10(T0), x, np.log10(np.maximum(cedt, 1e-30))], axis=1)
    return dict(pairs=np.stack([t1, y1], axis=1), features=f, cedt=cedt)


def _exact_uniform(case, seed):
    """The adiabatic one-level run on the whole grid: two-stage update with
    first-order then limited fluxes, outflow boundaries, the viscosity term."""
    cfg = _config(case, seed)
    p = cfg.params()
    cv, gam, ny, nx = p.cv, p.gamma, 16 * cfg.nbrooty, 16 * cfg.nbrootx
    dx, dy = p.dx[0], p.dy[0]
    u0, _, _ = P.initial_state(cfg)
    U = (u0[1:, :, 2:18, 2:18].reshape(cfg.nbrooty, cfg.nbrootx, 4, 16, 16).transpose(2, 0, 3, 1, 4)
         .reshape(4, ny, nx))

    def pad(a):
        return np.pad(a, ((0, 0), (2, 2), (2, 2)), mode="symmetric")

    def prim(a):
        r = np.maximum(a[0], 1e-15)
        vx, vy = a[1] / r, a[2] / r
        return np.stack([r, vx, vy, np.maximum((a[3] - 0.5 * r * (vx * vx + vy * vy)) / cv, 1e-15)])

    def cons(q):
        return np.stack([q[0], q[0] * q[1], q[0] * q[2], 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2) + cv * q[3]])

    def flux(q):
        e = 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2) + cv * q[3]
        return np.stack([q[0] * q[1], q[0] * q[1] * q[1] + q[3], q[0] * q[1] * q[2], q[1] * (e + q[3])])

    def avg(a, b):
        if case["limiter"] == 1:
            s = np.copysign(1., a)
            return s * np.maximum(0., np.minimum(np.abs(a), s * b))
        with np.errstate(all="ignore"):
            return np.where(a * b <= 0., 0., a * b * (a + b) / (a * a + b * b))

    def star(q, s, sst, right):
        smu = s - q[1]
        rs = q[0] * smu / (s - sst)
        ek = 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2) + cv * q[3]
        den = (q[3] if right else q[0]) * smu   # the reference's right-star energy
        us = np.stack([rs, rs * sst, rs * q[2], rs * (ek / q[0] + (sst - q[1]) * (sst + q[3] / den))])
        return flux(q) + s * (us - cons(q))

    def riemann(l, r):
        with np.errstate(all="ignore"):
            cl, cr = np.sqrt(gam * l[3] / l[0]), np.sqrt(gam * r[3] / r[0])
            sr, sl = np.maximum(l[1] + cl, r[1] + cr), np.minimum(l[1] - cl, r[1] - cr)
            if cfg.solver == "HLL":
                f = (sr * flux(l) - sl * flux(r) + sl * sr * (cons(r) - cons(l))) / (sr - sl)
            else:
                # the routine's own order: the right-star formula jumps at sst = 0
                ml, mr = sl - l[1], sr - r[1]
                sst = (mr * (r[0] * r[1]) - ml * (l[0] * l[1]) - r[3] + l[3]) / (mr * r[0] - ml * l[0])
                f = np.where(sst >= 0., star(l, sl, sst, False), star(r, sr, sst, True))
            return np.where(sl > 0., flux(l), np.where(sr < 0., flux(r), f))

    def faces(q, second):
        """Fluxes of the nx + 1 faces of every row of q (padded by 2)."""
        l, r = q[:, :, 1:-2], q[:, :, 2:-1]
        if second:
            ll, rr = q[:, :, :-3], q[:, :, 3:]
            l, r = l + 0.5 * avg(l - ll, r - l), r - 0.5 * avg(r - l, rr - r)
        return riemann(l, r)

    sw = [0, 2, 1, 3]

    def update(base, q, dt, second):
        F = faces(q[:, 2:-2], second)
        G = faces(q[sw][:, :, 2:-2].transpose(0, 2, 1), second)[sw].transpose(0, 2, 1)
        return base - dt / dx * (F[:, :, 1:] - F[:, :, :-1]) - dt / dy * (G[:, 1:] - G[:, :-1])

    t = 0.
    for _ in range(case["steps"]):
        q = prim(U)
        cs = np.sqrt(gam * q[3] / q[0])
        dt = p.cfl * min((dx / (np.abs(q[1]) + cs)).min(), (dy / (np.abs(q[2]) + cs)).min())
        t += dt
        H = update(U, prim(pad(U)), dt / 2., False)
        V = update(U, prim(pad(H)), dt, True)
        W = pad(U)[:, 1:-1, 1:-1]
        U = V + p.eta * (W[:, 1:-1, 2:] + W[:, 1:-1, :-2] + W[:, 2:, 1:-1] + W[:, :-2, 1:-1] - 4. * U)
    u = U.reshape(4, cfg.nbrooty, 16, cfg.nbrootx, 16).transpose(1, 3, 0, 2, 4).reshape(-1, 4, 16, 16)
    return dict(u=u, time=t, dt=dt, zones=float(256 * cfg.nbrootx * cfg.nbrooty * case["steps"]))
