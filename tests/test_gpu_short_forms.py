"""The stage kernels' short divisions and square roots against the oracle, on a
mesh large enough for the launches that use them (56 x 56 blocks): states with
velocities from ordinary ones down to the last denormal and zero, so that both
the short forms and the general ones they leave cells to are reached within a
launch.  Every interior cell equals the oracle's, bit for bit."""
import numpy as np
import pytest

from walicxe2d_amd import params as P
from walicxe2d_amd.capi import Simulation
from wxoracle import MeshState, Oracle

pytestmark = pytest.mark.gpu


def _state(cfg, n, rng):
    """Random conserved states: density and pressure over a few decades, the
    velocities of a block scaled by one power of ten each, many exactly zero."""
    neq = cfg.neq
    u = np.zeros((n + 1, neq, P.NP, P.NP))
    shape = (n, P.NP, P.NP)
    rho = 10.0 ** rng.uniform(-1, 1, shape)
    block = 10.0 ** np.where(rng.random(n) < 0.4, 0.0, rng.uniform(-322, 0, n))
    v = [0.3 * rng.normal(size=shape) * block[:, None, None] * (rng.random(shape) < 0.8) for _ in range(2)]
    p = 10.0 ** rng.uniform(-1, 1, shape)
    p[rng.random(n) < 0.3] = 1.0          # uniform pressure: the star speed is the tiny velocities' alone
    u[1:, 0], u[1:, 1], u[1:, 2] = rho, rho * v[0], rho * v[1]
    u[1:, 3] = 0.5 * rho * (v[0] ** 2 + v[1] ** 2) + cfg.sc["cv"] * p
    if neq >= 5:
        u[1:, 4] = rho * rng.choice([0.0, 1e-4, 0.3, 1.0], size=shape)
    if neq >= 6:
        u[1:, 5] = -rho
    return u


@pytest.mark.parametrize("opts", [
    dict(), dict(limiter=2), dict(solver="HLL"), dict(solver="HLL", limiter=2), dict(solver="HLL_HLLC", limiter=2),
    dict(limiter=4), dict(cylindrical=True), dict(cylindrical=True, limiter=2, solver="HLL_HLLC", neq=6, cooling="H"),
    dict(neq=5, cooling="H"), dict(neq=6, cooling="H", limiter=2), dict(cooling="DMC"), dict(compat=0, neq=5, cooling="H"),
], ids=lambda o: "-".join(f"{k}{v}" for k, v in o.items()) or "default")
def test_large_launch_equals_oracle(opts):
    side = 56
    kw = dict(neq=4, cooling="ADIABATIC", compat=P.COMPAT_HLLC_TYPO, cfl=0.2)
    kw.update(opts)
    cfg = P.config_c1(nbrootx=side, nbrooty=side, nblocks=side * side + 2, **kw)
    n = side * side
    O, pp = Oracle(), cfg.params()
    m = MeshState(n + 2, cfg.neq)
    O.basegrid(pp, m)
    u = _state(cfg, n, np.random.default_rng(len(str(opts))))
    m.u[1:n + 1] = u[1:]
    for nb in range(1, n + 1):
        m.primit[nb] = O.calcprim(pp, m.u[nb])
    lp, ic = P.root_layout(cfg)
    leaf = np.ones(n + 1, dtype=np.int32)
    leaf[0] = 0
    sim = Simulation(cfg)
    sim.upload(u, lp, leaf, ic, n, n)
    t = 0.0
    for step in range(2):
        dt = O.timestep(pp, m)
        assert sim.timestep() == dt, step
        t += dt
        assert O.tstep(pp, m, t, dt) == 0
        sim.tstep(t, dt)
        got = sim.download()[1:, :, 2:18, 2:18]
        want = m.u[1:n + 1, :, 2:18, 2:18]
        bad = np.argwhere(got != want)
        assert bad.size == 0, (step, len(bad), bad[0], got[tuple(bad[0])], want[tuple(bad[0])])
    sim.close()
