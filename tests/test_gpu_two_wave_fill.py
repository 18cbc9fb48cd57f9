"""The fill's two-wave form (launches of 8 192 blocks and more with n_HI)
against the oracle: a step's cells and the next step's dt to the bit, and the
refinement flags against those of the statistics kernel on the same state."""
import numpy as np
import pytest

from test_gpu_short_forms import _state
from walicxe2d_amd import params as P
from walicxe2d_amd.capi import Simulation
from wxoracle import MeshState, Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("neq,rx,ry", [(5, 64, 128), (5, 91, 91), (6, 128, 65)])   # the first such launch, and odd ones
def test_equals_oracle(neq, rx, ry):
    n = rx * ry
    cfg = P.config_c1(nbrootx=rx, nbrooty=ry, nblocks=n + 2, neq=neq, cooling="H", compat=P.COMPAT_HLLC_TYPO, cfl=0.2,
                      nlevs=2)
    O, pp = Oracle(), cfg.params()
    m = MeshState(n + 2, neq)
    O.basegrid(pp, m)
    u = _state(cfg, n, np.random.default_rng(neq + n))
    m.u[1:n + 1] = u[1:]
    for nb in range(1, n + 1):
        m.primit[nb] = O.calcprim(pp, m.u[nb])
    lp, ic = P.root_layout(cfg)
    leaf = np.ones(n + 1, dtype=np.int32)
    leaf[0] = 0
    sim = Simulation(cfg)
    sim.upload(u, lp, leaf, ic, n, n)
    dt = O.timestep(pp, m)
    assert sim.timestep() == dt
    assert O.tstep(pp, m, dt, dt) == 0
    sim.tstep(dt, dt)
    got = sim.download()
    bad = np.argwhere(got[1:, :, 2:18, 2:18] != m.u[1:n + 1, :, 2:18, 2:18])
    assert bad.size == 0, (len(bad), bad[0])
    assert sim.timestep() == O.timestep(pp, m)
    flags = sim.criteria()
    sim.upload(got, lp, leaf, ic, n, n)
    for a, b in zip(flags, sim.criteria()):
        assert np.array_equal(a, b)
    sim.close()
