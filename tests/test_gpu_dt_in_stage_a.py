"""wx_step's dt, which stage A takes itself on up to 512 blocks, against
wx_timestep's reduction and wx_tstep: time, dt and every cell to the bit."""
import numpy as np
import pytest

from test_gpu_short_forms import _state
from walicxe2d_amd import params as P
from walicxe2d_amd.capi import Simulation

pytestmark = pytest.mark.gpu


def _both(a, b, t):
    for s in range(3):
        ta, dta, _ = a.step(1, admesh=False)
        dtb = b.timestep()
        t += dtb
        b.tstep(t, dtb)
        assert np.array_equal([ta, dta], [t, dtb]), s
        assert np.array_equal(a.download(), b.download()), s
    a.close()
    b.close()


# one block, a wave's and a workgroup's edges, the last size and the first past it
@pytest.mark.parametrize("rx,ry", [(1, 1), (8, 8), (13, 5), (16, 32), (27, 19)])
@pytest.mark.parametrize("neq,cooling", [(4, "DMC"), (5, "H"), (6, "H")])
def test_random_states(rx, ry, neq, cooling):
    n = rx * ry
    cfg = P.config_c1(nbrootx=rx, nbrooty=ry, nblocks=n + 2, neq=neq, cooling=cooling, cfl=0.2)
    u = _state(cfg, n, np.random.default_rng(n + neq))
    lp, ic = P.root_layout(cfg)
    leaf = np.ones(n + 1, dtype=np.int32)
    leaf[0] = 0
    sims = [Simulation(cfg), Simulation(cfg)]
    for s in sims:
        s.upload(u, lp, leaf, ic, n, n)
    _both(*sims, 0.0)


def test_jet_source():
    cfg = P.config_c5(3, nbrootx=16, nbrooty=4, xmax=1.0, ymax=0.25, xphys=1.e17, nlevs=2, nblocks=200)
    sims = [Simulation(cfg), Simulation(cfg)]
    for s in sims:
        s.basegrid()
    _both(*sims, 0.0)
