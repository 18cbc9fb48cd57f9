"""A block whose CFL partial is NaN: the minimum over the blocks is the other
blocks', as long as each block's partial enters it once."""
import numpy as np
import pytest

from walicxe2d_amd import params as P
from walicxe2d_amd.capi import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rx,ry", [(3, 1), (5, 7)])
def test_nan_in_the_last_block(rx, ry):
    n = rx * ry
    cfg = P.config_c1(nbrootx=rx, nbrooty=ry, nblocks=n + 2)
    lp, ic = P.root_layout(cfg)
    leaf = np.ones(n + 1, dtype=np.int32)
    leaf[0] = 0
    u = np.zeros((n + 1, 4, P.NP, P.NP))
    u[1:, 0] = 1.0
    u[1:, 3] = np.linspace(1.0, 2.0, n)[:, None, None]   # the last block's dt alone is the smallest
    sim = Simulation(cfg)
    v = u.copy()
    v[n, 3] = 1.0
    sim.upload(v, lp, leaf, ic, n, n)
    dts = [sim.timestep()]
    v = u.copy()
    v[n - 1, 3] = 3.0
    want = []
    for last in (1.0, np.nan):   # the last block slow, then NaN: the one before it decides
        w = v.copy()
        w[n, 3] = 1.0
        w[n, 1] = 0.0 if last == 1.0 else np.nan
        sim.upload(w, lp, leaf, ic, n, n)
        want.append(sim.timestep())
    assert want[1] == want[0] < dts[0]
    sim.close()
