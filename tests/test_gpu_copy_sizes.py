"""States up and down unchanged, every cell of the padded tiles, at the edges of
the pieces of 32 MiB that a download goes by, and the primitives of a state at
rest."""
import numpy as np
import pytest

from walicxe2d_amd import params as P
from walicxe2d_amd.capi import Simulation

pytestmark = pytest.mark.gpu


# 12 800 bytes a block of four variables, 16 000 of five; block 0 is copied too
@pytest.mark.parametrize("neq,n", [(4, 1), (5, 64), (4, 2620), (4, 2621), (5, 4500)])
def test_round_trip(neq, n):
    cfg = P.config_c1(neq=neq, nbrootx=n, nbrooty=1, cooling="H" if neq >= 5 else "ADIABATIC", nblocks=n + 1)
    sim = Simulation(cfg)
    lp, ic = P.root_layout(cfg)
    leaf = np.ones(n + 1, dtype=np.int32)
    leaf[0] = 0
    u = np.random.default_rng(neq + n).uniform(1.0, 2.0, (n + 1, neq, P.NP, P.NP))
    u[:, 1:3] = 0.0
    sim.upload(u, lp, leaf, ic, n, n)
    assert np.array_equal(sim.download(), u)
    v, prim = sim.download(prim=True)
    assert np.array_equal(v, u) and np.array_equal(prim[1:, 0], u[1:, 0])
    sim.close()
