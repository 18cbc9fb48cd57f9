"""The device's cell order behind the boundary: a state goes up and comes back
unchanged, every cell of the padded tiles included, in both layouts."""
import numpy as np
import pytest

from walicxe2d_amd import params as P
from walicxe2d_amd.capi import WX_LAYOUT_FORTRAN, Simulation, _check, _d, _i, tree_to_fortran

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("neq,rx,ry", [(4, 1, 1), (5, 3, 1), (6, 2, 2), (4, 5, 3)])   # odd and even numbers of tile variables
def test_state_round_trip(neq, rx, ry):
    cooling = "H" if neq >= 5 else "ADIABATIC"
    cfg = P.config_c1(neq=neq, nbrootx=rx, nbrooty=ry, cooling=cooling, nblocks=rx * ry + 3)
    sim = Simulation(cfg)
    lp, ic = P.root_layout(cfg)
    n = rx * ry
    leaf = np.ones(n + 1, dtype=np.int32)
    leaf[0] = 0
    u = np.random.default_rng(neq * 100 + n).uniform(1.0, 2.0, (n + 1, neq, P.NP, P.NP))
    u[0] = 0.0
    sim.upload(u, lp, leaf, ic, n, n)
    assert np.array_equal(sim.download(), u)
    assert np.array_equal(sim.download(), u)   # a download leaves the device's state as it was
    # u(nb, ieq, i, j), nb fastest
    want = u[1:].transpose(2, 3, 1, 0)
    f = sim.download_fortran().reshape(P.NP, P.NP, neq, n)
    assert np.array_equal(f, want)
    flp, fleaf, fic, ld = tree_to_fortran(lp, leaf, ic, n)
    g = np.ascontiguousarray(want[::-1]).reshape(-1)
    _check(sim.L.wx_upload(sim.h, _d(g), WX_LAYOUT_FORTRAN, _i(flp), _i(fleaf), _i(fic), ld, n, n), "wx_upload")
    assert np.array_equal(sim.download()[1:], g.reshape(P.NP, P.NP, neq, n).transpose(3, 2, 0, 1))
    sim.close()


@pytest.mark.parametrize("cooling", ["ADIABATIC", "DMC"])
def test_refine_and_coarse_tiles(cooling):
    """The padded tiles of a refined and re-coarsened block, cell by cell:
    injection of the parent's cells, then 2x2 means of the sons with the outer
    ghosts copied from the nearest cell."""
    cfg = P.config_c1(neq=4, nbrootx=1, nbrooty=1, nlevs=2, cooling=cooling, nblocks=8)
    sim = Simulation(cfg)
    lp0, _ = P.root_layout(cfg)
    lp = np.zeros((7, 8), dtype=np.int32)
    lp[:2] = lp0
    ic = np.zeros((7, 2), dtype=np.int32)
    leaf = np.array([0, 1, 0, 0, 0, 0, 0], dtype=np.int32)
    u = np.random.default_rng(9).uniform(1.0, 2.0, (7, 4, P.NP, P.NP))
    sim.upload(u, lp, leaf, ic, 6, 1)
    sim.refine(1, 2, 3, 4, 5)
    got = sim.download()
    k = np.arange(-1, 19)
    for s in range(4):
        si, sj = (k + 1) // 2 + 8 * (s & 1), (k + 1) // 2 + 8 * (s >> 1)
        assert np.array_equal(got[2 + s], u[1][:, sj + 1][:, :, si + 1]), s
    v = np.random.default_rng(10).uniform(1.0, 2.0, (7, 4, P.NP, P.NP))
    sim.upload(v, lp, leaf, ic, 6, 1)
    sim.coarse(1, 2, 3, 4, 5)
    c = np.clip(k, 0, 17)
    want = np.empty((4, P.NP, P.NP))
    for y in range(20):
        for x in range(20):
            sx, sy = int(c[x] > 8), int(c[y] > 8)
            t = v[2 + sx + 2 * sy]
            a, b = 2 * (c[x] - 8 * sx), 2 * (c[y] - 8 * sy)   # array indices of cells 2 l - 1
            want[:, y, x] = 0.25 * (((t[:, b, a] + t[:, b, a + 1]) + t[:, b + 1, a]) + t[:, b + 1, a + 1])
    assert np.array_equal(sim.download()[1], want)
    sim.close()
