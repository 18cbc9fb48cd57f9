"""The default choice of the table builder on a new tree of 6 144 leaves and
more, which the device compiles, and the small changes after it, which the host
takes over, against the host's compilation throughout."""
import pytest

from test_gpu_builder import _pair
from walicxe2d_amd import params as P

pytestmark = pytest.mark.gpu


def test_new_tree_then_small_changes():
    cfg = P.config_c5(3, nbrootx=136, nbrooty=46, xmax=8.5, ymax=2.875, xphys=8.5e17, nlevs=3, nblocks=20000)
    assert _pair(cfg, 60, cfg.nblocks, 12, mode=3) >= 6144
