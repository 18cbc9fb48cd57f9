"""Runs whose units put the cell sizes outside the range of the stages' short
divisions: large launches take the general form and equal the oracle, as those
just inside do."""
import pytest

from test_gpu_short_forms import test_large_launch_equals_oracle as equals_oracle

pytestmark = pytest.mark.gpu


# 56 x 16 cells across the box: 2^73 and 2^74 lie on the two sides of cells of 2^64
@pytest.mark.parametrize("size", [2.0 ** 73, 2.0 ** 74, 2.0 ** -55, 2.0 ** -53])
def test_box_size(size):
    equals_oracle(dict(xmax=size, ymax=size))
