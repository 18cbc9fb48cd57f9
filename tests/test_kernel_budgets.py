"""More of the hot kernels' register budgets, from the same compiler report as
tests/test_kernel_resources.py."""
from test_kernel_resources import usage  # noqa: F401 (the fixture)


def test_two_wave_fill_only_at_the_same_occupancy(usage):  # noqa: F811
    """Two waves per block pay where as many waves fit a SIMD as with four."""
    forms = [k for k in usage if k.startswith("wx::k_fillI_cool<") and ", false, 128, false>" in k]
    assert forms
    for k in forms:
        assert usage[k]["waves"] >= usage[k.replace("128", "256")]["waves"], (k, usage[k])
