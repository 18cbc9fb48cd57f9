"""More of the hot kernels' register budgets, from the same compiler report as
tests/test_kernel_resources.py."""
import pytest

from test_kernel_resources import usage  # noqa: F401 (the fixture)


def test_two_wave_fill_only_at_the_same_occupancy(usage):  # noqa: F811
    """Two waves per block pay where as many waves fit a SIMD as with four."""
    forms = [k for k in usage if k.startswith("wx::k_fillI_cool<") and ", false, 128, false>" in k]
    assert forms
    for k in forms:
        assert usage[k]["waves"] >= usage[k.replace("128", "256")]["waves"], (k, usage[k])


@pytest.mark.parametrize("kernel,waves,scratch", [
    ("k_stageA_mild<5, 512>", 8, 32),                # a few spills that stay in the caches
    ("k_stageA_dt<5>", 4, 0),                        # few blocks: two workgroups a compute unit
    ("k_stageB<5, 256, false>", 5, 0),
    ("k_stageB<5, 512, false>", 5, 0),
    ("k_stageB_mild<5, 256>", 5, 0),
    ("k_stageB_mild<4, 256>", 5, 0),
    ("k_fillI_cool<5, false, 128, false>", 5, 0),
    ("k_fillI_cool<5, false, 256, false>", 5, 0),
    ("k_fillI_cool<5, false, 384, false>", 5, 0),
    ("k_fillI_cool<5, true, 256, false>", 4, 0),     # the learned cooling
])
def test_main_path_budgets(usage, kernel, waves, scratch):  # noqa: F811
    r = usage["wx::" + kernel]
    assert r["waves"] >= waves, (kernel, r)
    assert r["scratch"] <= scratch, (kernel, r)
