"""The surrogate kernels' register budgets, as the compiler reports them
(hipcc -Rpass-analysis=kernel-resource-usage on wx_surrogate.hip, gfx950).
Built for the device only; no GPU needed."""
import os
import re
import shutil
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT


@pytest.fixture(scope="module")
def usage(tmp_path_factory):
    if not os.path.exists(HIPCC) or shutil.which("c++filt") is None:
        pytest.skip("hipcc not available")
    cmd = [HIPCC, "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-fno-fast-math", "--offload-arch=gfx950",
           "-fno-gpu-rdc", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-c",
           os.path.join(ROOT, "walicxe2d_amd", "csrc", "wx_surrogate.hip"), "-o",
           str(tmp_path_factory.mktemp("ru") / "s.o"), "-Rpass-analysis=kernel-resource-usage"]
    err = subprocess.run(cmd, capture_output=True, text=True, check=True).stderr
    res, name = {}, None
    for line in err.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = subprocess.run(["c++filt", m.group(1)], capture_output=True, text=True).stdout.strip()
            name = name.split("(")[0].replace("void ", "")
            res[name] = {}
        for key, pat in (("scratch", r"ScratchSize \[bytes/lane\]: (\d+)"), ("sgpr_spill", r"SGPRs Spill: (\d+)"),
                         ("waves", r"Occupancy \[waves/SIMD\]: (\d+)")):
            m = re.search(pat, line)
            if m and name:
                res[name][key] = int(m.group(1))
    return res


def test_inference_of_few_samples_takes_one_group_a_wave(usage):
    # a wave of one group of 16 samples: no more registers than leave room for three
    r = usage["wx::k_sur_infer<1>"]
    assert r["waves"] >= 3 and r["scratch"] == 0, r
