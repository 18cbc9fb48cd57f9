"""wx_upload_tree's host part (set_tree, wx_mesh.cpp) is the copy of the tree's
arrays, and no slower than that: the shortest of 60 times against the shortest
of the plain copy loop, both in one program."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_set_tree_takes_the_time_of_its_copies(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = str(tmp_path / "set_tree_check")
    subprocess.run(["g++", "-std=c++17", "-O3", "-I", os.path.join(HERE, "hostsim"), "-I",
                    os.path.join(HERE, "..", "include"), os.path.join(HERE, "hostsim", "set_tree_check.cpp"),
                    os.path.join(HERE, "..", "walicxe2d_amd", "csrc", "wx_mesh.cpp"), "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe, "10240"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    ours, copy = map(float, r.stdout.split())
    assert ours < 1.6 * copy, (ours, copy)
