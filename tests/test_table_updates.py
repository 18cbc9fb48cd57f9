"""The tables kept up to date from the rows of a mesh change equal a full
compilation of the tree (tests/hostsim/update_check.cpp), for both kinds of
bottom boundary, the OUTFYB mode, and with and without a jet source."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "walicxe2d_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = str(tmp_path_factory.mktemp("upd") / "update_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-I", os.path.join(HERE, "hostsim"),
                    "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "hostsim", "update_check.cpp"),
                    os.path.join(CSRC, "wx_mesh.cpp"), "-o", exe, "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("rx,ry,nlevs,otherb,compat,left,bottom", [
    (32, 8, 3, 1, 3, 0, 1),     # jet: reflective axis
    (32, 8, 3, 0, 3, 0, 0),     # OUTFYB
    (12, 9, 4, 1, 3, 0, 0),     # OUTFYB with a source
    (5, 7, 4, 1, 0, 1, 0),
    (2, 2, 5, 0, 2, 0, 0),
    (3, 1, 4, 0, 0, 1, 1),
    (1, 1, 5, 1, 3, 0, 0),
])
def test_tables_from_rows_match_full_compilation(program, rx, ry, nlevs, otherb, compat, left, bottom):
    r = subprocess.run([program] + [str(v) for v in (rx, ry, nlevs, otherb, compat, left, bottom, 250)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
