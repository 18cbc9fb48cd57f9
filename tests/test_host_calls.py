"""Sequences of calls a host program makes, through the host runtime built for
the CPU under sanitizers (tests/hostsim/host_calls_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "walicxe2d_amd", "csrc")
SOURCES = [os.path.join(HERE, "hostsim", "host_calls_check.cpp")] + [
    os.path.join(CSRC, f) for f in ("wx_host.cpp", "wx_mesh.cpp", "wx_runtime.cpp", "wx_ensemble.cpp")]


def _build(tmp_path_factory, sanitizers):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    out = tmp_path_factory.mktemp("calls")
    flags = ["g++", "-std=c++17", "-O1", "-g", "-fsanitize=" + sanitizers]
    inc = ["-I", os.path.join(HERE, "hostsim"), "-I", os.path.join(HERE, "..", "include")]
    objs = [str(out / (os.path.basename(s) + ".o")) for s in SOURCES]
    for p in [subprocess.Popen(flags + inc + ["-c", s, "-o", o]) for s, o in zip(SOURCES, objs)]:
        assert p.wait() == 0
    exe = str(out / "host_calls_check")
    subprocess.run(flags + objs + ["-o", exe, "-lpthread"], check=True)
    return exe


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return _build(tmp_path_factory, "address,undefined")


@pytest.fixture(scope="module")
def program_tsan(tmp_path_factory):
    return _build(tmp_path_factory, "thread")


def _run(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr[-4000:]


def test_own_list_after_a_rejected_one(program):
    _run(program, "rejected_list")


def test_builder_of_new_trees(program):
    _run(program, "builder_of_new_trees")


def test_info_of_an_unchecked_tree(program):
    _run(program, "info_of_an_unchecked_tree")


def test_downloads_only_read(program, program_tsan):
    _run(program, "downloads")
    _run(program_tsan, "downloads")


def test_general_form_of_the_stages(program):
    _run(program, "general_form")


def test_profile_counts_launches(program):
    _run(program, "profile_counts")
