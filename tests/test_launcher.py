"""How the library launches kernels (marian-dev_amd/csrc/abi_common.h), on the CPU: tests/launcher_check.cpp brings a
runtime of its own."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")


def build(exe, *options):
    return subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-isystem", "/opt/rocm/include", "-I", CSRC,
                           *options, "-o", exe, os.path.join(ROOT, "tests", "launcher_check.cpp")], capture_output=True, text=True, timeout=300)


@pytest.fixture(scope="module", autouse=True)
def headers():
    if not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("HIP headers not available")


def test_launcher(tmp_path):
    exe = str(tmp_path / "launcher_check")
    r = build(exe)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout


def test_kernels_are_launched_by_name_only(tmp_path):
    """A function is kept for one kernel.  A place that launches a kernel through a pointer, and so may launch several, kept the
    function of the first for all of them (the 128 x 128 tiles over several matrices, with and without streamed stores): it does not compile."""
    assert build(str(tmp_path / "by_pointer"), "-DKERNEL_BY_POINTER").returncode != 0
