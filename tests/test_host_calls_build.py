"""The native host path belongs to the torch it was built against, and the C library is built without any torch."""
import os
import subprocess
import sys

from conftest import PKG, ROOT

CSRC = os.path.join(ROOT, PKG, "csrc")
LOAD = """
import importlib, sys, torch
{change}
_lib = importlib.import_module("marian-dev_amd._lib")
importlib.import_module("marian-dev_amd.integer")._host.prepare_a
print("loaded")
"""


def loading(change):
    return subprocess.run([sys.executable, "-c", LOAD.format(change=change)], cwd=ROOT, capture_output=True, text=True)


def test_host_calls_load_into_their_own_torch_only():
    assert loading("").stdout.strip().endswith("loaded")
    for other in ("2.9.1+rocm7.0", "2.10.0", "2.11.0+rocm7.0"):
        r = loading("torch.__version__ = {!r}".format(other))
        assert r.returncode != 0 and "loaded" not in r.stdout
        assert "MarianHipError" in r.stderr and "built for torch" in r.stderr and other in r.stderr, r.stderr


def test_the_c_library_is_built_without_torch():
    """`make` asks for no Python and names no torch; `make python` does"""
    def plan(*what):
        return subprocess.run(["make", "-C", CSRC, "-n", "-B", "PYTHON=false", *what], capture_output=True, text=True)
    r = plan()
    assert r.returncode == 0 and "libmarian_hip_int8.so" in r.stdout and "torch" not in r.stdout + r.stderr and "_host_calls" not in r.stdout
    assert "-ltorch" in plan("python").stdout
