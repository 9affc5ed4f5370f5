"""Runs the checks of tests/host_checks.cpp (host code behind the C interface;
built here once per session against the built library, no GPU needed)."""

import os
import subprocess

import pytest

from pyalign_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHECKS = ["graph_key", "wsb_extents", "fold_rule", "layouts", "noalloc_scratch", "pin_pool", "long_choice"]


@pytest.fixture(scope="session")
def host_checks(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "host_checks")
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["g++", "-D__HIP_PLATFORM_AMD__", "-O1", "-std=c++17", "-w", "-I", os.path.join(ROOT, "include"),
                    "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "host_checks.cpp"), _lib.LIB_PATH,
                    "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{libdir}:/opt/rocm/lib", "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("check", CHECKS)
def test_host_code(host_checks, check):
    r = subprocess.run([host_checks, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
