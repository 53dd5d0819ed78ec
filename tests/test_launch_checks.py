"""Checks that the host makes before a launch whose kernel relies on them
(tests/cpu/launch_checks_test.cpp, linked against the built library)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "vortexstark_amd")

CASES = ["tail_level_0", "tail_other_challenge", "tail_no_challenge", "proof_destination", "inputs_pointer_slot"]


@pytest.fixture(scope="module")
def binary(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("launch_checks") / "launch_checks_test")
    src = os.path.join(ROOT, "tests", "cpu", "launch_checks_test.cpp")
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"), "-c",
                    src, "-o", out + ".o"], check=True)
    subprocess.run([hipcc, out + ".o", "-o", out, os.path.join(PKG, "libvortex_hip.so"), f"-Wl,-rpath,{PKG}"],
                   check=True)
    return out


@pytest.mark.parametrize("case", CASES)
def test_refused(binary, case):
    r = subprocess.run([binary, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert f"PASS {case}" in r.stdout
