"""Rules that choose launches (host arithmetic of csrc/rg_plan.h), checked by
a small C++ program on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launch_plans_hold_their_rules(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = tmp_path / "plan_checks"
    subprocess.check_call([gxx, "-std=c++17", "-O1", "-Wall", "-I",
                           os.path.join(ROOT, "esys-escript.github.io_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "plan_checks.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
