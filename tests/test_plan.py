"""Decisions on sizes that need no device (epet_plan.hpp), compiled with g++."""
import os
import subprocess

from conftest import ROOT


def test_plan(tmp_path):
    exe = str(tmp_path / "test_plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(ROOT, "tests", "cpp", "test_plan.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
