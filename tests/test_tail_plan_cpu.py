"""The levels that the tail's LDS takes (plan_tail, mg_plan.hpp), on the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = os.environ.get("CXX", "g++")


@pytest.mark.skipif(not shutil.which(CXX), reason=f"no {CXX}")
def test_solved_coarsest_levels_fit(tmp_path):
    exe = tmp_path / "tail_plan"
    subprocess.run([CXX, "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "saras-cc_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "native", "tail_plan.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
