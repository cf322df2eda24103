"""The form that a colour pass takes (plan_pass, mg_plan.hpp), on the host: at 4 GB
an array, at 2^31 vectors, for odd rows and stored wall values."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = os.environ.get("CXX", "g++")


@pytest.mark.skipif(not shutil.which(CXX), reason=f"no {CXX}")
def test_forms(tmp_path):
    exe = tmp_path / "pass_plan"
    subprocess.run([CXX, "-O1", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "saras-cc_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "native", "pass_plan.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
