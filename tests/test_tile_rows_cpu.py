"""The rows that k_tile's planned tiles touch (mg_plan.hpp), on the host: none
outside the level, on thin periodic axes neither, and none missing."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = os.environ.get("CXX", "g++")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which(CXX):
        pytest.skip(f"no {CXX}")
    exe = tmp_path_factory.mktemp("tile") / "tile_rows"
    subprocess.run([CXX, "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "saras-cc_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "native", "tile_rows.cpp")], check=True)
    return str(exe)


@pytest.mark.parametrize("word", [4, 8])
@pytest.mark.parametrize("dim", [2, 3])
def test_rows_stay_inside(program, dim, word):
    r = subprocess.run([program, str(word), str(dim)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[:2000]
    plans, cut = map(int, re.search(r"plans (\d+) cut (\d+)", r.stdout).groups())
    assert plans > 1000
    # the sweep reaches plans whose last tile ends beyond the second image
    assert dim == 2 or cut > 50
