"""The launch plans of Merkle trees (whir_amd/csrc/tree_plan.h), compiled for the host and
checked over widths and numbers of trees (tree_plan_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CXX = shutil.which("g++") or shutil.which("clang++")


@pytest.mark.skipif(CXX is None, reason="needs a C++ compiler")
def test_tree_plans_cover_every_level(tmp_path):
    exe = tmp_path / "tree_plan_check"
    subprocess.run([CXX, "-O1", "-std=c++17", os.path.join(HERE, "tree_plan_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok ")
