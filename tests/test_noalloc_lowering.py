"""The lowering of mu_dtrsm_noalloc's solves on the CPU: no unit needs a
workspace (tests/noalloc_lowering_main.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_solves_need_no_workspace(tmp_path):
    exe, csrc = str(tmp_path / "noalloc"), os.path.join(ROOT, "mustard_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, os.path.join(ROOT, "tests", "noalloc_lowering_main.cpp"),
                    os.path.join(csrc, "mu_dag.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
