"""Single steps of the persistent scheduler on the CPU: tests/sched_pop_main.cpp
runs sched_pop of mu_sched.hpp (the code the gfx950 kernel runs) for one worker
whose lots and arrivals the case decides."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_scheduler_pop_steps(tmp_path):
    exe = str(tmp_path / "sched_pop")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-I",
                    os.path.join(ROOT, "mustard_amd", "csrc"),
                    os.path.join(ROOT, "tests", "sched_pop_main.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    lines = p.stdout.splitlines()
    assert p.returncode == 0 and lines and all(l.endswith(" ok") for l in lines), p.stdout + p.stderr
