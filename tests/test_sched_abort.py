"""An abort by the host in the middle of a busy persistent run, on the CPU:
tests/sched_abort_main.cpp runs the scheduler's host emulation on 16 workgroups
that never wait for an item; once one of them sees the abort word the
others have to leave at their next item."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_host_abort_ends_a_busy_run(tmp_path):
    exe, csrc = str(tmp_path / "sched_abort"), os.path.join(ROOT, "mustard_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I", csrc,
                    os.path.join(ROOT, "tests", "sched_abort_main.cpp"), os.path.join(csrc, "mu_sched_host.cpp"),
                    os.path.join(csrc, "mu_dag.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and p.stdout.endswith(" ok\n"), p.stdout + p.stderr
