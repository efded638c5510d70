"""The copy helpers that the per-frame handles share (CopyTeam,
vship_amd/csrc/parallel_copy.hpp), built with g++ and run on the CPU:
tests/copy_team_check.cpp says what is checked."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
def test_copy_team(tmp_path):
    exe = tmp_path / "copy_team_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-Wall", "-Werror", "-o", str(exe),
                    os.path.join(ROOT, "tests", "copy_team_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"
