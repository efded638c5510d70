"""The copy helpers that the per-frame handles share (CopyTeam,
vship_amd/csrc/parallel_copy.hpp) where CPUs, threads or helpers are short:
tests/copy_team_limits_check.cpp says what is checked."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("copy_team") / "copy_team_limits_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-Wall", "-Werror", "-o", str(exe),
                    os.path.join(ROOT, "tests", "copy_team_limits_check.cpp"), "-ldl"], check=True)
    return str(exe)


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
@pytest.mark.parametrize("what", ["asleep", "threads", "taken"])
def test_copy_team_limits(check, what):
    r = subprocess.run([check, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.splitlines()[-1] == "ok"
