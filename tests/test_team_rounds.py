"""The counters of the BFS and SSSP kernels on the host: workgroups that wait
outside a team may read their input at any time while the team's rounds run."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "tpds22-artifact_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ absent")
    exe = str(tmp_path_factory.mktemp("team") / "team_rounds_check")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-I", CSRC, os.path.join(HERE, "team_rounds_check.cpp"),
                        "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return lambda *args: subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)


def test_inputs_do_not_change_while_a_team_runs(check):
    r = check()
    assert r.returncode == 0 and "failures 0" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("mistake", ["shared", "report", "far"])
def test_the_check_finds(check, mistake):
    r = check("plant", mistake)
    assert r.returncode == 1 and "failures 0" not in r.stdout, r.stdout


def test_the_kernels_use_these_counters():
    """The kernels reach their counters through this header alone."""
    text = open(os.path.join(CSRC, "graph.hip")).read()
    assert '#include "team_rounds.hpp"' in text
    body = text[text.index("struct BfsArgs1"):text.index("struct PrArgs")]
    # no team where the grid's barrier has no limit
    assert len(re.findall(r"team\.init\(", body)) == len(re.findall(r"KIND != HS_BAR_COOP\);", body)) == 2
    assert not re.search(r"% 3\) \* kCtr|p\.ctr \+ \d|p\.ctr\[\d", body)
