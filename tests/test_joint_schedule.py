"""The order of the joint solves (joint_schedule.hpp): the definition's, found in
time that grows with the solves and not with their square.
"""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = tmp_path_factory.mktemp("joint_schedule") / "check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(HERE.parent / "blobs_amd" / "csrc"), "-o", str(out),
                    str(HERE / "joint_schedule_check.cpp")], check=True)
    return lambda *args: subprocess.run([str(out), *map(str, args)], capture_output=True, text=True, check=True,
                                        timeout=60).stdout


def test_levels_are_the_definitions(check):
    assert check("random").strip() == "ok"


def test_a_wide_component(check):
    solves, seconds = check("mesh", 500, 8).split()
    assert int(solves) == 2 * 500 * 499 * 8
    assert float(seconds) < 3.0
