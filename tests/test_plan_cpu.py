"""The emit's plan (kmc_plan.h) on the host: what a wave queues names the slot it
looked at, in volumes of any number of rows, every slot is looked at once, and small
or flat surfaces fall to many waves, and a large volume among many small ones in a
batch keeps its share of the workgroups."""
import os
import subprocess

import pytest

from tests.conftest import ROOT


@pytest.fixture(scope="module")
def plan_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "plan_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "kvs_amd", "csrc"),
                    os.path.join(ROOT, "tests", "plan", "plan_check.cpp"), "-o", exe], check=True, timeout=120)
    return exe


@pytest.mark.parametrize("what", ["slots", "places", "large", "shares", "unequal"])
def test_emit_slots(plan_check, what):
    r = subprocess.run([plan_check, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
