"""The host shim without a GPU: its source is compiled into programs that plan
and launch nothing (tests/cxx/plan_test.cpp: the launch planner over many
shapes; host_call_test.cpp: host-pointer calls whose launches fail)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(*command):
    exe = os.path.join(ROOT, "tests", "cxx", command[0])
    assert os.path.exists(exe), f"tests/cxx/{command[0]} missing: run __graft_entry__.build()"
    r = subprocess.run([exe, *command[1:]], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-1000:]


@pytest.mark.parametrize("what", ["scratch", "capture"])
def test_plans(what):
    _run("plan_test", what)


def test_host_call_that_fails_writes_nothing():
    _run("host_call_test")
