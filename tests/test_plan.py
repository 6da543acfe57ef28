"""The launch planner over many shapes without a GPU (tests/cxx/plan_test.cpp,
the host shim's source compiled into a program that plans and launches
nothing)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("what", ["scratch", "capture"])
def test_plans(what):
    exe = os.path.join(ROOT, "tests", "cxx", "plan_test")
    assert os.path.exists(exe), "tests/cxx/plan_test missing: run __graft_entry__.build()"
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-1000:]
