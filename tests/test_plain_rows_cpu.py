"""The plain kernel's batch rows where the device is short of memory: fewer
rows (and more launches) instead of a refused run."""
import os
import subprocess

import pytest

from tests.test_event_cpu import CLANG, HERE

pytestmark = pytest.mark.skipif(CLANG is None, reason="no clang++ for the CPU build")


def test_fewer_rows_where_memory_is_short(tmp_path):
    exe = str(tmp_path / "rows_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O1", "-ffp-contract=off", "-I", os.path.join(HERE, "cpu_event", "include"),
                           "-DLDS_FLOATS=1", "-o", exe, os.path.join(HERE, "cpu_event", "rows_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-2000:]
