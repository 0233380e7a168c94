"""The event loop's tuning, compiled for the CPU: what a caller sets, what it
reads back and what a run makes of it."""
import os
import subprocess

import pytest

from tests.test_event_cpu import CLANG, HERE

pytestmark = pytest.mark.skipif(CLANG is None, reason="no clang++ for the CPU build")


def test_tuning_read_and_set_again_changes_no_run(tmp_path):
    exe = str(tmp_path / "tuning_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O1", "-ffp-contract=off", "-I", os.path.join(HERE, "cpu_event", "include"),
                           "-DLDS_FLOATS=1", "-o", exe, os.path.join(HERE, "cpu_event", "tuning_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-2000:]
