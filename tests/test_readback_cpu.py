"""The copy of results into host buffers over a stand-in of the runtime:
small results take plain copies, and where the runtime gives no pinned memory
or no event the copy still succeeds, at that call and at the later ones."""
import os
import subprocess

import pytest

from tests.test_event_cpu import CLANG, HERE

pytestmark = pytest.mark.skipif(CLANG is None, reason="no clang++ for the CPU build")


def test_read_back_without_pinned_memory_or_events(tmp_path):
    exe = str(tmp_path / "readback_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O1", "-g", "-fsanitize=address", "-fno-omit-frame-pointer", "-pthread",
                           "-o", exe, os.path.join(HERE, "cpu_event", "readback_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr[-2000:])
