"""The head geometry's polygon tests (point in polygon, ray to the nearest
edge, distance to the nearest edge), which pick the deciding edge with cheap
arithmetic, against their plain forms, compiled for the CPU: bit for bit over
slabs, leaves, leaf ends and random polygons (lengths 1e-3 to 1e4 cm, edges
of no length), with points on and beside vertices and edges and directions
along the axes, at vertices and near zero.  The device's own reciprocals and
quotients are checked by test_gpu_reciprocals.py."""
import os
import subprocess

import pytest

from tests.test_event_cpu import CLANG, HERE

pytestmark = pytest.mark.skipif(CLANG is None, reason="no clang++ for the CPU build of the geometry")


def test_polygon_tests_equal_their_plain_forms(tmp_path):
    exe = str(tmp_path / "polygon_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O2", "-ffp-contract=off", "-I", os.path.join(HERE, "cpu_event", "include"),
                           "-DLDS_FLOATS=1", "-o", exe, os.path.join(HERE, "cpu_event", "polygon_check.cpp")])
    # the selections' reciprocals exact, as far off as the device's (1 ULP) and twice as far
    for ulps in ("0", "1", "2"):
        r = subprocess.run([exe, "6000", ulps], capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stdout + r.stderr[-2000:]
        assert r.stdout.startswith("checks 2400000")


def test_walk_quotients_and_logarithm_equal_their_plain_forms(tmp_path):
    """div_by against the division for the operands the photon walk gives it,
    and glog against its form with the exponent and mantissa taken apart."""
    exe = str(tmp_path / "walk_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-I",
                           os.path.join(HERE, "cpu_event", "include"), "-DLDS_FLOATS=1", "-o", exe,
                           os.path.join(HERE, "cpu_event", "walk_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-2000:]


def test_walk_takes_each_axis_bounds_from_its_own_array(tmp_path):
    """Kernels that stage nothing in LDS have the three bounds in allocations
    of their own, any distance apart; and a flight that leaves through the
    lowest face of an axis reads nothing before them (address checks on)."""
    exe = str(tmp_path / "walk_bounds_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O1", "-g", "-fsanitize=address", "-fno-omit-frame-pointer",
                           "-ffp-contract=off", "-I", os.path.join(HERE, "cpu_event", "include"), "-DLDS_FLOATS=1",
                           "-o", exe, os.path.join(HERE, "cpu_event", "walk_bounds_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr[-2000:])
