"""The photon walk's steps from voxel to voxel where its rules change over:
flights along an axis (faces never met on the others) and almost along it,
vacuum voxels (general steps inside, entered
and left), density factors its reciprocal does not take, turned gantries and
both axis orders.  Both methods against the oracle, history by history."""
import copy

import numpy as np
import pytest

from gegs_amd import source, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu


def _axis_beam(n, z0, seed):
    """Photons along +z (u = v = 0) and, every third, tilted by 1e-12 or 1e-3."""
    rng = np.random.default_rng(seed)
    s = np.zeros(n, dtype=source.SOURCE_DTYPE)
    s["e"] = rng.uniform(0.05, 6.0, n).astype(np.float32)
    s["x"] = rng.uniform(-3.9, 3.9, n).astype(np.float32)
    s["y"] = rng.uniform(-3.9, 3.9, n).astype(np.float32)
    s["z"] = z0
    s["u"] = np.where(np.arange(n) % 3 == 0, np.where(np.arange(n) % 2 == 0, 1e-12, 1e-3), 0.0).astype(np.float32)
    s["w"] = 1.0
    s["wt"] = 1.0
    return s


def _compare(ctx, wl, src, seed):
    ctx.load_workload(wl)
    ctx.set_source(src)
    ctx.set_tuning(None)
    o = oracle.run(wl, src, seed=seed, per_history=True)
    p = ctx.run(seed=seed, n_batches=3, method="plain", per_history=True)
    assert np.array_equal(p["steps"], o["steps"]) and np.array_equal(p["edep"], o["edep"])
    ctx.set_tuning(tail_particles=0xFFFFFFFF, photon_chunk=7)
    e = ctx.run(seed=seed, n_batches=3, method="event", per_history=True)
    ctx.set_tuning(None)
    assert np.array_equal(e["steps"], o["steps"])
    assert np.allclose(e["edep"], o["edep"], rtol=1e-12, atol=1e-12)
    for k in ("photon_steps", "region_gathers", "deposits", "interactions"):
        assert e["counters"][k] == p["counters"][k], k
    assert o["edep"].sum() > 0


@pytest.mark.parametrize("change_xyz", [False, True])
@pytest.mark.parametrize("angle", [0.0, 90.0, 37.0])
def test_axis_flights(gpu_ctx, change_xyz, angle):
    print("walk: axis flights, change_xyz %s, gantry %g" % (change_xyz, angle), flush=True)
    wl = workloads.water(n=16, voxel=0.5)
    wl.field = workloads.make_field(change_xyz, 100.0, angle)
    src = _axis_beam(3000, 90.0, 5)
    _compare(gpu_ctx, wl, src, 61)


@pytest.mark.parametrize("kind", ["vacuum", "odd_density"])
def test_vacuum_and_odd_densities(gpu_ctx, kind):
    """Blocks of vacuum in the CT, or of a density factor of 2^-45 (far below
    any ramp's)."""
    print("walk: %s voxels" % kind, flush=True)
    wl = copy.copy(workloads.ct(nx=24, ny=24, nz=20, voxel=1.25))
    reg = np.array(wl.regions)
    ph = wl.phantom
    idx = np.arange(ph.nvox)
    ix, iy, iz = idx % ph.nx, (idx // ph.nx) % ph.ny, idx // (ph.nx * ph.ny)
    hole = (ix // 3 + iy // 3 + iz // 3) % 4 == 0
    if kind == "vacuum":
        reg["med"][6:][hole] = 0xFFFF
    else:
        reg["rhof"][6:][hole] = np.float32(2.0 ** -45)
    wl._regions = reg
    _compare(gpu_ctx, wl, wl.source(2000, 8), 67)
