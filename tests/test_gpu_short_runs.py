"""Runs of few histories: the lanes of a wavefront that take histories, the
statistical batches that share a launch, and the event loop's tail launch
taken straight after the injection, at the sizes where their splits change
(one history, a wavefront's and the resident wavefronts' worth and one more,
the last run without sweeps and the first with them)."""
import numpy as np
import pytest

from gegs_amd import workloads

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 65, 2047, 2049, 8192, 8193]


@pytest.fixture(scope="module")
def water16():
    return workloads.water(n=16, voxel=30.0 / 16)


@pytest.mark.parametrize("n", SIZES)
def test_plain_and_event_histories_at_the_split_sizes(gpu_ctx, water16, n):
    """Both methods transport the same histories; a history's energy is summed
    in another order by each, within a few hundred roundings of binary64."""
    print("short runs: %d histories" % n, flush=True)
    ctx = gpu_ctx
    ctx.load_workload(water16)
    ctx.set_source(water16.source(n, 91))
    ctx.set_tuning(None)
    p = ctx.run(seed=19, n_batches=7, method="plain", per_history=True)
    e = ctx.run(seed=19, n_batches=7, method="event", per_history=True)
    assert p["counters"]["histories"] == e["counters"]["histories"] == n
    assert p["counters"]["overflow"] == 0 and e["counters"]["overflow"] == 0
    assert np.array_equal(p["steps"], e["steps"])
    for k in ("photon_steps", "electron_steps", "deposits", "interactions"):
        assert p["counters"][k] == e["counters"][k], k
    assert np.allclose(p["edep"], e["edep"], rtol=1e-13, atol=1e-13)
    for k in ("dose", "dose2"):
        assert np.allclose(p[k], e[k], rtol=1e-12, atol=1e-13 * max(1.0, p[k].max())), k


@pytest.mark.parametrize("n,n_batches", [(1, 1), (5, 13), (2049, 13), (9001, 6)])
def test_noalloc_batches_in_several_launches(gpu_ctx, n, n_batches):
    """On the 128x128x100 CT the scratch holds five dose rows: 13 batches are
    three launches (the last of three rows), 6 are two, 1 is one.  The
    allocating call holds every row: one launch.  Batch doses are sums of the
    same deposits, dose2 the same squares added in two or three parts."""
    import torch
    print("short runs: no-alloc, %d histories in %d batches" % (n, n_batches), flush=True)
    ctx = gpu_ctx
    wl = workloads.ct()
    ctx.load_workload(wl)
    ctx.set_source(wl.source(n, 17))
    p = ctx.run(seed=23, n_batches=n_batches, method="plain")
    dose = torch.empty(ctx.nvox, dtype=torch.float64, device="cuda")
    dose2 = torch.empty_like(dose)
    torch.cuda.synchronize()
    c = ctx.run_plain_noalloc(23, dose.data_ptr(), dose2.data_ptr(), n_batches=n_batches)
    assert c["histories"] == n and c["overflow"] == 0
    assert c["photon_steps"] == p["counters"]["photon_steps"]
    assert np.allclose(dose.cpu().numpy(), p["dose"], rtol=1e-13, atol=1e-13)
    assert np.allclose(dose2.cpu().numpy(), p["dose2"], rtol=1e-13, atol=1e-13)


def test_noalloc_deep_stacks_keep_their_room(gpu_ctx):
    """One block of stacks 28 000 deep takes 229 MB of the 256 MiB scratch: it
    fits beside one dose row of the CT, as before, not beside five."""
    import torch
    print("short runs: no-alloc, deep stacks", flush=True)
    ctx = gpu_ctx
    wl = workloads.ct()
    ctx.load_workload(wl)
    ctx.set_source(wl.source(100, 17))
    p = ctx.run(seed=29, n_batches=5, method="plain")
    dose = torch.empty(ctx.nvox, dtype=torch.float64, device="cuda")
    dose2 = torch.empty_like(dose)
    torch.cuda.synchronize()
    c = ctx.run_plain_noalloc(29, dose.data_ptr(), dose2.data_ptr(), n_batches=5, depth=28000)
    assert c["histories"] == 100 and c["overflow"] == 0
    assert np.allclose(dose.cpu().numpy(), p["dose"], rtol=1e-13, atol=1e-13)
