"""Tables that split bremsstrahlung and annihilation photons (nbr_split > 1):
the event loop's tail launch, which holds a particle's descendants on one
thread's stack, has the room that splitting takes, in short runs (the whole
run in that launch) and at the end of longer ones (after the sweeps)."""
import numpy as np
import pytest

from gegs_amd import native, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("load,nsplit,n,depth", [("ct", 2, 4000, 0), ("ct", 16, 4000, 200), ("jaws", 8, 4000, 200),
                                                 ("jaws", 8, 20000, 200), ("ct", 32, 20000, 400)])
def test_split_photons_fit_the_tail(load, nsplit, n, depth):
    print("splitting: %s, nbr_split %d, %d histories" % (load, nsplit, n), flush=True)
    wl = workloads.ct() if load == "ct" else workloads.ct_jaws_mlc()
    src = wl.source(n, 23)
    t = wl.tables.c
    t.nbr_split = nsplit
    ctx = native.Context(0)
    try:
        ctx.load_workload(wl)
        ctx.set_source(src)
        e = ctx.run(seed=13, n_batches=2, method="event", per_history=True)
        ctx.set_tuning(tail_particles=0xFFFFFFFF)
        w = ctx.run(seed=13, n_batches=2, method="event", per_history=True)
        p = ctx.run(seed=13, n_batches=2, method="plain", per_history=True, depth=depth)
        m = min(n, 1000)
        o = oracle.run(wl, src[:m], seed=13, per_history=True, threads=8)
    finally:
        t.nbr_split = 1
        ctx.close()
    assert o["counters"].overflow == 0 and p["counters"]["overflow"] == 0
    assert np.array_equal(p["steps"][:m], o["steps"]) and np.array_equal(p["edep"][:m], o["edep"])
    for r in (e, w):
        assert r["counters"]["overflow"] == 0
        assert np.array_equal(r["steps"], p["steps"])
        assert np.allclose(r["edep"], p["edep"], rtol=1e-12, atol=1e-12)
        assert list(r["counters"]["interactions"]) == list(p["counters"]["interactions"])
