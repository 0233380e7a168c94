"""The autotuner's walk over a context whose runs take a given time: it times
the library's defaults and keeps them unless something is faster by more than
the noise."""
import pytest

from gegs_amd import autotune


class Clock:
    def __init__(self, cost):
        self.now, self.cost, self.tuning, self.runs = 0.0, cost, None, []

    def perf_counter(self):
        return self.now

    def set_tuning(self, tuning=None):
        self.tuning = dict(tuning or {})

    def run(self, **kw):
        self.runs.append(dict(self.tuning))
        self.now += self.cost(self, self.tuning)


def _tune(monkeypatch, cost):
    ctx = Clock(cost)
    monkeypatch.setattr(autotune.time, "perf_counter", ctx.perf_counter)
    tuning, best, trials = autotune.autotune(ctx, 0, 1000)
    assert ctx.tuning == tuning
    return ctx, tuning, best, trials


def _given(t):
    """What of a tuning differs from the library's defaults (zero: the run's pick)."""
    defaults = dict(refill_min=16, refill_slots=64, flight_block=256, inject=6 << 20, threshold=6 << 20,
                    sweeps_per_graph=4)
    return {k: v for k, v in t.items() if v and v != defaults.get(k)}


def test_the_defaults_are_timed_and_kept(monkeypatch):
    """Every explicit tuning is slower than the defaults."""
    ctx, tuning, best, trials = _tune(monkeypatch, lambda c, t: 2.0 if _given(t) else 1.0)
    assert _given(tuning) == {} and best == 1000.0
    assert _given(trials[0][0]) == {}
    tried = [_given(t) for t, _ in trials]
    for want in (dict(photon_chunk=96), dict(electron_chunk=12), dict(grid=512), dict(grid=2048)):
        assert want in tried


@pytest.mark.parametrize("gain", [1.01, 1.2])
def test_a_change_is_kept_by_more_than_the_noise(monkeypatch, gain):
    ctx, tuning, best, _ = _tune(monkeypatch, lambda c, t: 1.0 / gain if _given(t) == dict(photon_chunk=64) else 1.0)
    assert _given(tuning) == (dict(photon_chunk=64) if gain > 1.02 else {})


def test_one_lucky_trial_is_not_kept(monkeypatch):
    """A tuning that was fast while it was tried and is not when timed again."""
    def cost(c, t):
        return 0.5 if _given(t) == dict(electron_chunk=32) and c.runs.count(c.tuning) <= 2 else 1.0
    ctx, tuning, best, _ = _tune(monkeypatch, cost)
    assert _given(tuning) == {} and best == 1000.0


def test_a_drift_of_the_machine_is_not_a_gain(monkeypatch):
    """Every run a little faster than the one before, whatever the tuning: the
    later trials win, and lose against the defaults timed before and after them."""
    ctx, tuning, best, _ = _tune(monkeypatch, lambda c, t: 0.985 ** len(c.runs))
    assert _given(tuning) == {}
