"""The launch-configuration tuner on the CPU, with stand-in simulations on a clock of their own."""
from osiris_amd import autotune


class Clock:
    now = 0.0

    def perf_counter(self):
        return self.now


class Sim:
    """A candidate whose calls of run take run_ms per step and `once` ms more one time, and whose
    kernels, each timed in a launch of its own, take kernel_ms."""

    def __init__(self, clock, run_ms, kernel_ms, once=0.0):
        self.clock, self.run_ms, self.kernel_ms, self.once, self.closed = clock, run_ms, kernel_ms, once, False

    def run(self, n):
        self.clock.now += (n * self.run_ms + self.once) * 1e-3
        self.once = 0.0

    def time_kernels(self, n):
        self.clock.now += n * self.kernel_ms * 1e-3
        return {"step": self.kernel_ms}

    def close(self):
        self.closed = True


def test_the_fastest_run_wins(monkeypatch):
    clock = Clock()
    monkeypatch.setattr(autotune, "time", clock, raising=False)
    cands = [{"tile": (8, 8)}, {"tile": (16, 16)}, {"tile": (32, 16)}]
    sims = [Sim(clock, 2.0, 1.0), Sim(clock, 1.5, 1.8, once=50.0), Sim(clock, 1.7, 1.2)]
    made = iter(sims)
    best, ms = autotune.tune(lambda cfg: next(made), "key", candidates=cands, warmup=0, cache=None)
    assert best["tile"] == (16, 16)
    assert [round(v, 6) for v in ms.values()] == [2.0, 1.5, 1.7]
    assert all(s.closed for s in sims)
