"""The autotuner times candidates once the GPU's clock has risen."""
import time

from pip_amd import autotune, problems


def test_candidates_are_timed_at_the_clock_of_a_run(tmp_path, monkeypatch):
    """A GPU whose first 30 ms of work after an idle spell are slow, by an
    amount that depends on the candidate: what a long run takes decides."""
    monkeypatch.setattr(autotune, "CACHE", str(tmp_path / "autotune.json"))
    now = [0.0]
    monkeypatch.setattr(time, "perf_counter", lambda: now[0])

    class Solver:
        def __init__(self, tile):
            now[0] += 0.2  # made while the GPU idles
            self.start = now[0]
            self.ms = 1.0 if tile == (16, 7, 1, 0) else 1.02
            self.cold = 1.2 if tile == (16, 7, 1, 0) else 1.05

        def step_ms(self):
            return self.ms * (self.cold if now[0] - self.start < 0.03 else 1.0)

        def enqueue(self, n):
            for _ in range(n):
                now[0] += 1e-3 * self.step_ms()

        def sync(self):
            pass

        def time_steps(self, n, stages=True):
            ms = 0.0
            for _ in range(n):
                ms += self.step_ms()
                now[0] += 1e-3 * self.step_ms()
            return dict(total_ms=ms)

        def close(self):
            pass

    assert autotune.tune_stage(Solver, problems.orszag_tang(64)[0])[0] == (16, 7, 1, 0)
