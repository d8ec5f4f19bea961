"""What the autotuner's cache is keyed by."""
import json

from pip_amd import autotune, problems


def test_keys_separate_the_time_orders():
    """Two-pass masks of RK2 and RK3 runs differ, and so do their stages."""
    cfg = problems.orszag_tang(64)[0]
    assert autotune.stage_key(cfg) != autotune.stage_key(cfg.replace(t_order=3))


def test_choices_for_earlier_kernels_are_not_taken(tmp_path, monkeypatch):
    """A cache written for the kernels before the present ones (whose keys had
    neither a version above 2 nor the time order)."""
    cfg = problems.orszag_tang(64)[0]
    stale = (f"stage2:{cfg.ndim}:{cfg.nx}x{cfg.ny}:nv{cfg.nvar_m}:ir{cfg.flag_ir}:ac{int(cfg.ac_field)}"
             f":col{cfg.flag_col}:imp{cfg.flag_pip_imp}:twopass")
    monkeypatch.setattr(autotune, "CACHE", str(tmp_path / "autotune.json"))
    autotune._save({stale: {"tile": [64, 7, 0, 0], "ms": {}}, "e:modes": {"best": ["persistent", 64], "ms": {}}})

    class Solver:
        def __init__(self, tile):
            self.ms = 1.0 if tile == (16, 7, 1, 0) else 2.0

        def enqueue(self, n):
            pass

        def sync(self):
            pass

        def time_steps(self, n, stages=True):
            return dict(total_ms=self.ms * n)

        def close(self):
            pass

    class Ens:
        def set_mode(self, mode):
            self.mode = mode

        def set_tile(self, tx):
            self.tx = tx

        def reset(self):
            pass

        def run(self, graph=True):
            return 1.0 if (self.mode, self.tx) == ("graph", 128) else 2.0

    assert autotune.tune_stage(Solver, cfg)[0] == (16, 7, 1, 0)
    assert autotune.tune_ensemble(Ens(), "e")[0] == ("graph", 128)
    # and what was tuned now is
    kept = json.load(open(autotune.CACHE))
    assert kept[autotune.stage_key(cfg)]["tile"] == [16, 7, 1, 0]
    assert autotune.tune_stage(None, cfg)[0] == (16, 7, 1, 0)
