"""The tuner times the library's own choice beside its launch shapes, and hands
out no shape that loses to it (no GPU: probe solvers and batches with planted
times)."""
import pytest

from bh_ringdown_amd import tune


class Probe:
    """Stands in for Solver and Batch: its time per stage is `us[shape]`."""
    us = {}

    def __init__(self, *a, **k):
        self.shape = None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        pass

    def set_tiling(self, *shape):
        self.shape = shape

    def step(self, n):
        Clock.now += n * 1e-6 * self.us.get(self.shape, 9.0)

    def timing(self):
        return 100, 0.1 * self.us.get(self.shape, 9.0)

    def set_cache_groups(self, n):
        pass

    def sync(self):
        pass

    add = enable_timing = set_cache_groups
    close = sync


class Clock:
    now = 0.0

    @classmethod
    def perf_counter(cls):
        return cls.now


@pytest.fixture
def probes(tmp_path, monkeypatch):
    monkeypatch.setattr(tune, "CACHE", str(tmp_path / "tuning.json"))
    monkeypatch.setattr(tune.teuk, "Solver", Probe)
    monkeypatch.setattr(tune.teuk, "Batch", Probe)
    monkeypatch.setattr(tune, "time", Clock)


@pytest.mark.parametrize("default,wins", [(3.0, True), (6.0, False)])
def test_solver_shapes_against_the_default(probes, monkeypatch, default, wins):
    monkeypatch.setattr(Probe, "us", {None: default, (2, 3, 4): 5.0})
    best, times = tune.tune_solver(2048, 136)
    assert best == (None if wins else (2, 3, 4)) and times[None] == pytest.approx(default)
    want = None if wins else {"waves_per_block": 2, "waves_per_eu": 3, "theta_rows": 4}
    assert tune.best_solver_tiling(2048, 136) == want


@pytest.mark.parametrize("default,wins", [(3.0, True), (6.0, False)])
def test_batch_schedules_against_the_default(probes, monkeypatch, default, wins):
    monkeypatch.setattr(Probe, "us", {None: default, (4, 2, 1, 16, 8): 5.0})
    shapes = [(2048, 136)] * 3
    best, times = tune.tune_batch(shapes, chunks=(16, 32), group_bytes=(1 << 20,))
    assert best == (None if wins else (4, 2, 1, 16, 1 << 20, 8)) and times[None] == pytest.approx(1e-6 * default)
    got = tune.best_batch_tiling(shapes)
    assert got is None if wins else got["order"] == 1 and got["theta_rows"] == 8
    assert tune.best_batch_groups(shapes) == (0 if wins else 1 << 20)


def test_committed_table_gives_no_shape_that_the_default_beats(probes):
    """Grids of the workloads, all faster without a shape (4096x32 and 16384x64
    RK4 have entries, for solvers kept off resident stepping)."""
    for N, M in ((8192, 32), (16384, 32), (8192, 64), (32768, 64), (65536, 128)):
        for integrator in (0, 1):
            assert tune.best_solver_tiling(N, M, integrator) is None, (N, M, integrator)
