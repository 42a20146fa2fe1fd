"""The wait of resident launches for their blocks (teuk_set_resident_wait):
what a solver, a batch and the no-allocation call do with values from zero to
infinity, set before the first step or between steps; and what
teuk_resident says of a batch's members."""
import math

import numpy as np
import pytest

from bh_ringdown_amd import teuk
from tests.test_gpu_resident import oracle, setup, start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seconds", [5e-3, 3600.0, 1e11, 1e300, math.inf])
def test_a_long_wait_is_not_taken_as_none(seconds):
    p, u0, _ = setup(1024, 32, 1, 2, 40)
    with start(p, u0, None, 40) as s:
        s.set_resident_wait(seconds)
        s.step(40)
        s.sync()
        assert s.resident()


@pytest.mark.parametrize("seconds", [-1.0, -math.inf, math.nan])
def test_what_is_no_wait_is_refused(seconds):
    p, u0, _ = setup(128, 16, 1, 2, 4)
    with start(p, u0, None, 4) as s:
        with pytest.raises(teuk.TeukError) as e:
            s.set_resident_wait(seconds)
        assert e.value.code == teuk.TEUK_EINVAL


def batch_of(specs, steps):
    solvers = [start(p, u0, None, steps) for p, u0, _ in specs]
    b = teuk.Batch(integrator=1)
    for s in solvers:
        assert b.add(s)
    return b, solvers


def test_wait_set_between_the_steps_of_a_batch():
    """It holds from the next step on: a wait of zero makes that launch give
    up, and no step is lost."""
    specs = [setup(1024, 32, 1, m, 96, seed=m) for m in (1, 2)]
    ref = []
    for p, u0, _ in specs:
        with start(p, u0, None, 96) as s:
            s.step(96)
            s.sync()
            ref.append(s.get_fields())
    b, solvers = batch_of(specs, 96)
    b.step(32)
    b.sync()
    assert all(s.resident() for s in solvers)
    solvers[1].set_resident_wait(0.0)
    b.step(32)
    b.sync()
    assert not any(s.resident() for s in solvers)      # they shared the launch
    b.step(32)
    b.sync()
    for s, u in zip(solvers, ref):
        assert s.progress()[0] == 96 and np.array_equal(s.get_fields(), u)
    b.close()
    for s in solvers:
        s.close()


def test_resident_of_members():
    """A member that is stepped in segments alone goes by stages in a batch;
    with a launch shape set for the batch all of them do."""
    specs = [setup(1024, 32, 1, 2, 8), setup(32768, 64, 1, 2, 8), setup(512, 136, 1, 2, 8)]
    b, solvers = batch_of(specs, 8)
    assert [s.resident() for s in solvers] == [True, False, False]
    b.step(4)
    b.sync()
    assert [s.resident() for s in solvers] == [True, False, False]
    b.set_tiling(1, 2, 0, 32, theta_rows=2)
    assert not any(s.resident() for s in solvers)
    b.set_tiling(1, 3, 0, 32, theta_rows=2, resident=True)      # the shape for those that do not fit
    assert [s.resident() for s in solvers] == [True, False, False]
    b.step(2)
    b.sync()
    assert teuk.lib().teuk_batch_set_resident(b._h, 0) == teuk.TEUK_OK
    b.step(2)
    b.sync()
    assert not any(s.resident() for s in solvers)
    for s, (p, u0, _) in zip(solvers, specs):
        with start(p, u0, None, 8) as one:
            one.step(8)
            assert np.array_equal(s.get_fields(), one.get_fields())
    b.close()
    assert [s.resident() for s in solvers] == [True, True, False]      # alone again
    for s in solvers:
        s.close()


@pytest.mark.parametrize("N,M,integrator,patience", [
    (1024, 32, 1, 0.0), (6080, 40, 0, 0.0), (16384, 64, 1, 0.0), (6144, 128, 0, 0.0), (32768, 64, 1, 0.0),
    (32768, 64, 0, 1e-8), (16384, 128, 1, 1e-8), (32768, 64, 1, 1e-8),
])
def test_launches_that_step_aside_are_tried_again(N, M, integrator, patience):
    """With no first wait every launch's first try steps aside; with a first
    wait of 0.5 to 1.5 ticks every other segment's, also after segments that
    have run.  The steps are taken by later launches."""
    print(f"step aside {N}x{M} integrator {integrator} patience {patience}", flush=True)
    parts = (1, 1, 1, 1, 1, 1, 2, 33, 6)
    steps = sum(parts)
    p, u0, rows = setup(N, M, integrator, 2, steps, N // 3, True)
    uo, psio, ho, _ = oracle(p, u0, rows, steps)
    with start(p, u0, rows, steps) as s:
        s.set_resident_patience(patience)
        s.enable_timing(True)
        for n in parts:
            s.step(n)
            assert s.progress()[0] == s.p.nsteps() - s.remaining()
        assert s.timing()[0] < (3, 4)[integrator] * steps      # those tried again are not timed
        assert s.resident() and s.progress()[0] == steps
        assert np.array_equal(s.get_fields(), uo) and np.array_equal(s.psi(), psio)
        assert np.array_equal(s.output()["h"], ho)
    with start(p, u0, rows, steps) as s:                        # queued at once
        s.set_resident_patience(patience)
        s.step(3)
        s.step(steps - 3)
        s.sync()
        assert s.resident() and s.progress()[0] == steps
        assert np.array_equal(s.get_fields(), uo) and np.array_equal(s.output()["h"], ho)


def test_batch_launches_that_step_aside_are_tried_again():
    specs = [setup(N, M, 1, 2, 70, seed=i) for i, (N, M) in enumerate([(1024, 32), (4096, 32), (512, 72), (8192, 64)])]
    ref = []
    for p, u0, _ in specs:
        with start(p, u0, None, 70) as s:
            s.step(70)
            s.sync()
            ref.append((s.get_fields(), s.output()["h"]))
    b, solvers = batch_of(specs, 70)
    solvers[2].set_resident_patience(0.0)
    for n in (5, 40, 25):
        b.step(n)
        b.sync()
    assert b.info()["active"] == 0
    for s, (u, h) in zip(solvers, ref):
        assert s.resident() and s.progress()[0] == 70
        assert np.array_equal(s.get_fields(), u) and np.array_equal(s.output()["h"], h)
    b.close()
    for s in solvers:
        s.close()


def test_launches_that_gave_up_are_not_timed():
    p, u0, _ = setup(1024, 32, 1, 2, 96)
    with start(p, u0, None, 96) as s:
        s.enable_timing(True)
        s.step(32)
        s.sync()
        assert s.timing()[0] == 4 * 32
        s.set_resident_wait(0.0)
        s.step(64)              # two launches that change nothing
        s.sync()
        n, ms = s.timing()
        assert n == 4 * 96 and 0.0 < ms < 100.0
    b, solvers = batch_of([setup(1024, 32, 1, 2, 32)], 32)
    solvers[0].enable_timing(True)      # a batch's steps are not a solver's own
    solvers[0].set_resident_wait(0.0)
    b.step(32)
    b.sync()
    assert solvers[0].timing()[0] == 0 and solvers[0].progress()[0] == 32
    b.close()
    solvers[0].close()
