"""Output records and fields read back at their edges: records formed a block
each, from row counts that fill one or several groups of terms or part of
one, with record intervals that do and do not divide the chunks of steps and
more records in a call than blocks; fields set and read between steps, with
infinities, NaN and signed zeros, for every integrator.  Against the CPU
oracle, or the call's own inputs, bit for bit."""
import numpy as np
import pytest

from bh_ringdown_amd import teuk
from tests.test_gpu_resident import oracle, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [16, 56, 64, 72, 128, 136, 200])
@pytest.mark.parametrize("Fr,parts", [(1, (33, 1, 70)), (3, (1, 1, 32, 70)), (40, (39, 1, 64))])
def test_records(M, Fr, parts):
    steps = sum(parts)
    p, u0, _ = setup(128, M, 1, 2, steps, je=63)
    p.Fr = Fr
    with teuk.Solver(p) as s:
        s.set_fields(u0)
        for n in parts:
            s.step(n)
        s.sync()
        out, u = s.output(), s.get_fields()
    uo, _, h, dedt = oracle(p, u0, None, steps)
    assert np.array_equal(u, uo)
    assert np.array_equal(out["k"], np.arange(0, steps, Fr))
    assert np.array_equal(out["h"], h[::Fr]) and np.array_equal(out["dedt"], dedt[::Fr])
    t = np.concatenate([[0.0], np.cumsum(np.full(steps - 1, p.dt))])   # repeated addition
    assert np.array_equal(out["t"], t[::Fr])


@pytest.mark.parametrize("N,M,integrator", [(128, 16, 0), (1216, 40, 1), (320, 136, 1), (192, 24, 2)])
def test_fields_round_trip(N, M, integrator):
    p, u0, _ = setup(N, M, integrator, 2, 40)
    odd = u0.copy()
    odd.ravel()[::7] = -0.0
    odd[0, 0, :4] = np.inf, -np.inf, np.nan, 5e-324
    odd[3, -1, -1] = np.nan
    with teuk.Solver(p) as s, teuk.Solver(p) as whole:
        s.set_fields(odd)
        assert s.get_fields().tobytes() == odd.tobytes()
        s.set_fields(u0)
        for n in (3, 20, 17):          # what set and get leave behind is not an input of the next step
            s.step(n)
            s.set_fields(s.get_fields())
        whole.set_fields(u0)
        whole.step(40)
        assert s.get_fields().tobytes() == whole.get_fields().tobytes()


@pytest.mark.parametrize("N,M,integrator", [(14336, 256, 0), (19136, 192, 1), (7168, 512, 1)])
def test_default_shape_of_tall_grids(N, M, integrator):
    """The smallest grids whose default is 8-row chunks."""
    p, u0, _ = setup(N, M, integrator, 2, 3, je=N // 2)
    with teuk.Solver(p) as s:
        s.set_fields(u0)
        s.step(3)
        s.sync()
        u, psi = s.get_fields(), s.psi()
    uo, psio, _, _ = oracle(p, u0, None, 3)
    assert np.array_equal(u, uo) and np.array_equal(psi, psio)
