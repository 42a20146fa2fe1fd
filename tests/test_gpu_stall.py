"""A resident launch whose blocks stop waiting for each other: every block
ends, the solve fails under its own code, and its batch neighbours end where
they end alone.  The condition is forced from the host: with a limit of no
further reads (teuk_set_exchange_reads) the first neighbour that is not there
yet counts as stopped."""
import numpy as np
import pytest

from bh_ringdown_amd import teuk
from tests.test_gpu_resident import setup, start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M,integrator", [(1024, 32, 1), (6080, 40, 0), (8192, 64, 1), (16384, 64, 0), (6144, 128, 1),
                                            (32768, 64, 1)])
def test_stopped_blocks_are_not_divergence(N, M, integrator):
    print(f"stall {N}x{M} integrator {integrator}", flush=True)
    p, u0, _ = setup(N, M, integrator, 2, 64)
    with start(p, u0, None, 64) as s:
        s.set_exchange_reads(0)
        s.step(32)
        assert s.status() == teuk.TEUK_ESTALLED
        s.step(32)                      # later launches end too
        with pytest.raises(teuk.TeukError) as e:
            s.sync()
        assert e.value.code == teuk.TEUK_ESTALLED and "wait" in teuk.strerror(e.value.code)
        with pytest.raises(teuk.TeukError) as e:
            s.set_exchange_reads(-1)
        assert e.value.code == teuk.TEUK_EINVAL


def test_stalled_member_leaves_its_neighbours():
    specs = [setup(1024, 32, 1, m, 64, seed=m) for m in (1, 2, 3)]
    ref = []
    for p, u0, _ in specs:
        with start(p, u0, None, 64) as s:
            s.step(64)
            s.sync()
            ref.append(s.get_fields())
    solvers = [start(p, u0, None, 64) for p, u0, _ in specs]
    solvers[1].set_exchange_reads(0)
    with teuk.Batch(integrator=1) as b:
        for s in solvers:
            assert b.add(s)
        b.step(64)
        with pytest.raises(teuk.TeukError) as e:
            b.sync()
        assert e.value.code == teuk.TEUK_ESTALLED
        assert [s.status() for s in solvers] == [teuk.TEUK_OK, teuk.TEUK_ESTALLED, teuk.TEUK_OK]
        for i in (0, 2):
            assert np.array_equal(solvers[i].get_fields(), ref[i])
    for s in solvers:
        s.close()
