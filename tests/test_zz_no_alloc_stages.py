"""teuk_solve_noalloc by the stage kernels: solves of more than 128 rows, and
resident launches that give up (a wait of zero), whose steps the stage kernels
run, with patches row after row where the launches' were column after column.
Against the CPU oracle, bit for bit."""
import math

import numpy as np
import pytest

from bh_ringdown_amd import teuk
from tests.test_gpu_resident import oracle, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wait", [None, 0.0, math.inf])
@pytest.mark.parametrize("N,M,integrator,m,steps,source", [
    (256, 136, 1, 2, 40, False),      # stages whatever the wait
    (256, 136, 0, -1, 65, True),
    (1024, 32, 1, 2, 70, True),       # resident, or given up: three launches' steps
    (4096, 32, 0, 1, 33, False),
    (704, 128, 1, 3, 32, True),
    (128, 16, 0, 2, 1, True),
])
def test_noalloc_equals_oracle(N, M, integrator, m, steps, source, wait):
    print(f"noalloc {N}x{M} integrator {integrator} steps {steps} source {source} wait {wait}", flush=True)
    p, u0, rows = setup(N, M, integrator, m, steps, N // 3, source)
    _, r_c, th = teuk.grid(p)
    sched = teuk.trajectory_schedule(rows, steps, p.dt) if source else None
    rc, u, out = teuk.solve_noalloc(p, r_c, th, steps, u0=u0, steps=sched, wait=wait)
    assert rc == teuk.TEUK_OK
    uo, _, h, dedt = oracle(p, u0, rows, steps)
    assert np.array_equal(u, uo)
    assert np.array_equal(out["k"], np.arange(steps))
    assert np.array_equal(out["h"], h[:steps]) and np.array_equal(out["dedt"], dedt[:steps])


def test_no_wait_refused():
    p, u0, _ = setup(128, 16, 1, 2, 4)
    _, r_c, th = teuk.grid(p)
    for wait in (-1.0, math.nan):
        with pytest.raises(teuk.TeukError) as e:
            teuk.solve_noalloc(p, r_c, th, 4, u0=u0, wait=wait)
        assert e.value.code == teuk.TEUK_EINVAL
