"""teuk_solve_noalloc beside another thread's solve: the other thread's step
calls queue their steps and return while the call runs, and both end with the
bits of a run alone.  With no other solve in the process yet the call has no
event to record behind its launches; a solve started while it runs follows
them all the same."""
import subprocess
import sys
import threading
import time

import numpy as np
import pytest

from bh_ringdown_amd import teuk
from tests.test_gpu_resident import setup, start

pytestmark = pytest.mark.gpu


def noalloc(p, u0, steps):
    _, r_c, th = teuk.grid(p)
    rc, u, out = teuk.solve_noalloc(p, r_c, th, steps, u0=u0)
    assert rc == teuk.TEUK_OK
    return u, out["h"]


def test_steps_beside_the_call_return_at_once():
    p, u0, _ = setup(4096, 32, 1, 2, 1000)
    q, v0, _ = setup(1024, 32, 1, 1, 60000, seed=2)
    p.Fr = q.Fr = 50
    alone = noalloc(p, u0, 1000)
    shares, steps = [], 0
    with start(q, v0, None, 60000) as s:
        for _ in range(6):
            got, span = [], []

            def call():
                t0 = time.perf_counter()
                got.append(noalloc(p, u0, 1000))
                span.extend((t0, time.perf_counter()))

            t = threading.Thread(target=call)
            t.start()
            longest = 0.0
            while t.is_alive():
                t0 = time.perf_counter()
                s.step(32)
                steps += 32
                longest = max(longest, time.perf_counter() - t0)
                time.sleep(5e-4)
            t.join()
            assert np.array_equal(got[0][0], alone[0]) and np.array_equal(got[0][1], alone[1])
            s.sync()
            shares.append(longest / (span[1] - span[0]))
        assert s.resident()
        u = s.get_fields()
    with start(q, v0, None, 60000) as s:
        s.step(steps)
        s.sync()
        assert np.array_equal(s.get_fields(), u)
    print("longest step call over the call's time:", [round(x, 3) for x in shares], flush=True)
    assert min(shares) < 0.3


CHILD = """
import threading, numpy as np
from bh_ringdown_amd import teuk
from tests.test_gpu_resident import setup, start
from tests.test_zz_no_alloc_threads import noalloc
p, u0, _ = setup(4096, 32, 1, 2, 1000)
q, v0, _ = setup(4096, 32, 1, 1, 320, seed=2)
p.Fr = q.Fr = 50
got = []
t = threading.Thread(target=lambda: got.append(noalloc(p, u0, 1000)))
t.start()                                  # the process's first launches
with start(q, v0, None, 320) as s:
    for _ in range(10):
        s.step(32)
    s.sync()
    assert s.resident()
    v = s.get_fields()
t.join()
u = noalloc(p, u0, 1000)
assert np.array_equal(got[0][0], u[0]) and np.array_equal(got[0][1], u[1])
with start(q, v0, None, 320) as s:
    s.step(320)
    s.sync()
    assert np.array_equal(s.get_fields(), v)
print("child: ok", flush=True)
"""


def test_first_solve_of_the_process():
    r = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "child: ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
