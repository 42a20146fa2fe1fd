"""Solves of several processes on one GPU at once.  Launches that need all CUs
meet; one that does not get its blocks in time steps aside and is tried again,
so that all of them stay resident, and each process ends with the bits of a run
alone."""
import subprocess
import sys

import numpy as np
import pytest

from tests.test_gpu_resident import setup, start

pytestmark = pytest.mark.gpu

CHILD = """
import sys, numpy as np
from tests.test_gpu_resident import setup, start
N, M, integrator, seed, out = int(sys.argv[1]), int(sys.argv[2]), int(sys.argv[3]), int(sys.argv[4]), sys.argv[5]
p, u0, rows = setup(N, M, integrator, 2, 960, source=True, seed=seed)
p.Fr = 8
with start(p, u0, rows, 960) as s:
    print("ready", flush=True)
    sys.stdin.readline()
    for _ in range(3):
        s.step(320)
        s.sync()
    np.savez(out, u=s.get_fields(), h=s.output()["h"], psi=s.psi())
    print("resident at the end:", s.resident(), flush=True)
"""


def test_processes_share_the_gpu(tmp_path):
    specs = [(4096, 32, 1, 1), (4096, 32, 1, 2), (16384, 64, 0, 3)]
    ref = []
    for N, M, integrator, seed in specs:
        p, u0, rows = setup(N, M, integrator, 2, 960, source=True, seed=seed)
        p.Fr = 8
        with start(p, u0, rows, 960) as s:
            s.step(960)
            s.sync()
            ref.append((s.get_fields(), s.output()["h"], s.psi()))
    children = [subprocess.Popen([sys.executable, "-c", CHILD, *map(str, spec), str(tmp_path / f"{i}.npz")],
                                 stdin=subprocess.PIPE, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
                for i, spec in enumerate(specs)]
    try:
        for c in children:
            line = c.stdout.readline()
            while line and line.strip() != "ready":
                line = c.stdout.readline()
            assert line, "a process ended before its first step"
        for c in children:      # together
            c.stdin.write("\n")
            c.stdin.flush()
        for i, c in enumerate(children):
            out, _ = c.communicate(timeout=60)
            print(specs[i], out.strip(), flush=True)
            assert c.returncode == 0, out[-2000:]
            assert "resident at the end: True" in out
            got = np.load(tmp_path / f"{i}.npz")
            for key, want in zip(("u", "h", "psi"), ref[i]):
                assert np.array_equal(got[key], want), (specs[i], key)
    finally:
        for c in children:
            if c.poll() is None:
                c.kill()
