"""Resident stepping (fields held on the chip between launches) against the
CPU oracle, bit for bit: the tile shapes' edges (one to eight columns per
thread, partly filled last blocks and phases, rows that fill a wave or not),
either integrator, odd modes, a source patch crossing block borders, the
extraction column next to a border and among the rho edge columns, initial
fields that do not satisfy the edge fills, and chunks of 1, 32 and 33 steps.
A launch that does not get its blocks onto the GPU hands its steps to the
stage kernels.  No tolerance: both sides evaluate the same expressions.
"""
import threading

import numpy as np
import pytest

from bh_ringdown_amd import teuk, workloads
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def setup(N, M, integrator, m, steps, je=-1, source=False, seed=4, a=0.6):
    L = min(0.39 * N, 1600.0)
    p = teuk.default_params(N, M, -0.25 * L, 0.75 * L, a, m, dt_over_dx=min(0.5, 1.6 * (np.pi / M) / (L / N)))
    p.T = steps * p.dt * (1.0 + 1e-12)
    p.Fr, p.integrator, p.j_extract = 1, integrator, je
    rng = np.random.default_rng(seed)
    u0 = workloads.gaussian_pulse(p, seed, center=p.xmin + 0.3 * L, width=max(3.0, 6.0 * p.dx))
    u0 += 1e-3 * rng.standard_normal(u0.shape)      # edge rows and columns too
    rows = workloads.plunge_rows(p, steps, seed=seed) if source else None
    return p, u0, rows


def start(p, u0, rows, steps):
    s = teuk.Solver(p)
    s.set_fields(u0)
    if rows is not None:
        s.set_trajectory(rows, steps)
    return s


def oracle(p, u0, rows, steps):
    _, r_c, th = teuk.grid(p)
    op = O.make_params(p.N, p.M, p.xmin, p.xmax, p.a, p.m, dt=p.dt, integrator=p.integrator,
                       j_extract=p.j_extract, ptsx=p.ptsx, ptsy=p.ptsy)
    ost = None
    if rows is not None:
        sched = teuk.trajectory_schedule(rows, steps, p.dt)
        ost = [O.SrcStep(*[getattr(x, f) for f, _ in teuk.SourceStep._fields_]) for x in sched]
    u = u0.copy()
    rc, psi, h, dedt = O.run(op, r_c, th, u, steps, src_steps=ost)
    assert rc == 0
    return u, psi, h, dedt


CASES = [  # N, M, integrator, m, steps, extraction column, source
    (128, 16, 1, 2, 33, -1, True),        # 16 blocks of 8 columns, one column per thread
    (136 * 8, 16, 0, -3, 20, 1, False),   # odd mode, extraction in the rho edge fill
    (192, 24, 1, 0, 33, 97, True),
    (1024, 32, 1, 2, 34, 703, True),
    (6080, 40, 0, -3, 20, 2400, False),   # two columns per thread, last block partly filled
    (8192, 32, 1, 2, 20, 8190, True),
    (4096, 64, 0, 1, 20, 2047, True),
    (8192, 64, 1, 2, 33, 2100, True),     # sweeps, two columns a phase
    (16384, 32, 0, 2, 20, 4111, True),
    (12288, 48, 1, -1, 12, 12286, True),  # 48 of 64 lanes
    (10304, 56, 0, 2, 12, 0, False),
    (9984, 24, 1, 2, 12, 2500, True),
    (16384, 64, 1, 2, 33, 4160, True),    # sweeps, four columns a phase, scalar column constants
    (16000, 64, 0, 3, 12, 15999, True),
    (32768, 32, 1, 2, 8, 8191, True),     # the same with constants from LDS
    (12288, 64, 1, 2, 12, 3070, True),    # three columns a phase
    (704, 128, 1, 2, 34, 300, True),      # two waves a column
    (6144, 128, 0, 2, 12, 6143, True),
    (128, 104, 1, -1, 20, 1, True),
    (3200, 72, 0, 3, 20, 1600, False),
    (3264, 96, 1, 0, 20, 3200, True),
    (32768, 64, 1, 2, 40, 21700, True),   # segments, the extraction column near a border
    (32768, 64, 0, 3, 12, 32766, False),
    (16384, 128, 1, 2, 33, 0, True),
    (65536, 24, 0, 2, 12, 30000, False),
    (11200, 96, 1, -2, 33, 5601, True),
]


@pytest.mark.parametrize("N,M,integrator,m,steps,je,source", CASES)
def test_resident_steps_equal_oracle(N, M, integrator, m, steps, je, source):
    print(f"resident {N}x{M} integ {integrator} m {m} steps {steps} je {je} source {source}", flush=True)
    p, u0, rows = setup(N, M, integrator, m, steps, je, source)
    with start(p, u0, rows, steps) as s:
        assert s.resident()
        s.step(1)
        s.step(steps - 1)       # 32-step launches and a rest
        s.sync()
        u, out, psi = s.get_fields(), s.output(), s.psi()
    uo, psio, ho, dedto = oracle(p, u0, rows, steps)
    assert np.isfinite(u).all()
    assert np.array_equal(u, uo)
    assert np.array_equal(psi, psio[:steps]) and np.array_equal(out["h"], ho[:steps])
    assert np.array_equal(out["dedt"], dedto[:steps])


def test_launch_shape_selects_the_stage_kernels():
    p, u0, _ = setup(1024, 32, 1, 2, 40)
    with start(p, u0, None, 40) as s:
        s.step(20)
        s.set_tiling(1, 2)      # from here on the stage kernels
        assert not s.resident()
        s.step(20)
        s.sync()
        u = s.get_fields()
    with start(p, u0, None, 40) as s:
        s.step(40)
        s.sync()
        assert np.array_equal(s.get_fields(), u)
    p, u0, _ = setup(1024, 136, 1, 2, 4)
    with start(p, u0, None, 4) as s:
        assert not s.resident()  # a column does not fit two waves


@pytest.mark.parametrize("N,M", [(1024, 32), (8192, 64), (16384, 128)])
def test_launch_that_gives_up_loses_no_step(N, M):
    """A wait of zero closes the launch's gate before any block can open it:
    the launch, and the ones queued behind it, change nothing, and the steps
    are run by the stage kernels when results are asked for."""
    p, u0, rows = setup(N, M, 1, 2, 80, N // 3, True)
    with start(p, u0, rows, 80) as s:
        s.step(80)
        s.sync()
        ref = s.get_fields(), s.output(), s.psi()
    with start(p, u0, rows, 80) as s:
        s.step(10)
        s.set_resident_wait(0.0)
        s.step(50)              # gives up; so does the launch after it
        assert s.progress()[0] == 60
        assert not s.resident()
        s.step(20)
        s.sync()
        out = s.output()
        assert np.array_equal(s.get_fields(), ref[0]) and np.array_equal(s.psi(), ref[2])
        for key in ref[1]:
            assert np.array_equal(out[key], ref[1][key]), key


def test_resident_solvers_on_several_threads():
    """Launches that each fill the GPU, from four threads at once."""
    specs = [setup(4096, 32, 1, 2, 96, seed=1), setup(4096, 32, 0, 1, 96, seed=2, source=True),
             setup(8192, 64, 1, -2, 96, seed=3), setup(1024, 16, 1, 3, 96, seed=5)]
    ref = []
    for p, u0, rows in specs:
        with start(p, u0, rows, 96) as s:
            s.step(96)
            s.sync()
            ref.append(s.get_fields())
    got = [None] * len(specs)

    def work(i):
        p, u0, rows = specs[i]
        with start(p, u0, rows, 96) as s:
            for _ in range(6):
                s.step(16)
            s.sync()
            got[i] = s.get_fields(), s.resident()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(specs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(len(specs)):
        assert np.array_equal(got[i][0], ref[i]) and got[i][1], i


BATCH = [  # N, M, m, steps, source: several row classes, narrow and wide tiles, two that do not fit
    (256, 16, 2, 40, True), (4096, 32, 2, 40, True), (8192, 32, -3, 33, False), (4096, 32, 0, 64, True),
    (16384, 32, 1, 20, False), (8192, 64, 2, 40, True), (2048, 64, 3, 12, False), (6080, 40, 2, 40, True),
    (1024, 24, -1, 70, False), (512, 72, 2, 40, True), (2048, 128, 1, 33, True), (512, 136, 2, 40, True),
    (32768, 48, 2, 20, True),
]


@pytest.mark.parametrize("integrator,wait", [(1, None), (0, None), (1, 0.0)])
def test_batch_of_resident_members_equal_alone(integrator, wait):
    """Members of one batch in shared resident launches, each as alone; with
    a wait of zero for one member its launch gives up and its members' steps
    are caught up with by the stage kernels."""
    specs = [setup(N, M, integrator, m, steps, N // 2 + 5, src, seed=i) for i, (N, M, m, steps, src) in enumerate(BATCH)]
    ref = []
    for (p, u0, rows), c in zip(specs, BATCH):
        with start(p, u0, rows, c[3]) as s:
            s.step(c[3])
            s.sync()
            ref.append((s.get_fields(), s.output(), s.psi()))
    solvers = [start(p, u0, rows, c[3]) for (p, u0, rows), c in zip(specs, BATCH)]
    if wait is not None:
        solvers[1].set_resident_wait(wait)
    with teuk.Batch(integrator=integrator) as b:
        for s in solvers:
            assert b.add(s)
        b.step(13)
        b.step(35)
        b.step(70)
        b.sync()
        assert b.info()["active"] == 0
        for s, (u, out, psi), c in zip(solvers, ref, BATCH):
            assert s.progress()[0] == c[3], c
            assert np.array_equal(s.get_fields(), u) and np.array_equal(s.psi(), psi), c
            o = s.output()
            assert np.array_equal(o["h"], out["h"]) and np.array_equal(o["t"], out["t"]), c
    for s in solvers:
        s.close()


@pytest.mark.parametrize("c", [
    (256, 16, 1, 2, 34, 0, True),         # exchange after every second stage; extraction in the rho edge fill
    (6080, 16, 0, 3, 33, 6079, True),     # RK3 pairs across steps; the last block as narrow as the halo
    (6080, 16, 1, 2, 20, 6077, False),
    (704, 32, 0, 2, 35, 11, True),
    (320, 24, 1, -1, 20, 318, True),      # rows that share a wave's lanes unevenly
    (8192, 16, 0, 2, 20, 40, True),       # two columns for some threads in the stage between
    (4096, 32, 1, -3, 33, 4095, True),
    (4096, 24, 0, 2, 20, 17, False),
    (1024, 48, 1, 2, 20, 9, True),        # every stage: one column per thread
    (8192, 32, 0, 1, 20, 2, True),        # two
    (1600, 56, 1, 2, 20, 1598, True),
], ids=str)
def test_small_tiles(c):
    N, M, integrator, m, steps, je, source = c
    p, u0, rows = setup(N, M, integrator, m, steps, je, source)
    uo, psio, ho, dedto = oracle(p, u0, rows, steps)
    with start(p, u0, rows, steps) as s:
        for n in (1, steps - 4, 3):
            s.step(n)
        s.sync()
        assert s.resident()
        u, out, psi = s.get_fields(), s.output(), s.psi()
    assert np.array_equal(u, uo) and np.array_equal(psi, psio)
    assert np.array_equal(out["h"], ho) and np.array_equal(out["dedt"], dedto)
