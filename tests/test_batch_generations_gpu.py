"""Which matrices a batch solve applies: those of the last run, prepare or graph replay that ran
on the GPU, for every set alike, whatever the kernels a run builds its tables with.  Results bit
for bit those of the plain per-set form on the same matrices."""
from __future__ import annotations

import pytest

import pfsolve_amd as pf

from test_batch_resident_gpu import Steps

pytestmark = pytest.mark.gpu


def test_run_then_other_matrices_then_solve():
    k = Steps(51)
    with pf.Batch(k.d.sets) as b:
        k.check(lambda: b.run(k.s), 0)
        k.use(k.mats[1])
        for _ in range(2):
            k.check(lambda: b.solve(k.s), 0)
        k.check(lambda: b.run(k.s), 1)
        k.use(k.mats[0])
        k.check(lambda: b.solve(k.s), 1)
        b.sync(k.s)


def test_replayed_run_then_other_matrices_then_solve():
    k = Steps(61)
    with pf.Batch(k.d.sets) as b:
        b.capture_graph(k.s)
        k.check(lambda: b.launch_graph(k.s), 0)
        k.use(k.mats[1])
        k.check(lambda: b.solve(k.s), 0)
        k.check(lambda: b.launch_graph(k.s), 1)
        k.use(k.mats[0])
        k.check(lambda: b.solve(k.s), 1)
        b.sync(k.s)


def test_solve_recorded_before_the_first_prepare():
    k = Steps(71)
    with pf.Batch(k.d.sets) as b:
        k.check(lambda: b.run(k.s), 0)
        b.capture_graph(k.s, solve_only=True)
        k.use(k.mats[1])
        k.check(lambda: b.launch_graph(k.s), 0)
        b.prepare(k.s)
        k.use(k.mats[0])
        for _ in range(2):
            k.check(lambda: b.launch_graph(k.s), 1)
        b.sync(k.s)


def test_recorded_prepare_counts_when_it_is_replayed():
    k = Steps(81)
    with pf.Batch(k.d.sets) as b:
        k.check(lambda: b.run(k.s), 0)
        g = k.t.cuda.CUDAGraph()
        with k.t.cuda.graph(g, stream=k.stream):
            b.prepare(k.s)
        k.use(k.mats[1])
        k.check(lambda: b.solve(k.s), 0)       # recorded, not run
        for which in (1, 0):
            k.use(k.mats[which])
            with k.t.cuda.stream(k.stream):
                g.replay()
            k.stream.synchronize()
            k.use(k.mats[1 - which])
            k.check(lambda: b.solve(k.s), which)
        b.sync(k.s)
