"""Batches with the default tuning: a run may build tables in LDS and leave none in memory
until resident tables are asked for.  Every order of run, prepare, solve and graph replays
gives what run = prepare + solve gives, bit for bit, with the matrices replaced in between."""
from __future__ import annotations

import numpy as np
import pytest

import pfsolve_amd as pf

from test_batch_gpu import BatchData, torch

pytestmark = pytest.mark.gpu

SETS = [(64, 5, 1, 1.0), (128, 7, 1, 0.5), (200, 9, 1, 1.0), (300, 40, 0, 1.0), (512, 6, 1, 1.0), (513, 5, 1, -1.0),
        (1024, 33, 1, 1.0), (1500, 4, 1, 1.0)]


class Steps:
    def __init__(self, seed):
        self.t = torch()
        self.d = BatchData(SETS, seed=seed)
        self.stream = self.t.cuda.Stream()
        self.s = self.stream.cuda_stream
        self.mats = [self.d.dmat.clone()]
        other = BatchData(SETS, seed=seed + 1)
        self.mats.append(other.dmat.clone())
        with pf.Batch(self.d.sets) as b:
            self.want = []
            for m in self.mats:      # the plain per-set form on each set of matrices
                self.use(m)
                self.d.reset()
                b.run_plain(self.s)
                self.want.append(self.result())
        assert not np.array_equal(*self.want)
        self.use(self.mats[0])

    def use(self, m):
        self.t.cuda.synchronize()
        self.d.dmat.copy_(m)
        self.t.cuda.synchronize()

    def result(self):
        self.stream.synchronize()
        return self.d.result()

    def check(self, call, which):
        self.d.reset()
        call()
        np.testing.assert_array_equal(self.result(), self.want[which])


def test_run_then_solve_then_new_matrices():
    k = Steps(21)
    with pf.Batch(k.d.sets) as b:
        k.check(lambda: b.run(k.s), 0)
        k.check(lambda: b.solve(k.s), 0)       # no tables were left: built from the matrices
        k.check(lambda: b.run(k.s), 0)         # resident tables are wanted now
        k.check(lambda: b.solve(k.s), 0)
        k.use(k.mats[1])
        k.check(lambda: b.solve(k.s), 0)       # the resident tables are those of the last run
        k.check(lambda: b.run(k.s), 1)
        k.check(lambda: b.solve(k.s), 1)
        b.sync(k.s)


def test_prepare_between_runs_and_changed_tuning():
    k = Steps(31)
    with pf.Batch(k.d.sets) as b:
        k.check(lambda: b.run(k.s), 0)
        k.use(k.mats[1])
        b.prepare(k.s)
        k.check(lambda: b.solve(k.s), 1)
        k.use(k.mats[0])
        k.check(lambda: b.solve(k.s), 1)
        k.check(lambda: b.run(k.s), 0)
        k.check(lambda: b.solve(k.s), 0)
        b.set_tuning(pf._abi.PfSolveBatchTuning())
        k.check(lambda: b.solve(k.s), 0)
        b.sync(k.s)


def test_recorded_runs_write_the_tables():
    k = Steps(41)
    with pf.Batch(k.d.sets) as b:
        k.check(lambda: b.run(k.s), 0)
        b.capture_graph(k.s)
        k.check(lambda: b.launch_graph(k.s), 0)
        b.prepare(k.s)
        k.use(k.mats[1])
        k.check(lambda: b.launch_graph(k.s), 1)
        k.check(lambda: b.solve(k.s), 1)
        k.use(k.mats[0])
        k.check(lambda: b.solve(k.s), 1)
        k.check(lambda: b.run(k.s), 0)
        b.capture_graph(k.s, solve_only=True)
        k.use(k.mats[1])
        k.check(lambda: b.launch_graph(k.s), 0)
        k.check(lambda: b.run(k.s), 1)
        k.check(lambda: b.launch_graph(k.s), 1)
        b.sync(k.s)


@pytest.mark.parametrize("sets,nsys", [(3, 700), (600, 2), (40, 130)])
def test_default_units_cover_every_pair(sets, nsys):
    """default unit sizes: many systems in few sets, many sets, sets that do not divide evenly"""
    specs = [(60 + 11 * (i % 45), nsys + i % 3, 1, 1.0) for i in range(sets)]
    d = BatchData(specs, seed=5, pad=0, off_sol=0)
    t = torch()
    with pf.Batch(d.sets) as b:
        d.reset()
        b.run(t.cuda.current_stream().cuda_stream)
        got = d.result()
        d.reset()
        b.run_plain(t.cuda.current_stream().cuda_stream)
        want = d.result()
    np.testing.assert_array_equal(got, want)
    d.check(got, sets=[0, sets // 2, sets - 1])
