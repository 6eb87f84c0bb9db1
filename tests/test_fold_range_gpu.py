"""Scalings at the lower end of FP64: the table folds ratios of neighbouring rows' scalings D into
the recurrences, which must not pass through 1 / D (beyond the largest double for D below 5.6e-309).
Against the __float128 oracle on the same stored matrices."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
import pfsolve_amd as pf
from jwgpu import run_plan, to_dev, torch

pytestmark = pytest.mark.gpu

# D = 2.5e-309 .. 5e-309 holds 50 bits: a rounding at that scale is 1e-15, and a row's result takes
# some ten of them through coefficients that add up to less than 2
TOL = 1e-13


def tiny(N, seed):
    offV, offT, offM = 0, 5 * N, 8 * N
    raw = O.raw_matrices(seed, N)
    buf = O.pack_fused(N, raw, 0, offV, offT, offM, 10 * N)
    md = np.abs(buf[offM:offM + N])
    buf[offM:offM + N] = md / md.max() * 2.5e-309 + 2.5e-309
    return buf, (offV, offT, offM)


def want(N, B, buf, off, x):
    p = O.problem(jw_type=1014, N=N, B=B, KL=2, KU=2, cfg_outStride=N, cfg_scaleC=1.0, cfg_offsetV=off[0],
                  cfg_offsetT=off[1], cfg_offsetM=off[2])
    return O.jw_f128(p, buf, x)


def check(got, ref, N, B):
    assert np.all(np.isfinite(got))
    for b in range(B):
        s = slice(b * N, (b + 1) * N)
        assert np.max(np.abs(got[s] - ref[s])) <= TOL * np.max(np.abs(ref[s])), (N, b)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("N", [64, 200, 256, 500, 1000, 2000, 4098])
def test_plan(N, variant):
    B = 3
    buf, off = tiny(N, N)
    x = O.uniform(N, -1, 1, B * N)
    got = run_plan(dict(size=[N, B, 1], jw_type=1014, doublePrecision=1, scaleC=1.0, offsetV=off[0], offsetT=off[1],
                        offsetM=off[2], kernelVariant=variant), buf, x)
    check(got, want(N, B, buf, off, x), N, B)


@pytest.mark.parametrize("resident", [False, True])
def test_batch(resident):
    t, B = torch(), 4
    sizes = [100, 250, 510, 1000, 2000]
    data = []
    for N in sizes:
        buf, off = tiny(N, N + 1)
        x = O.uniform(N, -1, 1, B * N)
        data.append((N, buf, off, x, to_dev(buf), to_dev(x)))
    with pf.Batch([dict(N=N, nsys=B, matrices=m.data_ptr(), offsetV=o[0], offsetT=o[1], offsetM=o[2], rhs=r.data_ptr(),
                        stride=N, naturalOrder=1) for N, _, o, _, m, r in data]) as b:
        s = t.cuda.current_stream().cuda_stream
        if resident:
            b.prepare(s)
            b.solve(s)
        else:
            b.run(s)
        t.cuda.synchronize()
    for N, buf, off, x, _, r in data:
        check(r.cpu().numpy(), want(N, B, buf, off, x), N, B)
