"""Systems at odd strides and offsets (8-byte aligned only) on the wave-per-system kernels:
against the __float128 oracle and against the general kernel (kernelVariant 1), which took
every such call before, over sizes at the edges of the rows-per-lane classes."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
from jwgpu import run_plan

pytestmark = pytest.mark.gpu

# FP64, diagonally dominant draws: both kernels round like eps times a small constant
TOL64 = 1e-13


def fused(N, perm, seed):
    offV, offT, offM = 0, 5 * N, 8 * N
    raw = O.raw_matrices(seed, N)
    return O.pack_fused(N, raw, perm, offV, offT, offM, 10 * N), (offV, offT, offM)


@pytest.mark.parametrize("pad,off", [(0, 0), (1, 0), (2, 1), (3, 5)])
@pytest.mark.parametrize("N", [1, 2, 3, 63, 64, 65, 127, 128, 129, 255, 257, 333, 511, 512, 513, 777, 1023, 1024, 1025, 1535, 1537, 1999, 2047, 2048])
def test_unaligned_fused_step(N, pad, off):
    B = 7
    stride = N + pad
    keep = (N // 3, N - N // 4) if N >= 8 else (0, N)
    perm = (N + off) % 2
    buf, (offV, offT, offM) = fused(N, perm, N + 3)
    x = O.uniform(N + off, -1, 1, B * stride + off + 3)
    cfg = dict(size=[N, B, 1], jw_type=14 if perm else 1014, doublePrecision=1, scaleC=0.5, offsetV=offV,
               offsetT=offT, offsetM=offM, outputBufferStride=[stride], offsetSolution=off,
               inputZeropad=list(keep), outputZeropad=[1, N] if N >= 8 else [0, 0])
    got = run_plan(cfg, buf, x)
    general = run_plan(dict(cfg, kernelVariant=1), buf, x)
    p = O.problem(jw_type=cfg["jw_type"], N=N, B=B, KL=2, KU=2, cfg_outStride=stride, cfg_offsetSolution=off,
                  cfg_scaleC=0.5, cfg_offsetV=offV, cfg_offsetT=offT, cfg_offsetM=offM, cfg_izp=list(keep),
                  cfg_ozp=[1, N] if N >= 8 else [0, 0])
    want = O.jw_f128(p, buf, x)
    lo = 1 if N >= 8 else 0
    inside = np.zeros(x.size, bool)
    for b in range(B):
        s = slice(b * stride + off + lo, b * stride + off + N)
        assert O.relerr_norm(got[s], want[s]) <= TOL64, (b, N)
        assert O.relerr_norm(got[s], general[s]) <= TOL64, (b, N)
        inside[s] = True
    np.testing.assert_array_equal(got[~inside], x[~inside])


def test_unaligned_many_systems():
    """more passes than one sweep of the persistent grid, an odd system count"""
    N, B = 65, 40001
    buf, (offV, offT, offM) = fused(N, 1, 1)
    x = O.uniform(4, -1, 1, B * N)
    cfg = dict(size=[N, B, 1], jw_type=14, doublePrecision=1, scaleC=1.0, offsetV=offV, offsetT=offT, offsetM=offM)
    got = run_plan(cfg, buf, x).reshape(B, N)
    general = run_plan(dict(cfg, kernelVariant=1), buf, x).reshape(B, N)
    err = np.abs(got - general).max(1) / np.abs(general).max(1)
    assert err.max() <= TOL64
