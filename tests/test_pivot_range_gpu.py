"""Tridiagonal solves whose products ld ud reach far beyond 1: the pivots p_r = 1 - ld_r ud_{r-1} /
p_{r-1} alternate between about that product and about 1 and are exact to rounding, so the scan of
the pivot maps has to keep its entries in range between them.  Odd sizes (an even number of rows is
nearly singular here) of every rows-per-thread class of a table build, against the __float128
oracle; the bound is some 50 roundings per row."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
from jwgpu import run_plan

pytestmark = pytest.mark.gpu


def matrix(N, exponent):
    rng = np.random.default_rng(N)
    buf = np.ones(3 * N)
    buf[:N] = 10.0 ** exponent * rng.uniform(1, 2, N)
    buf[2 * N:] = 10.0 ** exponent * rng.uniform(1, 2, N)
    return buf


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("exponent", [40, 60, 76, 79, 80])
@pytest.mark.parametrize("N", [17, 65, 201, 255, 333, 511, 777, 1023, 1501, 2047, 4099, 9999])
def test_large_off_diagonals(N, exponent, variant):
    B = 3
    buf = matrix(N, exponent)
    stride = N + 1
    x = O.uniform(3, -1, 1, B * stride)
    got = run_plan(dict(size=[N, B, 1], jw_type=1013, upperBanded=2, doublePrecision=1, scaleC=1.0,
                        kernelVariant=variant, outputBufferStride=[stride]), buf, x)
    p = O.problem(jw_type=1013, upperBanded=2, N=N, B=B, cfg_outStride=stride, cfg_scaleC=1.0)
    want = O.jw_f128(p, buf, x)
    for b in range(B):
        s = slice(b * stride, b * stride + N)
        assert np.all(np.isfinite(got[s]))
        assert O.relerr_norm(got[s], want[s]) <= 1e-14 * N, b
