"""A NaN or an infinity in one row of one system, single operators on systems at odd strides or
offsets: it reaches the rows that depend on that row, and no other row or system."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
from jwgpu import run_plan

pytestmark = pytest.mark.gpu


def reached(jw, ub, r, N):
    """rows that depend on row r: of the matvec (10, 11), then the bidiagonal solve (10, 12, 13)"""
    lo, hi = r, r
    if jw in (10, 11):
        lo, hi = (r - 1, r) if ub == 1 else (r, r + 1)
    if jw != 11:
        lo, hi = (lo, N - 1) if ub == 1 else (0, hi)
    if ub == 2:
        lo, hi = 0, N - 1
    return max(lo, 0), min(hi, N - 1)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("jw,ub", [(10, 1), (10, 0), (11, 1), (11, 0), (12, 1), (12, 0), (13, 2), (13, 1), (13, 0)])
@pytest.mark.parametrize("N", [60, 128, 200, 256, 500, 1000, 1500, 2048])
def test_rows_reached(N, jw, ub, value):
    B = 6000 if jw == 12 and N <= 256 else 3     # several sweeps of the grid: the compute / store split too
    S = N + 1 + N % 2
    buf = O.uniform(N, 0.05, 0.3, 3 * N)
    for r in (0, N // 3, N // 2 + 1, N - 1):
        x = O.uniform(N + r, 0.5, 1, B * S + 1)
        bad = B // 2
        x[bad * S + r] = value
        got = run_plan(dict(size=[N, B, 1], jw_type=1000 + jw, upperBanded=ub, doublePrecision=1, scaleC=1.0,
                            outputBufferStride=[S]), buf, x)
        lo, hi = reached(jw, ub, r, N)
        want = np.zeros(got.size, bool)
        want[bad * S + lo:bad * S + hi + 1] = True
        np.testing.assert_array_equal(~np.isfinite(got), want)
