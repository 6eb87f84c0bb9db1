"""Single operators and pairs of 1025 to 2048 rows over many passes per workgroup: wavefronts
that share a system pass their boundary rows on through LDS in every pass, also where no
recurrence follows whose barriers would keep the passes apart (jw 11, a matvec alone)."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
from jw_systems import mode_buffer
from jwgpu import run_plan

pytestmark = pytest.mark.gpu

# FP64, connection matrices of degree 4096: condition below 100
TOL64 = 1e-13


@pytest.mark.parametrize("jw,ub", [(1, 0), (1, 1), (0, 0), (0, 1), (2, 0), (2, 1)])
@pytest.mark.parametrize("N,B", [(1025, 5001), (1500, 4100), (2048, 3073)])
def test_many_passes(jw, ub, N, B):
    buf = mode_buffer(jw, ub, N, False, 0, 0, 4096.0, False)[0]
    x = O.uniform(7 + N, -1, 1, B * N)
    cfg = dict(size=[N, B, 1], jw_type=10 + jw, upperBanded=ub, doublePrecision=1, scaleC=1.0)
    got = run_plan(cfg, buf, x).reshape(B, N)
    chunks = run_plan(dict(cfg, kernelVariant=1), buf, x).reshape(B, N)
    err = np.abs(got - chunks).max(1) / np.abs(chunks).max(1)
    assert err.max() <= TOL64, (int(err.argmax()), err.max())
    some = [0, 1, 1023, 1024, 2050, B - 2, B - 1]
    xs = np.ascontiguousarray(x.reshape(B, N)[some]).ravel()
    p = O.problem(jw_type=10 + jw, upperBanded=ub, N=N, B=len(some), cfg_outStride=N, cfg_scaleC=1.0)
    want = O.jw_f128(p, buf, xs).reshape(len(some), N)
    for i, b in enumerate(some):
        assert O.relerr_norm(got[b], want[i]) <= TOL64, b


@pytest.mark.parametrize("ub", [0, 1])
def test_product_alone_is_the_same_every_time(ub):
    """a matvec rounds the same in every pass: equal systems, equal results"""
    N, B = 2048, 6000
    buf = mode_buffer(1, ub, N, False, 0, 0, 4096.0, False)[0]
    one = O.uniform(9, -1, 1, 2 * N)
    x = np.tile(one, B // 2)
    cfg = dict(size=[N, B, 1], jw_type=11, upperBanded=ub, doublePrecision=1, scaleC=1.0)
    got = run_plan(cfg, buf, x).reshape(B // 2, 2 * N)
    np.testing.assert_array_equal(got, np.broadcast_to(got[0], got.shape))
