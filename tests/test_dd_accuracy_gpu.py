"""Mean error of the double-double step over many matrices, beside that of the sequential
double-double algorithm (the CPU oracle's) on the same inputs: the scans and the table build may not
round more than it does.  Both against __float128; 192 systems put the mean's own spread at 2 to
3 %, hence the 5 %."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
from jwgpu import run_plan
from test_jw_gpu import dd_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("N", [64, 100])
def test_mean_error(N, variant):
    B, here, seq = 8, [], []
    for seed in range(24):
        buf, x, (a, b, c) = dd_inputs(N, B, 31 + N + seed)
        got = run_plan(dict(size=[N, B, 1], jw_type=14, quadDoubleDoublePrecision=1, scaleC=1.0, offsetV=a, offsetT=b,
                            offsetM=c, kernelVariant=variant), buf.ravel(), x.ravel()).reshape(-1, 2)
        p = O.problem(jw_type=14, N=N, B=B, KL=2, KU=2, cfg_outStride=N, cfg_scaleC=1.0, cfg_offsetV=a, cfg_offsetT=b,
                      cfg_offsetM=c)
        want, cpu = O.jw_f128_dd(p, buf, x), O.jw_dd(p, buf, x)
        for i in range(B):
            s = slice(i * N, (i + 1) * N)
            here.append(O.dd_relerr_norm(got[s], want[s]))
            seq.append(O.dd_relerr_norm(cpu[s], want[s]))
    print("N %d variant %d: mean %.3e, sequential %.3e" % (N, variant, np.mean(here), np.mean(seq)))
    assert np.mean(here) <= 1.05 * np.mean(seq)
