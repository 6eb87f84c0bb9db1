"""Long FP64 steps whose table builds take their entering pivot from the earlier builds' maps:
builds of 2048 rows, one, two, more than 64 of them and ragged ends, from matrices where the
scanned pivots hold (dominant) to ones where they do not and every build continues from the
one before it (m_r = ld_r ud_{r-1} within 1e-11 of 1/4).  Against the __float128 oracle: at
most 1e-13 or four times the error of the chunk kernel, whose pivots are handed on from build
to build."""
import numpy as np
import pytest

import _oracle as O
from jwgpu import run_plan
from test_jw_gpu import TOL64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("delta", [0.5, 1e-3, 1e-7, 1e-11])
@pytest.mark.parametrize("N", [2050, 4096, 4098, 6146, 20000, 140000])
def test_builds_take_the_entering_pivot_from_the_maps(N, delta):
    B = 2
    raw = [np.array(a) for a in O.raw_matrices(77 + N, N)]
    rng = np.random.default_rng(N)
    # stretches of rows near the parabolic fixed point between ordinary ones
    near = np.ones(N, bool)
    near[N // 3:N // 3 + N // 16] = False
    off = 0.5 * (1.0 - delta * (1.0 + rng.random(N)) / 2)
    for a in (1, 3):
        raw[a][near] = -(off * np.abs(raw[2]))[near]
    offV, offT, offM = 0, 5 * N, 8 * N
    buf = O.pack_fused(N, raw, 0, offV, offT, offM, 10 * N)
    x = O.uniform(5 + N, -1, 1, B * N)
    p = O.problem(jw_type=1014, N=N, B=B, KL=2, KU=2, cfg_outStride=N, cfg_scaleC=1.0, cfg_offsetV=offV,
                  cfg_offsetT=offT, cfg_offsetM=offM)
    want = O.jw_f128(p, buf, x)
    err = []
    for variant in (1, 0):
        cfg = dict(size=[N, B, 1], jw_type=1014, doublePrecision=1, scaleC=1.0, KL=2, KU=2, kernelVariant=variant,
                   offsetV=offV, offsetT=offT, offsetM=offM)
        got = run_plan(cfg, buf, x)
        err.append(max(O.relerr_norm(got[b * N:(b + 1) * N], want[b * N:(b + 1) * N]) for b in range(B)))
    print(N, delta, "chunk kernel %.2e, pair path %.2e" % tuple(err), flush=True)
    assert np.isfinite(err[0])
    assert err[1] <= max(TOL64, 4 * err[0])
