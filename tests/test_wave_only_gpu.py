"""kernelVariant 2 asks for the wave-per-system kernels and has no chunk path behind them: systems
of 1025 to 2048 rows at an odd stride or offset are refused, as they always were, and the aligned
ones and every smaller size run."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as O
from jwgpu import run_plan
from pfsolve_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,pad,off,taken", [(1025, 0, 0, False), (1500, 1, 0, False), (1500, 0, 3, False),
                                             (2048, 2, 1, False), (1500, 0, 0, True), (1025, 1, 2, True),
                                             (777, 0, 0, True), (500, 1, 1, True), (64, 1, 0, True)])
def test_unaligned_systems(N, pad, off, taken):
    B = 3
    offV, offT, offM = 0, 5 * N, 8 * N
    buf = O.pack_fused(N, O.raw_matrices(2, N), 0, offV, offT, offM, 10 * N)
    x = O.uniform(N, -1, 1, B * (N + pad) + off + 1)
    cfg = dict(size=[N, B, 1], jw_type=1014, doublePrecision=1, scaleC=1.0, offsetV=offV, offsetT=offT, offsetM=offM,
               outputBufferStride=[N + pad], offsetSolution=off, kernelVariant=2)
    if not taken:
        assert run_plan(cfg, buf, x, expect=1) == _abi.PFSOLVE_ERROR_UNSUPPORTED_FFT_LENGTH
        return
    got = run_plan(cfg, buf, x)
    general = run_plan(dict(cfg, kernelVariant=1), buf, x)
    assert np.max(np.abs(got - general)) <= 1e-13 * np.max(np.abs(general))
