"""Serving requests whose bundles lie in mapped host memory, which a kernel moves: tiles of
4096 elements, rows padded to an even stride on the device.  Every result against the
__float128 oracle and bit for bit what the same request gives from pageable memory (moving
rounds nothing), with nothing written around the results."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import pfsolve_amd as pf
from test_serve_gpu import Workload

pytestmark = pytest.mark.gpu

# element counts around a tile's end, one tile and many, odd and even rows, one row
SIZES = [(2, 1), (3, 1), (3, 5), (17, 241), (31, 133), (64, 64), (65, 63), (65, 64), (2047, 2), (2048, 2), (1025, 9),
         (1000, 41), (300, 1200)]
KINDS = {"pinned": ("p", "p", "h"), "pinned in": ("p", "h", "h"), "pinned out": ("h", "p", "p"),
         "device": ("d", "d", "d"), "device matrices": ("p", "p", "d")}


def place(kind, values, shift):
    """values at an address 8 * shift behind an aligned one, with a guard on both sides"""
    n = values.size
    if kind == "h":
        t = torch.full((n + shift + 8,), np.nan, dtype=torch.float64)
    elif kind == "p":
        t = torch.full((n + shift + 8,), np.nan, dtype=torch.float64).pin_memory()
    else:
        t = torch.full((n + shift + 8,), np.nan, dtype=torch.float64, device="cuda")
    t[shift:shift + n] = torch.from_numpy(values)
    return t


@pytest.mark.parametrize("kinds", list(KINDS))
def test_bundles_in_mapped_memory(kinds):
    kin, kout, kmat = KINDS[kinds]
    specs = [(N, nsys, i, i % 2, 1.0) for i, (N, nsys) in enumerate(SIZES)]
    w = Workload(specs, seed=5)
    st, res = pf.serve(w.reqs, hbm_budget=64 << 20, streams=2, max_batch=5)
    assert st.requests == len(specs)
    reqs, keep = [], []
    for i, (N, nsys, key, _, _) in enumerate(specs):
        shift = 1 + 2 * (i % 2)
        x, y = place(kin, w.ins[i], shift), place(kout, np.full(nsys * N, np.nan), shift)
        m = place(kmat, np.asarray(w.mats[key][0]), 0)
        keep.append((x, y, m, shift))
        reqs.append(dict(w.reqs[i], rhs_in=x.data_ptr() + 8 * shift, rhs_out=y.data_ptr() + 8 * shift,
                         matrices=m.data_ptr()))
    torch.cuda.synchronize()
    st, res = pf.serve(reqs, hbm_budget=64 << 20, streams=2, max_batch=5)
    assert st.requests == len(specs) and all(s == 0 for _, _, s in res)
    for i, (N, nsys, *_) in enumerate(specs):
        x, y, m, shift = keep[i]
        got = y.cpu().numpy()
        assert np.all(np.isnan(got[:shift])) and np.all(np.isnan(got[shift + nsys * N:])), (kinds, N, nsys)
        assert np.array_equal(got[shift:shift + nsys * N], w.outs[i]), (kinds, N, nsys)
        w.check(i)
