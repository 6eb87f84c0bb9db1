"""Rows next to a chunk that REDUCE of a long FP64 step reads.  A plan whose keep-ranges end
early may lie in a buffer that holds nothing behind them (systems `stride` = keep-range apart),
so every address has to lie inside the keep-range and inside the extent that a call's declared
buffer is checked against."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import _oracle as O
from pfsolve_amd import build

SHIM = r"""
#include "jw_plan.h"
/* largest element of the right-hand side buffer an edge load touches, -1 none; -2 a row outside
 * the input keep-range; extent: what jw_index_extent allows */
int64_t edge_max(int64_t N, int64_t rows, int64_t lo, int64_t hi, int64_t ohi, int64_t stride, int64_t off,
                 int64_t nsys, int64_t* extent, int64_t* count)
{
    jw_source_desc s = {0};
    jw_run_desc r = {0};
    int64_t mm, top = -1;
    s.N = N;
    s.mdS = -1;
    r.nsys = nsys; r.stride = stride; r.offSol = off;
    r.in_lo = lo; r.in_hi = hi; r.out_lo = 0; r.out_hi = ohi; r.N = (int32_t)N;
    if (jw_check_offsets(&s, &r) != PFSOLVE_SUCCESS) return -3;
    jw_index_extent(&s, &r, &mm, extent);
    *count = 0;
    for (int64_t rb = 0; rb < N; rb += rows) {
        if (lo < hi) {
            const int64_t idle = jw_long_idle_row(rb, lo, hi);
            if (idle < lo || idle >= hi) return -5;
        }
        for (int lane = 0; lane < 64; lane++)
            for (int k = 0; k < 2; k++) {
                const int64_t row = jw_long_edge_row(rb, rows, lane, k, lo, hi);
                if (row < 0) continue;
                if (row < lo || row >= hi) return -2;
                if (row >= rb && row < rb + rows) return -4;
                const int64_t e = (nsys - 1) * stride + off + row;
                if (e > top) top = e;
                ++*count;
            }
    }
    return top;
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    if not os.path.exists(build.LIB):
        build.build()
    d = tmp_path_factory.mktemp("edges")
    src, so = d / "edges.c", d / "edges.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", *build.C_FLAGS, "-shared", "-o", str(so), str(src), build.LIB,
                    "-Wl,-rpath," + os.path.dirname(build.LIB)], check=True)
    f = C.CDLL(str(so)).edge_max
    f.restype = C.c_int64
    f.argtypes = [C.c_int64] * 8 + [C.POINTER(C.c_int64)] * 2
    return f


# keep-ranges that end early, on both sides of chunk ends, empty ones and the whole system
@pytest.mark.parametrize("lo,hi,ohi", [(0, 512, 512), (0, 50000, 50000), (0, 511, 3), (0, 513, 513), (0, 514, 1),
                                       (700, 701, 701), (512, 1024, 5000), (0, 0, 100), (9, 9, 100),
                                       (99999, 100000, 100000), (0, 100000, 100000)])
@pytest.mark.parametrize("off,nsys", [(0, 1), (6, 4)])
def test_edge_rows_lie_inside_the_buffer(shim, lo, hi, ohi, off, nsys):
    N, rows = 100000, 512
    stride = max(hi, ohi) + max(hi, ohi) % 2
    extent, count = C.c_int64(), C.c_int64()
    top = shim(N, rows, lo, hi, ohi, stride, off, nsys, C.byref(extent), C.byref(count))
    assert -1 <= top <= extent.value
    # a row is read once for each chunk end it is within two rows of, on the other side
    ends = range(rows, N, rows)
    want = sum(sum(lo <= e + j < hi for j in (-1, -2, 0, 1)) for e in ends)
    assert count.value == want


# FP64, diagonally dominant draws: the step rounds like eps times a small constant
TOL64 = 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("keep", [(0, 512), (0, 1000), (510, 1026), (1023, 1024), (1, 1)])
def test_early_keep_ranges_against_the_oracle(keep):
    """systems the keep-range apart, NaN behind the last one: nothing of it enters a result"""
    from jwgpu import run_plan
    N, B = 4098, 5
    out = (0, 600)
    stride = max(keep[1], out[1]) + max(keep[1], out[1]) % 2
    offV, offT, offM = 0, 5 * N, 8 * N
    buf = O.pack_fused(N, O.raw_matrices(3, N), 0, offV, offT, offM, 10 * N)
    x = np.full(B * stride + N, np.nan)
    x[:B * stride] = O.uniform(8, -1, 1, B * stride)
    izp = list(keep)
    got = run_plan(dict(size=[N, B, 1], jw_type=1014, doublePrecision=1, scaleC=1.0, offsetV=offV, offsetT=offT,
                        offsetM=offM, outputBufferStride=[stride], inputZeropad=izp, outputZeropad=list(out)), buf, x)
    p = O.problem(jw_type=1014, N=N, B=B, KL=2, KU=2, cfg_outStride=stride, cfg_scaleC=1.0, cfg_offsetV=offV,
                  cfg_offsetT=offT, cfg_offsetM=offM, cfg_izp=izp, cfg_ozp=list(out))
    want = O.jw_f128(p, buf, x)
    for b in range(B):
        s = slice(b * stride, b * stride + out[1])
        assert np.all(np.isfinite(got[s]))
        assert np.max(np.abs(got[s] - want[s])) <= TOL64 * max(np.max(np.abs(want[s])), 1e-300)
        s = slice(b * stride + out[1], (b + 1) * stride)
        np.testing.assert_array_equal(got[s], x[s])
    assert np.all(np.isnan(got[B * stride:]))
