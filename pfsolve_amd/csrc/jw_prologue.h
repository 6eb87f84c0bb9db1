// jw_prologue.h -- the coefficient-table build of the JW step (device code,
// included by jw_device.hip and jw_main64.hip): one workgroup turns one matrix
// set in the reference storage into the table the main kernels apply.
//
// Reference semantics restated (paths relative to the reference root):
//   PfSolve/pfSolve_CodeGen/pfSolve_KernelsLevel1/pfSolve_ReadWrite.h:1561-1733
//   PfSolve/pfSolve_CodeGen/pfSolve_KernelsLevel1/pfSolve_TridiagonalSolve.h:1578-1929
#ifndef PFSOLVE_JW_PROLOGUE_H
#define PFSOLVE_JW_PROLOGUE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "jw_common.h"

// ------------------------------------------------------------------------
// table layout (elements of T):
//   coefficient pair p (0..4) of row-in-lane i, lane t:  ((p*R + i)*L + t)*2 + {0,1}
//     p0 = (vm2, vm1)  p1 = (v0, vp1)  p2 = (vp2, l)  p3 = (g, h)  p4 = (D, E)
//   scan multipliers of level k, lane t: SC + (k*L + t)*4 + {0: F, 1: B1, 2: B2}
// ------------------------------------------------------------------------
__host__ __device__ __forceinline__ int64_t tab_coef(int p, int i, int t, int c, int R, int L)
{
    return ((int64_t)(p * R + i) * L + t) * 2 + c;
}
__host__ __device__ __forceinline__ int64_t tab_scan(int k, int t, int j, int R, int L)
{
    return (int64_t)JW_NCOEF * R * L + ((int64_t)k * L + t) * 4 + j;
}
__host__ __device__ __forceinline__ int ilog2_rt(int v)
{
    int r = 0;
    while ((1 << r) < v) r++;
    return r;
}

// ------------------------------------------------------------------------
// prologue: one workgroup (256 threads) per matrix set
//
// Every per-row quantity is staged in LDS (arrays of R*L elements):
//   v[-2..2], l, g, h, D, E   (rows >= N are zero)
// then written in one of two table formats:
//   format 1: the pairs above + Hillis-Steele multipliers over L lanes
//             (jw_main_kernel);
//   format 2 (L = 64): scalings folded in, a_r = D_r g_r,
//       v'_d[r] = a_r v_d[r],  l'_r = a_r l_r / a_{r-1},  h'_r = D_r h_r / D_{r+1},
//     so that the three recurrences are W_r = u'_r - l'_r W_{r-1},
//     Z_r = W_r - h'_r Z_{r+1}, y_r = Z_r - E_r y_{r+1} (W = a w, Z = D z);
//     8 coefficients per row, and per recurrence and lane 8 multipliers of the
//     DPP scan: products over the 2^k lanes a row_shr/row_shl:2^k step
//     combines (k = 0..3), then the cross-row multipliers (forward: row
//     prefix and the row_bcast31 step; backward: one per later row start)
//     (jw_main64_kernel).  Table size JW_TAB64_ELEMS(R).
// Matrix loads are spread over all threads (every load of a thread's rows issued
// at once, the band kept in registers until the fold); the LU scan runs on
// wavefront 0.
// ------------------------------------------------------------------------
constexpr int kPrologueThreads = 512;
constexpr int kProRows = 4;   // rows per thread: a build's rows <= 4 x its threads
constexpr int kMaxRT = 8;     // rows per thread of the pivot scan: a build's rows <= 8 x NP

// rows per thread at most of a build of RL rows on at least 256 threads (row phases and
// pivot scan alike), for the MAXJ / MAXRT bounds of a build whose size is known at compile time
__host__ __device__ constexpr int pro_rows(int RL) { return RL <= 256 ? 1 : (RL + 255) / 256; }

// place of row r in prologue_body's LDS arrays (rows stay inside their 32)
__host__ __device__ __forceinline__ int prologue_at(int r) { return r ^ ((r >> 3) & 31); }

// LDS of prologue_body: four arrays of RL values (the last at least 32 long, since the pivot
// scan keeps its wavefront totals there) and 24 values of the refinement.  1024 rows: 32 KiB,
// so four batched builds fit a CU.
__host__ __device__ constexpr size_t prologue_lds_bytes(int RL, size_t elt)
{
    return (3 * (size_t)RL + (RL > 32 ? (size_t)RL : 32) + 24) * elt;
}

// The band coefficients v_{-2..2} of row r of the matvec (zero outside the matrix),
// P = storage position of row r in the permuted diagonals, in two parts: row_band_load
// issues the row's loads (positions outside the matrix read an in-bounds neighbour: a
// clamped column, or the row's own position), row_band_finish zeroes what lies outside by
// selects and applies the pre-scale.  No per-row branch separates the loads (the compiler
// waits for a load before the join of any branch around it), and a caller can issue the
// loads of several rows before finishing any.
template <typename T>
__device__ __forceinline__ void row_band_load(const jw_source_desc& d, const void* mat, int64_t r, int64_t N,
                                              int64_t P, T (&raw)[6])
{
    using A = Ar<T>;
    const int mf = d.mem_f64;
#pragma unroll
    for (int k = 0; k < 5; k++) raw[k] = A::zero();
    switch (d.band_kind) {
    case JW_BAND_DIAG:
        raw[2] = mem_load<T>(mat, d.mdA + P, mf);
        break;
    case JW_BAND_UPPER:
        raw[3] = mem_load<T>(mat, d.udA + P, mf);
        raw[2] = d.unit_diag ? A::one() : mem_load<T>(mat, d.mdA + P, mf);
        break;
    case JW_BAND_LOWER:
        raw[1] = mem_load<T>(mat, d.ldA + P, mf);
        raw[2] = d.unit_diag ? A::one() : mem_load<T>(mat, d.mdA + P, mf);
        break;
    case JW_BAND_GB:
#pragma unroll
        for (int off = -2; off <= 2; off++) {
            const int64_t col = r + off;
            const int64_t cc = col < 0 ? 0 : (col >= N ? N - 1 : col);
            // band rows outside [-KL, KU] are not in the storage: read the main one
            const int j = (off < -d.KL || off > d.KU) ? d.KU : d.KU - off;
            raw[2 + off] = mem_load<T>(mat, d.offV + (int64_t)j * N + cc, mf);
        }
        break;
    default:
        raw[2] = A::one();
        break;
    }
    raw[5] = d.mdS >= 0 ? mem_load<T>(mat, d.mdS + P, mf) : A::one();
}

template <typename T>
__device__ __forceinline__ void row_band_finish(const jw_source_desc& d, int64_t r, int64_t N, const T (&raw)[6],
                                                T (&v)[5])
{
    using A = Ar<T>;
    // columns of the matvec: N, or in a chained step the previous iteration's rows
    const int64_t ncols = d.Ncols > 0 ? d.Ncols : N;
#pragma unroll
    for (int k = 0; k < 5; k++) v[k] = raw[k];
    switch (d.band_kind) {
    case JW_BAND_UPPER:
        v[3] = A::sel(r + 1 < ncols, raw[3], A::zero());
        break;
    case JW_BAND_LOWER:
        v[1] = A::sel(r >= 1 && r - 1 < ncols, raw[1], A::zero());
        break;
    case JW_BAND_GB:
#pragma unroll
        for (int off = -2; off <= 2; off++) {
            const int64_t col = r + off;
            const bool ok = off >= -d.KL && off <= d.KU && col >= 0 && col < N;
            v[2 + off] = A::sel(ok, raw[2 + off], A::zero());
        }
        break;
    default:
        break;
    }
    if (d.mdS >= 0) {
#pragma unroll
        for (int k = 0; k < 5; k++) v[k] = A::mul(v[k], raw[5]);
    }
}

// The same in one piece (loads, then selects and the pre-scale), for builds that finish
// each row before loading the next (double-double: with the two-part form the compiler
// keeps the rows' band arrays in scratch memory, measured 3x slower loads).
template <typename T>
__device__ __forceinline__ void row_band(const jw_source_desc& d, const void* mat, int64_t r, int64_t N, int64_t P,
                                         T (&v)[5])
{
    using A = Ar<T>;
    const int mf = d.mem_f64;
    // columns of the matvec: N, or in a chained step the previous iteration's rows
    const int64_t ncols = d.Ncols > 0 ? d.Ncols : N;
#pragma unroll
    for (int k = 0; k < 5; k++) v[k] = A::zero();
    switch (d.band_kind) {
    case JW_BAND_DIAG:
        v[2] = mem_load<T>(mat, d.mdA + P, mf);
        break;
    case JW_BAND_UPPER: {
        const T u = mem_load<T>(mat, d.udA + P, mf);
        v[2] = d.unit_diag ? A::one() : mem_load<T>(mat, d.mdA + P, mf);
        v[3] = A::sel(r + 1 < ncols, u, A::zero());
        break;
    }
    case JW_BAND_LOWER: {
        const T l = mem_load<T>(mat, d.ldA + P, mf);
        v[2] = d.unit_diag ? A::one() : mem_load<T>(mat, d.mdA + P, mf);
        v[1] = A::sel(r >= 1 && r - 1 < ncols, l, A::zero());
        break;
    }
    case JW_BAND_GB: {
        T raw[5];
#pragma unroll
        for (int off = -2; off <= 2; off++) {
            const int64_t col = r + off;
            const int64_t cc = col < 0 ? 0 : (col >= N ? N - 1 : col);
            // band rows outside [-KL, KU] are not in the storage: read the main one
            const int j = (off < -d.KL || off > d.KU) ? d.KU : d.KU - off;
            raw[2 + off] = mem_load<T>(mat, d.offV + (int64_t)j * N + cc, mf);
        }
#pragma unroll
        for (int off = -2; off <= 2; off++) {
            const int64_t col = r + off;
            const bool ok = off >= -d.KL && off <= d.KU && col >= 0 && col < N;
            v[2 + off] = A::sel(ok, raw[2 + off], A::zero());
        }
        break;
    }
    default:
        v[2] = A::one();
        break;
    }
    if (d.mdS >= 0) {
        const T sc = mem_load<T>(mat, d.mdS + P, mf);
#pragma unroll
        for (int k = 0; k < 5; k++) v[k] = A::mul(v[k], sc);
    }
}

// storage position of row r of the system the descriptor reads
__device__ __forceinline__ int64_t source_pos(const jw_source_desc& d, int64_t r, int64_t N)
{
    return d.alt ? alt_pos(2 * r + d.alt_parity, d.alt_N)
                 : (d.permuted ? reorder_pos(r, N, d.Nalign, d.Msplit0) : r);
}

// No pivot hand-over between builds.
struct NoPivotHooks {
    static constexpr bool kAhead = false;
    __device__ void wait_carry(int) const {}
    template <typename T> __device__ void publish(int, const T*) const {}
};
// Nothing to issue behind the build's loads.
struct NoAfterLoads {
    __device__ void operator()() const {}
};

// Takes the folded coefficients of a build that writes no table (FORMAT 3).
struct NoSink {
    template <typename T> __device__ void operator()(int, int, int, const T (&)[8]) const {}
    __device__ void done(int) const {}
};

// DPP moves and readlane of either arithmetic type (lanes without a source receive 0)
template <int CTRL, int ROWMASK = 0xf>
__device__ __forceinline__ double lane_move(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWMASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWMASK, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <int CTRL, int ROWMASK = 0xf>
__device__ __forceinline__ dd lane_move(dd v)
{
    return dd_make(lane_move<CTRL, ROWMASK>(v.hi), lane_move<CTRL, ROWMASK>(v.lo));
}
__device__ __forceinline__ double lane_read(double v, int lane) { return readlane_d(v, lane); }
__device__ __forceinline__ dd lane_read(dd v, int lane) { return dd_make(readlane_d(v.hi, lane), readlane_d(v.lo, lane)); }

// The pivot map p -> (a p + b) / (c p + e) of consecutive rows, up to a factor.
// moebius_normalize rescales its entries by a power of two (exact), so that no product over-
// or underflows: after at most two rows (whose entries are linear in each m; four rows' hold
// m_r m_{r+2}, beyond range from |m| = 1e154 on) and after every product of two maps (a row
// with |m| = 1e120 has entries of that ratio, whose products of four underflow).
template <typename T>
__device__ __forceinline__ void moebius_normalize(T& a, T& b, T& c, T& e)
{
    using A = Ar<T>;
    const double mx = fmax(fmax(fabs(A::hi(a)), fabs(A::hi(b))), fmax(fabs(A::hi(c)), fabs(A::hi(e))));
    const int ex = -__builtin_amdgcn_frexp_exp(mx);
    a = A::ldexp_(a, ex); b = A::ldexp_(b, ex); c = A::ldexp_(c, ex); e = A::ldexp_(e, ex);
}
// X <- X * P (P: the maps of earlier rows, applied first)
template <typename T>
__device__ __forceinline__ void moebius_compose(T& a, T& b, T& c, T& e, T pa, T pb, T pc, T pe)
{
    using A = Ar<T>;
    T na = A::madd(A::mul(a, pa), b, pc);
    T nb = A::madd(A::mul(a, pb), b, pe);
    T nc = A::madd(A::mul(c, pa), e, pc);
    T ne = A::madd(A::mul(c, pb), e, pe);
    a = na; b = nb; c = nc; e = ne;
}
// inclusive scan over the wavefront (lower lanes applied first): Hillis-Steele inside 16-lane
// rows, then rows 1 and 3 take the ends of rows 0 and 2, rows 2 and 3 the end of row 1
template <typename T>
__device__ __forceinline__ void moebius_scan(T& a, T& b, T& c, T& e, int lane)
{
    const int tr = lane & 15;
#define JW_SCAN_STEP(CTRL, MASK, ON)                                                                        \
    do {                                                                                                    \
        const T pa = lane_move<CTRL, MASK>(a), pb = lane_move<CTRL, MASK>(b);                               \
        const T pc = lane_move<CTRL, MASK>(c), pe = lane_move<CTRL, MASK>(e);                               \
        if (ON) moebius_compose(a, b, c, e, pa, pb, pc, pe);                                                \
        moebius_normalize(a, b, c, e);                                                                      \
    } while (0)
    JW_SCAN_STEP(DPP_ROW_SHR(1), 0xf, tr >= 1);
    JW_SCAN_STEP(DPP_ROW_SHR(2), 0xf, tr >= 2);
    JW_SCAN_STEP(DPP_ROW_SHR(4), 0xf, tr >= 4);
    JW_SCAN_STEP(DPP_ROW_SHR(8), 0xf, tr >= 8);
    JW_SCAN_STEP(0x142 /* row_bcast15 */, 0xa, lane & 16);
    JW_SCAN_STEP(0x143 /* row_bcast31 */, 0xc, lane & 32);
#undef JW_SCAN_STEP
}
// residual bound of a scanned pivot that needs no refinement, relative: a few ulps
template <typename T> constexpr double pivot_tol() { return sizeof(T) == 8 ? 0x1p-51 : 0x1p-103; }

// One table build.  Local row r of the build is row rb + r of the system.  A build of a
// long system's later rows (rb > 0) takes from `carry` the pivot of the row before its
// first (carry[0] = g_{rb-1}) and that row's raw super-diagonal entry (carry[1] =
// ud_{rb-1}), so that its pivots continue the exact recurrence; it writes nsub tables of
// R * L rows each, one after the other (format 1: table_elems apart; format 2, L = 64:
// JW_TAB64_ELEMS(R) apart, the scalings folded across the build's ends too, so that the
// tables of consecutive builds continue each other's scaled recurrences).
// Hooks of a build that hands its pivots on (tridiagonal solves only): wait_carry(tid),
// called by every thread just before the barrier after which carry[0] is first read, and
// publish(tid, g), called by every thread once the g of every row is final (g: the last
// row's, in LDS).  With kAhead the carry need not be final: publish_map(a, b, c, e) gives
// the map of the build's rows (one thread, before wait_carry), and settle(tid, refine, g, p,
// m), called by every thread after the first pass (refine: that pass needs the refinement,
// g: its last row's, p, m: the thread's first pivot and map entry), returns whether the pass
// is to be made again (workgroup-uniform, carry[0] then final; it has a barrier).  `after` is
// called once the build's own loads are issued (FP64): loads
// issued there return behind them and overlap the build.
// TP: T*, or a pointer to global memory stated as such.  FORMAT 3 folds as format 2, but
// hands row-in-lane i, lane t of the thread's j-th row to sink(j, i, t, coefficients) and
// calls sink.done(j) after each j (every thread does); it forms no scan multipliers and
// writes no table.  MAXJ, MAXRT: rows per thread at most in the row phases (RL <= MAXJ nthr) and in the pivot
// scan (RL <= MAXRT NP); smaller bounds keep a small build's per-thread arrays in fewer
// registers.
//
// The build is a chain of short latencies (one workgroup, every launch of most kernels):
// what it costs is instructions and memory round trips on one path, not bandwidth.  Hence
// the row map below, cross-lane moves by DPP instead of ds_bpermute, one division per row
// on the path of the pivots, and LDS arrays in a swizzled order (prologue_at: rows 1, 8 or 16
// apart over the lanes meet at most two-way bank conflicts).  Steps before and
// after this form, whole launches: 1024 systems of 64 rows 10.1 and 7.2 us, 8192 systems of
// 256 rows (no pivots) 12.3 and 9.4, 16384 of 1000 rows 64.1 and 58.3, the tables of 1024
// sets of 1024 - 513 rows in one launch 47 and 30.
template <typename T, int FORMAT, typename H = NoPivotHooks, int MAXJ = kProRows, int MAXRT = kMaxRT,
          typename F = NoAfterLoads, typename TP, typename S = NoSink>
__device__ __forceinline__ void prologue_body(const jw_source_desc& d, const void* mat, TP table, int L, int R,
                                              unsigned char* smem_raw, int64_t rb = 0, const T* carry = nullptr,
                                              int nsub = 1, const H& hooks = H(), const F& after = F(),
                                              const S& sink = S())
{
    constexpr bool FOLD = FORMAT != 1;
    using A = Ar<T>;
    const int RLs = R * L;                 // rows of one table
    const int RL = RLs * nsub;             // rows of this build
    const int64_t tab_elems = (int64_t)JW_NCOEF * RLs + 4 * (int64_t)ilog2_rt(L) * L;
    // format-1 element (p, c) of local row r: table rr / RLs, row-in-lane and lane of rr % RLs
    auto tab1 = [&](int r, int p, int c) -> int64_t {
        const int k = r / RLs, rr = r - k * RLs;
        return k * tab_elems + tab_coef(p, rr % R, rr / R, c, R, L);
    };
    const bool has_carry = rb > 0 && carry != nullptr;
    auto at = [](int r) -> int { return prologue_at(r); };
    T* sl = reinterpret_cast<T*>(smem_raw);    // raw ld, then l (format 1) or l' (format 2)
    T* sh = sl + RL;                           // raw ud, then h or h'
    T* sE = sh + RL;                           // E (format 1) or D (format 2)
    T* sg = sE + RL;                           // g = 1 / pivot, then E (format 2)
    T* sx = sg + (RL > 32 ? RL : 32);          // the refinement's wavefront totals and flag
    const int tid = threadIdx.x;
    const int nthr = blockDim.x;
    const int64_t N = d.N;
    const int mf = d.mem_f64;
    const bool has_b1 = d.solve_kind == JW_SOLVE_UPPER || d.solve_kind == JW_SOLVE_TRI;
    const bool has_f = d.solve_kind == JW_SOLVE_LOWER || d.solve_kind == JW_SOLVE_TRI;

    // phase 1: raw solve coefficients per row (zeros outside the matrix) into LDS,
    // band coefficients into registers (format 1: straight into the table).  Row row_of(j)
    // of thread tid; RL or more: no row.
    // Format 1: consecutive threads take consecutive rows.  Format 2: a wavefront takes a
    // tile of LT table lanes x NI rows-in-lane (LT NI = 64, NI = min(R, 8)), lane l the
    // row of table lane l mod LT, row-in-lane l / LT.  Its rows are runs of NI consecutive
    // ones (the natural-order band: few cache lines per load), and 8 neighbouring lanes
    // write 128 consecutive bytes of the table (no bank conflicts in LDS, whole segments in
    // memory).  Consecutive rows alone write 16-byte pieces 1 KiB apart, rows R apart alone
    // read 64 lines per load: each cost the build over 1 us.
    const int ni2 = FOLD ? (R >= 8 ? 3 : (R == 4 ? 2 : 1)) : 0;   // log2 NI
    auto row_of = [&](int j) -> int {
        if (!FOLD) return tid + j * nthr;
        const int lt2 = 6 - ni2;
        const int b = (tid >> 6) + (nthr >> 6) * j;                  // tile: R of them per table
        const int k = R >= 16 ? b / R : b >> (ni2);                  // R == NI below 16
        const int bb = b - k * R;
        const int c = bb & ((1 << ni2) - 1), ib = bb >> ni2;
        const int t = (c << lt2) + (tid & ((1 << lt2) - 1)), i = (ib << ni2) + ((tid & 63) >> lt2);
        return k * RLs + t * R + i;
    };
    // no thread of the wavefront has a j-th row (wavefront-uniform)
    auto none = [&](int j) -> bool { return FOLD ? (tid >> 6) + (nthr >> 6) * j >= RL / 64 : j * nthr >= RL; };
    T vb[MAXJ][5], Dr[MAXJ], Er[MAXJ];
    // FP64: every row's loads first (rows outside the matrix read row 0's positions and
    // are discarded), then the selects, products and LDS stores, so that a thread's rows
    // cost one round of memory latency.  Double-double loads and finishes row by row (the
    // rows' double-double loads at once need more registers than they save time).
    constexpr bool PRE = sizeof(T) == 8;
    T raw[PRE ? MAXJ : 1][6], sr[PRE ? MAXJ : 1][4];
    if constexpr (PRE) {
#pragma unroll
        for (int j = 0; j < MAXJ; j++) {
            if (none(j)) continue;
            const int r = row_of(j);
            const int64_t gr = rb + r;
            const int64_t gq = (r < RL && gr < N) ? gr : 0;
            const int64_t P = source_pos(d, gq, N);
            sr[j][0] = has_f ? mem_load<T>(mat, d.ldS + P, mf) : A::zero();
            sr[j][1] = has_b1 ? mem_load<T>(mat, d.udS + P, mf) : A::zero();
            sr[j][2] = d.has_m ? mem_load<T>(mat, d.mdM + P, mf) : A::one();
            sr[j][3] = d.has_m ? mem_load<T>(mat, d.udM + P, mf) : A::zero();
            row_band_load<T>(d, mat, gq, N, P, raw[j]);
        }
    }
    // format 2 folds D of the rows next to the build into its first and last rows: a build
    // of a long system's rows takes D_{rb-1} and D_{rb+RL} from the matrix
    // (every thread reads them: one address each, workgroup-uniform conditions)
    T dprev = A::one(), dnext = A::one();
    if (FOLD && d.has_m) {
        if (rb >= 1 && rb - 1 < N) dprev = mem_load<T>(mat, d.mdM + source_pos(d, rb - 1, N), mf);
        if (rb + RL < N) dnext = mem_load<T>(mat, d.mdM + source_pos(d, rb + RL, N), mf);
    }
    after();
#pragma unroll
    for (int j = 0; j < MAXJ; j++) {
        const int r = row_of(j);
        const int64_t gr = rb + r;
        T ldv = A::zero(), udv = A::zero();
        Dr[j] = A::zero();
        Er[j] = A::zero();
#pragma unroll
        for (int k = 0; k < 5; k++) vb[j][k] = A::zero();
        if (none(j)) continue;
        if (r < RL && gr < N) {
            if constexpr (PRE) {
                row_band_finish<T>(d, gr, N, raw[j], vb[j]);
                ldv = A::sel(gr >= 1, sr[j][0], A::zero());
                udv = A::sel(gr + 1 < N, sr[j][1], A::zero());
                Dr[j] = sr[j][2];
                Er[j] = A::sel(gr + 1 < N, sr[j][3], A::zero());
            } else {
                const int64_t P = source_pos(d, gr, N);
                // the solve diagonals' loads first (the band's products need its own
                // loads), all at the row's position, zeroed by selects where the row has no
                // entry
                T ldr = A::zero(), udr = A::zero(), Dv = A::one(), Ev = A::zero();
                if (has_f) ldr = mem_load<T>(mat, d.ldS + P, mf);
                if (has_b1) udr = mem_load<T>(mat, d.udS + P, mf);
                if (d.has_m) {
                    Dv = mem_load<T>(mat, d.mdM + P, mf);
                    Ev = mem_load<T>(mat, d.udM + P, mf);
                }
                row_band<T>(d, mat, gr, N, P, vb[j]);
                ldv = A::sel(gr >= 1, ldr, A::zero());
                udv = A::sel(gr + 1 < N, udr, A::zero());
                Dr[j] = Dv;
                Er[j] = A::sel(gr + 1 < N, Ev, A::zero());
            }
        }
        if (r < RL) {
            sl[at(r)] = ldv;
            sh[at(r)] = udv;
            if (FOLD && d.has_m) sE[at(r)] = Dr[j];
            if constexpr (FORMAT == 1) {
                sE[at(r)] = Er[j];
                table[tab1(r, 4, 0)] = Dr[j];
                table[tab1(r, 4, 1)] = Er[j];
                table[tab1(r, 0, 0)] = vb[j][0];
                table[tab1(r, 0, 1)] = vb[j][1];
                table[tab1(r, 1, 0)] = vb[j][2];
                table[tab1(r, 1, 1)] = vb[j][3];
                table[tab1(r, 2, 0)] = vb[j][4];
            }
        }
    }
    if (tid == 0) sx[16] = A::zero();   // the refinement flag
    __syncthreads();
    // phase 2: factors of the unit-diagonal solve.  Pivots p_r = 1 - m_r / p_{r-1},
    // m_r = ld_r ud_{r-1}: the Moebius map p -> (p - m)/p is the 2x2 matrix
    // [[1,-m],[1,0]] on (num, den).  Thread t < NP composes the maps of its RT
    // consecutive rows; an inclusive scan over those threads (DPP inside each wavefront,
    // then the wavefront totals through LDS) gives every thread the map of all rows before
    // its own, applied to (1,1) the pivot of the row before its first; each thread then
    // runs the exact recurrence over its rows.
    // NP depends on the build's rows only (up to 256 threads for 2048 rows, one wavefront
    // more per further 512), so the rounding does not depend on the workgroup size (every
    // kernel that builds a table gives the same table, bit for bit).
    if (d.solve_kind == JW_SOLVE_TRI) {
        // participating threads (the workgroup has at least NP)
        const int NP = RL <= 256 ? (RL + 63) / 64 * 64
                                 : (RL <= 256 * kMaxRT ? 256 : (RL + 64 * kMaxRT - 1) / (64 * kMaxRT) * 64);
        // the wavefront totals live in g's array, which nothing reads or writes until the
        // per-row pass below (a barrier keeps that pass after every read)
        T* s_tot = sg;
        const int RT = (RL + NP - 1) / NP;
        const int r0 = tid < NP ? tid * RT : RL;   // threads >= NP own no rows
        const int lane = tid & 63, wv = tid >> 6;
        // the wavefronts past the first NP threads own no rows: they skip the scan
        // (wave-uniform) and only keep the barriers
        const bool part = wv < NP / 64;
        // super-diagonal entry of the row before this thread's first
        const T udp0 = (r0 >= 1 && r0 < RL) ? sh[at(r0 - 1)] : ((r0 == 0 && has_carry) ? carry[1] : A::zero());
        T ldv[MAXRT], udv[MAXRT];
        T a = A::one(), b = A::zero(), c = A::zero(), e = A::one();
        T xa = A::one(), xb = A::zero(), xc = A::zero(), xe = A::one();
        if (part) {
            T udp = udp0;
#pragma unroll
            for (int i = 0; i < MAXRT; i++) {
                ldv[i] = A::zero();
                udv[i] = A::zero();
                const int r = r0 + i;
                if (i >= RT || r >= RL) continue;
                ldv[i] = sl[at(r)];
                udv[i] = sh[at(r)];
                // (rows outside the matrix and row 0 have no sub-diagonal: m = 0)
                const T m = A::mul(ldv[i], udp);
                udp = udv[i];
                const T na = A::msub(a, m, c), nb = A::msub(b, m, e);
                c = a;
                e = b;
                a = na;
                b = nb;
                if ((i & 1) == 1) moebius_normalize(a, b, c, e);
            }
            // (a row alone goes into the scan's first product as it is, which is two rows then)
            if (MAXRT > 2 && RT > 1 && (RT & 1)) moebius_normalize(a, b, c, e);
            moebius_scan(a, b, c, e, lane);
            if (lane == 63) {
                s_tot[4 * wv + 0] = a;
                s_tot[4 * wv + 1] = b;
                s_tot[4 * wv + 2] = c;
                s_tot[4 * wv + 3] = e;
            }
            // this thread's exclusive map within the wavefront (lane - 1's inclusive)
            xa = lane_move<DPP_WAVE_SHR1>(a);
            xb = lane_move<DPP_WAVE_SHR1>(b);
            xc = lane_move<DPP_WAVE_SHR1>(c);
            xe = lane_move<DPP_WAVE_SHR1>(e);
            if (lane == 0) {
                xa = A::one(); xb = A::zero(); xc = A::zero(); xe = A::one();
            }
        }
        __syncthreads();   // the wavefront totals are in LDS
        if constexpr (H::kAhead) {
            // the map of all the build's rows, for the builds behind it
            if (tid == NP - 1) {
                for (int w = wv - 1; w >= 0; w--) {
                    moebius_compose(a, b, c, e, s_tot[4 * w + 0], s_tot[4 * w + 1], s_tot[4 * w + 2], s_tot[4 * w + 3]);
                    moebius_normalize(a, b, c, e);
                }
                hooks.publish_map(a, b, c, e);
            }
        }
        if (part && wv > 0) {
            // the maps of all earlier wavefronts, then the in-wavefront part on top (none of
            // it depends on a carry, so a build that waits for one has it ready)
            T wa = s_tot[0], wb = s_tot[1], wc = s_tot[2], we = s_tot[3];
            for (int w = 1; w < wv; w++) {
                T ta = s_tot[4 * w + 0], tb = s_tot[4 * w + 1], tc = s_tot[4 * w + 2], te = s_tot[4 * w + 3];
                moebius_compose(ta, tb, tc, te, wa, wb, wc, we);
                wa = ta; wb = tb; wc = tc; we = te;
                moebius_normalize(wa, wb, wc, we);
            }
            moebius_compose(xa, xb, xc, xe, wa, wb, wc, we);
            moebius_normalize(xa, xb, xc, xe);
        }
        hooks.wait_carry(tid);
        __syncthreads();   // the carry is in LDS, the totals are read: g's array is free
        // first pass over this thread's rows.  The prefix map applied to (1, 1) (the first
        // row has no sub-diagonal, so any start works), or after a carry to (1, g_in), gives
        // the pivot of the row before as num / den, so the first row's pivot is
        // (num - m den) / num: its g and p by two independent divisions; the others by the
        // exact recurrence p_r = 1 - ld_r ud_{r-1} g_{r-1},  g_r = 1 / p_r.  Double-double takes
        // den / num first and then the recurrence, products and differences by themselves: its
        // multiply-adds round more than the two apart (mean error of a step of 64 rows 2.25e-32
        // with them, 1.91e-32 so; in FP64, where they are fused, 1.71e-16 with, 1.74e-16 without).
        T pr[MAXRT];
        auto first_pass = [&] {
            if (!part) return;
            const T gin = has_carry ? carry[0] : A::one();
            constexpr bool DD = sizeof(T) > 8;
            const T num = DD && !has_carry ? A::add(xa, xb) : A::madd(xa, xb, gin);
            const T den = DD && !has_carry ? A::add(xc, xe) : A::madd(xc, xe, gin);
            T gprev = DD ? A::div(den, num) : A::one(), udprev = udp0;
#pragma unroll
            for (int i = 0; i < MAXRT; i++) {
                pr[i] = A::one();
                const int r = r0 + i;
                if (i >= RT || r >= RL) continue;
                T g = A::zero();
                if (rb + r < N) {
                    if (DD) {
                        pr[i] = A::sub(A::one(), A::mul(A::mul(ldv[i], gprev), udprev));
                        g = A::div(A::one(), pr[i]);
                    } else if (i == 0) {
                        const T q = A::msub(num, A::mul(ldv[0], udprev), den);
                        g = A::div(num, q);
                        pr[0] = A::div(q, num);
                    } else {
                        pr[i] = A::msub(A::one(), A::mul(ldv[i], gprev), udprev);
                        g = A::div(A::one(), pr[i]);
                    }
                    gprev = g;
                }
                udprev = udv[i];
                sg[at(r)] = g;
            }
        };
        first_pass();
        __syncthreads();   // every first-pass g is in sg

        // Refinement.  Near a parabolic fixed point of the pivot map (m_r -> 1/4, e.g. the
        // Gram matrices of Jones-Worland connection matrices at small degree) the scanned
        // products lose accuracy like eps k^1.5 over k rows, where the sequential recurrence
        // loses eps k^0.5.  The pivots p~ of the first pass have residuals
        //   rho_r = p~_r - (1 - m_r / p~_{r-1})   (rounding inside a thread, the scan's error
        // at its first row), and their errors e_r = p~_r - p_r obey, to first order,
        //   e_r = rho_r + c_r e_{r-1},  c_r = m_r / p~_{r-1}^2,  e_0 = rho_0 = 0:
        // an affine recurrence, solved by one more scan over the same partition (its own
        // rounding is relative to e, far below eps); p_r = p~_r - e_r.
        // Inside a thread rho is one rounding; the scan's error shows at a thread's first
        // row.  The refinement runs only when some first-row residual exceeds a few ulps
        // (the flag is raised by any thread, read by all: the choice is workgroup-uniform
        // and a function of the matrix alone, so every kernel still builds the same table).
        auto check = [&] {
            if (!part || r0 < 1 || rb + r0 >= N) return;
            const T rho0 = A::add(A::sub(pr[0], A::one()), A::mul(A::mul(ldv[0], udp0), sg[at(r0 - 1)]));
            if (!(fabs(A::hi(rho0)) <= pivot_tol<T>() * fabs(A::hi(pr[0])))) sx[16] = A::one();
        };
        check();
        __syncthreads();
        bool refine = A::hi(sx[16]) != 0.0;
        if constexpr (H::kAhead) {
            // a carry taken from the earlier builds' maps: when it does not hold (settle), the
            // pass is made again from the pivot that the build before ends with
            if (hooks.settle(tid, refine, sg + at(RL - 1), pr[0], A::mul(ldv[0], udp0))) {
                if (tid == 0) sx[16] = A::zero();
                first_pass();
                __syncthreads();
                check();
                __syncthreads();
                refine = A::hi(sx[16]) != 0.0;
            }
        }
        // not refined: every first-pass g is final (in sg since the barrier before the
        // check), so the last one goes to the next build at once
        if (!refine) hooks.publish(tid, sg + at(RL - 1));
        if (refine) {
            T rho[MAXRT], cc[MAXRT];
            T sc = A::one(), ss = A::zero();      // this thread's map e -> sc e + ss
            if (part) {
                T gm = (r0 >= 1 && r0 < RL) ? sg[at(r0 - 1)] : ((r0 == 0 && has_carry) ? carry[0] : A::one());
                T udprev = udp0;
#pragma unroll
                for (int i = 0; i < MAXRT; i++) {
                    rho[i] = A::zero();
                    cc[i] = A::zero();
                    const int r = r0 + i;
                    if (i >= RT || rb + r >= N) continue;
                    const T m = (rb + r >= 1) ? A::mul(ldv[i], udprev) : A::zero();
                    const T mg = A::mul(m, gm);
                    rho[i] = A::add(A::sub(pr[i], A::one()), mg);
                    cc[i] = A::mul(mg, gm);
                    ss = A::madd(rho[i], cc[i], ss);
                    sc = A::mul(cc[i], sc);
                    gm = sg[at(r)];
                    udprev = udv[i];
                }
                // inclusive scan of the maps inside the wavefront, wavefront totals to LDS
                for (int k = 0; k < 6; k++) {
                    const int sft = 1 << k;
                    const int src = lane >= sft ? lane - sft : lane;
                    const T pc = lane_fetch(sc, src), ps = lane_fetch(ss, src);
                    if (lane >= sft) {
                        ss = A::madd(ss, sc, ps);
                        sc = A::mul(sc, pc);
                    }
                }
                if (lane == 63) {
                    sx[2 * wv] = sc;
                    sx[2 * wv + 1] = ss;
                }
                const int src = lane >= 1 ? lane - 1 : lane;
                const T xs = lane_fetch(ss, src), xk = lane_fetch(sc, src);
                ss = lane == 0 ? A::zero() : xs;
                sc = lane == 0 ? A::one() : xk;
            }
            __syncthreads();
            if (part) {
                // error entering this thread's first row: earlier wavefronts' maps, then this
                // wavefront's exclusive part, applied to e = 0
                T ein = A::zero();
                for (int w = 0; w < wv; w++) ein = A::madd(sx[2 * w + 1], sx[2 * w], ein);
                ein = A::madd(ss, sc, ein);
#pragma unroll
                for (int i = 0; i < MAXRT; i++) {
                    const int r = r0 + i;
                    if (i >= RT || rb + r >= N) continue;
                    ein = A::madd(rho[i], cc[i], ein);
                    // a correction that is not finite (no dominance, products out of range)
                    // is not applied
                    const double eh = A::hi(ein);
                    const T p = (eh - eh == 0.0) ? A::sub(pr[i], ein) : pr[i];
                    sg[at(r)] = A::div(A::one(), p);
                }
            }
            // the corrected g of every row is in sg
            __syncthreads();
            hooks.publish(tid, sg + at(RL - 1));
        }
    } else {
        for (int r = tid; r < RL; r += nthr) sg[at(r)] = rb + r < N ? A::one() : A::zero();
        __syncthreads();
    }

    if constexpr (FOLD) {
        // nsub tables of 64 R rows each, JW_TAB64_ELEMS(R) apart, the scalings folded:
        // with l_r = ld_r g_{r-1}, h_r = ud_r g_r and a_r = D_r g_r,
        //   l'_r = a_r l_r / a_{r-1} = a_r ld_r / D_{r-1},  h'_r = D_r h_r / D_{r+1} = a_r ud_r / D_{r+1}
        // (a build's first and last rows take D of the rows next to the build).  l', h' and
        // E then replace ld, ud and g in LDS (a row reads only its own of those).
        const int64_t te2 = JW_TAB64_ELEMS(R);
#pragma unroll
        for (int j = 0; j < MAXJ; j++) {
            const int r = none(j) ? RL : row_of(j);
            if (r < RL) {
                const int kt = nsub > 1 ? r / RLs : 0, rr = r - kt * RLs;
                const int t = rr / R, i = rr % R;
                const T ar = A::mul(Dr[j], sg[at(r)]);
                T cf[8];
#pragma unroll
                for (int k = 0; k < 5; k++) cf[k] = A::mul(ar, vb[j][k]);
                T lp = A::zero(), hp = A::zero();
                if (rb + r >= 1 && rb + r < N) {
                    lp = A::mul(ar, sl[at(r)]);
                    if (d.has_m) lp = A::div(lp, r >= 1 ? sE[at(r - 1)] : dprev);
                }
                if (rb + r + 1 < N) {
                    hp = A::mul(ar, sh[at(r)]);
                    if (d.has_m) hp = A::div(hp, r + 1 < RL ? sE[at(r + 1)] : dnext);
                }
                cf[5] = lp;
                cf[6] = hp;
                cf[7] = Er[j];
                if constexpr (FORMAT == 3) {
                    sink(j, i, t, cf);
                } else {
                    const TP tk = table + kt * te2;
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        tk[tab_coef64(p, i, t, R)] = cf[2 * p];
                        tk[tab_coef64(p, i, t, R) + 1] = cf[2 * p + 1];
                    }
                    sl[at(r)] = lp;
                    sh[at(r)] = hp;
                    sg[at(r)] = Er[j];
                }
            }
            if constexpr (FORMAT == 3) sink.done(j);
        }
        if constexpr (FORMAT == 3) return;
        __syncthreads();
        // scan multipliers: wavefront item (wave-uniform) takes recurrence j = item % 3
        // (0: forward through l', 1: backward through h', 2: backward through E) of
        // table item / 3
        for (int item = tid >> 6; item < 3 * nsub; item += nthr >> 6) {
            const int kt = item / 3, j = item - 3 * kt;
            const int t = tid & 63;
            const TP tabk = table + kt * te2;
            const T* src = j == 0 ? sl : (j == 1 ? sh : sg);
            T v = A::one();
            for (int i = 0; i < R; i++) v = A::mul(v, A::neg(src[at(kt * RLs + t * R + i)]));
            // in-row Hillis-Steele: before step k the value covers the 2^k lanes a
            // shift of 2^k combines; after 4 steps, the row prefix (j = 0) or suffix
            const int tr = t & 15;
            const TP m = tabk + (int64_t)8 * R * 64 + (int64_t)j * 8 * 64 + t;
            if (j == 0) {
                m[0] = v;
                T u = lane_move<DPP_ROW_SHR(1)>(v);
                if (tr >= 1) v = A::mul(v, u);
                m[64] = v;
                u = lane_move<DPP_ROW_SHR(2)>(v);
                if (tr >= 2) v = A::mul(v, u);
                m[128] = v;
                u = lane_move<DPP_ROW_SHR(4)>(v);
                if (tr >= 4) v = A::mul(v, u);
                m[192] = v;
                u = lane_move<DPP_ROW_SHR(8)>(v);
                if (tr >= 8) v = A::mul(v, u);
            } else {
                m[0] = v;
                T u = lane_move<DPP_ROW_SHL(1)>(v);
                if (tr + 1 <= 15) v = A::mul(v, u);
                m[64] = v;
                u = lane_move<DPP_ROW_SHL(2)>(v);
                if (tr + 2 <= 15) v = A::mul(v, u);
                m[128] = v;
                u = lane_move<DPP_ROW_SHL(4)>(v);
                if (tr + 4 <= 15) v = A::mul(v, u);
                m[192] = v;
                u = lane_move<DPP_ROW_SHL(8)>(v);
                if (tr + 8 <= 15) v = A::mul(v, u);
            }
            const int rw = t >> 4;
            if (j == 0) {
                // forward cross-row combine in two broadcasts: rows 1,3 take the end of
                // rows 0,2 (multiplier: row prefix), then rows 2,3 take lane 31, which
                // row 3 reaches through all of row 2 (prefix of lane 47 times its own)
                const T pre47 = lane_read(v, 47);
                T m2 = A::zero();
                if (rw == 2) m2 = v;
                if (rw == 3) m2 = A::mul(pre47, v);
                m[256] = v;
                m[320] = m2;
                m[384] = A::zero();
                m[448] = A::zero();
            } else {
                // backward cross-row combine from the in-row results S_1..S_3 at the
                // row starts (lanes 16, 32, 48): a lane of row r adds
                //   suf_t * F_{r+1},  F_q = S_q + P_q F_{q+1},  P_q = suffix product of lane 16q,
                // i.e. c_k,t * S_k with c_k,t = suf_t * prod_{r<q<k} P_q for k > r, else 0
                const T P1 = lane_read(v, 16), P2 = lane_read(v, 32);
                T c1 = A::zero(), c2 = A::zero(), c3 = A::zero();
                if (rw == 0) { c1 = v; c2 = A::mul(v, P1); c3 = A::mul(c2, P2); }
                if (rw == 1) { c2 = v; c3 = A::mul(v, P2); }
                if (rw == 2) c3 = v;
                m[256] = c1;
                m[320] = c2;
                m[384] = c3;
                m[448] = A::zero();
            }
        }
    } else {
        // format 1: pairs (vm2,vm1) (v0,vp1) (vp2,l) (g,h) (D,E) + Hillis-Steele multipliers
        // (the band and D, E pairs were written in phase 1)
        for (int r = tid; r < RL; r += nthr) {
            // l_r = ld_r g_{r-1},  h_r = ud_r g_r  (zero outside the matrix)
            const T gm = r >= 1 ? sg[at(r - 1)] : (has_carry ? carry[0] : A::one());
            const T l = rb + r < N ? A::mul(sl[at(r)], gm) : A::zero();
            const T h = rb + r < N ? A::mul(sh[at(r)], sg[at(r)]) : A::zero();
            sl[at(r)] = l;
            sh[at(r)] = h;
            table[tab1(r, 2, 1)] = l;
            table[tab1(r, 3, 0)] = sg[at(r)];
            table[tab1(r, 3, 1)] = h;
        }
        __syncthreads();
        // scan multipliers: wavefront k (wave-uniform) takes table k
        if ((tid >> 6) < nsub) {
            const int kt = tid >> 6;
            const int t = tid & 63;
            const TP tabk = table + kt * tab_elems;
            const int rbase = kt * RLs;
            const bool active = t < L;
            const int log2L = ilog2_rt(L);
            T bf = A::one(), bb1 = A::one(), bb2 = A::one();
            if (active) {
                for (int i = 0; i < R; i++) {
                    const int r = at(rbase + t * R + i);
                    bf = A::mul(bf, A::neg(sl[r]));
                    bb1 = A::mul(bb1, A::neg(sh[r]));
                    bb2 = A::mul(bb2, A::neg(sE[r]));
                }
            }
            for (int k = 0; k < log2L; k++) {
                const int s = 1 << k;
                if (active) {
                    tabk[tab_scan(k, t, 0, R, L)] = bf;
                    tabk[tab_scan(k, t, 1, R, L)] = bb1;
                    tabk[tab_scan(k, t, 2, R, L)] = bb2;
                    tabk[tab_scan(k, t, 3, R, L)] = A::zero();
                }
                const int su = (t >= s) ? t - s : t;
                const int sdn = (t + s < L) ? t + s : t;
                T ubf = lane_fetch(bf, su);
                T ub1 = lane_fetch(bb1, sdn);
                T ub2 = lane_fetch(bb2, sdn);
                if (active && t >= s) bf = A::mul(bf, ubf);
                if (active && t + s < L) {
                    bb1 = A::mul(bb1, ub1);
                    bb2 = A::mul(bb2, ub2);
                }
            }
        }
    }
}

// Pivot hand-over between the table builds of a long system (tridiagonal solves): build b
// waits for build b-1's last pivot (flags[b-1], acquire) and publishes its own (release).
// The wait is bounded: when it runs out the device error flag is raised and the build goes
// on with a unit pivot, so the grid always drains.
constexpr int kLongMaxPolls = 1 << 22;

template <typename T>
struct ChainHooks {
    static constexpr bool kAhead = false;
    T* carry;        // LDS: carry[0] = g entering the build
    int* flags;      // per build: 1 once its last pivot is in gval
    T* gval;         // per build: g of its last row
    int* err;
    int64_t build;
    int chained;
    __device__ void wait_carry(int tid) const
    {
        if (!chained || build == 0 || tid != 0) return;
        int polls = 0;
        bool ok = true;
        // relaxed polls, one acquire once the flag is seen: an acquire per poll invalidates caches
        // under the builds that are not waiting
        while (__hip_atomic_load(&flags[build - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
            if (++polls > kLongMaxPolls) {
                ok = false;
                __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        carry[0] = ok ? gval[build - 1] : Ar<T>::one();
    }
    __device__ void publish(int tid, const T* g) const
    {
        if (!chained || tid != 0) return;
        gval[build] = *g;
        __hip_atomic_store(&flags[build], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
};

#endif  // PFSOLVE_JW_PROLOGUE_H
