// jw_main64.hip -- wave-per-system FP64 JW kernels for gfx950 (table format 2).
//
// One wavefront owns a pair of systems (the re/im halves of a complex system
// in XXII layout, or two consecutive real systems); lane t owns rows
// t*R .. t*R+R-1 of both.  Per pair:
//   1. input: the 16-byte chunks (row pairs) inside the input keep-range; the
//      compute / store split kernel and the chained steps load a lane's own chunks
//      straight into registers one pass ahead, the others contiguous chunks (64
//      lanes per instruction on one KiB) that LDS turns into a lane's rows: loaded
//      into registers one pass ahead, or by LDS DMA at the pass's start (queue
//      kernel 1 at R <= 8, long systems; XOR-swizzled slots so the blocked
//      read-back is bank-conflict free);
//      an odd range end is read by its owning lane alone;
//   2. banded matvec u' = a.(V x) with neighbour rows by DPP wave shifts;
//   3. three first-order recurrences (forward W, backward Z, backward y),
//      each: lane-local sweep, affine scan across the wavefront, lane-local
//      redo.  Scan: DPP row_shr/row_shl 1,2,4,8 inside 16-lane rows; across
//      rows DPP row_bcast15/row_bcast31 (forward) or readlane of the row
//      starts (backward);
//   4. row-0 scaleC; output written blocked to LDS, read back contiguous and
//      stored with 16-byte nontemporal stores (rows outside the output
//      keep-range untouched; an odd range end is written by its owning lane).
// Coefficients (8 per row, scalings folded) and scan multipliers come from the
// per-matrix-set table (format 2): built by each workgroup in its LDS (plans), or
// written by jw_prologue_kernel / jw_prologue_batch_kernel and staged once per
// workgroup or work unit in LDS (batches, serving, the plain per-set form).
// Systems of 1025 to 2048 rows: four wavefronts hold a pair (jw_wide64_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "jw_common.h"
#include "jw_prologue.h"

extern "C" void jwdev_set_error(const char* msg);

namespace {

constexpr int kLdsBytesMax = 160 * 1024;

template <int H>
__device__ __forceinline__ int swz(int c)
{
    return c ^ ((c >> 4) & (H - 1));
}

__device__ __forceinline__ void compiler_fence() { asm volatile("" ::: "memory"); }
__host__ __device__ __forceinline__ int64_t max_i64(int64_t a, int64_t b) { return a > b ? a : b; }

// A chunk (rows 2c, 2c + 1) at any 8-byte aligned address: gfx950 takes a 16-byte global
// access at dword alignment, so systems of odd stride or offset move by the same
// instructions as 16-byte aligned ones (LDS DMA does not: those paths stay aligned).
typedef double jw_d2u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ double2 load_chunk(const double* p)
{
    const jw_d2u t = *(const JW_GLOBAL jw_d2u*)p;
    return make_double2(t.x, t.y);
}

// store of a result chunk: written once and not read back by the step, so it is
// marked nontemporal (streamed to memory without allocating in the caches)
__device__ __forceinline__ void store_stream(double* p, double2 v)
{
    jw_d2u t;
    t.x = v.x;
    t.y = v.y;
    __builtin_nontemporal_store(t, (JW_GLOBAL jw_d2u*)p);
}

// A system's chunks [lo, hi) through a buffer resource: accesses outside read zeros and store
// nothing, without a branch around each.  vmcnt counts loads and stores in order, and only
// straight-line stores let the compiler wait for a pass's loads alone; with branches it waits
// for the stores behind them too, that is for the last pass's write acknowledgements: 256
// sets of 2000 rows, 64 systems each, 172 -> 129 us; 300 sets of 1024 rows, 74 -> 70; one
// plan of 30000 systems of 1024 rows, 104 -> 99.  The plain kernel for 1024 < N <= 2048 is
// no faster for it (1500 rows: 133 us by branches, 138 so) and neither are the chained steps
// up to 512 rows (115.2, 116.9); those keep the branches.  Offsets are whole chunks, so no
// access straddles the end.
struct chunk_range {
    __amdgpu_buffer_rsrc_t rsrc;
    int lo;
    __device__ __forceinline__ int offset(int c) const { return c >= lo ? c * 16 : 0x40000000; }
};
__device__ __forceinline__ chunk_range make_chunks(const double* system, int lo, int hi, bool on)
{
    // word 3 of the resource: the gfx9 raw-buffer default (data format 32)
    return chunk_range{__builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(system), 0, on ? hi * 16 : 0, 0x00020000),
                       lo};
}
__device__ __forceinline__ double2 load_chunk(const chunk_range& r, int c)
{
    typedef double d2v __attribute__((ext_vector_type(2)));
    const d2v t = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(r.rsrc, r.offset(c), 0, 0));
    return make_double2(t.x, t.y);
}
// (nontemporal: the store_stream above)
__device__ __forceinline__ void store_chunk(const chunk_range& r, int c, double2 v)
{
    typedef double d2v __attribute__((ext_vector_type(2)));
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    const d2v t = {v.x, v.y};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, t), r.rsrc, r.offset(c), 0, 2);
}

// keeps the scheduler from hoisting one phase's table loads into the previous
// phase, which would raise register pressure past the launch bound
__device__ __forceinline__ void phase_barrier() { __builtin_amdgcn_sched_barrier(0); }

// DPP move of a double with an explicit row mask; rows outside the mask and
// lanes without a source receive 0
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_rm(double v)
{
    int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWMASK, 0xf, false);
    int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWMASK, 0xf, false);
    return __hiloint2double(hi, lo);
}
constexpr int DPP_ROW_BCAST15 = 0x142;
constexpr int DPP_ROW_BCAST31 = 0x143;

// register budget: 512 / waves_per_eu VGPRs per lane (128 for R <= 8, 256 for R = 16)
template <int R>
constexpr int waves_per_eu()
{
    return R <= 8 ? 4 : 2;
}

template <int R>
constexpr int max_threads()
{
    return R <= 4 ? 1024 : (R == 8 ? 768 : 512);
}

// How the pair kernels (plain, batch queue kernels 1 and 4) move right-hand sides.  R = 16:
// contiguous loads into registers one pass ahead and a staging of one system (8 KiB), so
// that 8 wavefronts fit beside the 76 KiB table and no wavefront waits for its own loads;
// 16384 systems of 1000 rows: 57 us per step, 74.5 us when R = 16 staged pairs by LDS DMA
// (16 KiB each: 5 wavefronts, which waited for their loads) behind a table build launch.
// Smaller R: LDS DMA into a staging of two systems at the pass's start, where 12 and more
// wavefronts hide it (512 sets of 512 to 257 rows, solve: 51.5 us, 54.3 us one pass ahead).
__host__ __device__ constexpr bool pair_ahead(int R) { return R == 16; }
__host__ __device__ constexpr int64_t pair_stage_bytes(int R) { return (pair_ahead(R) ? 1LL : 2LL) * 64 * R * 8; }

// value of row r (which lane `lane` owns when r / R == lane) from the lane's registers
template <int R>
__device__ __forceinline__ double pick_row(const double (&x)[R], int i)
{
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < R; k++) v = (k == i) ? x[k] : v;
    return v;
}

// Everything one pass over a system pair needs besides the table.
struct jw_pass64 {
    double* rhs;
    int64_t nsys, stride, offSol;
    int in_lo, in_hi, out_lo, out_hi;     // keep-ranges, clipped to [0, N)
    int icl, ich, ocl, och;               // their full 16-byte chunks
    bool in_edge_lo, in_edge_hi, out_edge_lo, out_edge_hi;   // odd range ends
    int kl, ku;
    bool fwd, b1, b2, apply_scale;
    double row0_scale;                    // scaleC on lane 0, 1 elsewhere
};

__device__ __forceinline__ jw_pass64 make_pass64(double* rhs, int64_t nsys, int64_t stride, int64_t offSol,
                                                 int in_lo, int in_hi, int out_lo, int out_hi, int kl, int ku,
                                                 bool fwd, bool b1, bool b2, bool apply_scale, double scale,
                                                 int lane)
{
    jw_pass64 g;
    g.rhs = rhs;
    g.nsys = nsys;
    g.stride = stride;
    g.offSol = offSol;
    g.in_lo = in_lo;
    g.in_hi = in_hi;
    g.out_lo = out_lo;
    g.out_hi = out_hi;
    g.icl = (in_lo + 1) >> 1;
    g.ich = in_hi >> 1;
    g.ocl = (out_lo + 1) >> 1;
    g.och = out_hi >> 1;
    g.in_edge_lo = (in_lo & 1) && in_lo < in_hi;
    g.in_edge_hi = (in_hi & 1) && in_hi - 1 >= in_lo;   // never the row of in_edge_lo: lo odd => lo+1 even
    g.out_edge_lo = (out_lo & 1) && out_lo < out_hi;
    g.out_edge_hi = (out_hi & 1) && out_hi - 1 >= out_lo;
    g.kl = kl;
    g.ku = ku;
    g.fwd = fwd;
    g.b1 = b1;
    g.b2 = b2;
    g.apply_scale = apply_scale;
    g.row0_scale = lane == 0 ? scale : 1.0;
    return g;
}

template <int R>
__device__ __forceinline__ void zero_staging(double2* stg, int lane)
{
#pragma unroll
    for (int k = 0; k < R; k++) stg[64 * k + lane] = make_double2(0.0, 0.0);
}

// Leaving a work queue.  A queue is a counter pair {next unit, workgroups that have left};
// the last workgroup to leave puts both back to 0, so the next launch on the stream finds
// an empty queue with no clearing kernel or memset before it.  Every thread calls this
// after its workgroup's last claim; thread 0 counts.  The acquire-release increment orders
// every other workgroup's claims before the reset.
__device__ __forceinline__ void queue_leave(int* counter)
{
    if (threadIdx.x == 0) {
        const int n = __hip_atomic_fetch_add(counter + 1, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (n == (int)gridDim.x - 1) {
            __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(counter + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// The pieces of one pass over systems sys0 and sys0+1 (if it exists).  stg: a
// wavefront's staging for 2 systems (64 R double2); the input slots outside the
// keep-range hold zeros whenever the input DMA is issued.

// issue the input DMA (global -> LDS) of the pair; completion is vmcnt(0)
template <int R>
__device__ __forceinline__ void dma_pair(double2* stg, int lane, const jw_pass64& g, int64_t sys0)
{
    constexpr int H = R / 2;
    constexpr int SYSC = 64 * H;
    const bool ok1 = sys0 + 1 < g.nsys;
    const double* src0 = g.rhs + sys0 * g.stride + g.offSol;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        if (s == 1 && !ok1) continue;
        const double* src = src0 + s * g.stride;
#pragma unroll
        for (int k = 0; k < H; k++) {
            const int c = swz<H>(64 * k + lane);
            if (c >= g.icl && c < g.ich)
                __builtin_amdgcn_global_load_lds(
                    src + 2 * c, (__attribute__((address_space(3))) void*)(stg + s * SYSC + 64 * k), 16, 0, 0);
        }
    }
}

template <int R, bool LOOP = false>
__device__ __forceinline__ void read_edges(int lane, const jw_pass64& g, int64_t sys0, double (&x0)[R], double (&x1)[R]);

// blocked read-back of the landed input (lane t: rows t R .. t R + R-1), odd range
// ends read from global memory by their owning lane
template <int R>
__device__ __forceinline__ void read_pair(const double2* stg, int lane, const jw_pass64& g, int64_t sys0,
                                          double (&x0)[R], double (&x1)[R])
{
    constexpr int H = R / 2;
    constexpr int SYSC = 64 * H;
#pragma unroll
    for (int m = 0; m < H; m++) {
        const double2 v0 = stg[swz<H>(lane * H + m)];
        const double2 v1 = stg[SYSC + swz<H>(lane * H + m)];
        x0[2 * m] = v0.x;
        x0[2 * m + 1] = v0.y;
        x1[2 * m] = v1.x;
        x1[2 * m + 1] = v1.y;
    }
    read_edges<R>(lane, g, sys0, x0, x1);
}

// the odd ends of the input keep-range (rows whose 16-byte chunk is only half
// inside), read from global memory by their owning lane.  LOOP: waited for behind the branch,
// the wait would be every pass's, for all its loads and stores; so it is inside
template <int R, bool LOOP>
__device__ __forceinline__ void read_edges(int lane, const jw_pass64& g, int64_t sys0, double (&x0)[R], double (&x1)[R])
{
    const bool ok1 = sys0 + 1 < g.nsys;
    const JW_GLOBAL double* src0 = as_global(g.rhs) + sys0 * g.stride + g.offSol;
    if (g.in_edge_lo || g.in_edge_hi) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const bool on = e == 0 ? g.in_edge_lo : g.in_edge_hi;
            const int r = e == 0 ? g.in_lo : g.in_hi - 1;
            if (on && lane == r / R) {
                double v0 = src0[r];
                double v1 = ok1 ? src0[g.stride + r] : 0.0;
                if constexpr (LOOP) asm volatile("" : "+v"(v0), "+v"(v1));
#pragma unroll
                for (int k = 0; k < R; k++)
                    if (k == r % R) {
                        x0[k] = v0;
                        x1[k] = v1;
                    }
            }
        }
    }

}

// The banded matvec of a lane's rows: coef(p, i) is row i's coefficient pair (v_-2, v_-1),
// (v_0, v_1), (v_2, .) for p = 0, 1, 2, m and p the rows on either side of the lane's.  All five
// products are formed, with zeros where the band is narrower, so a NaN or infinity reaches the
// rows on both sides (and through zero scan multipliers some more).  EXACT (a single operator, one
// neighbour at most): rows outside the band count as zeros, and it spreads to the rows that depend
// on it only.  Systems at odd addresses take that form, since the general kernel (their other one)
// spreads it no further than a row or two; the fused step spreads it to every row in any case, and
// the aligned single operators never had it: the selects cost 8192 systems of 256 rows 9.5 -> 9.9 us.
struct band_side {
    double a1, a2, b1, b2;   // nearest and second row, of both systems
};
template <int R, bool EXACT, bool FENCE, class Coef>
__device__ __forceinline__ void band_rows(const Coef& coef, const jw_pass64& g, band_side m, band_side p,
                                          double (&x0)[R], double (&x1)[R])
{
#pragma unroll
    for (int i = 0; i < R; i++) {
        const double2 c0 = coef(0, i), c1 = coef(1, i);
        const double ia = x0[i], ib = x1[i];
        double n1a = (i + 1 < R) ? x0[(i + 1) % R] : p.a1;
        double n1b = (i + 1 < R) ? x1[(i + 1) % R] : p.b1;
        double ua = c1.x * ia, ub = c1.x * ib;
        if (EXACT) {
            m.a1 = g.kl ? m.a1 : 0.0;
            m.b1 = g.kl ? m.b1 : 0.0;
            n1a = g.ku ? n1a : 0.0;
            n1b = g.ku ? n1b : 0.0;
        }
        ua = __builtin_fma(c0.y, m.a1, ua);
        ub = __builtin_fma(c0.y, m.b1, ub);
        if (!EXACT) {
            ua = __builtin_fma(c0.x, m.a2, ua);
            ub = __builtin_fma(c0.x, m.b2, ub);
        }
        ua = __builtin_fma(c1.y, n1a, ua);
        ub = __builtin_fma(c1.y, n1b, ub);
        if (!EXACT) {
            const double vp2 = coef(2, i).x;
            ua = __builtin_fma(vp2, (i + 2 < R) ? x0[(i + 2) % R] : ((i + 2 == R) ? p.a1 : p.a2), ua);
            ub = __builtin_fma(vp2, (i + 2 < R) ? x1[(i + 2) % R] : ((i + 2 == R) ? p.b1 : p.b2), ub);
            m.a2 = m.a1;
            m.b2 = m.b1;
        }
        m.a1 = ia;
        m.b1 = ib;
        x0[i] = ua;
        x1[i] = ub;
        if (FENCE && (i & 3) == 3) phase_barrier();
    }
}
// the form of the kernels that build their table: all three recurrences, some, or some on
// systems at odd addresses
enum { kAllThree = 0, kSome = 1, kSomeExact = 2 };
int solve_form(const jw_run_desc& r)
{
    return r.fwd && r.b1 && r.b2 ? kAllThree : (r.vec2 || r.kl > 1 || r.ku > 1 || r.fused_io ? kSome : kSomeExact);
}

// adds c s; where not `on` c is 0, and EXACT does not look at s
template <bool EXACT>
__device__ __forceinline__ double add_from(double c, double s, bool on, double a)
{
    return __builtin_fma(c, !EXACT || on ? s : 0.0, a);
}

// banded matvec, the three recurrences and row-0 scaleC, in registers.
// ALL3: all three recurrences present (the fused step), decided at compile time.
// G > 1 (R = 2 only): sub-wavefront groups.  The 64 lanes form G groups of LG = 64 / G
// lanes, each solving its own pair of systems of N <= 2 LG rows; lane t is lane t mod LG of
// its group for the table (the set's 64-lane table, whose lanes from N / 2 on are zero
// rows).  What crosses lanes is cut at the group boundaries: the matvec's neighbour rows
// and the recurrences' carries are 0 at a group's ends, and the scans' cross-row stages
// run inside a group only (G = 2: the row_bcast15 stage and the readlane of the group's
// second row start; G = 4: none).  The stages left out are the ones that, for a single
// system of N <= 2 LG rows, only move its zero rows, so a group computes what the pair
// kernel computes for the same pair.
// What a chunk of a long system (64 R of its rows, a pass of its own) takes from outside
// and hands out, per system of the pair.  In: lane 0 holds the two rows before the chunk
// (h1 = row -1, h2 = row -2) and the forward carry cw (W' of row -1); lane 63 holds the two
// rows after it (h1 = row C, h2 = row C + 1) and the backward carries cz, cy (Z' and y of
// row C); every other lane holds zeros.  Out: wl = W' of the lane's last row (the chunk's
// last row on lane 63), zf = Z' of the lane's first row (the chunk's first row on lane 0).
struct jw_edge64 {
    double h1[2], h2[2], cw[2], cz[2], cy[2];
    double wl[2], zf[2];
};

template <int R, bool ALL3, int G = 1, bool EDGE = false, bool EXACT = false>
__device__ __forceinline__ void compute_pair(const double* tab, int lane, const jw_pass64& g, double (&x0)[R],
                                             double (&x1)[R], jw_edge64* e = nullptr)
{
    static_assert(!EDGE || G == 1, "chunk edges: whole wavefronts only");
    static_assert(G == 1 || (R == 2 && (G == 2 || G == 4)), "sub-wavefront groups: R = 2, G = 2 or 4");
    constexpr int SC = 8 * R * 64;            // start of the scan multipliers
    constexpr int LG = 64 / G;
    const int tl = G == 1 ? lane : (lane & (LG - 1));   // lane within the group: the table's lane
    const bool gfirst = G > 1 && tl == 0, glast = G > 1 && tl == LG - 1;
    // ---- 2. banded matvec (coefficients carry the folded row scaling) ----
    {
        double m1a = 0.0, m2a = 0.0, p1a = 0.0, p2a = 0.0;
        double m1b = 0.0, m2b = 0.0, p1b = 0.0, p2b = 0.0;
        if (g.kl >= 1) { m1a = dpp_d<DPP_WAVE_SHR1>(x0[R - 1]); m1b = dpp_d<DPP_WAVE_SHR1>(x1[R - 1]); }
        if (g.kl >= 2) { m2a = dpp_d<DPP_WAVE_SHR1>(x0[R - 2]); m2b = dpp_d<DPP_WAVE_SHR1>(x1[R - 2]); }
        if (g.ku >= 1) { p1a = dpp_d<DPP_WAVE_SHL1>(x0[0]); p1b = dpp_d<DPP_WAVE_SHL1>(x1[0]); }
        if (g.ku >= 2) { p2a = dpp_d<DPP_WAVE_SHL1>(x0[1]); p2b = dpp_d<DPP_WAVE_SHL1>(x1[1]); }
        if (gfirst) { m1a = 0.0; m1b = 0.0; m2a = 0.0; m2b = 0.0; }
        if (glast) { p1a = 0.0; p1b = 0.0; p2a = 0.0; p2b = 0.0; }
        if constexpr (EDGE) {
            // the rows next to the chunk enter where the wave shifts bring zeros
            if (lane == 0) {
                if (g.kl >= 1) { m1a = e->h1[0]; m1b = e->h1[1]; }
                if (g.kl >= 2) { m2a = e->h2[0]; m2b = e->h2[1]; }
            }
            if (lane == 63) {
                if (g.ku >= 1) { p1a = e->h1[0]; p1b = e->h1[1]; }
                if (g.ku >= 2) { p2a = e->h2[0]; p2b = e->h2[1]; }
            }
        }
        auto coef = [&](int p, int i) -> double2 {
            const double* c = tab + tab_coef64(p, i, tl, R);
            return p == 2 ? make_double2(*c, 0.0) : *reinterpret_cast<const double2*>(c);
        };
        band_rows<R, EXACT, (R >= 16)>(coef, g, band_side{m1a, m2a, m1b, m2b}, band_side{p1a, p2a, p1b, p2b}, x0, x1);
    }
    if (R >= 16) phase_barrier();

    // ---- 3a. forward recurrence W_r = u'_r - l'_r W_{r-1} ----
    if (ALL3 || g.fwd) {
        double lr[R];
#pragma unroll
        for (int i = 0; i < R; i++) lr[i] = tab[tab_coef64(2, i, tl, R) + 1];
        if constexpr (EDGE) {
            // W' entering the chunk: its first row becomes u'_0 - l'_0 cw
            if (lane == 0) {
                x0[0] = __builtin_fma(-lr[0], e->cw[0], x0[0]);
                x1[0] = __builtin_fma(-lr[0], e->cw[1], x1[0]);
            }
        }
        double a = x0[0], b = x1[0];
#pragma unroll
        for (int i = 1; i < R; i++) {
            a = __builtin_fma(-lr[i], a, x0[i]);
            b = __builtin_fma(-lr[i], b, x1[i]);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double f = tab[SC + k * 64 + tl];
            double sa, sb;
            switch (k) {
            case 0: sa = dpp_d<DPP_ROW_SHR(1)>(a); sb = dpp_d<DPP_ROW_SHR(1)>(b); break;
            case 1: sa = dpp_d<DPP_ROW_SHR(2)>(a); sb = dpp_d<DPP_ROW_SHR(2)>(b); break;
            case 2: sa = dpp_d<DPP_ROW_SHR(4)>(a); sb = dpp_d<DPP_ROW_SHR(4)>(b); break;
            default: sa = dpp_d<DPP_ROW_SHR(8)>(a); sb = dpp_d<DPP_ROW_SHR(8)>(b); break;
            }
            a = __builtin_fma(f, sa, a);
            b = __builtin_fma(f, sb, b);
        }
        if (G <= 2) {
            // rows 1 and 3 take the ends of rows 0 and 2; rows 2 and 3 then take lane 31
            const double fp = tab[SC + 4 * 64 + tl];
            const double sa = dpp_rm<DPP_ROW_BCAST15, 0xa>(a), sb = dpp_rm<DPP_ROW_BCAST15, 0xa>(b);
            a = __builtin_fma(fp, sa, a);
            b = __builtin_fma(fp, sb, b);
            if (G == 1) {
                const double fp2 = tab[SC + 5 * 64 + tl];
                const double ta = dpp_rm<DPP_ROW_BCAST31, 0xc>(a), tb = dpp_rm<DPP_ROW_BCAST31, 0xc>(b);
                a = __builtin_fma(fp2, ta, a);
                b = __builtin_fma(fp2, tb, b);
            }
        }
        double wa = dpp_d<DPP_WAVE_SHR1>(a), wb = dpp_d<DPP_WAVE_SHR1>(b);
        if (gfirst) { wa = 0.0; wb = 0.0; }
#pragma unroll
        for (int i = 0; i < R; i++) {
            wa = __builtin_fma(-lr[i], wa, x0[i]);
            wb = __builtin_fma(-lr[i], wb, x1[i]);
            x0[i] = wa;
            x1[i] = wb;
        }
    }

    if (R >= 16) phase_barrier();
    // ---- 3b/3c. backward recurrences Z_r = W_r - h'_r Z_{r+1}, y_r = Z_r - E_r y_{r+1} ----
#pragma unroll
    for (int stage = 0; stage < 2; stage++) {
        if (R >= 16 && stage == 1) phase_barrier();
        if constexpr (EDGE) {
            if (stage == 0) { e->wl[0] = x0[R - 1]; e->wl[1] = x1[R - 1]; }
            if (stage == 1) { e->zf[0] = x0[0]; e->zf[1] = x1[0]; }
        }
        if (!ALL3 && stage == 0 && !g.b1) continue;
        if (!ALL3 && stage == 1 && !g.b2) continue;
        double hh[R];
#pragma unroll
        for (int i = 0; i < R; i++) hh[i] = tab[tab_coef64(3, i, tl, R) + stage];
        if constexpr (EDGE) {
            // Z' (stage 0) or y (stage 1) entering the chunk from the row after it
            if (lane == 63) {
                const double ca = stage == 0 ? e->cz[0] : e->cy[0], cb = stage == 0 ? e->cz[1] : e->cy[1];
                x0[R - 1] = __builtin_fma(-hh[R - 1], ca, x0[R - 1]);
                x1[R - 1] = __builtin_fma(-hh[R - 1], cb, x1[R - 1]);
            }
        }
        const int j = 1 + stage;
        double a = x0[R - 1], b = x1[R - 1];
#pragma unroll
        for (int i = R - 2; i >= 0; i--) {
            a = __builtin_fma(-hh[i], a, x0[i]);
            b = __builtin_fma(-hh[i], b, x1[i]);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double f = tab[SC + (j * 8 + k) * 64 + tl];
            double sa, sb;
            switch (k) {
            case 0: sa = dpp_d<DPP_ROW_SHL(1)>(a); sb = dpp_d<DPP_ROW_SHL(1)>(b); break;
            case 1: sa = dpp_d<DPP_ROW_SHL(2)>(a); sb = dpp_d<DPP_ROW_SHL(2)>(b); break;
            case 2: sa = dpp_d<DPP_ROW_SHL(4)>(a); sb = dpp_d<DPP_ROW_SHL(4)>(b); break;
            default: sa = dpp_d<DPP_ROW_SHL(8)>(a); sb = dpp_d<DPP_ROW_SHL(8)>(b); break;
            }
            a = __builtin_fma(f, sa, a);
            b = __builtin_fma(f, sb, b);
        }
        if (G == 1) {
            // every row adds the in-row results of the later row starts (lanes 16, 32, 48),
            // weighted by matrix-only multipliers (zero for rows at or after that start)
            const double c1 = tab[SC + (j * 8 + 4) * 64 + lane];
            const double c2 = tab[SC + (j * 8 + 5) * 64 + lane];
            const double c3 = tab[SC + (j * 8 + 6) * 64 + lane];
            const double a1 = readlane_d(a, 16), a2 = readlane_d(a, 32), a3 = readlane_d(a, 48);
            const double b1 = readlane_d(b, 16), b2 = readlane_d(b, 32), b3 = readlane_d(b, 48);
            a = add_from<EXACT>(c1, a1, lane < 16, a);
            b = add_from<EXACT>(c1, b1, lane < 16, b);
            a = add_from<EXACT>(c2, a2, lane < 32, a);
            b = add_from<EXACT>(c2, b2, lane < 32, b);
            a = add_from<EXACT>(c3, a3, lane < 48, a);
            b = add_from<EXACT>(c3, b3, lane < 48, b);
        } else if (G == 2) {
            // the group's second row start: lane 16 of group 0, lane 48 of group 1
            const double c1 = tab[SC + (j * 8 + 4) * 64 + tl];
            const double a16 = readlane_d(a, 16), a48 = readlane_d(a, 48);
            const double b16 = readlane_d(b, 16), b48 = readlane_d(b, 48);
            const bool g0 = lane < 32;
            a = __builtin_fma(c1, g0 ? a16 : a48, a);
            b = __builtin_fma(c1, g0 ? b16 : b48, b);
        }
        double za = dpp_d<DPP_WAVE_SHL1>(a), zb = dpp_d<DPP_WAVE_SHL1>(b);
        if (glast) { za = 0.0; zb = 0.0; }
#pragma unroll
        for (int i = R - 1; i >= 0; i--) {
            za = __builtin_fma(-hh[i], za, x0[i]);
            zb = __builtin_fma(-hh[i], zb, x1[i]);
            x0[i] = za;
            x1[i] = zb;
        }
    }

    // ---- row-0 scaleC (pfSolve_TridiagonalSolve.h:1918-1927) ----
    if (g.apply_scale) {
        x0[0] *= g.row0_scale;
        x1[0] *= g.row0_scale;
    }

}

// results written blocked into the staging
template <int R>
__device__ __forceinline__ void write_blocked(double2* stg, int lane, const double (&x0)[R], const double (&x1)[R])
{
    constexpr int H = R / 2;
    constexpr int SYSC = 64 * H;
    compiler_fence();
#pragma unroll
    for (int m = 0; m < H; m++) {
        stg[swz<H>(lane * H + m)] = make_double2(x0[2 * m], x0[2 * m + 1]);
        stg[SYSC + swz<H>(lane * H + m)] = make_double2(x1[2 * m], x1[2 * m + 1]);
    }
}

// contiguous read of the staging and 16-byte stores of the output keep-range;
// odd range ends stored by lane 0
template <int R>
__device__ __forceinline__ void store_pair(const double2* stg, int lane, const jw_pass64& g, int64_t sys0)
{
    constexpr int H = R / 2;
    constexpr int SYSC = 64 * H;
    const bool ok1 = sys0 + 1 < g.nsys;
    compiler_fence();
    // all LDS reads first (always in bounds), so that they overlap, then the stores
    double2 v[2][H];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int k = 0; k < H; k++) v[s][k] = stg[s * SYSC + swz<H>(64 * k + lane)];
    // keeps the compiler from sinking each read into its store's branch
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int k = 0; k < H; k++) asm volatile("" : "+v"(v[s][k].x), "+v"(v[s][k].y));
#pragma unroll
    for (int s = 0; s < 2; s++) {
        if (s == 1 && !ok1) continue;
        double* dst = g.rhs + (sys0 + s) * g.stride + g.offSol;
#pragma unroll
        for (int k = 0; k < H; k++) {
            const int c = 64 * k + lane;
            if (c >= g.ocl && c < g.och) store_stream(dst + 2 * c, v[s][k]);
        }
    }
    if (g.out_edge_lo || g.out_edge_hi) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const bool on = e == 0 ? g.out_edge_lo : g.out_edge_hi;
            const int r = e == 0 ? g.out_lo : g.out_hi - 1;
            if (on && lane == 0) {
                JW_GLOBAL double* dst = as_global(g.rhs) + sys0 * g.stride + g.offSol + r;
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    if (s == 1 && !ok1) continue;
                    const double2 v = stg[s * SYSC + swz<H>(r >> 1)];
                    dst[s * g.stride] = (r & 1) ? v.y : v.x;
                }
            }
        }
    }
}

// zeros back into the slots the input DMA skips
template <int R>
__device__ __forceinline__ void rezero_input(double2* stg, int lane, const jw_pass64& g)
{
    constexpr int H = R / 2;
    constexpr int SYSC = 64 * H;
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int k = 0; k < H; k++) {
            const int c = swz<H>(64 * k + lane);
            if (!(c >= g.icl && c < g.ich)) stg[s * SYSC + 64 * k + lane] = make_double2(0.0, 0.0);
        }
    }
}

// One whole pass in one wavefront (input, compute, output through one staging).
template <int R, bool ALL3>
__device__ __forceinline__ void jw_pair64(const double* tab, double2* stg, int lane, const jw_pass64& g,
                                          int64_t sys0)
{
    dma_pair<R>(stg, lane, g, sys0);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the DMA writes have landed in LDS
    compiler_fence();
    double x0[R], x1[R];
    read_pair<R>(stg, lane, g, sys0, x0, x1);
    compute_pair<R, ALL3>(tab, lane, g, x0, x1);
    write_blocked<R>(stg, lane, x0, x1);
    store_pair<R>(stg, lane, g, sys0);
    rezero_input<R>(stg, lane, g);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): LDS traffic done before the next DMA lands
    compiler_fence();
}

// One pass of sub-wavefront groups (R = 2): the 2G consecutive systems sys0 .. sys0+2G-1
// (those below sys_end) in one wavefront, group gi solving systems sys0 + 2 gi and
// sys0 + 2 gi + 1.  Staging: system slot k (system sys0 + k) is chunks [k LG, (k+1) LG)
// of the wavefront's 128 chunks (chunk m = rows 2m, 2m+1).  Every chunk is written each
// pass (by the input DMA or as zeros), so the pass needs no zeroed staging.
template <int G>
__device__ __forceinline__ void jw_groups64(const double* tab, double2* stg, int lane, const jw_pass64& g,
                                            int64_t sys0, int64_t sys_end)
{
    constexpr int LG = 64 / G;
    const int tl = lane & (LG - 1), gi = lane / LG;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int c = 64 * j + lane;
        const int64_t sys = sys0 + c / LG;
        const int m = c & (LG - 1);
        if (sys < sys_end && m >= g.icl && m < g.ich)
            __builtin_amdgcn_global_load_lds(g.rhs + sys * g.stride + g.offSol + 2 * m,
                                             (__attribute__((address_space(3))) void*)(stg + 64 * j), 16, 0, 0);
        else
            stg[c] = make_double2(0.0, 0.0);
    }
    __builtin_amdgcn_s_waitcnt(0);   // the DMA and the zero writes have landed
    compiler_fence();
    const int64_t s0 = sys0 + 2 * gi, s1 = s0 + 1;
    double x0[2], x1[2];
    {
        const double2 v0 = stg[2 * gi * LG + tl], v1 = stg[(2 * gi + 1) * LG + tl];
        x0[0] = v0.x;
        x0[1] = v0.y;
        x1[0] = v1.x;
        x1[1] = v1.y;
    }
    // the odd ends of the input keep-range, by their owning lanes
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const bool on = e == 0 ? g.in_edge_lo : g.in_edge_hi;
        const int r = e == 0 ? g.in_lo : g.in_hi - 1;
        if (on && tl == r / 2) {
            const double v0 = s0 < sys_end ? as_global(g.rhs)[s0 * g.stride + g.offSol + r] : 0.0;
            const double v1 = s1 < sys_end ? as_global(g.rhs)[s1 * g.stride + g.offSol + r] : 0.0;
            if (r & 1) { x0[1] = v0; x1[1] = v1; } else { x0[0] = v0; x1[0] = v1; }
        }
    }
    compute_pair<2, true, G>(tab, lane, g, x0, x1);
    compiler_fence();
    stg[2 * gi * LG + tl] = make_double2(x0[0], x0[1]);
    stg[(2 * gi + 1) * LG + tl] = make_double2(x1[0], x1[1]);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the results are in the staging
    compiler_fence();
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int c = 64 * j + lane;
        const int64_t sys = sys0 + c / LG;
        const int m = c & (LG - 1);
        const double2 v = stg[c];
        if (sys < sys_end && m >= g.ocl && m < g.och)
            store_stream(g.rhs + sys * g.stride + g.offSol + 2 * m, v);
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const bool on = e == 0 ? g.out_edge_lo : g.out_edge_hi;
        const int r = e == 0 ? g.out_lo : g.out_hi - 1;
        if (on && tl == r / 2) {
            if (s0 < sys_end) as_global(g.rhs)[s0 * g.stride + g.offSol + r] = (r & 1) ? x0[1] : x0[0];
            if (s1 < sys_end) as_global(g.rhs)[s1 * g.stride + g.offSol + r] = (r & 1) ? x1[1] : x1[0];
        }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the staging is read before the next pass writes it
    compiler_fence();
}

// Direct blocked loads (kernels that load one pass ahead): lane t fetches its own R
// rows, 16-byte chunks t H .. t H + H-1, of both systems, straight into the
// registers the recurrences use.  One instruction's 64 accesses are spread over
// a 64 x 16H-byte span that its H sibling instructions complete, so every line
// is fetched from memory once and the other accesses hit the cache; no LDS
// transposition is needed.
template <int R>
__device__ __forceinline__ void load_pair_direct(double2 (&pf)[2][R / 2], int lane, const jw_pass64& g, int64_t sys0)
{
    constexpr int H = R / 2;
    const bool ok1 = sys0 + 1 < g.nsys;
    const double* src0 = g.rhs + sys0 * g.stride + g.offSol;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const double* src = src0 + s * g.stride;
#pragma unroll
        for (int m = 0; m < H; m++) {
            const int c = lane * H + m;
            double2 v = make_double2(0.0, 0.0);
            if (c >= g.icl && c < g.ich && (s == 0 || ok1)) v = load_chunk(src + 2 * c);
            pf[s][m] = v;
        }
    }
}

// the directly loaded chunks as rows, the odd keep-range ends from global memory
template <int R>
__device__ __forceinline__ void unpack_pair(const double2 (&pf)[2][R / 2], int lane, const jw_pass64& g, int64_t sys0,
                                            double (&x0)[R], double (&x1)[R])
{
#pragma unroll
    for (int m = 0; m < R / 2; m++) {
        x0[2 * m] = pf[0][m].x;
        x0[2 * m + 1] = pf[0][m].y;
        x1[2 * m] = pf[1][m].x;
        x1[2 * m + 1] = pf[1][m].y;
    }
    read_edges<R>(lane, g, sys0, x0, x1);
}

// Contiguous loads one pass ahead: lane l takes chunk 64 k + l of instruction k (one KiB per
// instruction); unpack_ahead turns them into a lane's own rows through the staging of one
// system.  For R = 16, where load_pair_direct's lanes stand 128 bytes apart: each of a
// line's 8 sibling loads misses the L1 once the wavefronts' rows exceed it, and the line
// comes from the L2 8 times (1024 sets of 1024 to 513 rows, solve: 251 us direct, 187 us
// contiguous; chained steps of 1000 rows, K = 4: 76 and 67 us).  At R <= 8 the chained steps
// measured the same or up to 4 % faster direct.
template <int R, bool BUF = true>
__device__ __forceinline__ void load_pair_ahead(double2 (&pf)[2][R / 2], int lane, const jw_pass64& g, int64_t sys0)
{
    constexpr int H = R / 2;
    const double* src0 = g.rhs + sys0 * g.stride + g.offSol;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const double* src = src0 + s * g.stride;
        const bool ok = s == 0 || sys0 + 1 < g.nsys;
        const chunk_range r = make_chunks(src, g.icl, g.ich, ok);
#pragma unroll
        for (int k = 0; k < H; k++) {
            const int c = 64 * k + lane;
            if constexpr (BUF) {
                pf[s][k] = load_chunk(r, c);
            } else {
                double2 v = make_double2(0.0, 0.0);
                if (c >= g.icl && c < g.ich && ok) v = load_chunk(src + 2 * c);
                pf[s][k] = v;
            }
        }
    }
}

template <int R, bool LOOP = true>
__device__ __forceinline__ void unpack_ahead(const double2 (&pf)[2][R / 2], double2* stg, int lane, const jw_pass64& g,
                                             int64_t sys0, double (&x0)[R], double (&x1)[R])
{
    constexpr int H = R / 2;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        double(&x)[R] = s == 0 ? x0 : x1;
        compiler_fence();   // LDS keeps a wavefront's order: the previous reads come first
#pragma unroll
        for (int k = 0; k < H; k++) stg[swz<H>(64 * k + lane)] = pf[s][k];
        compiler_fence();
#pragma unroll
        for (int m = 0; m < H; m++) {
            const double2 v = stg[swz<H>(lane * H + m)];
            x[2 * m] = v.x;
            x[2 * m + 1] = v.y;
        }
    }
    read_edges<R, LOOP>(lane, g, sys0, x0, x1);
}

// the first pair's loads end here, so that the pass loop's wait counts only what a pass issues
template <int R>
__device__ __forceinline__ void hold_pair(double2 (&pf)[2][R / 2])
{
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int k = 0; k < R / 2; k++) asm volatile("" : "+v"(pf[s][k].x), "+v"(pf[s][k].y));
}

// one system's results through a staging of 32 R chunks to contiguous 16-byte stores of
// the output keep-range; odd range ends by their owning lanes
template <int R, bool BUF = true>
__device__ __forceinline__ void store_system(double2* stg, int lane, const jw_pass64& g, int64_t sys,
                                             const double (&x)[R], bool on)
{
    constexpr int H = R / 2;
    compiler_fence();   // the staging's previous reads are issued (LDS keeps their order)
#pragma unroll
    for (int m = 0; m < H; m++) stg[swz<H>(lane * H + m)] = make_double2(x[2 * m], x[2 * m + 1]);
    compiler_fence();
    double2 v[H];
#pragma unroll
    for (int k = 0; k < H; k++) v[k] = stg[swz<H>(64 * k + lane)];
#pragma unroll
    for (int k = 0; k < H; k++) asm volatile("" : "+v"(v[k].x), "+v"(v[k].y));
    double* dst = g.rhs + sys * g.stride + g.offSol;
    const chunk_range out = make_chunks(dst, g.ocl, g.och, on);
#pragma unroll
    for (int k = 0; k < H; k++) {
        const int c = 64 * k + lane;
        if constexpr (BUF) store_chunk(out, c, v[k]);
        else if (c >= g.ocl && c < g.och) store_stream(dst + 2 * c, v[k]);
    }
    if (BUF && !on) return;
    if (g.out_edge_lo && lane == g.out_lo / R) as_global(dst)[g.out_lo] = pick_row<R>(x, g.out_lo % R);
    if (g.out_edge_hi && lane == (g.out_hi - 1) / R) as_global(dst)[g.out_hi - 1] = pick_row<R>(x, (g.out_hi - 1) % R);
}

// the results of systems sys0 and sys0 + 1 (on: sys0 is one)
template <int R, bool BUF>
__device__ __forceinline__ void store_pair(double2* stg, int lane, const jw_pass64& g, int64_t sys0,
                                           const double (&x0)[R], const double (&x1)[R], bool on)
{
    if constexpr (BUF) {
        store_system<R, true>(stg, lane, g, sys0, x0, on);
        store_system<R, true>(stg, lane, g, sys0 + 1, x1, on && sys0 + 1 < g.nsys);
    } else if (on) {
        store_system<R, false>(stg, lane, g, sys0, x0, true);
        if (sys0 + 1 < g.nsys) store_system<R, false>(stg, lane, g, sys0 + 1, x1, true);
    }
}

// Pairs q, q + step, ... below q1 through one wavefront: each pair's rows were loaded into
// registers a pass ahead (pf holds the first pair's on entry), results leave through a
// staging of one system.  geo() gives the pass geometry, rebuilt every pass from the kernel
// arguments, so that nothing derived from them stays live in registers across the loop.
template <int R, bool ALL3, bool EXACT = false, class Geo>
__device__ __forceinline__ void stream_pairs(const double* tab, double2* stg, int lane, const Geo& geo, int64_t q,
                                             int64_t q1, int64_t step, double2 (&pf)[2][R / 2])
{
    hold_pair<R>(pf);
    while (q < q1) {
        const jw_pass64 g = geo();
        double x0[R], x1[R];
        unpack_ahead<R>(pf, stg, lane, g, 2 * q, x0, x1);
        const int64_t qn = q + step;
        if (qn < q1) load_pair_ahead<R>(pf, lane, g, 2 * qn);
        compute_pair<R, ALL3, 1, false, EXACT>(tab, lane, g, x0, x1);
        store_pair<R, true>(stg, lane, g, 2 * q, x0, x1, true);
        q = qn;
    }
}

// A set's table (NTAB doubles, whole 1 KiB blocks) from global memory into LDS at `smem`
template <int NTAB>
__device__ __forceinline__ void copy_table_lds(unsigned char* smem, const void* table, int wave, int nwaves, int lane)
{
    static_assert(NTAB * 8 % 1024 == 0, "the table is whole 1 KiB blocks");
    copy_to_lds(smem, table, NTAB * 8, wave, nwaves, lane);
}

// BUILD: the table is built in LDS from the caller's matrices (the stagings as scratch)
// and pairs are loaded ahead at every R; otherwise it is copied from global memory.
template <int R, bool ALL3, bool BUILD, bool EXACT = false>
__global__ __launch_bounds__(max_threads<R>()) void jw_main64_kernel(jw_run_desc d, jw_source_desc src, const void* mat)
{
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    extern __shared__ __align__(16) unsigned char smem[];
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* stg = reinterpret_cast<double2*>(smem + NTAB * 8 + wave * (BUILD ? 512LL * R : pair_stage_bytes(R)));
    const int64_t npass = (d.nsys + 1) >> 1, step = (int64_t)gridDim.x * nwaves;
    int64_t q = (int64_t)blockIdx.x * nwaves + wave;
    // rebuilt every pass from the kernel arguments, so that nothing derived from
    // them stays live in registers across the loop
    auto geo = [&] {
        return make_pass64(reinterpret_cast<double*>(d.rhs), d.nsys, d.stride, d.offSol, (int)d.in_lo, (int)d.in_hi,
                           (int)d.out_lo, (int)d.out_hi, d.kl, d.ku, d.fwd, d.b1, d.b2, d.apply_scale, d.scale_hi,
                           lane);
    };
    if constexpr (BUILD || pair_ahead(R)) {
        // the first pair's loads go out behind the build's (or before the table copy)
        double2 pf[2][R / 2];
        auto first = [&] { if (q < npass) load_pair_ahead<R>(pf, lane, geo(), 2 * q); };
        if constexpr (BUILD) {
            prologue_body<double, 2, NoPivotHooks, R <= 8 ? 1 : 2, pro_rows(64 * R)>(
                src, mat, reinterpret_cast<double*>(smem), 64, R, smem + NTAB * 8, 0, nullptr, 1, NoPivotHooks(), first);
        } else {
            first();
            copy_table_lds<NTAB>(smem, d.table, wave, nwaves, lane);
        }
        __syncthreads();
        stream_pairs<R, ALL3, EXACT>(tab, stg, lane, geo, q, npass, step, pf);
    } else {
        copy_table_lds<NTAB>(smem, d.table, wave, nwaves, lane);
        zero_staging<R>(stg, lane);
        __syncthreads();
        for (; q < npass; q += step) jw_pair64<R, ALL3>(tab, stg, lane, geo(), 2 * q);
    }
}

// ---------------------------------------------------------------------------
// Long FP64 systems on the pair machinery (16-byte aligned systems).  Chunk c of a long
// system (rows c C .. c C + C - 1, C = 512, R = 8) is one wavefront pass over a pair of
// systems like a whole 512-row system, with the chunk's format-2 table (the scalings
// continue across chunks) and the edges of jw_edge64.  The modes of the chunk
// decomposition (jw_long.hip: COEF, REDUCE, FINISH, the reduced solve between REDUCE and
// FINISH) run the same arithmetic, so the carries the reduced solve composes from COEF's
// responses are the ones FINISH applies.
// ---------------------------------------------------------------------------
constexpr int kLong64R = 8;

// reduced data of chunk c, system s: array a (the layout of jw_long_desc)
__device__ __forceinline__ int64_t long_at(const jw_long_desc& d, int a, int64_t c, int64_t s)
{
    return ((int64_t)a * d.red_sys + s) * d.nchunks + c;
}

template <int MODE, bool ALL3>
__device__ __forceinline__ void long64_pass(const double* tab, double2* stg, int lane, const jw_pass64& g,
                                            const jw_long_desc& d, int64_t c, int64_t sys0)
{
    constexpr int R = kLong64R;
    constexpr int C = 64 * R;
    const jw_run_desc& rd = d.run;
    const double* rhs = reinterpret_cast<const double*>(rd.rhs);
    double* red = reinterpret_cast<double*>(d.red);
    const int64_t rb = c * C;
    jw_edge64 e;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        e.h1[s] = 0.0;
        e.h2[s] = 0.0;
        e.cw[s] = 0.0;
        e.cz[s] = 0.0;
        e.cy[s] = 0.0;
    }
    // The edges, loaded while the DMA is in flight: lane 0 and lane 63 take them.  Every lane
    // loads (where it needs nothing, from inside the keep-range: the buffer need not hold a
    // system's other rows) and selects afterwards: with a branch around each load the compiler
    // waited for it there, four round trips one after another in FINISH.  With the stores below
    // moved behind the arithmetic: 512 systems of 100000 rows 332 -> 318 us, 1000 of 20000 rows
    // 138 -> 130.
    double l1[2], l2[2], ca[2], cb[2];
    bool k1[2], k2[2];
    if constexpr (MODE == JW_LONG_COEF) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            // unit carries, zero right-hand sides: system 0 takes w, 1 takes z, 2 takes y
            const int64_t sys = sys0 + s;
            if (lane == 0 && sys == 0) e.cw[s] = 1.0;
            if (lane == 63 && sys == 1) e.cz[s] = 1.0;
            if (lane == 63 && sys == 2) e.cy[s] = 1.0;
        }
    } else {
        dma_pair<R>(stg, lane, g, sys0);
        const bool first = lane == 0, last = lane == 63;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool have = sys0 + s < g.nsys;
            const int64_t sys = have ? sys0 + s : sys0;
            if constexpr (MODE == JW_LONG_REDUCE) {
                // rows next to the chunk, before any chunk is written, as offsets from a row that
                // may be read (the same for the wavefront; an empty keep-range has none: the
                // reduced data stand in)
                const bool rows = rd.in_lo < rd.in_hi, edge = have && rd.band;
                const int64_t idle = rows ? jw_long_idle_row(rb, rd.in_lo, rd.in_hi) : 0;
                const JW_GLOBAL double* x =
                    rows ? as_global(rhs) + sys * rd.stride + rd.offSol + idle : as_global(red);
                const int64_t b1 = jw_long_edge_row(rb, C, 0, 0, rd.in_lo, rd.in_hi);
                const int64_t b2 = jw_long_edge_row(rb, C, 0, 1, rd.in_lo, rd.in_hi);
                const int64_t a1 = jw_long_edge_row(rb, C, 63, 0, rd.in_lo, rd.in_hi);
                const int64_t a2 = jw_long_edge_row(rb, C, 63, 1, rd.in_lo, rd.in_hi);
                k1[s] = edge && ((first && b1 >= 0) || (last && a1 >= 0));
                k2[s] = edge && ((first && b2 >= 0) || (last && a2 >= 0));
                l1[s] = x[k1[s] ? (first ? (int)(b1 - idle) : (int)(a1 - idle)) : 0];
                l2[s] = x[k2[s] ? (first ? (int)(b2 - idle) : (int)(a2 - idle)) : 0];
            } else {
                // the same rows as REDUCE read them (the step runs in place), and the carries
                k1[s] = k2[s] = have && rd.band && ((first && c > 0) || (last && c + 1 < d.nchunks));
                const JW_GLOBAL double* r = as_global(red);
                l1[s] = r[k1[s] ? (first ? long_at(d, 6, c - 1, sys) : long_at(d, 3, c + 1, sys))
                                : long_at(d, 7, c, sys)];
                l2[s] = r[k1[s] ? (first ? long_at(d, 5, c - 1, sys) : long_at(d, 4, c + 1, sys))
                                : long_at(d, 7, c, sys)];
                ca[s] = r[long_at(d, last ? 8 : 7, c, sys)];
                cb[s] = r[long_at(d, 9, c, sys)];
            }
        }
    }
    double x0[R], x1[R];
    if constexpr (MODE == JW_LONG_COEF) {
#pragma unroll
        for (int i = 0; i < R; i++) {
            x0[i] = 0.0;
            x1[i] = 0.0;
        }
    } else {
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the DMA writes have landed in LDS
        compiler_fence();
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool have = sys0 + s < g.nsys;
            e.h1[s] = k1[s] ? l1[s] : 0.0;
            e.h2[s] = k2[s] ? l2[s] : 0.0;
            if constexpr (MODE == JW_LONG_FINISH) {
                e.cw[s] = have && lane == 0 ? ca[s] : 0.0;
                e.cz[s] = have && lane == 63 ? ca[s] : 0.0;
                e.cy[s] = have && lane == 63 ? cb[s] : 0.0;
            }
        }
        read_pair<R>(stg, lane, g, sys0, x0, x1);
    }
    // REDUCE: the rows the neighbouring chunks' banded matvec needs, as read (lane 0: the
    // first two, lane 63: the last two), stored with the boundary values: stored here, their
    // acknowledgements were waited for before the arithmetic
    double n0[2], n1[2];
    if constexpr (MODE == JW_LONG_REDUCE) {
        n0[0] = lane == 0 ? x0[0] : x0[R - 2];
        n1[0] = lane == 0 ? x0[1] : x0[R - 1];
        n0[1] = lane == 0 ? x1[0] : x1[R - 2];
        n1[1] = lane == 0 ? x1[1] : x1[R - 1];
    }
    compute_pair<R, ALL3, 1, true>(tab, lane, g, x0, x1, &e);
    if constexpr (MODE == JW_LONG_FINISH) {
        write_blocked<R>(stg, lane, x0, x1);
        store_pair<R>(stg, lane, g, sys0);
        rezero_input<R>(stg, lane, g);
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): LDS traffic done before the next DMA lands
        compiler_fence();
    } else {
        // boundary values: W' at the chunk's last row, Z' and y at its first
        double* coef = red + (int64_t)JW_LONG_ARRAYS * d.nchunks * d.red_sys;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int64_t sys = sys0 + s;
            if (sys >= g.nsys) continue;
            const double y0 = s == 0 ? x0[0] : x1[0];
            if constexpr (MODE == JW_LONG_COEF) {
                if (lane == 63) coef[9 * c + 3 * sys + 0] = e.wl[s];
                if (lane == 0) {
                    coef[9 * c + 3 * sys + 1] = e.zf[s];
                    coef[9 * c + 3 * sys + 2] = y0;
                }
            } else if (lane == 0 || lane == 63) {
                red[long_at(d, lane == 0 ? 3 : 5, c, sys)] = n0[s];
                red[long_at(d, lane == 0 ? 4 : 6, c, sys)] = n1[s];
                red[long_at(d, lane == 0 ? 1 : 0, c, sys)] = lane == 0 ? e.zf[s] : e.wl[s];
                if (lane == 0) red[long_at(d, 2, c, sys)] = y0;
            }
        }
    }
}

// A persistent grid: workgroup b takes the units [b per_wg, (b + 1) per_wg) of the
// (chunk, pair of systems) space in chunk order, stages each chunk's table in LDS once and
// spreads the chunk's pairs over its wavefronts.
template <int MODE, bool ALL3>
__global__ __launch_bounds__(max_threads<kLong64R>()) void jw_long64_kernel(jw_long_desc d, int64_t per_wg)
{
    constexpr int R = kLong64R;
    constexpr int C = 64 * R;
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    extern __shared__ __align__(16) unsigned char smem[];
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* stg = reinterpret_cast<double2*>(smem + NTAB * 8) + (size_t)wave * 64 * R;
    const jw_run_desc& rd = d.run;
    const int64_t nc = d.nchunks;
    const int64_t ppc = (rd.nsys + 1) >> 1;
    const int64_t u0 = (int64_t)blockIdx.x * per_wg;
    const int64_t u1 = u0 + per_wg < nc * ppc ? u0 + per_wg : nc * ppc;
    for (int64_t c = u0 / ppc; c < nc && c * ppc < u1; c++) {
        __syncthreads();   // the previous chunk's passes are done: its table may go
        copy_table_lds<NTAB>(smem, reinterpret_cast<const double*>(d.table) + c * d.tab_elems, wave, nwaves, lane);
        zero_staging<R>(stg, lane);   // this chunk's keep-range may be narrower
        __syncthreads();
        // keep-ranges relative to the chunk, inside its rows of the system
        const int64_t rb = c * C;
        const int64_t cn = (int64_t)rd.N - rb < C ? (int64_t)rd.N - rb : C;
        auto clip = [&](int64_t v) -> int {
            const int64_t w = v - rb;
            return (int)(w < 0 ? 0 : (w > cn ? cn : w));
        };
        const int ilo = clip(rd.in_lo), olo = clip(rd.out_lo);
        const int ihi = clip(rd.in_hi) > ilo ? clip(rd.in_hi) : ilo;
        const int ohi = clip(rd.out_hi) > olo ? clip(rd.out_hi) : olo;
        const int64_t q0 = (u0 > c * ppc ? u0 : c * ppc) - c * ppc;
        const int64_t q1 = (u1 < (c + 1) * ppc ? u1 : (c + 1) * ppc) - c * ppc;
        for (int64_t q = q0 + wave; q < q1; q += nwaves) {
            const jw_pass64 g = make_pass64(reinterpret_cast<double*>(rd.rhs), rd.nsys, rd.stride, rd.offSol + rb, ilo,
                                            ihi, olo, ohi, rd.kl, rd.ku, rd.fwd, rd.b1, rd.b2,
                                            MODE == JW_LONG_FINISH && c == 0 && rd.apply_scale, rd.scale_hi, lane);
            long64_pass<MODE, ALL3>(tab, stg, lane, g, d, c, 2 * q);
        }
    }
}

// The front of a long FP64 step in one launch: the chunks' table builds, then COEF and
// REDUCE of the first slice of systems behind them.  Workgroups take tickets in start
// order.  The first nbuild build the tables, NSUB chunks each (the pivots' way through them:
// below), mark the build's tables written (tflags) and leave.  The others drain a queue
// of units in chunk order (unit 0 of a chunk: COEF on two wavefronts; unit j > 0: REDUCE of
// pairs [(j-1) P, j P)), waiting for each chunk's tables before
// staging them, so that the reduction runs while later tables are still being built.  A
// worker's ticket comes after every build's, so every build it waits for has started, and
// builds wait only for earlier builds: the launch drains whatever the residency.  All
// waits are bounded (the device error flag is raised when one runs out).
// sync: [0] ticket, [1] queue counter, [kLong64Tflags + b] build b's tables written;
// lines: the builds' maps and pivots (below); both set by jw_long64_clear_kernel before the launch.
constexpr int kLong64Nsub = 4;   // chunks per table build: 2, 3, 4 and 6 measured 87, 88, 89
                                 // and 93 us (100000 rows, 64 systems), 309, 275, 260 and
                                 // 246 us (10^6 rows, 8 systems: 490 builds' maps at 4)
constexpr int kLong64PairsPerUnit = 2 * (max_threads<kLong64R>() / 64);
constexpr int kLong64UnitsPerWorker = 2;
constexpr int kLong64Tflags = 32;   // the table flags start one 128-byte line after the counters

// The pivots' way through the builds.  Every build publishes the map of its rows; a build
// composes the maps of all builds before it (one wavefront, 64 at a time) for the pivot that
// enters it, runs its rows, publishes its last pivot and checks its first one against the
// last of the build before, as a build's threads check theirs.  If that holds for it and for
// every build before it, its pivots stand.  If not (near a parabolic fixed point the scanned
// products lose accuracy) it takes the final last pivot of the build before and makes its
// pass again, refined where needed: from the first such build on, one build after another.
// So the builds wait for three hand-overs, not for one per build before them: 100000 rows,
// 2 systems 159 -> 111 us, 64 systems 128 -> 87, 512 systems 319 -> 312; 8 systems of 10^6
// rows 1290 -> 257.  Where the scanned pivots do not hold (ld_r ud_{r-1} within 1e-7 of 1/4
// everywhere, 64 systems of 100000 rows) the extra hand-overs cost 202 -> 227.
// A word of a build's line holds all ones (a NaN pattern never published: a NaN is
// published as the canonical one) until it is written; it carries its own readiness, so
// relaxed atomics suffice, no flag, no release or acquire.  The waits are bounded: when one
// runs out the device error flag is raised and the build goes on with a one, so the grid
// always drains.
constexpr unsigned long long kPivotEmpty = ~0ull;
constexpr int kPivotLine = 8;   // words per build: the map (4), then
enum { kPivotFirst = 4, kPivotState = 5, kPivotFinal = 6 };   // last pivot, whether it holds, and finally

struct AheadHooks {
    static constexpr bool kAhead = true;
    double* carry;                  // LDS: carry[0] = g entering the build, carry[2]: settle's answer
    unsigned long long* lines;
    int* err;
    int64_t build;
    __device__ void put(int64_t b, int word, double v) const
    {
        const unsigned long long u = v != v ? 0x7FF8000000000000ull : (unsigned long long)__double_as_longlong(v);
        __hip_atomic_store(&lines[b * kPivotLine + word], u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ double get(int64_t b, int word) const
    {
        int polls = 0;
        unsigned long long v;
        while ((v = __hip_atomic_load(&lines[b * kPivotLine + word], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ==
               kPivotEmpty) {
            if (++polls > kLongMaxPolls) {
                __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return 1.0;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        return __longlong_as_double((long long)v);
    }
    __device__ void publish_map(double a, double b, double c, double e) const
    {
        put(build, 0, a);
        put(build, 1, b);
        put(build, 2, c);
        put(build, 3, e);
    }
    // (wavefront 0; the pivot before row 0 may be any, the first row has no sub-diagonal)
    __device__ void wait_carry(int tid) const
    {
        if (build == 0 || tid >= 64) return;
        double ta = 1.0, tb = 0.0, tc = 0.0, te = 1.0;
        for (int64_t b0 = 0; b0 < build; b0 += 64) {
            double a = 1.0, b = 0.0, c = 0.0, e = 1.0;
            if (b0 + tid < build) {
                a = get(b0 + tid, 0);
                b = get(b0 + tid, 1);
                c = get(b0 + tid, 2);
                e = get(b0 + tid, 3);
            }
            moebius_scan(a, b, c, e, tid);
            a = readlane_d(a, 63);
            b = readlane_d(b, 63);
            c = readlane_d(c, 63);
            e = readlane_d(e, 63);
            moebius_compose(a, b, c, e, ta, tb, tc, te);
            moebius_normalize(a, b, c, e);
            ta = a; tb = b; tc = c; te = e;
        }
        // g = 1 / p of p = (ta + tb) / (tc + te)
        if (tid == 0) carry[0] = (tc + te) / (ta + tb);
    }
    __device__ bool settle(int tid, bool refine, const double* gl, double p, double m) const
    {
        if (tid < 64) {
            if (tid == 0) {
                put(build, kPivotFirst, *gl);
                bool bad = refine;
                if (build > 0) {
                    const double rho = (p - 1.0) + m * get(build - 1, kPivotFirst);
                    bad = bad || !(fabs(rho) <= pivot_tol<double>() * fabs(p));
                }
                put(build, kPivotState, bad ? 1.0 : 0.0);
            }
            bool bad = false;
            for (int64_t b = tid; b <= build; b += 64) bad = bad || get(b, kPivotState) != 0.0;
            const bool again = __ballot(bad) != 0;
            if (tid == 0) {
                if (again && build > 0) carry[0] = get(build - 1, kPivotFinal);
                carry[2] = again ? 1.0 : 0.0;
            }
        }
        __syncthreads();
        return carry[2] != 0.0;
    }
    __device__ void publish(int tid, const double* gl) const
    {
        if (tid == 0) put(build, kPivotFinal, *gl);
    }
};

__device__ __forceinline__ void wait_table(int* flag, int* err)
{
    int polls = 0;
    // relaxed polls (no cache invalidation per poll), one acquire once the flag is seen
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
        if (++polls > kLongMaxPolls) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        __builtin_amdgcn_s_sleep(16);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

template <bool ALL3>
__global__ __launch_bounds__(max_threads<kLong64R>()) void jw_long64_front_kernel(jw_source_desc src, const void* mat,
                                                                                 jw_long_desc d, int* sync,
                                                                                 unsigned long long* lines, int* err,
                                                                                 int nbuild, int chained, int P)
{
    constexpr int R = kLong64R;
    constexpr int C = 64 * R;
    constexpr int SR = kLong64Nsub * C;
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_id;
    int* queue = sync + 1;
    int* tflags = sync + kLong64Tflags;
    double* table = reinterpret_cast<double*>(const_cast<void*>(d.table));
    if (threadIdx.x == 0) s_id = __hip_atomic_fetch_add(&sync[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int tk = s_id;
    if (tk < nbuild) {
        const int64_t rb = (int64_t)tk * SR;
        // the pivot carry follows the build's row arrays; thread 0 reads the raw
        // super-diagonal entry of the row before the build (the build's first barrier
        // publishes it)
        double* carry = reinterpret_cast<double*>(smem + prologue_lds_bytes(SR, sizeof(double)));
        if (chained && threadIdx.x == 0)
            carry[1] = rb > 0 ? mem_load<double>(mat, src.udS + source_pos(src, rb - 1, src.N), src.mem_f64) : 0.0;
        const AheadHooks hooks{carry, lines, err, tk};
        prologue_body<double, 2, AheadHooks>(src, mat, table + (int64_t)tk * kLong64Nsub * NTAB, 64, R, smem, rb,
                                            chained ? carry : nullptr, kLong64Nsub, hooks);
        // every wavefront waits for its own table stores (written into the L2), then one
        // agent-scope release by thread 0 writes the L2 back and sets the flag (one L2
        // writeback per build: a fence in every wavefront measured 3x longer under the
        // workers' load, and slowed them)
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(&tflags[tk], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* stg = reinterpret_cast<double2*>(smem + NTAB * 8) + (size_t)wave * 64 * R;
    const jw_run_desc& rd = d.run;
    const int64_t nc = d.nchunks;
    const int64_t ppc = (rd.nsys + 1) >> 1;
    const int upc = 1 + (int)((ppc + P - 1) / P);
    const int nunits = (int)nc * upc;
    int64_t cur = -1;
    for (;;) {
        __syncthreads();   // the previous unit is finished: s_id and the table may change
        if (threadIdx.x == 0) s_id = __hip_atomic_fetch_add(queue, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const int u = __builtin_amdgcn_readfirstlane(s_id);
        if (u >= nunits) break;
        const int64_t c = u / upc;
        const int j = u - (int)c * upc;
        if (c != cur) {
            if (threadIdx.x == 0) wait_table(&tflags[c / kLong64Nsub], err);
            __syncthreads();
            copy_table_lds<NTAB>(smem, table + c * NTAB, wave, nwaves, lane);
            zero_staging<R>(stg, lane);   // this chunk's keep-range may be narrower
            __syncthreads();
            cur = c;
        }
        const int64_t rb = c * C;
        const int64_t cn = (int64_t)rd.N - rb < C ? (int64_t)rd.N - rb : C;
        auto clip = [&](int64_t v) -> int {
            const int64_t w = v - rb;
            return (int)(w < 0 ? 0 : (w > cn ? cn : w));
        };
        const int ilo = clip(rd.in_lo), olo = clip(rd.out_lo);
        const int ihi = clip(rd.in_hi) > ilo ? clip(rd.in_hi) : ilo;
        const int ohi = clip(rd.out_hi) > olo ? clip(rd.out_hi) : olo;
        if (j == 0) {
            // COEF: the 3 unit-carry systems, passes 0 and 1 on wavefronts 0 and 1
            if (wave < 2) {
                const jw_pass64 g = make_pass64(reinterpret_cast<double*>(rd.rhs), 3, rd.stride, rd.offSol + rb, ilo,
                                                ihi, olo, ohi, rd.kl, rd.ku, rd.fwd, rd.b1, rd.b2, false, 1.0, lane);
                long64_pass<JW_LONG_COEF, ALL3>(tab, stg, lane, g, d, c, 2 * (int64_t)wave);
            }
        } else {
            const int64_t q0 = (int64_t)(j - 1) * P;
            const int64_t q1 = q0 + P < ppc ? q0 + P : ppc;
            for (int64_t q = q0 + wave; q < q1; q += nwaves) {
                const jw_pass64 g = make_pass64(reinterpret_cast<double*>(rd.rhs), rd.nsys, rd.stride, rd.offSol + rb,
                                                ilo, ihi, olo, ohi, rd.kl, rd.ku, rd.fwd, rd.b1, rd.b2, false, 1.0,
                                                lane);
                long64_pass<JW_LONG_REDUCE, ALL3>(tab, stg, lane, g, d, c, 2 * q);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// 1024 < N <= 2048: a group of four wavefronts owns a pair of systems, 512 rows (R = 8 per
// lane) each; a workgroup is two groups.  The 8 coefficients of a lane's 8 rows do not
// change from pair to pair and stay in its registers (128 VGPRs), so no pass reads a table:
// LDS holds the scan multipliers (48 KiB) and a staging of 4 KiB per wavefront.  (The whole
// table, 128 KiB, leaves no LDS for stagings; streamed through the L2 by one wavefront per
// system it set the pace: 8192 systems of 2000 rows 142 us, 56 us
// this way.)
// What crosses wavefronts goes through LDS: the two rows on each side for the matvec, and
// per recurrence each wavefront's end value for a zero carry; a wavefront's carry follows
// from those of the wavefronts before it (matrix-only factors), and enters a lane's rows
// by one more multiplier, the product over the lanes before it.  A barrier per exchange, four
// per pass with all three recurrences, two with one or none; the
// arithmetic takes a third of the time the pass's memory traffic does.
// Tables in memory (batches, the plain per-set form) are the format-2 tables of 32 rows per
// lane, whose coefficients are read once per matrix set.
// ---------------------------------------------------------------------------
constexpr int kWideW = 4;                       // wavefronts per group
constexpr int kWideR = 8;                       // rows per lane
constexpr int kWideRows = 64 * kWideR;          // rows per wavefront
constexpr int kWideThreads = 512;
constexpr int kWideGroups = kWideThreads / 64 / kWideW;
// LDS while solving: stagings, multipliers of the 4 wavefront places (3 recurrences x 8 x
// 64), exchange; while building: the build's scratch and two 512-row coefficient slots
constexpr int kWideMult = kWideGroups * kWideW * kWideRows * 8;
constexpr int kWideExch = kWideMult + kWideW * 24 * 64 * 8;
constexpr int kWideExchDoubles = kWideGroups * kWideW * (2 * 4 + 3 * 2) + 3 * kWideW;
constexpr int kWideSlots = (int)((prologue_lds_bytes(kWideW * kWideRows, 8) + 1023) / 1024 * 1024);
constexpr int kWideLds = kWideSlots + 2 * kWideRows * 64 > kWideExch + kWideExchDoubles * 8
                             ? kWideSlots + 2 * kWideRows * 64 : kWideExch + kWideExchDoubles * 8;

// the coefficients of a lane's rows: (v_-2, v_-1), (v_0, v_1), (v_2, l'), (h', E)
struct wide_coef {
    double2 p[4][kWideR];
};

// from a format-2 table of 32 rows per lane in global memory: row w 512 + 8 lane + k of the
// system is row-in-lane 8 (lane mod 4) + k of table lane 16 w + lane / 4
__device__ __forceinline__ void wide_load_table(wide_coef& c, const void* table, int w, int lane)
{
    const double* tab = reinterpret_cast<const double*>(table);
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int k = 0; k < kWideR; k++) {
            const int e = tab_coef64(p, 8 * (lane & 3) + k, 16 * w + (lane >> 2), 32);
            c.p[p][k] = load_chunk(tab + e);
        }
}

// a build's rows (FORMAT 3 of prologue_body on 8 wavefronts: the j-th row of every thread
// belongs to wavefront place j) through two LDS slots into the registers of their owners
struct wide_sink {
    double* slots;
    wide_coef& c;
    int w, lane;
    __device__ __forceinline__ void operator()(int j, int i, int t, const double (&cf)[8]) const
    {
        double* s = slots + (j & 1) * (kWideRows * 8);
#pragma unroll
        for (int p = 0; p < 4; p++)
            *reinterpret_cast<double2*>(s + tab_coef64(p, i, t, kWideR)) = make_double2(cf[2 * p], cf[2 * p + 1]);
    }
    __device__ __forceinline__ void done(int j) const
    {
        // a slot is written again two rows on, behind the next barrier
        __syncthreads();
        if (w != j) return;
        const double* s = slots + (j & 1) * (kWideRows * 8);
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int k = 0; k < kWideR; k++)
                c.p[p][k] = *reinterpret_cast<const double2*>(s + tab_coef64(p, k, lane, kWideR));
    }
};

// scan multipliers of wavefront place w from its coefficients, by group 0: as the format-2
// build's (jw_prologue.h) over the wavefront's 64 lanes, with the carry's multiplier (the
// product over the lanes before, or behind) in place 7 and the whole wavefront's product in tot
__device__ __forceinline__ void wide_multipliers(const wide_coef& c, double* mult, double* tot, int w, int t)
{
    const int tr = t & 15, rw = t >> 4;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        double v = 1.0;
#pragma unroll
        for (int k = 0; k < kWideR; k++)
            v *= -(j == 0 ? c.p[2][k].y : (j == 1 ? c.p[3][k].x : c.p[3][k].y));
        double* m = mult + (w * 24 + j * 8) * 64 + t;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int s = 1 << k;
            m[64 * k] = v;
            const bool from = j == 0 ? tr >= s : tr + s <= 15;
            double u;
            switch (k) {
            case 0: u = j == 0 ? dpp_d<DPP_ROW_SHR(1)>(v) : dpp_d<DPP_ROW_SHL(1)>(v); break;
            case 1: u = j == 0 ? dpp_d<DPP_ROW_SHR(2)>(v) : dpp_d<DPP_ROW_SHL(2)>(v); break;
            case 2: u = j == 0 ? dpp_d<DPP_ROW_SHR(4)>(v) : dpp_d<DPP_ROW_SHL(4)>(v); break;
            default: u = j == 0 ? dpp_d<DPP_ROW_SHR(8)>(v) : dpp_d<DPP_ROW_SHL(8)>(v); break;
            }
            if (from) v *= u;
        }
        if (j == 0) {
            const double T0 = readlane_d(v, 15), T1 = readlane_d(v, 31), T2 = readlane_d(v, 47), T3 = readlane_d(v, 63);
            m[64 * 4] = v;
            m[64 * 5] = rw == 2 ? v : (rw == 3 ? T2 * v : 0.0);
            const double before = dpp_d<DPP_ROW_SHR(1)>(v);   // in every lane; a row's first takes 1
            const double rows = rw == 0 ? 1.0 : (rw == 1 ? T0 : (rw == 2 ? T0 * T1 : T0 * T1 * T2));
            m[64 * 7] = (tr == 0 ? 1.0 : before) * rows;
            if (t == 0) tot[w] = T0 * T1 * T2 * T3;
        } else {
            const double T0 = readlane_d(v, 0), T1 = readlane_d(v, 16), T2 = readlane_d(v, 32), T3 = readlane_d(v, 48);
            m[64 * 4] = rw == 0 ? v : 0.0;
            m[64 * 5] = rw == 0 ? v * T1 : (rw == 1 ? v : 0.0);
            m[64 * 6] = rw == 0 ? v * T1 * T2 : (rw == 1 ? v * T2 : (rw == 2 ? v : 0.0));
            const double behind = dpp_d<DPP_ROW_SHL(1)>(v);
            const double rows = rw == 3 ? 1.0 : (rw == 2 ? T3 : (rw == 1 ? T2 * T3 : T1 * T2 * T3));
            m[64 * 7] = (tr == 15 ? 1.0 : behind) * rows;
            if (t == 0) tot[j * kWideW + w] = T0 * T1 * T2 * T3;
        }
    }
}

// the step on a pair, in registers; every wavefront of the workgroup calls it (barriers)
template <bool ALL3, bool EXACT>
__device__ __forceinline__ void wide_compute(const wide_coef& c, const double* mult, double* exch, int grp, int w,
                                             int lane, const jw_pass64& g, double (&x0)[kWideR], double (&x1)[kWideR])
{
    constexpr int R = kWideR;
    double* rows = exch + (grp * kWideW + w) * 8;   // first two and last two rows of both systems
    double* ends = exch + kWideGroups * kWideW * 8;                     // per recurrence, group, place, system
    const double* tot = ends + 3 * kWideGroups * kWideW * 2;
    if (lane == 0) {
        rows[0] = x0[0]; rows[1] = x0[1];
        rows[4] = x1[0]; rows[5] = x1[1];
    }
    if (lane == 63) {
        rows[2] = x0[R - 2]; rows[3] = x0[R - 1];
        rows[6] = x1[R - 2]; rows[7] = x1[R - 1];
    }
    __syncthreads();
    {
        double m1a = 0.0, m2a = 0.0, p1a = 0.0, p2a = 0.0;
        double m1b = 0.0, m2b = 0.0, p1b = 0.0, p2b = 0.0;
        const bool lo = lane == 0 && w > 0, hi = lane == 63 && w + 1 < kWideW;
        if (g.kl >= 1) {
            m1a = dpp_d<DPP_WAVE_SHR1>(x0[R - 1]);
            m1b = dpp_d<DPP_WAVE_SHR1>(x1[R - 1]);
            if (lo) { m1a = rows[-8 + 3]; m1b = rows[-8 + 7]; }
        }
        if (g.kl >= 2) {
            m2a = dpp_d<DPP_WAVE_SHR1>(x0[R - 2]);
            m2b = dpp_d<DPP_WAVE_SHR1>(x1[R - 2]);
            if (lo) { m2a = rows[-8 + 2]; m2b = rows[-8 + 6]; }
        }
        if (g.ku >= 1) {
            p1a = dpp_d<DPP_WAVE_SHL1>(x0[0]);
            p1b = dpp_d<DPP_WAVE_SHL1>(x1[0]);
            if (hi) { p1a = rows[8]; p1b = rows[8 + 4]; }
        }
        if (g.ku >= 2) {
            p2a = dpp_d<DPP_WAVE_SHL1>(x0[1]);
            p2b = dpp_d<DPP_WAVE_SHL1>(x1[1]);
            if (hi) { p2a = rows[8 + 1]; p2b = rows[8 + 5]; }
        }
        auto coef = [&](int p, int i) -> double2 { return c.p[p][i]; };
        band_rows<R, EXACT, false>(coef, g, band_side{m1a, m2a, m1b, m2b}, band_side{p1a, p2a, p1b, p2b}, x0, x1);
    }
    // forward recurrence
    if (ALL3 || g.fwd) {
        const double* m = mult + (w * 24) * 64 + lane;
        double* e = ends + (grp * kWideW) * 2;
        double a = x0[0], b = x1[0];
#pragma unroll
        for (int i = 1; i < R; i++) {
            a = __builtin_fma(-c.p[2][i].y, a, x0[i]);
            b = __builtin_fma(-c.p[2][i].y, b, x1[i]);
        }
        a = __builtin_fma(m[0], dpp_d<DPP_ROW_SHR(1)>(a), a);
        b = __builtin_fma(m[0], dpp_d<DPP_ROW_SHR(1)>(b), b);
        a = __builtin_fma(m[64], dpp_d<DPP_ROW_SHR(2)>(a), a);
        b = __builtin_fma(m[64], dpp_d<DPP_ROW_SHR(2)>(b), b);
        a = __builtin_fma(m[128], dpp_d<DPP_ROW_SHR(4)>(a), a);
        b = __builtin_fma(m[128], dpp_d<DPP_ROW_SHR(4)>(b), b);
        a = __builtin_fma(m[192], dpp_d<DPP_ROW_SHR(8)>(a), a);
        b = __builtin_fma(m[192], dpp_d<DPP_ROW_SHR(8)>(b), b);
        a = __builtin_fma(m[256], dpp_rm<DPP_ROW_BCAST15, 0xa>(a), a);
        b = __builtin_fma(m[256], dpp_rm<DPP_ROW_BCAST15, 0xa>(b), b);
        a = __builtin_fma(m[320], dpp_rm<DPP_ROW_BCAST31, 0xc>(a), a);
        b = __builtin_fma(m[320], dpp_rm<DPP_ROW_BCAST31, 0xc>(b), b);
        if (lane == 63) *reinterpret_cast<double2*>(e + 2 * w) = make_double2(a, b);
        double wa = dpp_d<DPP_WAVE_SHR1>(a), wb = dpp_d<DPP_WAVE_SHR1>(b);
        const double pt = m[448];
        __syncthreads();
        // W' entering the wavefront
        double ca = 0.0, cb = 0.0;
        for (int k = 0; k < w; k++) {
            const double2 s = *reinterpret_cast<const double2*>(e + 2 * k);
            ca = __builtin_fma(tot[k], ca, s.x);
            cb = __builtin_fma(tot[k], cb, s.y);
        }
        wa = __builtin_fma(pt, ca, wa);
        wb = __builtin_fma(pt, cb, wb);
#pragma unroll
        for (int i = 0; i < R; i++) {
            wa = __builtin_fma(-c.p[2][i].y, wa, x0[i]);
            wb = __builtin_fma(-c.p[2][i].y, wb, x1[i]);
            x0[i] = wa;
            x1[i] = wb;
        }
    }
    // backward recurrences
#pragma unroll
    for (int stage = 0; stage < 2; stage++) {
        if (!ALL3 && stage == 0 && !g.b1) continue;
        if (!ALL3 && stage == 1 && !g.b2) continue;
        const double* m = mult + (w * 24 + 8 * (1 + stage)) * 64 + lane;
        double* e = ends + ((1 + stage) * kWideGroups + grp) * kWideW * 2;
        auto h = [&](int i) -> double { return stage == 0 ? c.p[3][i].x : c.p[3][i].y; };
        double a = x0[R - 1], b = x1[R - 1];
#pragma unroll
        for (int i = R - 2; i >= 0; i--) {
            a = __builtin_fma(-h(i), a, x0[i]);
            b = __builtin_fma(-h(i), b, x1[i]);
        }
        a = __builtin_fma(m[0], dpp_d<DPP_ROW_SHL(1)>(a), a);
        b = __builtin_fma(m[0], dpp_d<DPP_ROW_SHL(1)>(b), b);
        a = __builtin_fma(m[64], dpp_d<DPP_ROW_SHL(2)>(a), a);
        b = __builtin_fma(m[64], dpp_d<DPP_ROW_SHL(2)>(b), b);
        a = __builtin_fma(m[128], dpp_d<DPP_ROW_SHL(4)>(a), a);
        b = __builtin_fma(m[128], dpp_d<DPP_ROW_SHL(4)>(b), b);
        a = __builtin_fma(m[192], dpp_d<DPP_ROW_SHL(8)>(a), a);
        b = __builtin_fma(m[192], dpp_d<DPP_ROW_SHL(8)>(b), b);
        {
            const double a1 = readlane_d(a, 16), a2 = readlane_d(a, 32), a3 = readlane_d(a, 48);
            const double b1 = readlane_d(b, 16), b2 = readlane_d(b, 32), b3 = readlane_d(b, 48);
            a = add_from<EXACT>(m[256], a1, lane < 16, a);
            b = add_from<EXACT>(m[256], b1, lane < 16, b);
            a = add_from<EXACT>(m[320], a2, lane < 32, a);
            b = add_from<EXACT>(m[320], b2, lane < 32, b);
            a = add_from<EXACT>(m[384], a3, lane < 48, a);
            b = add_from<EXACT>(m[384], b3, lane < 48, b);
        }
        if (lane == 0) *reinterpret_cast<double2*>(e + 2 * w) = make_double2(a, b);
        double za = dpp_d<DPP_WAVE_SHL1>(a), zb = dpp_d<DPP_WAVE_SHL1>(b);
        const double pt = m[448];
        __syncthreads();
        // Z' (or y) entering the wavefront from the one behind it
        double ca = 0.0, cb = 0.0;
        for (int k = kWideW - 1; k > w; k--) {
            const double2 s = *reinterpret_cast<const double2*>(e + 2 * k);
            ca = __builtin_fma(tot[(1 + stage) * kWideW + k], ca, s.x);
            cb = __builtin_fma(tot[(1 + stage) * kWideW + k], cb, s.y);
        }
        za = __builtin_fma(pt, ca, za);
        zb = __builtin_fma(pt, cb, zb);
#pragma unroll
        for (int i = R - 1; i >= 0; i--) {
            za = __builtin_fma(-h(i), za, x0[i]);
            zb = __builtin_fma(-h(i), zb, x1[i]);
            x0[i] = za;
            x1[i] = zb;
        }
    }
    if (g.apply_scale) {
        x0[0] *= g.row0_scale;
        x1[0] *= g.row0_scale;
    }
    // A recurrence's barrier comes after every wavefront has read its neighbours' rows; a
    // product alone has none, and the next pass must not write rows still to be read
    if (!ALL3 && !g.fwd && !g.b1 && !g.b2) __syncthreads();
}

// pass geometry of wavefront place w: its 512 rows of the system as a system of their own
__device__ __forceinline__ jw_pass64 wide_pass(double* rhs, int64_t nsys, int64_t stride, int64_t offSol, int64_t N,
                                               int64_t in_lo, int64_t in_hi, int64_t out_lo, int64_t out_hi, int kl,
                                               int ku, bool fwd, bool b1, bool b2, bool apply_scale, double scale,
                                               int w, int lane)
{
    const int64_t rb = (int64_t)w * kWideRows;
    int64_t n = N - rb;
    n = n < 0 ? 0 : (n > kWideRows ? kWideRows : n);
    auto clip = [&](int64_t v) -> int {
        const int64_t u = v - rb;
        return (int)(u < 0 ? 0 : (u > n ? n : u));
    };
    const int il = clip(in_lo), ih = clip(in_hi), ol = clip(out_lo), oh = clip(out_hi);
    return make_pass64(rhs, nsys, stride, offSol + rb, il, ih > il ? ih : il, ol, oh > ol ? oh : ol, kl, ku, fwd, b1, b2,
                       apply_scale && w == 0, scale, lane);
}

// pairs p0 + 2 s + group for s = 0, step, ... (systems first + 2 pair, below the geometry's
// nsys), one per group and pass, for a workgroup whose wavefronts hold their coefficients;
// pf: the first pass's rows
template <bool ALL3, bool BUF, bool EXACT = false, class Geo>
__device__ __forceinline__ void wide_stream(const wide_coef& c, unsigned char* smem, int grp, int w, int lane,
                                            const Geo& geo, int64_t first, int64_t p, int64_t p1, int64_t step,
                                            double2 (&pf)[2][kWideR / 2])
{
    constexpr int R = kWideR;
    const double* mult = reinterpret_cast<const double*>(smem + kWideMult);
    double* exch = reinterpret_cast<double*>(smem + kWideExch);
    double2* stg = reinterpret_cast<double2*>(smem) + (size_t)(grp * kWideW + w) * 32 * R;
    if constexpr (BUF) hold_pair<R>(pf);
    // every wavefront makes every pass (barriers)
    for (; p < p1; p += step) {
        jw_pass64 g = geo();
        const int64_t q = p + grp, sys0 = first + 2 * q;
        const bool on = q < p1;
        // a group past the last pair goes through the pass on what its registers hold and
        // reads and stores nothing
        g.in_edge_lo = g.in_edge_lo && on;
        g.in_edge_hi = g.in_edge_hi && on;
        double x0[R], x1[R];
        unpack_ahead<R, BUF>(pf, stg, lane, g, sys0, x0, x1);
        const int64_t qn = q + step;
        if (qn < p1) load_pair_ahead<R, BUF>(pf, lane, g, first + 2 * qn);
        wide_compute<ALL3, EXACT>(c, mult, exch, grp, w, lane, g, x0, x1);
        store_pair<R, BUF>(stg, lane, g, sys0, x0, x1, on);
    }
}

template <bool ALL3, bool BUILD, bool EXACT = false>
__global__ __launch_bounds__(kWideThreads) void jw_wide64_kernel(jw_run_desc d, jw_source_desc src, const void* mat)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave / kWideW, w = wave % kWideW;
    const int64_t npass = (d.nsys + 1) >> 1, step = (int64_t)gridDim.x * kWideGroups;
    const int64_t p = (int64_t)blockIdx.x * kWideGroups;
    auto geo = [&] {
        return wide_pass(reinterpret_cast<double*>(d.rhs), d.nsys, d.stride, d.offSol, d.N, d.in_lo, d.in_hi, d.out_lo,
                         d.out_hi, d.kl, d.ku, d.fwd, d.b1, d.b2, d.apply_scale, d.scale_hi, w, lane);
    };
    double2 pf[2][kWideR / 2] = {};
    auto first = [&] { if (p + grp < npass) load_pair_ahead<kWideR, false>(pf, lane, geo(), 2 * (p + grp)); };
    wide_coef c;
    if constexpr (BUILD) {
        const wide_sink sink{reinterpret_cast<double*>(smem + kWideSlots), c, w, lane};
        prologue_body<double, 3, NoPivotHooks, kWideW, kMaxRT>(src, mat, static_cast<double*>(nullptr), 64, kWideR, smem,
                                                               0, nullptr, kWideW, NoPivotHooks(), first, sink);
    } else {
        wide_load_table(c, d.table, w, lane);
        first();
    }
    __syncthreads();   // the build's LDS is free
    if (grp == 0)
        wide_multipliers(c, reinterpret_cast<double*>(smem + kWideMult),
                         reinterpret_cast<double*>(smem + kWideExch) + kWideGroups * kWideW * (8 + 3 * 2), w, lane);
    __syncthreads();
    wide_stream<ALL3, false, EXACT>(c, smem, grp, w, lane, geo, 0, p, npass, step, pf);
}

// ---------------------------------------------------------------------------
// Chained steps (numConsecutiveJWIterations = K): a wavefront owns a pair of systems
// through all K iterations, whose right-hand sides stay in its registers in between (one
// read and one write of HBM per K-step instead of K).  The input keep-range applies to the
// first iteration's rows, the output keep-range to the last one's.
//
// An iteration is a bidiagonal matvec and a unit-bidiagonal solve: per row the diagonal,
// one off-diagonal and the solve's off-diagonal, and the 7 scan multipliers of its one
// recurrence.  As a table of its own (JW_CHAIN_TAB, 15.5 KiB at R = 8 against the 44 KiB of
// format 2) the K tables fit in LDS, where every workgroup builds them from the matrices
// (no pivots: the build is the loads and one product scan), so the step is one launch and
// the loop touches HBM for right-hand sides only.  Bound: HBM.  65536 systems, N = 512 ->
// 509, K = 4: 114 us per step; 240 us when a launch of its own wrote format-2 tables
// and every pass read 24 KiB of them per iteration through the L2.
// A chain whose tables leave no room for 4 wavefronts' stagings (N = 512: K >= 10; N = 1024:
// K >= 5) keeps the first ones in LDS and reads the others, written by
// jw_chain_tables_kernel, through the L2.
// ---------------------------------------------------------------------------
// doubles of one iteration's table: (v0, voff) of row-in-lane i, lane t at (64 i + t) 2, the
// solve's off-diagonal at 128 R + 64 i + t, multiplier k at 192 R + 64 k + t
__host__ __device__ constexpr int chain_tab_elems(int R) { return (3 * R + 7) * 64; }

// row r of an iteration's table
template <int R, bool UP>
__device__ __forceinline__ void chain_row(const jw_source_desc& d, const double* mat, double* tab, int r)
{
    const int64_t N = d.N, ncols = d.Ncols > 0 ? d.Ncols : N;
    const bool band = d.band_kind != JW_BAND_NONE, solve = d.solve_kind != JW_SOLVE_NONE;
    const int64_t offA = UP ? d.udA : d.ldA, offS = UP ? d.ldS : d.udS;
    const bool in = r < N;
    const int64_t P = source_pos(d, in ? r : 0, N);
    // entries of the matvec and the solve inside the matrix; the others are read at an
    // in-bounds position and dropped by the selects
    const double v0 = !band || d.unit_diag ? 1.0 : mat[d.mdA + P];
    const double vo = band ? mat[offA + P] : 0.0;
    const double so = solve ? mat[offS + P] : 0.0;
    const bool vin = UP ? r + 1 < ncols : r >= 1 && r - 1 < ncols;
    const bool sin = UP ? r >= 1 : r + 1 < N;
    const int i = r % R, t = r / R;
    *reinterpret_cast<double2*>(tab + (64 * i + t) * 2) = make_double2(in ? v0 : 0.0, in && vin ? vo : 0.0);
    tab[128 * R + 64 * i + t] = in && sin ? so : 0.0;
}

// rows of the tables of iterations k0 .. k1 - 1 (that of k0 at tab): wavefronts take 64 rows at a
// time over all tables, so that short systems keep them busy (N = 100, K = 16, 4000 systems: 14.9
// us, 24.9 us with one table after another)
template <int R, bool UP>
__device__ __forceinline__ void chain_rows(const jw_chain_jobs& jobs, int k0, int k1, double* tab, int wave,
                                           int nwaves, int lane)
{
    for (int b = wave; b < (k1 - k0) * R; b += nwaves) {
        const int k = b / R;
        chain_row<R, UP>(jobs.src[k0 + k], reinterpret_cast<const double*>(jobs.matrices[k0 + k]),
                         tab + (int64_t)k * chain_tab_elems(R), (b - k * R) * 64 + lane);
    }
}

// the scan multipliers of one table by one wavefront, once its rows are written: as the
// format-2 build's (jw_prologue.h), for the forward (UP: the upper matvec's lower solve) or
// the backward recurrence
template <int R, bool UP>
__device__ __forceinline__ void chain_multipliers(double* tab, int t)
{
    double v = 1.0;
#pragma unroll
    for (int i = 0; i < R; i++) v *= -tab[128 * R + 64 * i + t];
    double* m = tab + 192 * R;
    const int tr = t & 15, rw = t >> 4;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int s = 1 << k;
        m[64 * k + t] = v;
        const bool from = UP ? tr >= s : tr + s <= 15;
        const double w = lane_fetch(v, from ? (UP ? t - s : t + s) : t);
        if (from) v *= w;
    }
    if (UP) {
        const double pre47 = lane_fetch(v, 47);
        m[64 * 4 + t] = v;
        m[64 * 5 + t] = rw == 2 ? v : (rw == 3 ? pre47 * v : 0.0);
        m[64 * 6 + t] = 0.0;
    } else {
        const double P1 = lane_fetch(v, 16), P2 = lane_fetch(v, 32);
        m[64 * 4 + t] = rw == 0 ? v : 0.0;
        m[64 * 5 + t] = rw == 0 ? v * P1 : (rw == 1 ? v : 0.0);
        m[64 * 6 + t] = rw == 0 ? v * P1 * P2 : (rw == 1 ? v * P2 : (rw == 2 ? v : 0.0));
    }
}

// A lane's part of an iteration's table: read where it is used from LDS, or from global memory
// into registers as a whole (left to the compiler, in the kernel for tables in LDS, the loads came
// one after another, 14 round trips through the L2 per iteration: N = 512, K = 16, 2000 systems
// 46 us, 30 us this way)
template <int R>
struct chain_lds {
    const double* tab;
    int lane;
    __device__ __forceinline__ double2 v(int i) const { return *reinterpret_cast<const double2*>(tab + (64 * i + lane) * 2); }
    __device__ __forceinline__ double s(int i) const { return tab[128 * R + 64 * i + lane]; }
    __device__ __forceinline__ double m(int k) const { return tab[192 * R + 64 * k + lane]; }
    __device__ __forceinline__ void before_band() {}
    __device__ __forceinline__ void before_solve() {}
};
template <int R>
struct chain_regs {
    const double* tab;
    int lane;
    double2 vv[R];
    double ss[R], mm[7];
    __device__ __forceinline__ double2 v(int i) const { return vv[i]; }
    __device__ __forceinline__ double s(int i) const { return ss[i]; }
    __device__ __forceinline__ double m(int k) const { return mm[k]; }
    __device__ __forceinline__ void load_band()
    {
#pragma unroll
        for (int i = 0; i < R; i++) vv[i] = load_chunk(tab + (64 * i + lane) * 2);
    }
    __device__ __forceinline__ void load_solve()
    {
        const JW_GLOBAL double* t = as_global(tab) + 128 * R + lane;
#pragma unroll
        for (int i = 0; i < R; i++) ss[i] = t[64 * i];
#pragma unroll
        for (int k = 0; k < 7; k++) mm[k] = t[64 * (R + k)];
    }
    // waits for the loads: none is put off to its use
    __device__ __forceinline__ void hold_band()
    {
#pragma unroll
        for (int i = 0; i < R; i++) asm volatile("" : "+v"(vv[i].x), "+v"(vv[i].y));
    }
    __device__ __forceinline__ void hold_solve()
    {
#pragma unroll
        for (int i = 0; i < R; i++) asm volatile("" : "+v"(ss[i]));
#pragma unroll
        for (int k = 0; k < 7; k++) asm volatile("" : "+v"(mm[k]));
    }
    // R = 16: in two parts, for the registers
    __device__ __forceinline__ void before_band()
    {
        load_band();
        if (R < 16) load_solve();
        hold_band();
        if (R < 16) hold_solve();
    }
    __device__ __forceinline__ void before_solve()
    {
        if (R < 16) return;
        load_solve();
        hold_solve();
    }
};

// one iteration on a pair in registers (the steps of compute_pair for these operators)
template <int R, bool UP, class Tab>
__device__ __forceinline__ void chain_pair(Tab tab, bool band, bool solve, bool apply_scale, double row0_scale,
                                           double (&x0)[R], double (&x1)[R])
{
    tab.before_band();
    if (band) {
        double na = UP ? dpp_d<DPP_WAVE_SHL1>(x0[0]) : dpp_d<DPP_WAVE_SHR1>(x0[R - 1]);
        double nb = UP ? dpp_d<DPP_WAVE_SHL1>(x1[0]) : dpp_d<DPP_WAVE_SHR1>(x1[R - 1]);
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int i = UP ? R - 1 - k : k;   // from the end whose neighbour came from the next lane
            const double2 v = tab.v(i);
            const double xa = x0[i], xb = x1[i];
            x0[i] = __builtin_fma(v.y, na, v.x * xa);
            x1[i] = __builtin_fma(v.y, nb, v.x * xb);
            na = xa;
            nb = xb;
        }
    }
    if (!solve) return;
    tab.before_solve();
    double s[R];
#pragma unroll
    for (int i = 0; i < R; i++) s[i] = tab.s(i);
    // row order of the recurrence: forward (UP) or backward
    double a = x0[UP ? 0 : R - 1], b = x1[UP ? 0 : R - 1];
#pragma unroll
    for (int k = 1; k < R; k++) {
        const int i = UP ? k : R - 1 - k;
        a = __builtin_fma(-s[i], a, x0[i]);
        b = __builtin_fma(-s[i], b, x1[i]);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const double f = tab.m(k);
        double sa, sb;
        switch (k) {
        case 0: sa = dpp_d<UP ? DPP_ROW_SHR(1) : DPP_ROW_SHL(1)>(a); sb = dpp_d<UP ? DPP_ROW_SHR(1) : DPP_ROW_SHL(1)>(b); break;
        case 1: sa = dpp_d<UP ? DPP_ROW_SHR(2) : DPP_ROW_SHL(2)>(a); sb = dpp_d<UP ? DPP_ROW_SHR(2) : DPP_ROW_SHL(2)>(b); break;
        case 2: sa = dpp_d<UP ? DPP_ROW_SHR(4) : DPP_ROW_SHL(4)>(a); sb = dpp_d<UP ? DPP_ROW_SHR(4) : DPP_ROW_SHL(4)>(b); break;
        default: sa = dpp_d<UP ? DPP_ROW_SHR(8) : DPP_ROW_SHL(8)>(a); sb = dpp_d<UP ? DPP_ROW_SHR(8) : DPP_ROW_SHL(8)>(b); break;
        }
        a = __builtin_fma(f, sa, a);
        b = __builtin_fma(f, sb, b);
    }
    if (UP) {
        const double f4 = tab.m(4), f5 = tab.m(5);
        const double sa = dpp_rm<DPP_ROW_BCAST15, 0xa>(a), sb = dpp_rm<DPP_ROW_BCAST15, 0xa>(b);
        a = __builtin_fma(f4, sa, a);
        b = __builtin_fma(f4, sb, b);
        const double ta = dpp_rm<DPP_ROW_BCAST31, 0xc>(a), tb = dpp_rm<DPP_ROW_BCAST31, 0xc>(b);
        a = __builtin_fma(f5, ta, a);
        b = __builtin_fma(f5, tb, b);
    } else {
        const double a1 = readlane_d(a, 16), a2 = readlane_d(a, 32), a3 = readlane_d(a, 48);
        const double b1 = readlane_d(b, 16), b2 = readlane_d(b, 32), b3 = readlane_d(b, 48);
        const double c1 = tab.m(4), c2 = tab.m(5), c3 = tab.m(6);
        a = __builtin_fma(c1, a1, a);
        b = __builtin_fma(c1, b1, b);
        a = __builtin_fma(c2, a2, a);
        b = __builtin_fma(c2, b2, b);
        a = __builtin_fma(c3, a3, a);
        b = __builtin_fma(c3, b3, b);
    }
    double wa = UP ? dpp_d<DPP_WAVE_SHR1>(a) : dpp_d<DPP_WAVE_SHL1>(a);
    double wb = UP ? dpp_d<DPP_WAVE_SHR1>(b) : dpp_d<DPP_WAVE_SHL1>(b);
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int i = UP ? k : R - 1 - k;
        wa = __builtin_fma(-s[i], wa, x0[i]);
        wb = __builtin_fma(-s[i], wb, x1[i]);
        x0[i] = wa;
        x1[i] = wb;
    }
    if (apply_scale) {
        x0[0] *= row0_scale;
        x1[0] *= row0_scale;
    }
}

__host__ __device__ constexpr int chain_max_waves(int R) { return R <= 8 ? 16 : 8; }

// LDS: the first kl tables, then one system's staging per wavefront.  GLOB: the tables of
// iterations kl .. K-1 are in global memory (at most 8 wavefronts, for the registers)
template <int R, bool UP, bool GLOB>
__global__ __launch_bounds__(64 * (GLOB ? 8 : chain_max_waves(R))) void jw_chain64_kernel(jw_run_desc d,
                                                                                        jw_chain_jobs jobs, int kl)
{
    constexpr int TE = chain_tab_elems(R);
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    const int K = jobs.K;
    const double* gtab = reinterpret_cast<const double*>(jobs.table);
    double* ltab = reinterpret_cast<double*>(smem);
    double2* stg = reinterpret_cast<double2*>(smem + (size_t)kl * TE * 8) + (size_t)wave * 32 * R;
    const int64_t npass = (d.nsys + 1) >> 1, step = (int64_t)gridDim.x * nwaves;
    int64_t q = (int64_t)blockIdx.x * nwaves + wave;
    const jw_pass64 g = make_pass64(reinterpret_cast<double*>(d.rhs), d.nsys, d.stride, d.offSol, (int)d.in_lo,
                                    (int)d.in_hi, (int)d.out_lo, (int)d.out_hi, 0, 0, false, false, false,
                                    d.apply_scale, d.scale_hi, lane);
    const bool solve = d.fwd || d.b1;
    // the first pair's loads overlap the table build
    double2 pf[2][R / 2];
    // (a lane's own rows, but contiguous chunks at R = 16: load_pair_ahead)
    auto load = [&](int64_t p) {
        if constexpr (pair_ahead(R)) load_pair_ahead<R>(pf, lane, g, 2 * p);
        else load_pair_direct<R>(pf, lane, g, 2 * p);
    };
    if (q < npass) load(q);
    chain_rows<R, UP>(jobs, 0, kl, ltab, wave, nwaves, lane);
    __syncthreads();
    if (solve)
        for (int k = wave; k < kl; k += nwaves) chain_multipliers<R, UP>(ltab + k * TE, lane);
    __syncthreads();
    if constexpr (pair_ahead(R)) hold_pair<R>(pf);
    while (q < npass) {
        double x0[R], x1[R];
        if constexpr (pair_ahead(R)) unpack_ahead<R>(pf, stg, lane, g, 2 * q, x0, x1);
        else unpack_pair<R>(pf, lane, g, 2 * q, x0, x1);
        const int64_t qn = q + step;
        if (qn < npass) load(qn);
        for (int k = 0; k < kl; k++)
            chain_pair<R, UP>(chain_lds<R>{ltab + k * TE, lane}, d.band, solve, g.apply_scale, g.row0_scale, x0, x1);
        if constexpr (GLOB) {
            for (int k = kl; k < K; k++) {
                chain_regs<R> t;
                t.tab = gtab + (int64_t)k * TE;
                t.lane = lane;
                chain_pair<R, UP>(t, d.band, solve, g.apply_scale, g.row0_scale, x0, x1);
            }
        }
        store_pair<R, pair_ahead(R)>(stg, lane, g, 2 * q, x0, x1, true);
        q = qn;
    }
}

// the tables of the iterations from kl on, one workgroup of a thread per row each
template <int R, bool UP>
__global__ __launch_bounds__(64 * R) void jw_chain_tables_kernel(jw_chain_jobs jobs, int kl)
{
    const int k = kl + blockIdx.x;
    double* tab = reinterpret_cast<double*>(jobs.table) + (int64_t)k * chain_tab_elems(R);
    chain_rows<R, UP>(jobs, k, k + 1, tab, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), blockDim.x >> 6,
                      threadIdx.x & 63);
    __syncthreads();   // the rows are visible to the workgroup
    if (jobs.src[k].solve_kind != JW_SOLVE_NONE && threadIdx.x < 64) chain_multipliers<R, UP>(tab, threadIdx.x);
}

// Fused block operators (compute / store split kernel, IOMODE 1 and 2): the pair
// of a pass is the re/im of complex system q of an interleaved (re, im) array.
// Input (block layout 4): rows of the input keep-range, each scaled by the input
// operator, other rows zero; output (IOMODE 1, block layout 7): rows of the
// output keep-range, each scaled by the output operator, then added to the
// complex output when accumulating; IOMODE 2 writes the two real systems (the
// layout-4 packed form) like the plain step.  The arithmetic per element is the
// block kernel's (jw_block_kernel), so the fused step equals the chain of plans.
template <int R>
__device__ __forceinline__ void load_pair_packed(double2 (&pf)[2][R / 2], int lane, const jw_run_desc& d, int64_t q)
{
    constexpr int H = R / 2;
    const double2* src = reinterpret_cast<const double2*>(d.in_c) + (q * d.in_stride_c + d.in_off_c);
    const bool zero_in = d.in_op == 1 && d.in_scale == 0.0;   // baked ScaleC of 0: zeros, input not read
#pragma unroll
    for (int m = 0; m < H; m++) {
        const int r0 = lane * R + 2 * m, r1 = r0 + 1;   // the lane's own rows, as in load_pair_direct
        double2 e0 = make_double2(0.0, 0.0), e1 = make_double2(0.0, 0.0);
        if (!zero_in && r0 >= d.in_lo && r0 < d.in_hi) e0 = src[r0];
        if (!zero_in && r1 >= d.in_lo && r1 < d.in_hi) e1 = src[r1];
        pf[0][m] = make_double2(e0.x, e1.x);
        pf[1][m] = make_double2(e0.y, e1.y);
    }
}

// the input operator on a lane's rows, once they are in registers (rows >= N are zero)
template <int R>
__device__ __forceinline__ void scale_input(double (&x0)[R], double (&x1)[R], int lane, const jw_run_desc& d,
                                            const double* fin)
{
    if (d.in_op < 1 || d.in_op > 4) return;
#pragma unroll
    for (int i = 0; i < R; i++) {
        const double f = fin[lane * R + i];
        x0[i] *= f;
        x1[i] *= f;
    }
}

// per-row factors of the block operators, once per workgroup into LDS (rows >= N
// get 1, so their zeros stay exact zeros even where a factor would be NaN)
__device__ __forceinline__ void block_factors(double* fin, double* fout, int rows, const jw_run_desc& d)
{
    for (int r = threadIdx.x; r < rows; r += blockDim.x) {
        const bool in = r < d.N;
        fin[r] = in && d.in_op >= 1 && d.in_op <= 4 ? jw_block_scale(d.in_op, r, d.in_lshift, d.in_scale) : 1.0;
        fout[r] = in && d.out_op >= 1 && d.out_op <= 4 ? jw_block_scale(d.out_op, r, d.out_lshift, d.out_scale) : 1.0;
    }
}

template <int R>
__device__ __forceinline__ void store_pair_packed(const double2* stg, int lane, const jw_run_desc& d, int64_t q,
                                                  const double* fout)
{
    constexpr int H = R / 2;
    constexpr int SYSC = 64 * H;
    double2* dst = reinterpret_cast<double2*>(d.out_c) + (q * d.out_stride_c + d.out_off_c);
    const double* s0 = reinterpret_cast<const double*>(stg);
    const double* s1 = reinterpret_cast<const double*>(stg + SYSC);
    const bool zero_out = d.out_op == 1 && d.out_scale == 0.0;
    const bool scaled = d.out_op >= 1 && d.out_op <= 4;
    // the previous output first (all loads in flight together), then the staging
    double2 prev[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int r = 64 * k + lane;
        prev[k] = make_double2(0.0, 0.0);
        if (d.out_acc && r >= d.out_lo && r < d.out_hi) prev[k] = dst[r];
    }
    double re[R], im[R], f[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int r = 64 * k + lane;   // complex row r: chunk r / 2, half r % 2, of both systems
        const int e = 2 * swz<H>(r >> 1) + (r & 1);
        re[k] = s0[e];
        im[k] = s1[e];
        f[k] = scaled ? fout[r] : 1.0;
    }
#pragma unroll
    for (int k = 0; k < R; k++) asm volatile("" : "+v"(re[k]), "+v"(im[k]), "+v"(f[k]));
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int r = 64 * k + lane;
        if (r < d.out_lo || r >= d.out_hi) continue;
        double a = re[k], b = im[k];
        if (zero_out) {
            a = 0.0;
            b = 0.0;
        } else if (scaled) {
            a *= f[k];
            b *= f[k];
        }
        if (d.out_acc) {
            a += prev[k].x;
            b += prev[k].y;
        }
        store_stream(reinterpret_cast<double*>(dst + r), make_double2(a, b));
    }
}

// Compute / store split.  The first `ncomp` wavefronts of a workgroup compute,
// the others store.  Every workgroup first builds the coefficient table in its
// LDS.  A compute wavefront owns an output staging; per pass it takes the rows
// of its pair that it loaded straight into registers one pass earlier, issues
// the loads of its next pair at once, computes, waits until a storer has
// emptied its staging, writes the results there and raises its `full` flag.  Storer
// wavefronts poll the flags of their compute wavefronts, stream full stagings
// to global memory (nontemporal stores) and lower the flag.  Compute
// wavefronts issue no global stores, so their vmcnt waits never wait for write
// acknowledgements; stores stay in flight while compute goes on.
// Every wait on a flag is bounded (kSpinLimit polls without progress); a
// wavefront that runs out stops and raises *err, so the grid always drains.
constexpr int kSpinLimit = 1 << 22;

// Flags and pair indices are relaxed workgroup-scope atomics in LDS: they
// compile to plain LDS accesses with no wait on outstanding global loads (a
// volatile access would wait for them and stall the prefetch).  The writer
// waits lgkmcnt(0) for its staging writes before it raises a flag.
__device__ __forceinline__ int lds_flag(int* f)
{
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ __forceinline__ void lds_set(int* f, int v)
{
    __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// waits until *f == v; false when `polls` polls ran out
__device__ __forceinline__ bool wait_flag(int* f, int v, int polls = kSpinLimit)
{
    for (int it = 0; it < polls; it++) {
        if (lds_flag(f) == v) return true;
        __builtin_amdgcn_s_sleep(2);
    }
    return false;
}

template <int R>
constexpr int split_threads()
{
    return R <= 4 ? 1024 : (R == 8 ? 768 : 320);
}

template <int R, bool ALL3, int IOMODE, bool EXACT = false>
__global__ __launch_bounds__(split_threads<R>())
__attribute__((amdgpu_waves_per_eu(split_threads<R>() / 256, split_threads<R>() / 256))) void jw_main64s_kernel(jw_run_desc d, int ncomp, int* err,
                                                                        jw_source_desc src, const void* mat)
{
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_full[16], s_done[16];
    __shared__ long long s_pair[16];
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* out_base = reinterpret_cast<double2*>(smem + NTAB * 8);
    const int64_t npass = (d.nsys + 1) >> 1;
    const int64_t step = (int64_t)gridDim.x * ncomp;
    const int polls = d.wait_polls > 0 ? d.wait_polls : (d.wait_polls < 0 ? 0 : kSpinLimit);
    int64_t q = (int64_t)blockIdx.x * ncomp + wave;
    // every workgroup builds the coefficient table in its own LDS from the
    // caller's matrices (no separate prologue launch); the staging area, unused
    // until the barrier below, is the build's scratch.  A compute wavefront's first pair
    // is loaded into registers behind the build's loads, so its latency overlaps the build
    // (before them, the build would wait for every wavefront's first pair)
    double2 pf[2][R / 2];
    auto first = [&] {
        if (wave >= ncomp || q >= npass) return;
        if (IOMODE != 0) {
            load_pair_packed<R>(pf, lane, d, q);
        } else {
            const jw_pass64 g = make_pass64(reinterpret_cast<double*>(d.rhs), d.nsys, d.stride, d.offSol,
                                            (int)d.in_lo, (int)d.in_hi, (int)d.out_lo, (int)d.out_hi, d.kl, d.ku,
                                            d.fwd, d.b1, d.b2, d.apply_scale, d.scale_hi, lane);
            load_pair_direct<R>(pf, lane, g, 2 * q);
        }
    };
    prologue_body<double, 2, NoPivotHooks, 1, pro_rows(64 * R)>(src, mat, reinterpret_cast<double*>(smem), 64, R,
                                                               smem + NTAB * 8, 0, nullptr, 1, NoPivotHooks(), first);
    // block operator factors past the staging and the build's scratch
    double* fin = reinterpret_cast<double*>(
        smem + NTAB * 8 + max_i64(2LL * 64 * R * 8 * ncomp, (int64_t)prologue_lds_bytes(64 * R, 8)));
    double* fout = fin + 64 * R;
    if (IOMODE != 0) block_factors(fin, fout, 64 * R, d);
    if (wave < ncomp) {
        if (lane == 0) {
            lds_set(&s_full[wave], 0);
            lds_set(&s_done[wave], 0);
        }
    }
    __syncthreads();
    int* vfull = s_full;
    int* vdone = s_done;

    if (wave < ncomp) {
        bool ok = true;
        double2* stg = out_base + (size_t)wave * 64 * R;
        // fused block input: whole systems, zero-filled past N by the packed loads, so
        // the keep-range is [0, N rounded up to even) and read_pair has no edge rows
        const int in_lo = IOMODE != 0 ? 0 : (int)d.in_lo;
        const int in_hi = IOMODE != 0 ? (int)(d.N + (d.N & 1)) : (int)d.in_hi;
        while (q < npass) {
            const jw_pass64 g = make_pass64(reinterpret_cast<double*>(d.rhs), d.nsys, d.stride, d.offSol, in_lo,
                                            in_hi, (int)d.out_lo, (int)d.out_hi, d.kl, d.ku, d.fwd, d.b1, d.b2,
                                            d.apply_scale, d.scale_hi, lane);
            // the rows prefetched a whole pass ago, then the next pair's loads at once
            double x0[R], x1[R];
            unpack_pair<R>(pf, lane, g, 2 * q, x0, x1);
            const int64_t qn = q + step;
            if (qn < npass) {
                if (IOMODE != 0) load_pair_packed<R>(pf, lane, d, qn);
                else load_pair_direct<R>(pf, lane, g, 2 * qn);
            }
            if (IOMODE != 0) scale_input<R>(x0, x1, lane, d, fin);
            compute_pair<R, ALL3, 1, false, EXACT>(tab, lane, g, x0, x1);
            if (!wait_flag(vfull + wave, 0, polls)) { ok = false; break; }
            write_blocked<R>(stg, lane, x0, x1);
            if (lane == 0) __hip_atomic_store(&s_pair[wave], (long long)q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): staging and pair index written
            compiler_fence();
            if (lane == 0) lds_set(vfull + wave, 1);
            q = qn;
        }
        if (ok) ok = wait_flag(vfull + wave, 0, polls);
        __builtin_amdgcn_s_waitcnt(0);
        compiler_fence();
        if (lane == 0) {
            lds_set(vdone + wave, 1);
            if (!ok) *err = 1;
        }
        return;
    }

    // storer wavefront j serves compute wavefronts j, j + nstore, ...
    const int nstore = nwaves - ncomp;
    const int j = wave - ncomp;
    int idle = 0;
    for (;;) {
        bool all_done = true, progress = false;
        for (int w = j; w < ncomp; w += nstore) {
            if (lds_flag(vfull + w)) {
                compiler_fence();   // the pair index and staging reads stay after the flag read
                const long long qq = __hip_atomic_load(&s_pair[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                const int64_t q = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)qq) |
                                  ((int64_t)__builtin_amdgcn_readfirstlane((int)(qq >> 32)) << 32);
                const jw_pass64 g = make_pass64(reinterpret_cast<double*>(d.rhs), d.nsys, d.stride, d.offSol,
                                                (int)d.in_lo, (int)d.in_hi, (int)d.out_lo, (int)d.out_hi, d.kl,
                                                d.ku, d.fwd, d.b1, d.b2, d.apply_scale, d.scale_hi, lane);
                if (IOMODE == 1) store_pair_packed<R>(out_base + (size_t)w * 64 * R, lane, d, q, fout);
                else store_pair<R>(out_base + (size_t)w * 64 * R, lane, g, 2 * q);
                __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the staging has been read
                compiler_fence();
                if (lane == 0) lds_set(vfull + w, 0);
                progress = true;
                all_done = false;
            } else if (!lds_flag(vdone + w)) {
                all_done = false;   // the flag is read before `done`: a raised done with an empty staging is final
            }
        }
        if (all_done) break;
        if (progress) {
            idle = 0;
        } else {
            if (++idle >= polls) {
                if (lane == 0) *err = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
}

// Uneven-size batch: a persistent grid drains a queue of work units (a matrix
// set and a range of its system pairs), in the order the host sorted them
// (largest N first).  A workgroup takes the next unit with one atomic add on
// the queue counter, stages the set's table in LDS when the set changes and
// spreads the unit's pairs over its wavefronts.  Every workgroup leaves the
// loop once the counter passes the last unit.
template <int R>
__global__ __launch_bounds__(max_threads<R>()) void jw_batch64_kernel(const jw_batch_item* items,
                                                                      const jw_batch_unit* units, int nunits,
                                                                      int* counter, int spw)
{
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_unit;
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* stg = reinterpret_cast<double2*>(smem + NTAB * 8 + wave * pair_stage_bytes(R));
    int cur = -1;
    for (;;) {
        __syncthreads();   // the previous unit is finished: s_unit and the table may change
        if (threadIdx.x == 0) s_unit = atomicAdd(counter, 1);
        __syncthreads();
        const int u = __builtin_amdgcn_readfirstlane(s_unit);
        if (u >= nunits) break;
        const jw_batch_unit un = units[u];
        const jw_batch_item& it = items[un.item];
        if constexpr (pair_ahead(R)) {
            auto geo = [&] {
                return make_pass64(reinterpret_cast<double*>(it.rhs), it.nsys, it.stride, it.offSol, 0, it.N, 0, it.N,
                                   it.kl, it.ku, true, true, true, it.apply_scale != 0, it.scale, lane);
            };
            // the unit's first pairs are loaded before the table copy
            double2 pf[2][R / 2];
            const int64_t q = un.pair0 + wave;
            if (q < un.pair1) load_pair_ahead<R>(pf, lane, geo(), 2 * q);
            if (un.item != cur) {
                copy_table_lds<NTAB>(smem, it.table, wave, nwaves, lane);
                __syncthreads();
                cur = un.item;
            }
            stream_pairs<R, true>(tab, stg, lane, geo, q, un.pair1, nwaves, pf);
            continue;
        }
        if (un.item != cur) {
            copy_table_lds<NTAB>(smem, it.table, wave, nwaves, lane);
            zero_staging<R>(stg, lane);   // the new set's keep-range may be narrower
            __syncthreads();
            cur = un.item;
        }
        if constexpr (R == 2) {
            // sub-wavefront groups: G pairs (2G systems) per wavefront pass
            const int G = spw >= 8 && it.N <= 32 ? 4 : (spw >= 4 && it.N <= 64 ? 2 : 1);
            if (G > 1) {
                const int tl = lane & (64 / G - 1);
                const jw_pass64 g = make_pass64(reinterpret_cast<double*>(it.rhs), it.nsys, it.stride, it.offSol, 0,
                                                it.N, 0, it.N, it.kl, it.ku, true, true, true, it.apply_scale != 0,
                                                it.scale, tl);
                const int64_t sys_end = it.nsys < 2 * (int64_t)un.pair1 ? it.nsys : 2 * (int64_t)un.pair1;
                for (int q = un.pair0 + wave * G; q < un.pair1; q += nwaves * G) {
                    if (G == 2) jw_groups64<2>(tab, stg, lane, g, 2 * (int64_t)q, sys_end);
                    else jw_groups64<4>(tab, stg, lane, g, 2 * (int64_t)q, sys_end);
                }
                continue;
            }
        }
        for (int q = un.pair0 + wave; q < un.pair1; q += nwaves) {
            const jw_pass64 g = make_pass64(reinterpret_cast<double*>(it.rhs), it.nsys, it.stride, it.offSol, 0,
                                            it.N, 0, it.N, it.kl, it.ku, true, true, true, it.apply_scale != 0,
                                            it.scale, lane);
            jw_pair64<R, true>(tab, stg, lane, g, 2 * (int64_t)q);
        }
    }
    queue_leave(counter);
}

// LDS of the build-in-LDS queue kernel: the table, then the wavefronts' stagings, which
// also hold the table build's scratch while a set's table is built
__host__ __device__ constexpr int64_t batch64b_lds_bytes(int R, int waves)
{
    const int64_t stagings = pair_stage_bytes(R) * waves, scratch = (int64_t)prologue_lds_bytes(64 * R, 8);
    return (int64_t)JW_TAB64_ELEMS(R) * 8 + (stagings > scratch ? stagings : scratch);
}

// The batch queue with the table built in LDS: as jw_batch64_kernel, but a workgroup
// whose set changes builds the set's format-2 table from the caller's matrices in its
// own LDS (prologue_body, the staging as scratch) instead of copying a table that a
// separate launch wrote to global memory: no table build launch before the queue, no
// table written and read back through HBM; the build's latency is paid per set change
// by the workgroup, while the other workgroups keep HBM busy.  Needs at least 256
// threads and 4 threads per 16 rows (prologue_body's partition).
// FULL: a full workgroup, whose threads take one or two rows each of a build.
// (R = 16: the build out of line, before the unit's first loads; in line, its registers
// spill the solve loop's: 266 us per step of the 1024-degree batch, 196 us out of line)
template <int R, int MAXJ>
__device__ __noinline__ void build_table_lds(const jw_prologue_job* job)
{
    extern __shared__ __align__(16) unsigned char smem_build[];   // named here: addressed as LDS
    // the argument is the same in every lane, which the callee cannot know: the job through
    // scalar loads (a descriptor in vector registers would make every branch on it divergent)
    typedef const __attribute__((address_space(4))) uint32_t const_word;
    const uint64_t p = reinterpret_cast<uint64_t>(job);
    const_word* w = (const_word*)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)p) |
                                  ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32));
    union {
        jw_prologue_job j;
        uint32_t u[sizeof(jw_prologue_job) / 4];
    } x;
#pragma unroll
    for (size_t i = 0; i < sizeof(jw_prologue_job) / 4; i++) x.u[i] = w[i];
    prologue_body<double, 2, NoPivotHooks, MAXJ, pro_rows(64 * R)>(
        x.j.src, x.j.matrices, reinterpret_cast<double*>(smem_build), 64, R, smem_build + JW_TAB64_ELEMS(R) * 8);
}

template <int R, bool FULL>
__global__ __launch_bounds__(max_threads<R>()) void jw_batch64b_kernel(const jw_batch_item* items,
                                                                       const jw_batch_unit* units, int nunits,
                                                                       int* counter, const jw_prologue_job* jobs,
                                                                       int keep)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    constexpr int MAXJ = FULL ? (R <= 8 ? 1 : 2) : pro_rows(64 * R);
    __shared__ int s_unit;
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* stg = reinterpret_cast<double2*>(smem + NTAB * 8 + wave * pair_stage_bytes(R));
    int cur = -1;
    for (;;) {
        __syncthreads();   // the previous unit is finished: s_unit, the table and the staging may change
        if (threadIdx.x == 0) s_unit = atomicAdd(counter, 1);
        __syncthreads();
        const int u = __builtin_amdgcn_readfirstlane(s_unit);
        if (u >= nunits) break;
        const jw_batch_unit un = units[u];
        const jw_batch_item& it = items[un.item];
        const int64_t q = un.pair0 + wave;
        auto geo = [&] {
            return make_pass64(reinterpret_cast<double*>(it.rhs), it.nsys, it.stride, it.offSol, 0, it.N, 0, it.N,
                               it.kl, it.ku, true, true, true, it.apply_scale != 0, it.scale, lane);
        };
        if (un.item != cur) {
            cur = un.item;
            if constexpr (pair_ahead(R)) {
                build_table_lds<R, MAXJ>(jobs + cur);
                __syncthreads();   // the build's scratch (the stagings) is free again
            } else {
                const jw_prologue_job& job = jobs[cur];
                prologue_body<double, 2, NoPivotHooks, MAXJ, pro_rows(64 * R)>(
                    job.src, job.matrices, reinterpret_cast<double*>(smem), 64, R, smem + NTAB * 8);
                __syncthreads();
                zero_staging<R>(stg, lane);
                __syncthreads();
            }
        }
        // the set's first unit writes the table for later solves (behind the first pairs' loads)
        auto write_table = [&] {
            if (!keep || un.pair0 != 0) return;
            double* out = reinterpret_cast<double*>(jobs[un.item].table);
            for (int i = 2 * threadIdx.x; i < NTAB; i += 2 * blockDim.x)
                store_stream(out + i, *reinterpret_cast<const double2*>(tab + i));
        };
        if constexpr (pair_ahead(R)) {
            double2 pf[2][R / 2];
            if (q < un.pair1) load_pair_ahead<R>(pf, lane, geo(), 2 * q);
            write_table();
            stream_pairs<R, true>(tab, stg, lane, geo, q, un.pair1, nwaves, pf);
        } else {
            write_table();
            for (int64_t p = q; p < un.pair1; p += nwaves) jw_pair64<R, true>(tab, stg, lane, geo(), 2 * p);
        }
    }
    queue_leave(counter);
}

// 16-byte stores of a pair straight from the registers (lane t: chunks t H .. t H + H-1
// of both systems, the output keep-range's full chunks), the odd range ends by their
// owning lane
template <int R>
__device__ __forceinline__ void store_pair_direct(int lane, const jw_pass64& g, int64_t sys0, const double (&x0)[R],
                                                  const double (&x1)[R])
{
    constexpr int H = R / 2;
    const bool ok1 = sys0 + 1 < g.nsys;
    double* dst0 = g.rhs + sys0 * g.stride + g.offSol;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        if (s == 1 && !ok1) continue;
        JW_GLOBAL jw_d2u* dst = (JW_GLOBAL jw_d2u*)(dst0 + s * g.stride);
        const double(&x)[R] = s == 0 ? x0 : x1;
#pragma unroll
        for (int m = 0; m < H; m++) {
            const int c = lane * H + m;
            // cached stores: the H stores of a lane each fill part of 64 lines that the
            // sibling stores complete, and L2 merges them before the write-back
            if (c >= g.ocl && c < g.och) dst[c] = jw_d2u{x[2 * m], x[2 * m + 1]};
        }
    }
    if (g.out_edge_lo || g.out_edge_hi) {
        JW_GLOBAL double* base = as_global(g.rhs) + sys0 * g.stride + g.offSol;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const bool on = e == 0 ? g.out_edge_lo : g.out_edge_hi;
            const int r = e == 0 ? g.out_lo : g.out_hi - 1;
            if (on && lane == r / R) {
#pragma unroll
                for (int k = 0; k < R; k++)
                    if (k == r % R) {
                        base[r] = x0[k];
                        if (ok1) base[g.stride + r] = x1[k];
                    }
            }
        }
    }
}

// The batch queue with direct I/O: LDS holds the set's table only (no staging), so more
// wavefronts share one table; every wavefront loads its pairs straight into registers
// one pass ahead, computes and stores straight from registers (nontemporal 16-byte
// stores).  Units and the table hand-over as in jw_batch64_kernel.
constexpr int kBatchDirectThreads = 512;
template <int R>
__global__ __launch_bounds__(kBatchDirectThreads) void jw_batch64d_kernel(const jw_batch_item* items,
                                                                          const jw_batch_unit* units, int nunits,
                                                                          int* counter)
{
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_unit;
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    int cur = -1;
    for (;;) {
        __syncthreads();   // the previous unit is finished: s_unit and the table may change
        if (threadIdx.x == 0) s_unit = atomicAdd(counter, 1);
        __syncthreads();
        const int u = __builtin_amdgcn_readfirstlane(s_unit);
        if (u >= nunits) break;
        const jw_batch_unit un = units[u];
        const jw_batch_item& it = items[un.item];
        const jw_pass64 g = make_pass64(reinterpret_cast<double*>(it.rhs), it.nsys, it.stride, it.offSol, 0, it.N, 0,
                                        it.N, it.kl, it.ku, true, true, true, it.apply_scale != 0, it.scale, lane);
        int64_t q = un.pair0 + wave;
        // the first pair's loads go out before the table copy
        double2 pf[2][R / 2];
        if (q < un.pair1) load_pair_direct<R>(pf, lane, g, 2 * q);
        if (un.item != cur) {
            copy_table_lds<NTAB>(smem, it.table, wave, nwaves, lane);
            __syncthreads();
            cur = un.item;
        }
        while (q < un.pair1) {
            const int64_t qn = q + nwaves;
            double x0[R], x1[R];
            unpack_pair<R>(pf, lane, g, 2 * q, x0, x1);
            if (qn < un.pair1) load_pair_direct<R>(pf, lane, g, 2 * qn);
            compute_pair<R, true>(tab, lane, g, x0, x1);
            store_pair_direct<R>(lane, g, 2 * q, x0, x1);
            q = qn;
        }
    }
    queue_leave(counter);
}

// The same queue for 1024 < N <= 2048: two pairs of systems per pass of a workgroup, the
// coefficients in its registers (above); the unit ranges count systems, not pairs.
__global__ __launch_bounds__(kWideThreads) void jw_batch64w_kernel(const jw_batch_item* items, const jw_batch_unit* units,
                                                                   int nunits, int* counter, int /* systems per pass */)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_unit;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave / kWideW, w = wave % kWideW;
    int cur = -1;
    wide_coef c;
    for (;;) {
        __syncthreads();   // the previous unit is finished: s_unit and the multipliers may change
        if (threadIdx.x == 0) s_unit = atomicAdd(counter, 1);
        __syncthreads();
        const int u = __builtin_amdgcn_readfirstlane(s_unit);
        if (u >= nunits) break;
        const jw_batch_unit un = units[u];
        const jw_batch_item& it = items[un.item];
        const int64_t sys_end = it.nsys < un.pair1 ? it.nsys : un.pair1;
        const int64_t npass = (sys_end - un.pair0 + 1) >> 1;
        auto geo = [&] {
            return wide_pass(reinterpret_cast<double*>(it.rhs), sys_end, it.stride, it.offSol, it.N, 0, it.N, 0, it.N,
                             it.kl, it.ku, true, true, true, it.apply_scale != 0, it.scale, w, lane);
        };
        double2 pf[2][kWideR / 2] = {};
        if (grp < npass) load_pair_ahead<kWideR>(pf, lane, geo(), un.pair0 + 2 * grp);
        if (un.item != cur) {
            wide_load_table(c, it.table, w, lane);
            if (grp == 0)
                wide_multipliers(c, reinterpret_cast<double*>(smem + kWideMult),
                                 reinterpret_cast<double*>(smem + kWideExch) + kWideGroups * kWideW * (8 + 3 * 2), w,
                                 lane);
            __syncthreads();
            cur = un.item;
        }
        wide_stream<true, true>(c, smem, grp, w, lane, geo, un.pair0, 0, npass, kWideGroups, pf);
    }
    queue_leave(counter);
}

// The batch queue with the compute / store split (R <= 16): the first `ncomp`
// wavefronts of a workgroup compute, the others store, as in jw_main64s_kernel.
// Per work unit the workgroup stages the set's table in LDS (when the set
// changes), compute wavefronts run the unit's pairs with the next pair's loads
// in registers one pass ahead, and storers stream the results.  Every
// wavefront meets at two barriers per unit: the table and the stagings change
// only while nobody uses them.  A wait that runs out of polls raises *err and
// the workgroup's abort flag; every wavefront then leaves at the next unit.
template <int R>
constexpr int bsplit_threads()
{
    return R <= 4 ? 1024 : (R == 8 ? 768 : 512);
}

template <int R>
__global__ __launch_bounds__(bsplit_threads<R>()) void jw_batch64s_kernel(const jw_batch_item* items,
                                                                          const jw_batch_unit* units, int nunits,
                                                                          int* counter, int ncomp, int* err,
                                                                          int wait_polls)
{
    // polls before a bounded wait gives up: 0 the default, negative none
    const int polls = wait_polls > 0 ? wait_polls : (wait_polls < 0 ? 0 : kSpinLimit);
    constexpr int NTAB = JW_TAB64_ELEMS(R);
    constexpr int STG = 64 * R;   // staging chunks (16 bytes) of a computing wavefront: two systems
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_full[16], s_done[16];
    __shared__ long long s_pair[16];
    __shared__ int s_unit, s_abort;
    const double* tab = reinterpret_cast<const double*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    double2* out_base = reinterpret_cast<double2*>(smem + NTAB * 8);
    if (threadIdx.x == 0) s_abort = 0;
    if (wave < ncomp && lane == 0) lds_set(&s_full[wave], 0);
    int cur = -1;
    for (;;) {
        __syncthreads();   // the previous unit is finished: stagings empty, the table unused
        // the abort flag is only raised inside a unit, so every wavefront sees the same answer
        if (threadIdx.x == 0) s_unit = s_abort ? nunits : atomicAdd(counter, 1);
        if (wave < ncomp && lane == 0) lds_set(&s_done[wave], 0);
        __syncthreads();
        const int u = __builtin_amdgcn_readfirstlane(s_unit);
        if (u >= nunits) break;
        const jw_batch_unit un = units[u];
        const jw_batch_item& it = items[un.item];
        const jw_pass64 g = make_pass64(reinterpret_cast<double*>(it.rhs), it.nsys, it.stride, it.offSol, 0, it.N, 0,
                                        it.N, it.kl, it.ku, true, true, true, it.apply_scale != 0, it.scale, lane);
        int64_t q = un.pair0 + wave;
        // a compute wavefront's first pair of the unit is loaded before the table copy
        double2 pf[2][R / 2];
        if (wave < ncomp && q < un.pair1) load_pair_direct<R>(pf, lane, g, 2 * q);
        if (un.item != cur) {
            copy_table_lds<NTAB>(smem, it.table, wave, nwaves, lane);
            __syncthreads();
            cur = un.item;
        }
        if (wave < ncomp) {
            bool ok = true;
            double2* stg = out_base + (size_t)wave * STG;
            while (q < un.pair1) {
                const int64_t qn = q + ncomp;
                double x0[R], x1[R];
                unpack_pair<R>(pf, lane, g, 2 * q, x0, x1);
                if (qn < un.pair1) load_pair_direct<R>(pf, lane, g, 2 * qn);
                compute_pair<R, true>(tab, lane, g, x0, x1);
                if (!wait_flag(&s_full[wave], 0, polls)) { ok = false; break; }
                write_blocked<R>(stg, lane, x0, x1);
                if (lane == 0)
                    __hip_atomic_store(&s_pair[wave], (long long)q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): staging and pair index written
                compiler_fence();
                if (lane == 0) lds_set(&s_full[wave], 1);
                q = qn;
            }
            if (ok) ok = wait_flag(&s_full[wave], 0, polls);
            __builtin_amdgcn_s_waitcnt(0);
            compiler_fence();
            if (lane == 0) {
                lds_set(&s_done[wave], 1);
                if (!ok) {
                    *err = 1;
                    lds_set(&s_abort, 1);
                }
            }
            continue;
        }
        // storer wavefront j serves compute wavefronts j, j + nstore, ...
        const int nstore = nwaves - ncomp;
        const int j = wave - ncomp;
        int idle = 0;
        for (;;) {
            bool all_done = true, progress = false;
            for (int w = j; w < ncomp; w += nstore) {
                if (lds_flag(&s_full[w])) {
                    compiler_fence();   // the pair index and staging reads stay after the flag read
                    const long long qq =
                        __hip_atomic_load(&s_pair[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    const int64_t qs = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)qq) |
                                       ((int64_t)__builtin_amdgcn_readfirstlane((int)(qq >> 32)) << 32);
                    store_pair<R>(out_base + (size_t)w * STG, lane, g, 2 * qs);
                    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the staging has been read
                    compiler_fence();
                    if (lane == 0) lds_set(&s_full[w], 0);
                    progress = true;
                    all_done = false;
                } else if (!lds_flag(&s_done[w])) {
                    all_done = false;   // `full` is read before `done`: done with an empty staging is final
                }
            }
            if (all_done) break;
            if (progress) {
                idle = 0;
            } else {
                if (++idle >= polls) {
                    if (lane == 0) {
                        *err = 1;
                        lds_set(&s_abort, 1);
                    }
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
        }
    }
    queue_leave(counter);
}

// the kernels on tables in memory (the fused step)
const void* pick64(int R)
{
    switch (R) {
    case 2: return reinterpret_cast<const void*>(&jw_main64_kernel<2, true, false>);
    case 4: return reinterpret_cast<const void*>(&jw_main64_kernel<4, true, false>);
    case 8: return reinterpret_cast<const void*>(&jw_main64_kernel<8, true, false>);
    case 16: return reinterpret_cast<const void*>(&jw_main64_kernel<16, true, false>);
    case 32: return reinterpret_cast<const void*>(&jw_wide64_kernel<true, false>);
    default: return nullptr;
    }
}

// the kernels that build their table, for a solve_form
template <int R>
const void* build_ptr(int form)
{
    return form == kAllThree ? reinterpret_cast<const void*>(&jw_main64_kernel<R, true, true>)
           : form == kSome   ? reinterpret_cast<const void*>(&jw_main64_kernel<R, false, true>)
                             : reinterpret_cast<const void*>(&jw_main64_kernel<R, false, true, true>);
}

const void* pick64b(int R, int form)
{
    switch (R) {
    case 2: return build_ptr<2>(form);
    case 4: return build_ptr<4>(form);
    case 8: return build_ptr<8>(form);
    case 16: return build_ptr<16>(form);
    case 32: return form == kAllThree ? reinterpret_cast<const void*>(&jw_wide64_kernel<true, true>)
                    : form == kSome   ? reinterpret_cast<const void*>(&jw_wide64_kernel<false, true>)
                                      : reinterpret_cast<const void*>(&jw_wide64_kernel<false, true, true>);
    default: return nullptr;
    }
}

template <int MODE>
const void* long64_ptr(bool all3)
{
    return all3 ? reinterpret_cast<const void*>(&jw_long64_kernel<MODE, true>)
                : reinterpret_cast<const void*>(&jw_long64_kernel<MODE, false>);
}

const void* pick_long64(int mode, bool all3)
{
    switch (mode) {
    case JW_LONG_REDUCE: return long64_ptr<JW_LONG_REDUCE>(all3);
    case JW_LONG_FINISH: return long64_ptr<JW_LONG_FINISH>(all3);
    default: return nullptr;
    }
}

constexpr int kLong64Waves = max_threads<kLong64R>() / 64;

const void* pick_long64_front(bool all3)
{
    return all3 ? reinterpret_cast<const void*>(&jw_long64_front_kernel<true>)
                : reinterpret_cast<const void*>(&jw_long64_front_kernel<false>);
}

// zeroes the counters and table flags, empties the pivot slots
__global__ void jw_long64_clear_kernel(int* p, int n, unsigned long long* lines, int nwords)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += gridDim.x * blockDim.x) lines[i] = kPivotEmpty;
}

// clears the work-queue counters (a kernel, so that it can sit in a captured graph)
__global__ void jw_zero_counters_kernel(int* p, int n)
{
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

template <int R>
const void* batch_ptr()
{
    return reinterpret_cast<const void*>(&jw_batch64_kernel<R>);
}

const void* pick_batch64(int R)
{
    switch (R) {
    case 32: return reinterpret_cast<const void*>(&jw_batch64w_kernel);
    case 2: return batch_ptr<2>();
    case 4: return batch_ptr<4>();
    case 8: return batch_ptr<8>();
    case 16: return batch_ptr<16>();
    default: return nullptr;
    }
}

const void* pick_batch64s(int R)
{
    switch (R) {
    case 2: return reinterpret_cast<const void*>(&jw_batch64s_kernel<2>);
    case 4: return reinterpret_cast<const void*>(&jw_batch64s_kernel<4>);
    case 8: return reinterpret_cast<const void*>(&jw_batch64s_kernel<8>);
    case 16: return reinterpret_cast<const void*>(&jw_batch64s_kernel<16>);
    default: return nullptr;
    }
}

int bsplit_threads_rt(int R) { return R <= 4 ? 1024 : (R == 8 ? 768 : 512); }

template <int R>
const void* split_ptr(int form, int io)
{
    const bool all3 = form == kAllThree;
    if constexpr (R > 2)
        if (io == 0)
            return all3            ? reinterpret_cast<const void*>(&jw_main64s_kernel<R, true, 0>)
                   : form == kSome ? reinterpret_cast<const void*>(&jw_main64s_kernel<R, false, 0>)
                                   : reinterpret_cast<const void*>(&jw_main64s_kernel<R, false, 0, true>);
    if (io == 1)
        return all3 ? reinterpret_cast<const void*>(&jw_main64s_kernel<R, true, 1>)
                    : reinterpret_cast<const void*>(&jw_main64s_kernel<R, false, 1>);
    return all3 ? reinterpret_cast<const void*>(&jw_main64s_kernel<R, true, 2>)
                : reinterpret_cast<const void*>(&jw_main64s_kernel<R, false, 2>);
}

// io: 0 plain step (R = 4, 8; every form), 1 complex in and out (block layouts 4 and 7),
// 2 complex in (layout 4), real systems out
const void* pick_split(int R, int form, int io)
{
    switch (R) {
    case 2: return io ? split_ptr<2>(form, io) : nullptr;
    case 4: return split_ptr<4>(form, io);
    case 8: return split_ptr<8>(form, io);
    default: return nullptr;
    }
}

// compute / storer wavefronts of the split kernel: compute wavefronts up to
// what LDS holds (table + output staging each), at most 8 for R = 8 and 12
// below, so that every SIMD holds the same number (2 or 3: a SIMD with one more
// than the others is the slowest), and storers for the rest of the launch bound
// (12 wavefronts for R = 8, 16 below).
bool split_shape(int R, int* ncomp, int* nstore)
{
    const int maxw = R <= 4 ? 16 : (R == 8 ? 12 : 5);
    const int cmax = R <= 4 ? 12 : (R == 8 ? 8 : 2);
    const int64_t table = jwdev_table64_elems(R) * 8;
    const int64_t per = 2LL * 64 * R * 8;   // output staging of 2 systems
    const int64_t avail = kLdsBytesMax - 256 - table - 2LL * 64 * R * 8;   // less the block factors
    int c = (int)(avail / per);
    if (c > cmax) c = cmax;
    if (c < 1 || c >= maxw) return false;
    *ncomp = c;
    *nstore = maxw - c;
    return true;
}

int max_waves64(int R) { return R <= 4 ? 16 : (R == 8 ? 12 : 8); }

thread_local char g_err64[256];

}  // namespace

extern "C" {

int64_t jwdev_table64_elems(int R) { return JW_TAB64_ELEMS(R); }
int jwdev_main64b_waves(int R);

/* waves per workgroup: as many as LDS (table + 2 systems of staging per wave)
 * and the kernel's launch bound allow */
int jwdev_main64_waves(int R)
{
    if (!pick64(R)) return 0;
    if (R == 32) return kWideThreads / 64;   /* the kernel's shape is fixed */
    const int64_t table = JW_TAB64_ELEMS(R) * 8;
    int w = (int)((kLdsBytesMax - table) / pair_stage_bytes(R));
    if (w > max_waves64(R)) w = max_waves64(R);
    return w < 1 ? 0 : w;
}

int64_t jwdev_main64_lds_bytes(int R, int waves)
{
    if (R == 32) return kWideLds;
    return JW_TAB64_ELEMS(R) * 8 + pair_stage_bytes(R) * waves;
}

/* pairs of systems per workgroup and pass */
int jwdev_main64_pairs(int R, int waves) { return R == 32 ? kWideGroups : waves; }

/* workgroups per CU of a kernel (0: it cannot run) */
static int occupancy_of(const void* f, int threads, int lds)
{
    int nb = 0;
    if (!f || hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, threads, lds) != hipSuccess)
        return 0;
    return nb;
}

int jwdev_main64_occupancy(int R, int waves)
{
    return occupancy_of(pick64(R), 64 * waves, (int)jwdev_main64_lds_bytes(R, waves));
}

int jwdev_main64(const jw_run_desc* r, int R, int waves, int grid, void* stream)
{
    if (!r->rhs || !r->table || solve_form(*r) != kAllThree) {
        snprintf(g_err64, sizeof(g_err64), "main64: no rhs or table, or not a fused step");
        return -1;
    }
    const void* f = pick64(R);
    if (!f) { snprintf(g_err64, sizeof(g_err64), "no 64-lane kernel for R=%d", R); return -1; }
    const size_t lds = (size_t)jwdev_main64_lds_bytes(R, waves);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    /* the source and matrices are read by the building variants only */
    jw_source_desc none;
    memset(&none, 0, sizeof(none));
    const void* nomat = NULL;
    void* args[] = {const_cast<jw_run_desc*>(r), &none, &nomat};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * waves), args, lds, reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

/* the same with the table built in the kernel (systems at any 8-byte address): wavefronts
 * per workgroup (the launch bound), workgroups per CU, launch */
static int64_t main64b_lds_bytes(int R)
{
    if (R == 32) return kWideLds;
    return (int64_t)JW_TAB64_ELEMS(R) * 8 + max_i64(512LL * R * jwdev_main64b_waves(R), (int64_t)prologue_lds_bytes(64 * R, 8));
}

int jwdev_main64b_waves(int R)
{
    switch (R) {
    case 2: return max_threads<2>() / 64;
    case 4: return max_threads<4>() / 64;
    case 8: return max_threads<8>() / 64;
    case 16: return max_threads<16>() / 64;
    case 32: return kWideThreads / 64;
    default: return 0;
    }
}

int jwdev_main64b_occupancy(int R)
{
    const int w = jwdev_main64b_waves(R);
    int best = 1 << 30;
    for (int form = kAllThree; w && form <= kSomeExact; form++) {
        const int nb = occupancy_of(pick64b(R, form), 64 * w, (int)main64b_lds_bytes(R));
        if (nb < best) best = nb;
    }
    return w ? best : 0;
}

int jwdev_main64b(const jw_run_desc* r, const jw_source_desc* src, const void* matrices, int R, int grid, void* stream)
{
    const void* f = pick64b(R, solve_form(*r));
    if (!r->rhs || !matrices || !f || grid < 1) {
        snprintf(g_err64, sizeof(g_err64), "main64b: no rhs or matrices, or no kernel for R=%d", R);
        return -1;
    }
    const size_t lds = (size_t)main64b_lds_bytes(R);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {const_cast<jw_run_desc*>(r), const_cast<jw_source_desc*>(src), &matrices};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * jwdev_main64b_waves(R)), args, lds,
                        reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

}  // extern "C"

namespace {
template <int R, bool UP>
const void* chain_ptr(bool glob)
{
    // (R <= 4: 16 tables fit)
    if constexpr (R >= 8)
        if (glob) return reinterpret_cast<const void*>(&jw_chain64_kernel<R, UP, true>);
    return glob ? nullptr : reinterpret_cast<const void*>(&jw_chain64_kernel<R, UP, false>);
}

// the chain kernel, with some of its tables in global memory or none
const void* pick_chain(int R, bool up, bool glob)
{
    switch (R) {
    case 2: return up ? chain_ptr<2, true>(glob) : chain_ptr<2, false>(glob);
    case 4: return up ? chain_ptr<4, true>(glob) : chain_ptr<4, false>(glob);
    case 8: return up ? chain_ptr<8, true>(glob) : chain_ptr<8, false>(glob);
    case 16: return up ? chain_ptr<16, true>(glob) : chain_ptr<16, false>(glob);
    default: return nullptr;
    }
}

// the build of the tables in global memory
const void* pick_chain_tables(int R, bool up)
{
    if (R == 8)
        return up ? reinterpret_cast<const void*>(&jw_chain_tables_kernel<8, true>)
                  : reinterpret_cast<const void*>(&jw_chain_tables_kernel<8, false>);
    if (R == 16)
        return up ? reinterpret_cast<const void*>(&jw_chain_tables_kernel<16, true>)
                  : reinterpret_cast<const void*>(&jw_chain_tables_kernel<16, false>);
    return nullptr;
}

int64_t chain_stage_bytes(int R) { return 64LL * R * 8; }   // one system per wavefront

// Tables in LDS and wavefronts per workgroup: every table with at least 4 stagings after
// them (one wavefront per SIMD), else as many tables as leave room for 8 stagings: N = 1000, K = 8,
// 16384 systems: 109 us with none of the 8 tables in LDS, 93 with 3, 106 with 4 and 6 stagings;
// N = 512, K = 12, 20000 systems: 104 with none of the 12, 86 with 4, 75 with 8.
void chain_split(int R, int K, int* kl, int* waves)
{
    const int64_t tab = (int64_t)chain_tab_elems(R) * 8;
    int64_t w = (kLdsBytesMax - K * tab) / chain_stage_bytes(R);
    *kl = K;
    if (w < 4) {
        w = 8;
        *kl = (int)((kLdsBytesMax - w * chain_stage_bytes(R)) / tab);
    }
    *waves = w > chain_max_waves(R) ? chain_max_waves(R) : (int)w;
}

size_t chain_lds_bytes(int R, int kl, int waves)
{
    return (size_t)(kl * (int64_t)chain_tab_elems(R) * 8 + waves * chain_stage_bytes(R));
}
}  // namespace

extern "C" {

/* wavefronts per workgroup, workgroups per CU of a chained step (0: not available) */
int jwdev_chain64_shape(int R, int K, int* waves)
{
    if (!pick_chain(R, true, false) || K < 1 || K > JW_CHAIN_MAX) return 0;
    int kl = 0;
    chain_split(R, K, &kl, waves);
    const int lds = (int)chain_lds_bytes(R, kl, *waves);
    int best = -1;
    for (int up = 0; up < 2; up++) {
        const void* f = pick_chain(R, up, kl < K);
        if (!f || hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 0;
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 64 * *waves, lds) != hipSuccess) return 0;
        if (best < 0 || nb < best) best = nb;
    }
    return best;
}

int jwdev_chain64(const jw_run_desc* r, const jw_chain_jobs* jobs, int up, int grid, void* stream)
{
    if (!r->rhs || jobs->K < 1 || jobs->K > JW_CHAIN_MAX || grid < 1 || !pick_chain(jobs->R, up, false)) {
        snprintf(g_err64, sizeof(g_err64), "chain64: no rhs, or a bad chain");
        return -1;
    }
    int kl = 0, waves = 0;
    chain_split(jobs->R, jobs->K, &kl, &waves);
    if (kl < jobs->K && (!jobs->table || !pick_chain_tables(jobs->R, up))) {
        snprintf(g_err64, sizeof(g_err64), "chain64: no tables");
        return -1;
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    jw_run_desc rr = *r;
    jw_chain_jobs jj = *jobs;
    if (kl < jobs->K) {
        void* args[] = {&jj, &kl};
        if (hipLaunchKernel(pick_chain_tables(jobs->R, up), dim3(jobs->K - kl), dim3(64 * jobs->R), args, 0, s) !=
            hipSuccess)
            return -3;
    }
    const void* f = pick_chain(jobs->R, up, kl < jobs->K);
    const size_t lds = chain_lds_bytes(jobs->R, kl, waves);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {&rr, &jj, &kl};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * waves), args, lds, s);
    return e == hipSuccess ? 0 : -3;
}

int jwdev_batch64_occupancy(int R, int waves)
{
    const void* f = pick_batch64(R);
    if (!f || waves < 1 || waves > max_waves64(R) || (R == 32 && waves != max_waves64(R))) return 0;
    const int lds = (int)jwdev_main64_lds_bytes(R, waves);
    if (lds > kLdsBytesMax) return 0;
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 64 * waves, lds) != hipSuccess) return 0;
    return nb;
}

int jwdev_batch64(const jw_batch_item* d_items, const jw_batch_unit* d_units, int nunits, int* d_counter, int R,
                  int waves, int grid, int spw, void* stream)
{
    const void* f = pick_batch64(R);
    if (!f) { snprintf(g_err64, sizeof(g_err64), "no batch kernel for R=%d", R); return -1; }
    if (waves < 1 || waves > max_waves64(R) || (R == 32 && waves != max_waves64(R)) || grid < 1) {
        snprintf(g_err64, sizeof(g_err64), "bad batch launch");
        return -1;
    }
    const size_t lds = (size_t)jwdev_main64_lds_bytes(R, waves);
    if (lds > (size_t)kLdsBytesMax) { snprintf(g_err64, sizeof(g_err64), "batch LDS %zu too large", lds); return -1; }
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {const_cast<jw_batch_item**>(&d_items), const_cast<jw_batch_unit**>(&d_units), &nunits,
                    &d_counter, &spw};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * waves), args, lds, reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

static const void* pick_batch64b(int R, int waves)
{
    const bool full = waves == max_waves64(R);
    switch (R) {
    case 2: return full ? reinterpret_cast<const void*>(&jw_batch64b_kernel<2, true>)
                        : reinterpret_cast<const void*>(&jw_batch64b_kernel<2, false>);
    case 4: return full ? reinterpret_cast<const void*>(&jw_batch64b_kernel<4, true>)
                        : reinterpret_cast<const void*>(&jw_batch64b_kernel<4, false>);
    case 8: return full ? reinterpret_cast<const void*>(&jw_batch64b_kernel<8, true>)
                        : reinterpret_cast<const void*>(&jw_batch64b_kernel<8, false>);
    case 16: return full ? reinterpret_cast<const void*>(&jw_batch64b_kernel<16, true>)
                         : reinterpret_cast<const void*>(&jw_batch64b_kernel<16, false>);
    default: return nullptr;
    }
}

/* the table build needs >= 256 threads and 4 threads per 16 rows */
static bool batch64b_shape_ok(int R, int waves)
{
    return pick_batch64b(R, waves) && waves >= 4 && waves <= max_waves64(R) && 4 * 64 * waves >= 64 * R &&
           batch64b_lds_bytes(R, waves) <= kLdsBytesMax;
}

int jwdev_batch64b_occupancy(int R, int waves)
{
    if (!batch64b_shape_ok(R, waves)) return 0;
    const void* f = pick_batch64b(R, waves);
    const int lds = (int)batch64b_lds_bytes(R, waves);
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 64 * waves, lds) != hipSuccess) return 0;
    return nb;
}

int jwdev_batch64b(const jw_batch_item* d_items, const jw_batch_unit* d_units, int nunits, int* d_counter, int R,
                   int waves, int grid, const jw_prologue_job* d_jobs, int keep, void* stream)
{
    if (!batch64b_shape_ok(R, waves) || grid < 1 || !d_jobs) {
        snprintf(g_err64, sizeof(g_err64), "bad build-in-LDS batch launch (R=%d, waves=%d)", R, waves);
        return -1;
    }
    const void* f = pick_batch64b(R, waves);
    const size_t lds = (size_t)batch64b_lds_bytes(R, waves);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {const_cast<jw_batch_item**>(&d_items), const_cast<jw_batch_unit**>(&d_units), &nunits,
                    &d_counter, const_cast<jw_prologue_job**>(&d_jobs), &keep};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * waves), args, lds, reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

static const void* pick_batch64d(int R)
{
    switch (R) {
    case 2: return reinterpret_cast<const void*>(&jw_batch64d_kernel<2>);
    case 4: return reinterpret_cast<const void*>(&jw_batch64d_kernel<4>);
    case 8: return reinterpret_cast<const void*>(&jw_batch64d_kernel<8>);
    case 16: return reinterpret_cast<const void*>(&jw_batch64d_kernel<16>);
    default: return nullptr;
    }
}

int jwdev_batch64d_occupancy(int R, int waves)
{
    const void* f = pick_batch64d(R);
    if (!f || waves < 1 || 64 * waves > kBatchDirectThreads) return 0;
    const int lds = JW_TAB64_ELEMS(R) * 8;
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 64 * waves, lds) != hipSuccess) return 0;
    return nb;
}

int jwdev_batch64d(const jw_batch_item* d_items, const jw_batch_unit* d_units, int nunits, int* d_counter, int R,
                   int waves, int grid, void* stream)
{
    const void* f = pick_batch64d(R);
    if (!f) { snprintf(g_err64, sizeof(g_err64), "no direct batch kernel for R=%d", R); return -1; }
    if (waves < 1 || 64 * waves > kBatchDirectThreads || grid < 1) {
        snprintf(g_err64, sizeof(g_err64), "bad direct batch launch");
        return -1;
    }
    const size_t lds = (size_t)JW_TAB64_ELEMS(R) * 8;
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {const_cast<jw_batch_item**>(&d_items), const_cast<jw_batch_unit**>(&d_units), &nunits,
                    &d_counter};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * waves), args, lds, reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

int jwdev_zero_counters(int* d_counters, int n, void* stream)
{
    if (n < 1 || n > 64) return -1;
    hipLaunchKernelGGL(jw_zero_counters_kernel, dim3(1), dim3(64), 0, reinterpret_cast<hipStream_t>(stream),
                       d_counters, n);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

/* batch queue with the compute / store split (R <= 16).  Compute wavefronts:
 * `ncomp` when 1 <= ncomp and the table plus their stagings fit in LDS with a
 * storer left over, else the default (12 for R <= 4, 8 for R = 8, 4 for
 * R = 16: the same number on every SIMD); storers fill the launch bound. */
int jwdev_batch64s_shape(int R, int ncomp, int* ncomp_out, int* nstore_out)
{
    if (!pick_batch64s(R)) return 0;
    const int nw = bsplit_threads_rt(R) / 64;
    const int64_t per = 2LL * 64 * R * 8;
    const int64_t avail = kLdsBytesMax - 512 - jwdev_table64_elems(R) * 8;
    int cmax = (int)(avail / per);
    if (cmax > nw - 1) cmax = nw - 1;
    const int cdef = R <= 4 ? 12 : (R == 8 ? 8 : 4);
    int c = ncomp >= 1 ? ncomp : cdef;
    if (c > cmax) c = cmax < cdef ? cmax : cdef;
    if (c < 1) return 0;
    *ncomp_out = c;
    *nstore_out = nw - c;
    return 1;
}

int64_t jwdev_batch64s_lds_bytes(int R, int ncomp)
{
    return jwdev_table64_elems(R) * 8 + 2LL * 64 * R * 8 * ncomp;
}

int jwdev_batch64s_occupancy(int R, int ncomp)
{
    int c = 0, st = 0;
    if (!jwdev_batch64s_shape(R, ncomp, &c, &st)) return 0;
    const void* f = pick_batch64s(R);
    const int lds = (int)jwdev_batch64s_lds_bytes(R, c);
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 64 * (c + st), lds) != hipSuccess) return 0;
    return nb;
}

int jwdev_batch64s(const jw_batch_item* d_items, const jw_batch_unit* d_units, int nunits, int* d_counter, int R,
                   int ncomp, int grid, int* d_err, int wait_polls, void* stream)
{
    int c = 0, st = 0;
    if (!jwdev_batch64s_shape(R, ncomp, &c, &st) || grid < 1) {
        snprintf(g_err64, sizeof(g_err64), "no split batch kernel for R=%d", R);
        return -1;
    }
    const void* f = pick_batch64s(R);
    const size_t lds = (size_t)jwdev_batch64s_lds_bytes(R, c);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {const_cast<jw_batch_item**>(&d_items), const_cast<jw_batch_unit**>(&d_units), &nunits,
                    &d_counter, &c, &d_err, &wait_polls};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * (c + st)), args, lds, reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

/* compute / store split kernel (R <= 8): shape, occupancy, launch */
int jwdev_main64s_shape(int R, int* ncomp, int* nstore)
{
    if (!pick_split(R, kAllThree, 2)) return 0;
    return split_shape(R, ncomp, nstore) ? 1 : 0;
}

int64_t jwdev_main64s_lds_bytes(int R, int ncomp)
{
    // output staging of the compute wavefronts, at least the table build's scratch,
    // and the block operators' row factors (in and out) of the fused form
    const int64_t staging = 2LL * 64 * R * 8 * ncomp;
    const int64_t scratch = (int64_t)prologue_lds_bytes(64 * R, 8);
    return jwdev_table64_elems(R) * 8 + max_i64(staging, scratch) + 2LL * 64 * R * 8;
}

int jwdev_main64s_occupancy(int R)
{
    int c = 0, st = 0;
    if (!jwdev_main64s_shape(R, &c, &st)) return 0;
    int best = -1;
    for (int v = 0; v < 9; v++) {
        const void* f = pick_split(R, v % 3, v / 3);
        if (!f) continue;
        const int nb = occupancy_of(f, 64 * (c + st), (int)jwdev_main64s_lds_bytes(R, c));
        if (best < 0 || nb < best) best = nb;
    }
    return best;
}

int jwdev_main64s(const jw_run_desc* r, const jw_source_desc* src, const void* matrices, int R, int grid, int* d_err,
                  void* stream)
{
    if (!r->rhs || !matrices || !d_err) {
        snprintf(g_err64, sizeof(g_err64), "main64s: no rhs, matrices or flag");
        return -1;
    }
    int c = 0, st = 0;
    if (!jwdev_main64s_shape(R, &c, &st)) { snprintf(g_err64, sizeof(g_err64), "no split kernel for R=%d", R); return -1; }
    const void* f = pick_split(R, solve_form(*r), (int)r->fused_io);
    if (!f) { snprintf(g_err64, sizeof(g_err64), "no split kernel for R=%d, I/O %d", R, (int)r->fused_io); return -1; }
    const size_t lds = (size_t)jwdev_main64s_lds_bytes(R, c);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return -2;
    void* args[] = {const_cast<jw_run_desc*>(r), &c, &d_err, const_cast<jw_source_desc*>(src), &matrices};
    e = hipLaunchKernel(f, dim3(grid), dim3(64 * (c + st)), args, lds, reinterpret_cast<hipStream_t>(stream));
    return e == hipSuccess ? 0 : -3;
}

/* Long FP64 systems (16-byte aligned) on the pair machinery: one workgroup of 12
 * wavefronts per CU (the chunk's table and a staging of 2 x 512 rows per wavefront) */
int64_t jwdev_long64_table_bytes(int64_t N)
{
    const int64_t nbuild = (N + (int64_t)kLong64Nsub * 64 * kLong64R - 1) / ((int64_t)kLong64Nsub * 64 * kLong64R);
    return nbuild * (kLong64Nsub * JW_TAB64_ELEMS(kLong64R) + kPivotLine) * 8;
}

int64_t jwdev_long64_lds_bytes(void)
{
    return (int64_t)JW_TAB64_ELEMS(kLong64R) * 8 + 2LL * 64 * kLong64R * 8 * kLong64Waves;
}

int jwdev_long64_occupancy(void)
{
    int best = -1;
    for (int m = JW_LONG_REDUCE; m <= JW_LONG_FINISH + 1; m++) {
        for (int v = 0; v < 2; v++) {
            const void* f = m <= JW_LONG_FINISH ? pick_long64(m, v == 0) : pick_long64_front(v == 0);
            const int lds = (int)jwdev_long64_lds_bytes();
            if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 0;
            int nb = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 64 * kLong64Waves, lds) != hipSuccess) return 0;
            if (best < 0 || nb < best) best = nb;
        }
    }
    return best < 0 ? 0 : best;
}

/* the front of a step (jw_long64_front_kernel): the table builds of every chunk, COEF and
 * REDUCE of the slice in d (its first systems) in one launch, after a fill kernel that
 * zeroes the 32 + nbuild ints of sync and empties the builds' pivot lines behind the tables */
int jwdev_long64_front(const jw_source_desc* src, const void* matrices, const jw_long_desc* d, int* sync, int* err,
                       int cu_count, int occupancy, void* stream)
{
    const int C = 64 * kLong64R;
    const int64_t SR = (int64_t)kLong64Nsub * C;
    if (!matrices || !d->table || !d->red || !d->run.rhs || !sync || !err) {
        jwdev_set_error("long64 front: no matrices, table, reduced data, rhs or hand-over scratch");
        return -1;
    }
    const int64_t nbuild = (src->N + SR - 1) / SR;
    if (src->N < 1 || nbuild > (1 << 20) || d->nchunks < 1 || (int64_t)d->nchunks * C < d->run.N ||
        d->nchunks > nbuild * kLong64Nsub || d->tab_elems != JW_TAB64_ELEMS(kLong64R) || cu_count < 1 ||
        occupancy < 1 || d->run.nsys < 1 || d->run.nsys > d->red_sys) {
        jwdev_set_error("long64 front: bad size, chunk count, table size, slice or grid");
        return -1;
    }
    if (((uintptr_t)d->run.rhs % 16) != 0 || (d->run.stride % 2) != 0 || (d->run.offSol % 2) != 0) {
        jwdev_set_error("long64 front: systems not 16-byte aligned");
        return -1;
    }
    const int64_t ppc = (d->run.nsys + 1) / 2;
    /* pairs per unit: about two units a worker, in whole rounds of its wavefronts, since a unit
     * of another chunk costs a table copy (512 systems of 100000 rows, units of 24 pairs: 330
     * us, two units a worker: 320; one: 338, for the workers that get a second) */
    const int64_t workers = (int64_t)cu_count * occupancy;
    int64_t P = ((int64_t)d->nchunks * ppc + kLong64UnitsPerWorker * workers - 1) / (kLong64UnitsPerWorker * workers);
    P = (P + kLong64Waves - 1) / kLong64Waves * kLong64Waves;
    if (P < kLong64PairsPerUnit) P = kLong64PairsPerUnit;
    if (P > ppc) P = ppc;
    const int64_t units = (int64_t)d->nchunks * (1 + (ppc + P - 1) / P);
    if (units > (1LL << 30)) {
        jwdev_set_error("long64 front: too many work units");
        return -1;
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int nclear = (int)(kLong64Tflags + nbuild);
    unsigned long long* lines = reinterpret_cast<unsigned long long*>(
        reinterpret_cast<double*>(const_cast<void*>(d->table)) + nbuild * kLong64Nsub * JW_TAB64_ELEMS(kLong64R));
    const int nwords = (int)nbuild * kPivotLine;
    hipLaunchKernelGGL(jw_long64_clear_kernel, dim3((unsigned)((nwords + 32 + 255) / 256)), dim3(256), 0, s, sync,
                       nclear, lines, nwords);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        jwdev_set_error("long64 front: clear launch failed");
        return -3;
    }
    const void* f = pick_long64_front(d->run.fwd && d->run.b1 && d->run.b2);
    const size_t lds = (size_t)jwdev_long64_lds_bytes();
    if (prologue_lds_bytes((int)SR, sizeof(double)) + 3 * sizeof(double) > lds) {
        jwdev_set_error("long64 front: table build does not fit");
        return -1;
    }
    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
        jwdev_set_error("long64 front: hipFuncSetAttribute failed");
        return -2;
    }
    /* every build's workgroup, then a full GPU of workers */
    const int64_t grid = nbuild + (int64_t)cu_count * occupancy;
    jw_source_desc sd = *src;
    const void* mat = matrices;
    jw_long_desc dd = *d;
    int nb = (int)nbuild;
    int chained = src->solve_kind == JW_SOLVE_TRI, pu = (int)P;
    void* args[] = {&sd, (void*)&mat, &dd, &sync, &lines, &err, &nb, &chained, &pu};
    e = hipLaunchKernel(f, dim3((unsigned)grid), dim3(64 * kLong64Waves), args, lds, s);
    if (e != hipSuccess) {
        jwdev_set_error("long64 front: launch failed");
        return -3;
    }
    return 0;
}

int jwdev_long64(const jw_long_desc* d, int cu_count, int occupancy, void* stream)
{
    const int C = 64 * kLong64R;
    if (!d->table || !d->red || !d->run.rhs) {
        jwdev_set_error("long64: no table, reduced data or rhs");
        return -1;
    }
    if ((d->mode != JW_LONG_REDUCE && d->mode != JW_LONG_FINISH) || d->nchunks < 1 ||
        (int64_t)d->nchunks * C < d->run.N || d->tab_elems != JW_TAB64_ELEMS(kLong64R) || cu_count < 1 ||
        occupancy < 1) {
        jwdev_set_error("long64: bad mode, chunk count, table size or grid");
        return -1;
    }
    if (d->run.nsys > d->red_sys) {
        jwdev_set_error("long64: slice exceeds reduced data");
        return -1;
    }
    /* the DMA moves 16-byte row pairs: aligned systems only */
    if (((uintptr_t)d->run.rhs % 16) != 0 || (d->run.stride % 2) != 0 || (d->run.offSol % 2) != 0) {
        jwdev_set_error("long64: systems not 16-byte aligned");
        return -1;
    }
    const int64_t nsys = d->run.nsys;
    if (nsys < 1) return 0;
    const int64_t total = (int64_t)d->nchunks * ((nsys + 1) / 2);
    int64_t grid = (int64_t)cu_count * occupancy;
    const int64_t need = (total + kLong64Waves - 1) / kLong64Waves;
    if (grid > need) grid = need;
    if (grid < 1) grid = 1;
    int64_t per_wg = (total + grid - 1) / grid;
    grid = (total + per_wg - 1) / per_wg;
    const void* f = pick_long64(d->mode, d->run.fwd && d->run.b1 && d->run.b2);
    const size_t lds = (size_t)jwdev_long64_lds_bytes();
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
        jwdev_set_error("long64: hipFuncSetAttribute failed");
        return -2;
    }
    void* args[] = {const_cast<jw_long_desc*>(d), &per_wg};
    e = hipLaunchKernel(f, dim3((unsigned)grid), dim3(64 * kLong64Waves), args, lds,
                        reinterpret_cast<hipStream_t>(stream));
    if (e != hipSuccess) {
        jwdev_set_error("long64: launch failed");
        return -3;
    }
    return 0;
}

}  // extern "C"
