// tcw_map.hip -- transient-CW F-statistic maps on MI355X (gfx950).
//
// Device path for one or many templates:
//   1. stage_kernel    binned detector merge (lalpulsar mergeMultiFstatAtomsBinned,
//                      called at pyfstat/tcw_fstat_map_funcs.py:706) fused with an
//                      FP64 prefix scan of the float32 merged bins (rect windows);
//                      stage_exp_kernel: the same merge into a float32 atom table
//                      (exp windows);
//   2. map kernels     window sums -> cond-guarded F per (t0, tau) cell, with the
//                      max/argmax, logsumexp and row/column posterior sums fused
//                      into the producer (pyfstat/tcw_fstat_map_funcs.py:809-828);
//   3. finalize_kernel per-template combination of the partials into FstatMap
//                      fields (maxF, t0_ML, tau_ML, lnBtSG, t0_MP, tau_MP).
// Host side: the C ABI declared in include/tcw_hip.h.
//
// Index maths and window semantics follow the reference kernels
// pyfstat/pyCUDAkernels/cudaTransientFstatRectWindow.cu:21-124 and
// pyfstat/pyCUDAkernels/cudaTransientFstatExpWindow.cu:27-134 (uint32
// wrap-around, clamping, incremental rect sums, cond < 1e4 guard, F = 2
// fallback); the arithmetic is new (prefix differences, FP64 determinant).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "tcw_common.h"
#include "tcw_hip.h"
#include "tcw_step.h"

// Device memory of tcw_map_noalloc: the single-map plan's buffers (descriptors,
// prefix or atom tables, reduction partials) are carved out of this array, so
// that call allocates nothing.  Each device holds its own copy from module
// load until the process ends; host code never uses this name as an address
// (it is a host-side stand-in there), only the pointer hipGetSymbolAddress
// returns for the current device (noalloc_scratch_ptr below).
static __device__ __align__(256) unsigned char scratch[TCW_NOALLOC_SCRATCH_BYTES];

namespace {

// ----------------------------------------------------------------------------
// constants and device-side descriptors
// ----------------------------------------------------------------------------

constexpr int NC = TCW_NCOL;
constexpr int WG = 256;           // threads per workgroup (4 wave64)
constexpr int TILE_COLS = 256;    // tau columns per work item (rect_step_kernel: 256, 128 or
                                  // 64; exp_walk_kernel: 64)
constexpr int MERGED_STRIDE = 8;  // floats per atom in the atom table (7 columns + kind)
// the kind column: 0 for a bin of zeros, 1 for one with data, BIN_ODD for one
// with an infinity or NaN (more than any count of bins with data)
constexpr float BIN_ODD = 2147483648.0f;
constexpr double COND_MAX = 1e4;  // rect.cu:104
// cond < K  <=>  T^2 < Q*D  with T = A+B, D = AB-C^2 > 0, Q = (K+1)^2/K, because
// cond = (T+s)/(T-s), s^2 = T^2-4D, and (1+cond)^2/cond = T^2/D grows with cond.
constexpr double QCOND = (COND_MAX + 1.0) * (COND_MAX + 1.0) / COND_MAX;

enum Mode : int32_t {
    MODE_RECT_FAST = 0,     // regular grid: dt0 == dtau == a*TAtom, no wrap-around
    MODE_RECT_GENERIC = 1,  // any rectangular window range, exact uint32 semantics
    MODE_EXP_DIRECT = 2,    // exponential window, direct weighted sum (any grid)
    MODE_EXP_FAST = 3,      // exponential window on the atom grid: recurrence in t0
    MODE_COUNT = 4
};

// Rows per work item when not tuned.  rect_fast: 192 (1024 templates of 250 to
// 2000 rows and columns: maps 1880 us; 128 rows 1955, 256 rows 1915).
constexpr int RB_DEFAULT[MODE_COUNT] = {192, 16, 16, 128};
// Rect items aimed at when rows are not tuned: eight a CU, since five fit a CU
// at a time (256 templates of 48 x 48 to 240 x 240: maps 22 us, 26 at 1024
// items, 29 at 512; 1024 templates of 125 x 125: 35 us, 37 at 1024, 38 at 4096).
constexpr int64_t SMALL_BATCH_ITEMS = 2048;
// exp_walk_kernel items aimed at when rows are not tuned: one a CU; fewer rows
// repeat the direct sum, more leave CUs idle.  Rows by 32, so that eight waves
// get four each at least.  Measured (maps, us, at 32 | 64 | 128 | 256 rows):
// 32 templates of 125 x 125 cells 30 | 37 | 47 | 47; 4 of 500 x 500 89 | 63 | 74 |
// 132; 64 of 500 x 500 1004 | 583 | 373 | 352.
constexpr int64_t WALK_ITEMS = 256;
constexpr int WALK_MAX_ROWS = 256;
// Exp rows on the atom grid when untuned and under DIRECT_INIT_MIN_BLOCKS column
// blocks: about EXP_SMALL_CHUNKS chunks over all columns, those above the map
// included (they are walked too): shorter ones leave more to the scan and to
// finalize, longer ones leave CUs idle.  Measured (pass, us, at 16 | 32 | 64 |
// 128 | 256 rows): one map of 2000 x 2000 cells 137 | 100 | 82 | 84 | 124; one of
// 150 x 150 39 | 43 | 51 | 69 | 84; 8 of 300 x 150 46 | 45 | 54 | 71 | 113; 128 of
// 300 x 150 172 | 124 | 116 | 107 | 123; 32 of 1000 x 1000 876 | 542 | 411 | 363 |
// 354.
constexpr int64_t EXP_SMALL_CHUNKS = 512;
constexpr int EXP_SMALL_MIN_ROWS = 16, EXP_SMALL_MAX_ROWS = 256;
// Rows of the layout that bounds tcw_map_noalloc's maps (tcw_plan::compact):
// rect items of 16 to 128 rows, about 512 of them, exp chunks of 64 under
// DIRECT_INIT_MIN_BLOCKS column blocks.
constexpr int COMPACT_RECT_ROWS = 128, COMPACT_EXP_ROWS = 64;
constexpr int64_t COMPACT_RECT_ITEMS = 512;

struct TmplDev {
    int64_t seg_begin, seg_end;  // detector segments of this template
    int64_t merged_off;          // floats, atom table [bins][8]      (exp modes)
    int64_t prefix_off;          // doubles, prefix entries [N+1][7]  (rect modes)
    int64_t F_off;               // floats, map [N_t0][N_tau]
    int64_t item_begin;          // first work item of this template
    int64_t rowpart_off;         // float, [n_colblk][N_t0], relative to the item max
    int64_t colpart_off;         // float, [n_rowblk][N_tau], relative to the item max
    uint32_t N, TAtom, t_min;    // binned atoms, atom length, t0_data
    uint32_t TA_rcp;             // floor((2^32 - 1) / TAtom), for div_TA
    uint32_t type, t0, dt0, tau, dtau;  // effective window (after NONE -> RECT)
    uint32_t N_t0, N_tau;
    uint32_t n_rowblk, n_colblk;
    int32_t mode;
    int32_t rb_rows;             // rows per work item
    int32_t tile;                // columns per work item
    int32_t q0, q00, a;          // MODE_RECT_FAST index maths; a also MODE_EXP_FAST
    int32_t k00, L0, Ls, H;      // MODE_EXP_FAST: first start atom, window lengths
                                 // L(n) = L0 + Ls*n atoms, atoms [0, H) reachable
    int32_t n_seg;               // MODE_EXP_FAST: row chunks (>= n_rowblk)
    int32_t init_empty;          // MODE_EXP_FAST: the top chunk's direct sum is empty
    int32_t walk;                // MODE_EXP_DIRECT, MODE_RECT_GENERIC: exp_walk_kernel's or
                                 // rect_step_kernel's, not the generic kernel's
    int64_t etab_off;            // MODE_EXP_FAST: doubles, [n_seg + INIT_PARTS][7][N_tau]
    uint32_t o_t0, o_t0Band, o_tau, o_tauBand;  // caller's window (posterior modes)
};

// Per-template flags: set by the stage kernels, FLAG_SINGLE_ATOM raised by the
// strict map kernels.
constexpr int FLAG_SINGLE_ATOM = 1;  // a window spans a single atom
// a merged bin has a negative or NaN a^2 or b^2, or a non-finite ab: window
// traces need not grow with the window, nor determinants be numbers
constexpr int FLAG_NO_BOUND = 2;

struct SegDev {
    int64_t begin, end;
};

// the Python binding (pyfstat_amd/_hiplib.py) mirrors these layouts
static_assert(sizeof(tcw_stats) == 104, "tcw_stats layout");
static_assert(sizeof(tcw_atoms) == 128, "tcw_atoms layout");
static_assert(sizeof(tcw_window) == 28, "tcw_window layout");

struct ItemDev {
    int32_t t, rb, cb, pad;
};

struct ItemPart {
    float maxF;
    int32_t idx;
    float M, S;  // M = the item's max F times LOG2E (float); S = sum of exp(F - M/LOG2E)
};

// ----------------------------------------------------------------------------
// stage: binned merge + FP64 prefix (rect) / float32 atom table (exp)
// ----------------------------------------------------------------------------

constexpr int SR_BINS = 4;           // consecutive bins per thread per round
constexpr int SR_PASS_LANES = 32;    // lanes per output pass
constexpr int SR_PASS = SR_PASS_LANES * SR_BINS * NC;  // doubles per wave and output pass
// Threads of a template's workgroup: one round for the shorter templates
// (128: N <= 512, 256: N <= 1024).  Longer ones take several rounds of 256
// threads, or, if they are few, of 1024: a CU holds one such workgroup, whose
// waves share the template's rounds, but all of them wait for each other at
// every barrier.  Measured (before timestamps were loaded ahead, which takes 3 to
// 10 us off either), N = 1000..4000 and 1000..8000, 256 | 1024 threads:
// 128 templates 57 | 40 us, 288 62 | 45, 512 105 | 92, 768 122 | 124, 1024
// 133 | 154; the line lies where the two meet.
constexpr int SR_CLASSES = 3;
constexpr int SR_THREADS[SR_CLASSES] = {128, 256, 256};
constexpr int SR_WIDE_THREADS = 1024;
constexpr int64_t SR_WIDE_TMPLS = 640;
static_assert(SR_THREADS[2] == SR_THREADS[1], "one kernel");
constexpr int stage_class(uint32_t N) {
    return N <= SR_THREADS[0] * SR_BINS ? 0 : N <= SR_THREADS[1] * SR_BINS ? 1 : 2;
}

// DPP controls of a wave scan: shifts within the 16-lane rows, and the last
// lane of a row (of the lower half) to the next row (the upper half)
constexpr int DPP_ROW_SHR = 0x110;
constexpr int DPP_ROW_BCAST15 = 0x142;
constexpr int DPP_ROW_BCAST31 = 0x143;

// the DPP source's value, 0.0 on lanes without one or in rows outside ROWS
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_d(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, ROWS, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// inclusive scan over the 64 lanes, in log depth, without LDS
__device__ __forceinline__ double wave_scan(double x) {
    x += dpp_d<DPP_ROW_SHR + 1>(x);
    x += dpp_d<DPP_ROW_SHR + 2>(x);
    x += dpp_d<DPP_ROW_SHR + 4>(x);
    x += dpp_d<DPP_ROW_SHR + 8>(x);
    x += dpp_d<DPP_ROW_BCAST15, 0xa>(x);
    return x + dpp_d<DPP_ROW_BCAST31, 0xc>(x);
}

// x / TAtom and x % TAtom: the product with the reciprocal is at most one short
__device__ __forceinline__ uint32_t div_TA(uint32_t x, const TmplDev &td, uint32_t &rem) {
    uint32_t q = __umulhi(x, td.TA_rcp);
    rem = x - q * td.TAtom;
    const bool more = rem >= td.TAtom;
    rem -= more ? td.TAtom : 0;
    return q + more;
}

typedef double d2 __attribute__((ext_vector_type(2)));
typedef d2 d2_u __attribute__((aligned(8)));  // the table starts at any double

// Rectangular-window templates: the exclusive prefix P[b] = sum of merged
// bins < b per column, [N+1][7] doubles.  One workgroup of NT threads per
// template, rounds of 4 NT bins, 4 consecutive bins per thread.
//  - merge: per detector, the bins of up to 4 NT timestamps are formed
//    (coalesced loads), and the first atom of every bin is marked where the bin
//    changes; each thread then reads its bins' atoms from the columns.  A
//    bin's merged value is the float32 sum over detectors X = 0,1,... (in that
//    order) of the detector's atoms in the bin (in atom order), from 0 -- the
//    additions of lalpulsar's binned merge, in its order, so merged atoms are
//    bit-identical;
//  - scan (FP64): thread totals, a scan within the wave in log depth, the wave
//    totals and the carry of earlier rounds in LDS.  A prefix value carries
//    ~20 roundings of 2^-53 relative to the largest partial sum;
//  - output: the LDS buffer is reused to transpose the prefix values, 32 lanes
//    of each wave per pass, so every global store is a contiguous run of the
//    [N+1][7] table (a thread's own 4 bins span 224 bytes).
// Bound: the waves' own instructions (about 1100 a round, half of them the
// output passes) on the few CUs that a batch of long templates fills, with the
// round's chain (two dependent loads, the barriers, the scan) exposed; stores
// and loads left out save 1 and 9 of 40 us.  The binary searches of a thread's
// first bins, a scan through LDS and 8-byte LDS words took: 1024 templates of
// N = 1000..8000 147 us, 128 of N = 1000..4000 and two detectors 49, 1024 of 500
// and two detectors 23.4; without them 136, 40 and 20.6; with the next
// detector's timestamps loaded ahead and the segments read once 125, 37 and 18.6
// (ahead across rounds too: the same).
template <int NT>
__global__ __launch_bounds__(NT) void stage_kernel(
    const TmplDev *__restrict__ tds, const int32_t *__restrict__ tmpls,
    const SegDev *__restrict__ segs, const uint32_t *__restrict__ ts,
    const float *__restrict__ cols, int64_t cstride, double *__restrict__ prefix,
    int *__restrict__ flags) {
    constexpr int NW = NT / 64;
    constexpr int ROUND = NT * SR_BINS;
    // per chunk of ROUND atoms: their bins, and the bins' first atoms; then the
    // output passes' transpose buffers
    __shared__ __align__(16) double s_buf[NW * SR_PASS];
    static_assert(NW * SR_PASS * 2 >= 2 * ROUND, "bins and first atoms share the buffer");
    int *s_bin = reinterpret_cast<int *>(s_buf);
    int *s_first = s_bin + ROUND;
    __shared__ double s_tot[NW][NC + 1];  // wave totals
    // a detector's first atom not yet merged, and its end
    __shared__ int64_t s_cur[TCW_MAX_DETECTORS], s_end[TCW_MAX_DETECTORS];
    __shared__ int s_cnt, s_flag;

    const int t = tmpls[blockIdx.x];
    const TmplDev td = tds[t];
    const int N = (int)td.N;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nseg = (int)(td.seg_end - td.seg_begin);
    double *__restrict__ P = prefix + td.prefix_off;
    if (tid == 0) s_flag = 0;
    if (tid < nseg) {
        const SegDev sg = segs[td.seg_begin + tid];
        s_cur[tid] = sg.begin;
        s_end[tid] = sg.end;
    }
    double carry[NC];  // sum of all earlier rounds
#pragma unroll
    for (int c = 0; c < NC; c++) carry[c] = 0.0;
    __syncthreads();

    for (int base = 0; base < N; base += ROUND) {
        const int nb = min(ROUND, N - base);  // bins of this round
        float v[SR_BINS][NC];
#pragma unroll
        for (int j = 0; j < SR_BINS; j++)
#pragma unroll
            for (int c = 0; c < NC; c++) v[j][c] = 0.0f;
        // a chunk's timestamps; the first chunk's of the next detector are loaded
        // while this one is merged
        uint32_t tx[SR_BINS];
        auto fetch = [&](int64_t c0, int64_t seg_end) {
#pragma unroll
            for (int u = 0; u < SR_BINS; u++) {
                const int64_t i = c0 + u * NT + tid;
                tx[u] = i < seg_end ? ts[i] : 0;
            }
        };
        fetch(s_cur[0], s_end[0]);
        for (int X = 0; X < nseg; X++) {
            const int64_t seg_end = s_end[X];
            int64_t c0 = s_cur[X];
            bool have = true;  // tx holds the chunk at c0 (block-uniform)
            while (c0 < seg_end) {  // block-uniform
                const int na = (int)min((int64_t)ROUND, seg_end - c0);
                if (!have) fetch(c0, seg_end);
                int bin[SR_BINS];
#pragma unroll
                for (int u = 0; u < SR_BINS; u++) {
                    const int i = u * NT + tid;
                    const uint32_t x = tx[u];
                    uint32_t rem;
                    // -1: before the first bin (in none); nb: in a later round
                    const int b = (int)min(div_TA(x - td.t_min, td, rem), 0x7fffffffu) - base;
                    bin[u] = i >= na ? nb : x < td.t_min ? -1 : min(b, nb);
                    s_bin[i] = bin[u];
                    s_first[i] = -1;
                }
                if (tid == 0) s_cnt = na;
                have = false;
                if (X + 1 < nseg) fetch(s_cur[X + 1], s_end[X + 1]);
                __syncthreads();
#pragma unroll
                for (int u = 0; u < SR_BINS; u++) {
                    const int i = u * NT + tid;
                    const int before = i > 0 ? s_bin[i - 1] : -1;
                    if (bin[u] != before || i == 0) {
                        if (bin[u] >= 0 && bin[u] < nb) s_first[bin[u]] = i;
                        if (bin[u] == nb && i < na) s_cnt = i;
                    }
                }
                __syncthreads();
                const int cnt = s_cnt;
                int k[SR_BINS];
                const float *__restrict__ col = cols + c0;
                // (a 32-bit offset from a uniform address: no 64-bit sums)
                auto at = [&](int c, int k) {
                    return *reinterpret_cast<const float *>(
                        reinterpret_cast<const char *>(col + c * cstride) + (uint32_t)k * 4u);
                };
#pragma unroll
                for (int j = 0; j < SR_BINS; j++) k[j] = s_first[tid * SR_BINS + j];
                float y[SR_BINS][NC];  // the bins' first atoms, all loads in flight
#pragma unroll
                for (int j = 0; j < SR_BINS; j++)
#pragma unroll
                    for (int c = 0; c < NC; c++) y[j][c] = at(c, max(k[j], 0));
#pragma unroll
                for (int j = 0; j < SR_BINS; j++) {
                    if (k[j] < 0) continue;
#pragma unroll
                    for (int c = 0; c < NC; c++) v[j][c] += y[j][c];
                    for (int q = k[j] + 1; q < cnt && s_bin[q] == tid * SR_BINS + j; q++) {
#pragma unroll
                        for (int c = 0; c < NC; c++) v[j][c] += at(c, q);
                    }
                }
                __syncthreads();  // bins consumed before the next chunk
                c0 += cnt;
                if (cnt < na) break;
            }
            if (have && X + 1 < nseg) fetch(s_cur[X + 1], s_end[X + 1]);  // none of X's left
            if (tid == 0) s_cur[X] = c0;  // read again after the next round's barriers
        }
        bool odd = false;  // what FLAG_NO_BOUND is for (NaN compares false)
#pragma unroll
        for (int j = 0; j < SR_BINS; j++)
            odd |= !(v[j][0] >= 0.0f) | !(v[j][1] >= 0.0f) | !(fabsf(v[j][2]) < INFINITY);
        if (odd) s_flag = FLAG_NO_BOUND;
        // inclusive scan of the thread totals within the wave (bins >= N hold 0)
        double ex[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            double sum = 0.0;
#pragma unroll
            for (int j = 0; j < SR_BINS; j++) sum += (double)v[j][c];
            const double x = wave_scan(sum);
            if (lane == 63) s_tot[wave][c] = x;
            ex[c] = __shfl_up(x, 1);
            if (lane == 0) ex[c] = 0.0;
        }
        __syncthreads();
        // exclusive prefix at the thread's first bin: the carry, the earlier
        // waves' totals in order, the earlier lanes
#pragma unroll 4
        for (int w = 0; w < wave; w++)
#pragma unroll
            for (int c = 0; c < NC; c++) carry[c] += s_tot[w][c];
#pragma unroll
        for (int c = 0; c < NC; c++) ex[c] += carry[c];
#pragma unroll 4
        for (int w = wave; w < NW; w++)
#pragma unroll
            for (int c = 0; c < NC; c++) carry[c] += s_tot[w][c];
        // the thread's 4 bins are 28 consecutive doubles of the table: through
        // LDS in 16-byte words, so that a store covers 1 KB of it in one run
        d2 *out = reinterpret_cast<d2 *>(s_buf + wave * SR_PASS);
#pragma unroll 1
        for (int pass = 0; pass < 64 / SR_PASS_LANES; pass++) {
            const int wb = wave * (64 * SR_BINS) + pass * (SR_PASS_LANES * SR_BINS);
            const int cnt = min(SR_PASS_LANES * SR_BINS, nb - wb) * NC;
            if (cnt <= 0) break;  // wave-uniform
            if (lane / SR_PASS_LANES == pass) {
                double r[SR_BINS * NC];
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    r[c] = ex[c];
#pragma unroll
                    for (int j = 1; j < SR_BINS; j++)
                        r[j * NC + c] = r[(j - 1) * NC + c] + (double)v[j - 1][c];
                }
                d2 *row = out + (lane % SR_PASS_LANES) * (SR_BINS * NC / 2);
#pragma unroll
                for (int q = 0; q < SR_BINS * NC / 2; q++) row[q] = d2{r[2 * q], r[2 * q + 1]};
            }
            // the buffer is the wave's own: order its LDS accesses, no barrier
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            double *dst = P + (int64_t)(base + wb) * NC;
#pragma unroll
            for (int q = 0; q < SR_PASS / 2; q += 64) {
                const int i = q + lane;
                if (2 * i + 1 < cnt)
                    *reinterpret_cast<d2_u *>(dst + 2 * i) = out[i];
                else if (2 * i < cnt)
                    dst[2 * i] = out[i][0];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();  // the buffer holds bins again in the next round
    }
    if (tid == 0) {
#pragma unroll
        for (int c = 0; c < NC; c++) P[(int64_t)N * NC + c] = carry[c];
        flags[t] = s_flag;
    }
}

// Bins of a template's atom table: the recurrence path reads none at or
// past H (the first atom no window reaches), the direct path any of the N.
__host__ __device__ __forceinline__ uint32_t exp_table_bins(const TmplDev &td) {
    return td.mode == MODE_EXP_FAST ? (uint32_t)td.H : td.N;
}

// Exponential-window templates: the merged atoms as the float32 table
// [exp_table_bins][8] (7 columns + padding), the same float32 detector-order
// sums as stage_kernel (the kernels that read it widen them to FP64, exactly).
// A workgroup owns 256 * SXB consecutive bins of one template: per detector,
// the block's atoms are bounded (bound_two: 9.9 us for 32 templates of 1000 bins
// with a block-wide search per detector, now 8.2) and copied into LDS in chunks with coalesced loads; each thread then sums its SXB bins
// from LDS (atoms in order, detectors in order).  Grid: (bin blocks, exp
// templates), y-strided.  SXB = 4 (1024-bin blocks) for batches, 1 (256-bin
// blocks) when 1024-bin blocks would give fewer than SX_NARROW_BELOW
// workgroups (one large map would otherwise occupy a handful of CUs).
constexpr int SX_NARROW_BELOW = 256;
constexpr int SX_CHUNK = 1024;  // atoms staged per pass
// the finished rows are restaged in LDS (row stride SX_ROW floats, odd so the
// lanes' writes spread over the banks) and written to the table with
// consecutive lanes on consecutive floats
constexpr int SX_ROW = MERGED_STRIDE + 1;

// For sorted ts[lo, hi): the first index with ts >= key (hi if none), by one
// wave: a round samples 64 evenly spaced timestamps (one load a lane) and keeps
// the gap where the key falls, so n atoms take about log_64(n) loads in turn.
__device__ __forceinline__ int64_t wave_lower_bound(const uint32_t *__restrict__ ts, int64_t lo,
                                                    int64_t hi, uint64_t key, int lane) {
    while (hi > lo) {
        const int64_t n = hi - lo;
        const int64_t sd = n <= 64 ? 1 : (n + 63) / 64;
        const bool pred = lane * sd < n && (uint64_t)ts[lo + lane * sd] < key;
        const int64_t c = __popcll(__ballot(pred));  // samples below the key
        if (c == 0) return lo;
        hi = min(lo + c * sd, hi);  // the answer is in (sample c-1, sample c]
        lo += (c - 1) * sd + 1;
    }
    return lo;
}

// The first atoms with ts >= key0 and >= key1 of detector segments s and s + 1
// (if below s_end) into r[0], r[1] and r[2], r[3]: each wave of a 256-thread
// block searches one of the four.  The caller synchronises before the next call.
__device__ __forceinline__ void bound_two(const uint32_t *__restrict__ ts,
                                          const SegDev *__restrict__ segs, int64_t s,
                                          int64_t s_end, uint64_t key0, uint64_t key1,
                                          int64_t (&r)[4]) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (s + (wave >> 1) < s_end) {
        const SegDev sg = segs[s + (wave >> 1)];
        const int lane = threadIdx.x & 63;
        const int64_t k = wave_lower_bound(ts, sg.begin, sg.end, wave & 1 ? key1 : key0, lane);
        if (lane == 0) r[wave] = k;
    }
    __syncthreads();
}

template <int SXB>
__global__ __launch_bounds__(256) void stage_exp_kernel(
    const TmplDev *__restrict__ tds, const int32_t *__restrict__ exp_tmpls, int64_t n_exp,
    const SegDev *__restrict__ segs, const uint32_t *__restrict__ ts,
    const float *__restrict__ cols, int64_t cstride, float *__restrict__ merged,
    int *__restrict__ flags) {
    // atom staging during the merge, the finished rows afterwards
    constexpr int SX_RAW = (NC + 1) * SX_CHUNK > 256 * SXB * SX_ROW ? (NC + 1) * SX_CHUNK
                                                                     : 256 * SXB * SX_ROW;
    __shared__ float s_raw[SX_RAW];
    uint32_t *s_ts = reinterpret_cast<uint32_t *>(s_raw);
    float(*s_x)[SX_CHUNK] = reinterpret_cast<float(*)[SX_CHUNK]>(s_raw + SX_CHUNK);
    __shared__ int64_t s_rng[4];
    const int tid = threadIdx.x;
    for (int64_t e = blockIdx.y; e < n_exp; e += gridDim.y) {
        // before any map kernel: clear the template's single-atom flag
        if (blockIdx.x == 0 && tid == 0) flags[exp_tmpls[e]] = 0;
        const TmplDev td = tds[exp_tmpls[e]];
        constexpr int SX_BINS = SXB;
        constexpr int SX_BINS_BLOCK = 256 * SXB;
        const uint32_t B0 = blockIdx.x * (uint32_t)SX_BINS_BLOCK;
        const uint32_t NB = exp_table_bins(td);
        if (B0 >= NB) continue;  // block-uniform
        const uint32_t B1 = min(NB, B0 + (uint32_t)SX_BINS_BLOCK);
        const uint64_t TA = td.TAtom;
        const uint64_t tb_lo = (uint64_t)td.t_min + (uint64_t)B0 * TA;
        const uint64_t tb_hi = (uint64_t)td.t_min + (uint64_t)B1 * TA;
        const uint32_t b0 = B0 + (uint32_t)tid * SX_BINS;  // this thread's first bin
        float v[SX_BINS][NC];
#pragma unroll
        for (int j = 0; j < SX_BINS; j++)
#pragma unroll
            for (int c = 0; c < NC; c++) v[j][c] = 0.0f;
        for (int64_t X = td.seg_begin; X < td.seg_end; X++) {
            const int two = (int)(X - td.seg_begin) & 1;  // bounded two at a time
            if (two == 0) bound_two(ts, segs, X, td.seg_end, tb_lo, tb_hi, s_rng);
            const int64_t ka = s_rng[2 * two], kb = s_rng[2 * two + 1];
            __syncthreads();  // s_rng is rewritten for the next two
            for (int64_t c0 = ka; c0 < kb; c0 += SX_CHUNK) {
                const int na = (int)min((int64_t)SX_CHUNK, kb - c0);
                for (int i = tid; i < na; i += 256) {
                    s_ts[i] = ts[c0 + i];
#pragma unroll
                    for (int c = 0; c < NC; c++) s_x[c][i] = cols[c * cstride + c0 + i];
                }
                __syncthreads();
                if (b0 < B1) {
                    const uint64_t t_lo = (uint64_t)td.t_min + (uint64_t)b0 * TA;
                    int lo = 0, hi = na;  // first staged atom with ts >= t_lo
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if ((uint64_t)s_ts[mid] < t_lo)
                            lo = mid + 1;
                        else
                            hi = mid;
                    }
                    int k = lo;
#pragma unroll
                    for (int j = 0; j < SX_BINS; j++) {
                        const uint64_t t_hi = t_lo + (uint64_t)(j + 1) * TA;
                        for (; k < na && (uint64_t)s_ts[k] < t_hi; k++) {
#pragma unroll
                            for (int c = 0; c < NC; c++) v[j][c] += s_x[c][k];
                        }
                    }
                }
                __syncthreads();
            }
        }
        // the last staging pass ended with a barrier: s_raw is free
#pragma unroll
        for (int j = 0; j < SX_BINS; j++) {
            float *r = s_raw + (tid * SX_BINS + j) * SX_ROW;
            bool some = false, odd = false;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                r[c] = v[j][c];
                some |= v[j][c] != 0.0f;
                odd |= !(fabsf(v[j][c]) < INFINITY);
            }
            r[NC] = odd ? BIN_ODD : some ? 1.0f : 0.0f;
        }
        __syncthreads();
        float *base = merged + td.merged_off + (int64_t)B0 * MERGED_STRIDE;
        const int nq = (int)(B1 - B0) * MERGED_STRIDE;
        for (int q = tid; q < nq; q += 256)
            base[q] = s_raw[(q / MERGED_STRIDE) * SX_ROW + q % MERGED_STRIDE];
        __syncthreads();  // s_raw is staged again for the next template
    }
}

// ----------------------------------------------------------------------------
// per-cell F
// ----------------------------------------------------------------------------

// F from window sums: determinant, numerator and condition guard in FP64
// (rect.cu:98-118 / exp.cu:109-129; F = 2 when the guard fails); the final
// quotient in float32 (the stored map is float32).
__device__ __forceinline__ double cell_D(double A, double B, double C) {
    return fma(A, B, -(C * C));
}

// The quotient, whatever the condition number; Df is the determinant as float.
// The map is float32: the quotient of the FP64 numerator and determinant
// (each rounded to float) through v_rcp_f32 is within ~3e-7 relative, and
// v_rcp_f64 issues at ~1/3.5 the rate of an FP64 FMA.
__device__ __forceinline__ double cell_num(double A, double B, double C, double far, double fai,
                                           double fbr, double fbi) {
    const double p = fma(far, far, fai * fai);
    const double q = fma(fbr, fbr, fbi * fbi);
    const double r = fma(far, fbr, fai * fbi);
    return fma(B, p, fma(A, q, (-2.0 * C) * r));
}

__device__ __forceinline__ float cell_quot(double A, double B, double C, double far, double fai,
                                           double fbr, double fbi, float &Df) {
    const double num = cell_num(A, B, C, far, fai, fbr, fbi);
    Df = (float)cell_D(A, B, C);
    return (float)num * __builtin_amdgcn_rcpf(Df);
}

// The condition test is FP64 (two multiplies and a compare: one conversion
// fewer than on float T and D).  A, B >= 0 (sums of squares), so T <= 0 only
// for an empty window, where D = 0 and the test fails as well.
__device__ __forceinline__ bool cell_ok(double A, double B, double C) {
    const double T = A + B;
    return T * T < QCOND * cell_D(A, B, C);
}

__device__ __forceinline__ float cell_F(double A, double B, double C, double far,
                                        double fai, double fbr, double fbi) {
    float Df;
    const float F = cell_quot(A, B, C, far, fai, fbr, fbi, Df);
    return cell_ok(A, B, C) ? F : 2.0f;
}

// uint32 index maths of rect.cu:21-31 (start) and rect.cu:59-69 (end).
__device__ __forceinline__ uint32_t idx_start(uint32_t t, uint32_t t_min, uint32_t TA,
                                              uint32_t N) {
    int32_t i = (int32_t)((uint32_t)(t - t_min + TA / 2) / TA);
    if (i < 0) i = 0;
    uint32_t u = (uint32_t)i;
    return u >= N ? N - 1 : u;
}

__device__ __forceinline__ uint32_t idx_end_q(uint32_t q, uint32_t N) {
    int32_t i = (int32_t)(q - 1u);
    if (i < 0) i = 0;
    uint32_t u = (uint32_t)i;
    return u >= N ? N - 1 : u;
}

// ----------------------------------------------------------------------------
// fused reductions
// ----------------------------------------------------------------------------

constexpr float LOG2E = 1.4426950408889634f;

// 2^(aL - bL) = exp(a - b) for references kept in log2 units (aL = a*LOG2E);
// exp2(-inf) = 0
__device__ __forceinline__ float exp2_diff(float aL, float bL) {
    return __builtin_amdgcn_exp2f(aL - bL);
}


// Cross-lane moves without LDS: DPP within 16-lane rows (quad permutes and
// row rotations; every source lane lies inside the row, so all lanes are
// written) and gfx950's row swaps across rows.
constexpr int DPP_QUAD_XOR1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int DPP_QUAD_XOR2 = 0x4E;  // quad_perm [2,3,0,1]
constexpr int DPP_ROW_ROR4 = 0x124;  // row_ror:4
constexpr int DPP_ROW_ROR8 = 0x128;  // row_ror:8

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// Combine over the four 16-lane rows at each row position: v_permlane16_swap
// pairs rows (0,1) and (2,3), v_permlane32_swap the two halves; every lane of
// a position ends with the same bits.
template <typename Op>
__device__ __forceinline__ float rows16_reduce(float v, Op op) {
    const unsigned u = __float_as_uint(v);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const float s = op(__uint_as_float(p[0]), __uint_as_float(p[1]));
    const unsigned us = __float_as_uint(s);
    const auto q = __builtin_amdgcn_permlane32_swap(us, us, false, false);
    return op(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

__device__ __forceinline__ float rows16_sum(float v) {
    return rows16_reduce(v, [](float a, float b) { return a + b; });
}

// Sum over the 4 quads of a 16-lane row at each quad position.
__device__ __forceinline__ float quads_sum(float v) {
    v += dpp_f<DPP_ROW_ROR4>(v);
    return v + dpp_f<DPP_ROW_ROR8>(v);
}

__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_f<DPP_QUAD_XOR1>(v);
    v += dpp_f<DPP_QUAD_XOR2>(v);
    return rows16_sum(quads_sum(v));
}

// wave maximum, the same value on every lane
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_f<DPP_QUAD_XOR1>(v));
    v = fmaxf(v, dpp_f<DPP_QUAD_XOR2>(v));
    v = fmaxf(v, dpp_f<DPP_ROW_ROR4>(v));
    v = fmaxf(v, dpp_f<DPP_ROW_ROR8>(v));
    return rows16_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

__device__ __forceinline__ void argmax_merge(float &bv, int &bi, float v, int i) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

// wave minimum of non-negative integers, the same on every lane
__device__ __forceinline__ int wave_min_idx(int v) {
    v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_QUAD_XOR1, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_QUAD_XOR2, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_ROW_ROR4, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_ROW_ROR8, 0xf, 0xf, false));
    const auto p = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    v = min((int)p[0], (int)p[1]);
    const auto q = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return min((int)q[0], (int)q[1]);
}

// Wave argmax, the first index on ties: the maximum first, then the smallest
// index among the lanes that hold it, both by DPP (~30 instructions; pairwise
// exchanges of value and index through LDS take ~130).  No lane's value is
// NaN (a running maximum starts from -inf and drops NaN).
__device__ __forceinline__ void wave_argmax(float &bv, int &bi) {
    const float m = wave_max(bv);
    bi = wave_min_idx(bv == m ? bi : 0x7fffffff);
    bv = m;
}

constexpr int MAX_RB = 512;
constexpr float REF_SLACK = 60.0f;  // e^60 * cells per item stays far below FLT_MAX

// Wave sums of R per-lane values.  Returns the sum of one of them, and in
// `row` which one (-1: this lane holds none).  R = 1: lane 0 holds the sum.
// R = 4: two halving exchange steps within each quad first (lanes pair up and
// keep half of the rows each), then one value per lane is summed over the
// quads (row rotations) and the rows (row swaps); row r ends up on lane
// 2*(r&1) + (r>>1).
template <int R>
__device__ __forceinline__ float rows_sum(const float (&v)[R], int lane, int &row);

template <>
__device__ __forceinline__ float rows_sum<1>(const float (&v)[1], int lane, int &row) {
    row = lane == 0 ? 0 : -1;
    return wave_sum(v[0]);
}

template <>
__device__ __forceinline__ float rows_sum<4>(const float (&v)[4], int lane, int &row) {
    const bool b = lane & 1;
    // step 1: b = 0 keeps rows {0,1}, b = 1 keeps rows {2,3}
    const float s0 = b ? v[0] : v[2];
    const float s1 = b ? v[1] : v[3];
    const float u0 = (b ? v[2] : v[0]) + dpp_f<DPP_QUAD_XOR1>(s0);
    const float u1 = (b ? v[3] : v[1]) + dpp_f<DPP_QUAD_XOR1>(s1);
    // step 2: c = 0 keeps the first of the pair, c = 1 the second
    const bool c = lane & 2;
    const float z = (c ? u1 : u0) + dpp_f<DPP_QUAD_XOR2>(c ? u0 : u1);
    row = lane < 4 ? 2 * (b ? 1 : 0) + (c ? 1 : 0) : -1;
    return rows16_sum(quads_sum(z));
}

// Per-work-item reduction state.  A lane owns NCOLS columns; every sub-tile
// brings R wave-uniform rows x those columns, with invalid cells set to -inf.
//  - argmax (add): lane maximum of the sub-tile; only when it beats the lane's
//    best is the first (row-major) position searched;
//  - BtSG: sum of 2^(F*LOG2E - ML), ML = Mw*LOG2E rounded to float, Mw the
//    wave's running maximum (accumulators rescaled when it grows) -- one FMA
//    and one exp2 per cell; each sum is relative to its reference in log2
//    units (ML), i.e. to exp(F - ML/LOG2E).  Column sums stay in registers
//    across sub-tiles (their sum is the item total), row sums are
//    wave-reduced and parked in LDS with ML.
template <bool BTSG, int NCOLS = 4>
struct Reducer {
    float best;
    int bidx;
    float Mw;
    float ML;
    float Scol[NCOLS];

    __device__ void init() {
        best = -INFINITY;
        bidx = 0x7fffffff;
        Mw = -INFINITY;
        ML = -INFINITY;
#pragma unroll
        for (int c = 0; c < NCOLS; c++) Scol[c] = 0.0f;
    }

    // the lane's sum over all its cells (relative to ML)
    __device__ float total() const {
        float s = Scol[0];
#pragma unroll
        for (int c = 1; c < NCOLS; c++) s += Scol[c];
        return s;
    }

    template <int R, typename Row>
    __device__ static float block_max(const Row (&F)[R]) {
        float lm = -INFINITY;
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < NCOLS; c++) lm = fmaxf(lm, F[r][c]);
        return lm;
    }

    // F[r][c]: cell values (-inf when invalid); row index m0 + r; colidx[c]
    // column index of the lane's c-th column; rl0: item-local row of r = 0.
    template <int R, typename Row>
    __device__ void add(const Row (&F)[R], int m0, const int (&colidx)[NCOLS], int N_tau,
                        int lane, int rl0, float *sh_rowM, float *sh_rowS) {
        const float lm = block_max(F);
        if (lm > best || (lm == best && lm != -INFINITY)) {
            // the first cell (row-major) equal to lm: selects from the last
            // cell to the first, no branches (a search with an early exit
            // compiles to a chain of masked branches, one per cell)
            int pos = 0;
#pragma unroll
            for (int q = R * NCOLS - 1; q >= 0; q--) pos = F[q / NCOLS][q % NCOLS] == lm ? q : pos;
            const int rr = pos / NCOLS, cc = pos % NCOLS;
            // a lane's columns are evenly spaced (64 apart): arithmetic, not a
            // selection the compiler would turn into a private array
            int col = colidx[0];
            if constexpr (NCOLS > 1) col += cc * (colidx[1] - colidx[0]);
            argmax_merge(best, bidx, lm, (m0 + rr) * N_tau + col);
        }
        sums(F, lm, lane, rl0, sh_rowM, sh_rowS);
    }

    // the BtSG sums of a sub-tile whose lane maximum is lm
    template <int R, typename Row>
    __device__ void sums(const Row (&F)[R], float lm, int lane, int rl0, float *sh_rowM,
                         float *sh_rowS) {
        if (!BTSG) return;
        // exp(F - Mw) only has to stay finite, so the wave reference Mw is
        // raised (wave maximum, accumulators rescaled) only when some lane
        // sees a value more than REF_SLACK above it
        if (__any(lm > Mw + REF_SLACK)) {
            const float wm = wave_max(lm);
            const float wmL = wm * LOG2E;
            const float sc = exp2_diff(ML, wmL);
#pragma unroll
            for (int c = 0; c < NCOLS; c++) Scol[c] *= sc;
            Mw = wm;
            ML = wmL;
        }
        if (Mw == -INFINITY) return;  // wave-uniform: no valid cell yet
        // (-ML in a register of its own: a multiply-add of two registers and a
        // literal issues in ~2.7 cycles, of three registers in 4)
        float nML = -ML;
        asm("" : "+v"(nML));
        float sr[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            sr[r] = 0.0f;
#pragma unroll
            for (int c = 0; c < NCOLS; c++) {
                const float e = __builtin_amdgcn_exp2f(fmaf(F[r][c], LOG2E, nML));
                sr[r] = c == 0 ? e : sr[r] + e;
                Scol[c] += e;
            }
        }
        int row;
        const float srw = rows_sum<R>(sr, lane, row);
        if (row >= 0) {
            sh_rowM[rl0 + row] = ML;
            sh_rowS[rl0 + row] = srw;
        }
    }
};

// End of a work item (red.best, red.bidx already the wave's): combine the 4 waves, then write the item partial
// {max, argmax, M, S} and, for BtSG, the row and column partial sums rescaled
// to the item reference M (so each is a single float).  M is in log2 units:
// the partial sums are relative to exp(M / LOG2E).
struct FinShared {
    float best[4];
    int bidx[4];
    float M[4], S[4];
    float col[4][TILE_COLS];
};

template <bool BTSG, int NCOLS, typename ColMap>
__device__ void finish_item(Reducer<BTSG, NCOLS> &red, int wave, int lane, const TmplDev &td,
                            const ItemDev &it, int64_t item_id, int nrows_item,
                            ItemPart *ipart, float *rowpart, float *colpart,
                            const float *sh_rowM, const float *sh_rowS, FinShared &fs,
                            ColMap colmap) {
    float(&sh_best)[4] = fs.best;
    int(&sh_bidx)[4] = fs.bidx;
    float(&sh_M)[4] = fs.M;
    float(&sh_S)[4] = fs.S;
    float(&sh_col)[4][TILE_COLS] = fs.col;

    float stot = 0.0f;
    if (BTSG) stot = wave_sum(red.total());
    if (lane == 0) {
        sh_best[wave] = red.best;
        sh_bidx[wave] = red.bidx;
        sh_M[wave] = red.ML;
        sh_S[wave] = stot;
    }
    if (BTSG) {
#pragma unroll
        for (int c = 0; c < NCOLS; c++) sh_col[wave][colmap(lane, c)] = red.Scol[c];
    }
    __syncthreads();
    const int tid = threadIdx.x;
    const float M = fmaxf(fmaxf(sh_M[0], sh_M[1]), fmaxf(sh_M[2], sh_M[3]));
    if (BTSG) {
        const int n = it.cb * td.tile + tid;
        if (tid < td.tile && n < (int)td.N_tau) {
            float S = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; w++)
                if (sh_M[w] != -INFINITY) S += sh_col[w][tid] * exp2_diff(sh_M[w], M);
            colpart[td.colpart_off + (int64_t)it.rb * td.N_tau + n] = S;
        }
        for (int rl = tid; rl < nrows_item; rl += WG) {
            const int m = it.rb * td.rb_rows + rl;
            rowpart[td.rowpart_off + (int64_t)it.cb * td.N_t0 + m] =
                sh_rowS[rl] * exp2_diff(sh_rowM[rl], M);
        }
    }
    if (tid == 0) {
        float bv = sh_best[0];
        int bi = sh_bidx[0];
#pragma unroll
        for (int w = 1; w < 4; w++) argmax_merge(bv, bi, sh_best[w], sh_bidx[w]);
        float S = 0.0f;
        if (BTSG) {
#pragma unroll
            for (int w = 0; w < 4; w++)
                if (sh_M[w] != -INFINITY) S += sh_S[w] * exp2_diff(sh_M[w], M);
        }
        ipart[item_id] = ItemPart{bv, bi, M, S};
    }
}

// ----------------------------------------------------------------------------
// rectangular window, regular grid: prefix differences with diagonal reuse
// ----------------------------------------------------------------------------
//
// With dt0 = dtau = a*TAtom and no uint32 wrap-around, the window of cell
// (m, n) is atoms [i(m), j(m+n)) of the prefix table, where
//   i(m)   = min(q0 + a*m, N-1)                      (rect.cu:21-31)
//   j(D)   = min(max(q00 + a*D - 1, 0), N-1) + 1     (rect.cu:54-69), D = m+n,
// and j >= i always, so the incremental sum of rect.cu:75-91 equals
// P[j] - P[i].  A lane computes a 4 x C block of cells (4 rows, C columns),
// whose cells touch 3 + C diagonals; the item's j(D) range is staged in LDS in
// groups of C diagonals, each group's 7 components x C diagonals contiguous
// (padded to an odd number of doubles: the lanes' 8-byte reads then spread
// over all banks), so that all of a lane's reads are at constant offsets from
// one address.
//
// C is 4 where the item's columns need it (a wave spans 64 C columns), 2 or 1
// in the last column block of a template and for maps of at most 128 or 64
// columns: the lanes of a 256-column wave past N_tau would idle (half of them
// on a 125-column map; 1024 such maps of 125 rows: 59 us with C = 4, 37 us
// with C = 2).
//
// Bound: VALU issue (every SIMD cycle is taken).  A 16-cell step issues ~490
// instructions, 306 of them FP64 -- 7 differences, 2 for the determinant and
// 10 for the numerator per cell, which is what the formula takes -- at ~4.4
// cycles each, and 32 transcendentals at ~8.3.  The FP64 matrix instructions
// do not run beside vector work on this chip (measured), so the differences
// stay on the VALU.  1024 templates of 1000 to 8000 bins, 1.57e9 cells, BtSG:
// maps 2150 -> 1880 us (0.83e12 cells/s, 3.3 TB/s of map written) with the
// shared condition test, the diagonal order, the narrow last blocks, the
// position of the maximum found once per item, and 192 rows an item.
template <int C>
constexpr int LDS_GS = C * NC + 1 - (C * NC) % 2;
// entry (diagonal d, component k) of the staged range
template <int C>
__host__ __device__ __forceinline__ int lds_at(int d, int k) {
    return d / C * LDS_GS<C> + k * C + d % C;
}
// doubles of LDS for nd diagonals
template <int C>
constexpr int lds_doubles(int nd) {
    return (nd + C - 1) / C * LDS_GS<C>;
}
// columns per lane of the column block that starts `rem` columns before N_tau
__host__ __device__ __forceinline__ int rect_lane_cols(int rem) {
    return rem > 128 ? 4 : rem > 64 ? 2 : 1;
}
// dynamic LDS of an item of rb rows: the rows' references and sums, then the
// staged range, which the item's final reduction reuses
constexpr int rect_item_lds(int rb, int C) {
    const int nd = rb + 64 * C - 1;
    return rb * 2 * (int)sizeof(float) +
           (C == 4 ? lds_doubles<4>(nd) : C == 2 ? lds_doubles<2>(nd) : lds_doubles<1>(nd)) *
               (int)sizeof(double);
}
static_assert(rect_item_lds(16, 1) - 16 * 2 * sizeof(float) >= sizeof(FinShared) &&
                  rect_item_lds(16, 2) - 16 * 2 * sizeof(float) >= sizeof(FinShared),
              "the staged range holds the final reduction");

// The condition test of a lane's cells at once.  With a^2, b^2 >= 0 in every
// bin (the stage kernel flags templates where that fails) the trace T of a
// window is at most that of the window from the block's first start to its
// last end, so T_all^2 < Q min(D) implies T^2 < Q D for every cell, and the
// quotients stand as they are; otherwise the wave repeats the test cell by
// cell.  The slack covers the determinants' rounding to float (6e-8) and that
// of the prefix sums (1e-11 of the window on 8000 bins).  Windows fail the
// shared test only when they are a few bins long, i.e. in a template's first
// column block, whose items test cell by cell from the start.  Per 16 cells: 8
// minima and ~8 FP64 operations in place of 80.
// Determinants outside float's range: min(D) starts at FLT_MAX, below what was
// rounded to infinity, and GUARD_ROUND is Q times half the spacing of the floats
// next to zero, which is what rounding may have added to a D there.
constexpr double GUARD_SLACK = 1.0 + 1e-5;
constexpr double GUARD_ROUND = QCOND * 0.5 * 1.401298464324817e-45;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
// A lane's cells of one row, in one register tuple as their store needs them;
// rows of a map start at any 4-byte boundary.
template <int C>
struct RowCells;
template <>
struct RowCells<4> {
    typedef f32x4 type;
    typedef f32x4 store __attribute__((aligned(4)));
};
template <>
struct RowCells<2> {
    typedef f32x2 type;
    typedef f32x2 store __attribute__((aligned(4)));
};
template <>
struct RowCells<1> {
    struct type {
        float v;
        __device__ float &operator[](int) { return v; }
        __device__ float operator[](int) const { return v; }
    };
    typedef type store;
};

// Word 3 of a raw buffer resource: 32-bit data format, as gfx9 raw buffer
// accesses require.
constexpr int BUF_RSRC_WORD3 = 0x00020000;

// Work-item order.  Blocks go to the 8 XCDs round-robin (block b on XCD
// b % 8) and every XCD has its own L2, so XCD x is given a contiguous run of
// work items: the items of one template, which read the same prefix table,
// then share one L2.
#ifndef TCW_XCD_REMAP
#define TCW_XCD_REMAP 1
#endif
__device__ __forceinline__ int64_t block_slot() {
#if TCW_XCD_REMAP
    const int64_t G = gridDim.x, b = blockIdx.x;
    const int64_t q = G >> 3, r = G & 7, x = b & 7;
    return x * q + min(x, r) + (b >> 3);
#else
    return blockIdx.x;
#endif
}

// The wave's maximum (into `best`, on every lane) and the first cell
// (row-major) that holds it, from each lane's maximum and the step that
// brought it.  The cells of that step are evaluated again, by the same
// operations: the 4 C cells of the one lane that holds the maximum on as many
// lanes, or row by row where several lanes hold it.  This runs once a wave and
// item; keeping the position as the steps go by costs a 71-instruction search
// whenever any lane of the wave sees a new maximum (about three of eight
// steps).
template <int C>
__device__ __forceinline__ int rect_first_max(float &best, int bstep, const TmplDev &td,
                                              const double *__restrict__ P,
                                              const double *__restrict__ lds, int row0, int col0,
                                              int wave, int lane) {
    const float wm = wave_max(best);
    const int s = wave_min_idx(best == wm ? bstep : 0x7fffffff);
    uint64_t held = __ballot(best == wm && bstep == s);
    best = wm;
    if (wm == -INFINITY) return 0x7fffffff;
    const int N_t0 = (int)td.N_t0, N_tau = (int)td.N_tau;
    const int rl0 = s * 16 + wave * 4;
    auto value = [&](int r, int col) {  // cell (row0 + rl0 + r, col0 + col)
        const double *__restrict__ pi =
            P + (int64_t)min(td.q0 + td.a * (row0 + rl0 + r), (int)td.N - 1) * NC;
        double S[NC];
#pragma unroll
        for (int k = 0; k < NC; k++) S[k] = lds[lds_at<C>(rl0 + r + col, k)] - pi[k];
        return cell_F(S[0], S[1], S[2], S[3], S[4], S[5], S[6]);
    };
    if (__popcll(held) == 1) {
        const int r = lane / C & 3;
        const int col = __builtin_ctzll(held) * C + lane % C;
        const bool in = lane < 4 * C && row0 + rl0 + r < N_t0 && col0 + col < N_tau;
        const uint64_t at = __ballot(in && value(r, col) == wm);
        if (at) {
            const int q = __builtin_ctzll(at);
            return (row0 + rl0 + q / C) * N_tau + col0 + __builtin_ctzll(held) * C + q % C;
        }
    }
    for (int r = 0; r < 4 && row0 + rl0 + r < N_t0; r++) {
        int first = C;  // the lane's first column of row r that holds the maximum
#pragma unroll
        for (int c = C - 1; c >= 0; c--)
            if (col0 + lane * C + c < N_tau && value(r, lane * C + c) == wm) first = c;
        const uint64_t at = __ballot(first < C);
        if (at) {
            const int l = __builtin_ctzll(at);
            return (row0 + rl0 + r) * N_tau + col0 + l * C + __builtin_amdgcn_readlane(first, l);
        }
    }
    // (not found again, should the two condition tests ever disagree: a cell of
    // the step, inside the map)
    return (row0 + rl0) * N_tau + col0 + __builtin_ctzll(held) * C;
}

// One work item.  FIRST: the template's first column block (cell-by-cell
// condition test).
template <bool BTSG, bool STRICT, int C, bool FIRST>
__device__ __forceinline__ void rect_fast_item(const TmplDev &td, const ItemDev &it,
                                               int64_t item_id, const double *__restrict__ P,
                                               float *__restrict__ Ft, ItemPart *ipart,
                                               float *rowpart, float *colpart, int *flags,
                                               double *lds) {
    const int RB = td.rb_rows;
    const int row0 = it.rb * RB;
    const int col0 = it.cb * TILE_COLS;
    const int N_t0 = (int)td.N_t0, N_tau = (int)td.N_tau;
    const int nd = RB + 64 * C - 1;
    const int D0 = row0 + col0;
    const int Nm1 = (int)td.N - 1;
    float *sh_rowM = reinterpret_cast<float *>(lds);
    float *sh_rowS = sh_rowM + RB;
    lds += RB;

    for (int d = threadIdx.x; d < nd; d += WG) {
        int64_t q = (int64_t)td.q00 + (int64_t)td.a * (D0 + d) - 1;
        q = min(max(q, (int64_t)0), (int64_t)Nm1);
        const double *__restrict__ src = P + (q + 1) * NC;
#pragma unroll
        for (int c = 0; c < NC; c++) lds[lds_at<C>(d, c)] = src[c];
    }
    __syncthreads();

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    Reducer<BTSG, C> red;
    red.init();
    int bstep = 0;  // the step that brought the lane's maximum
    bool single = false;
    const int c0 = col0 + lane * C;  // the lane's first column
    int colidx[C];
#pragma unroll
    for (int c = 0; c < C; c++) colidx[c] = c0 + c;
    const bool cols_full = col0 + 64 * C <= N_tau;
    const bool no_bound = !FIRST && (flags[it.t] & FLAG_NO_BOUND);
    const uint32_t rowb = (uint32_t)N_tau * (uint32_t)sizeof(float);

    for (int s = 0; s < RB / 16; s++) {
        const int rl0 = s * 16 + wave * 4;
        const int m0 = row0 + rl0;
        if (m0 >= N_t0) break;
        const int nvr = min(N_t0 - m0, 4);
        // lane's diagonals d = rl0 + C*lane + x, x = 0 .. C + 2; rl0 + C*lane
        // is a multiple of C, so lds_at(d, k) = lb + lds_at(x, k)
        const double *__restrict__ lb = lds + lds_at<C>(rl0 + lane * C, 0);
        // window starts: wave-uniform, read through the scalar cache
        int i0[4];
        double Pi[4][NC];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            i0[r] = min(td.q0 + td.a * (m0 + r), Nm1);
#pragma unroll
            for (int k = 0; k < NC; k++) Pi[r][k] = P[(int64_t)i0[r] * NC + k];
        }
        typename RowCells<C>::type F[4];
        float Dmin = FLT_MAX;
        double Tall = 0.0;
        // Diagonal by diagonal: its entry meets the starts of up to four rows.
        // The starts sit in scalar registers, so a lane holds one diagonal's 7
        // sums at a time (87 VGPRs, five waves a SIMD; row by row it holds C of
        // them: 96-104, four or five waves).
#pragma unroll
        for (int x = 0; x < C + 3; x++) {
            double w[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) w[k] = lb[lds_at<C>(x, k)];
            // the window from the block's first start to its last end
            if (!FIRST && x == C + 2) Tall = (w[0] - Pi[0][0]) + (w[1] - Pi[0][1]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int c = x - r;
                if (c < 0 || c >= C) continue;
                float f;
                if constexpr (FIRST) {
                    f = cell_F(w[0] - Pi[r][0], w[1] - Pi[r][1], w[2] - Pi[r][2], w[3] - Pi[r][3],
                               w[4] - Pi[r][4], w[5] - Pi[r][5], w[6] - Pi[r][6]);
                } else {
                    float Df;
                    f = cell_quot(w[0] - Pi[r][0], w[1] - Pi[r][1], w[2] - Pi[r][2],
                                  w[3] - Pi[r][3], w[4] - Pi[r][4], w[5] - Pi[r][5],
                                  w[6] - Pi[r][6], Df);
                    Dmin = fminf(Dmin, Df);
                }
                // (finished here: not after the shared test, nor together with
                // the other diagonals' cells)
                asm volatile("" : "+v"(f));
                F[r][c] = f;
                if (STRICT) {
                    int64_t q = (int64_t)td.q00 + (int64_t)td.a * (m0 + r + colidx[c]) - 1;
                    q = min(max(q, (int64_t)0), (int64_t)Nm1);
                    single |= (q == i0[r]) && (r < nvr) && (colidx[c] < N_tau);
                }
            }
        }
        if constexpr (!FIRST) {
            const bool ok_all =
                fma(Tall * GUARD_SLACK, Tall, GUARD_ROUND) < QCOND * (double)Dmin;
            if (no_bound || !__all(ok_all)) {  // wave-uniform: cell by cell
                // (an address the compiler cannot match with the one above: it
                // would keep the differences of all cells alive, and spill)
                int at = rl0 + lane * C;
                asm volatile("" : "+v"(at));
                const double *__restrict__ lb = lds + lds_at<C>(at, 0);
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        const int x = r + c;
                        if (!cell_ok(lb[lds_at<C>(x, 0)] - Pi[r][0], lb[lds_at<C>(x, 1)] - Pi[r][1],
                                     lb[lds_at<C>(x, 2)] - Pi[r][2]))
                            F[r][c] = 2.0f;
                    }
            }
        }
        if (cols_full && nvr == 4) {
#pragma unroll
            for (int r = 0; r < 4; r++)
                *(typename RowCells<C>::store *)(Ft + (int64_t)(m0 + r) * N_tau + c0) = F[r];
        } else {
            // partial sub-tiles store through a buffer resource over their rows
            // inside the map: the lane's column c at byte voff of a row, or far
            // outside the resource for a column past N_tau (the hardware drops
            // the store; rows past the map lie beyond the resource as well), so
            // no branch per cell (the offsets are formed here: held over the
            // loop, they cost registers)
            int first = c0, nvc = N_tau - c0;
            asm volatile("" : "+v"(first), "+v"(nvc));
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                Ft + (int64_t)m0 * N_tau, (short)0, (int)((uint32_t)nvr * rowb), BUF_RSRC_WORD3);
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int c = 0; c < C; c++) {
                    const uint32_t voff = c < nvc ? (uint32_t)(first + c) * 4u : 0x80000000u;
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(F[r][c]), rs,
                                                          (int)voff, (int)(r * rowb), 0);
                    F[r][c] = (r < nvr) && (c < nvc) ? F[r][c] : -INFINITY;
                }
        }
        const float lm = red.block_max(F);
        bstep = lm > red.best ? s : bstep;
        red.best = fmaxf(red.best, lm);
        red.sums(F, lm, lane, rl0, sh_rowM, sh_rowS);
    }
    if (STRICT && single) atomicOr(flags + it.t, FLAG_SINGLE_ATOM);
    red.bidx = rect_first_max<C>(red.best, bstep, td, P, lds, row0, col0, wave, lane);
    __syncthreads();  // the staged range is consumed: the final reduction reuses it
    finish_item(red, wave, lane, td, it, item_id, min(RB, N_t0 - row0), ipart, rowpart, colpart,
                sh_rowM, sh_rowS, *reinterpret_cast<FinShared *>(lds),
                [](int ln, int c) { return ln * C + c; });
}

template <bool BTSG, bool STRICT>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(4, 8))) void rect_fast_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items, int64_t item0,
    const double *__restrict__ prefix, float *__restrict__ Fout,
    ItemPart *__restrict__ ipart, float *__restrict__ rowpart,
    float *__restrict__ colpart, int *__restrict__ flags) {
    extern __shared__ double lds_raw[];  // one dynamic LDS symbol per file
    const int64_t item_id = item0 + block_slot();
    const ItemDev it = items[item_id];
    const TmplDev td = tds[it.t];
    const double *P = prefix + td.prefix_off;
    float *Ft = Fout + td.F_off;
    const int C = rect_lane_cols((int)td.N_tau - it.cb * TILE_COLS);
#define RECT_ITEM(cols, first)                                                              \
    rect_fast_item<BTSG, STRICT, cols, first>(td, it, item_id, P, Ft, ipart, rowpart, colpart, \
                                              flags, lds_raw)
    if (it.cb == 0) {  // block-uniform
        if (C == 4)
            RECT_ITEM(4, true);
        else if (C == 2)
            RECT_ITEM(2, true);
        else
            RECT_ITEM(1, true);
    } else {
        if (C == 4)
            RECT_ITEM(4, false);
        else if (C == 2)
            RECT_ITEM(2, false);
        else
            RECT_ITEM(1, false);
    }
#undef RECT_ITEM
}

// ----------------------------------------------------------------------------
// rectangular window, steps of an atom or more, without wrap-around
// ----------------------------------------------------------------------------
//
// Row m starts at t0 + m dt0 + TAtom/2 - t_min = TAtom q + phi, column n lasts
// tau + n dtau = TAtom Q + R, and (rect.cu:21-31, 54-69; nothing wraps, so the
// ends grow with n and no running maximum is needed)
//   i = min(q, N-1),   j = min(max(q + Q + [phi + R >= TAtom], 1), N) >= i,
// a compare and an add with carry per cell.  The item's range of prefix entries
// is staged in LDS where it fits: entry e at e*7 + (e >> pad) doubles, pad the
// lanes' stride of entries if that is even, rounded down to a power of two, so
// that the lanes' reads spread over the banks; wider steps read the table in
// place.  A lane owns the columns lane, + 64, + 128, + 192 of the block (as many
// as the block has groups of 64) and a wave 4 rows at a time, whose starts are read through the scalar cache.
//
// Bound: VALU issue and latency together (63 instructions a cell, 24 of them
// FP64; 69% of the cycles issue, at ~3 waves a SIMD).  128 templates of 1000 to
// 4000 bins, steps of 2 and 3 bins, 37e6 cells: maps 195 us with the generic
// kernel (an integer division and an uncoalesced 56-byte read a cell), 90 us
// so, 210 us with these indices but the table read in place.
// Rows per item at most and items aimed at, untuned (the maps above: 64 rows
// 100 us, 32 rows 110, 96 rows 115, all with 256 columns an item).
constexpr int STEP_RB = 64;
constexpr int64_t STEP_ITEMS = 1024;
using tcwc::step_bytes;
using tcwc::step_in_lds;
using tcwc::step_range;
using tcwc::step_shape;
using tcwc::STEP_LDS_AIM;
using tcwc::STEP_LDS_MOST;
using tcwc::StepRange;
using tcwc::StepShape;

// dynamic LDS of an item: the rows' references and sums, and the staged range
// (none if it does not fit) or the final reduction in its place
__host__ __device__ __forceinline__ int step_lds(int rb, const StepShape &sh) {
    const int range = step_in_lds(sh) ? step_bytes(sh) : 0;
    return rb * 2 * (int)sizeof(float) + (range < (int)sizeof(FinShared) ? (int)sizeof(FinShared) : range);
}

template <bool BTSG, bool STRICT, bool LDS, int C>
__device__ __forceinline__ void rect_step_item(const TmplDev &td, const ItemDev &it,
                                               int64_t item_id, const double *__restrict__ P,
                                               float *__restrict__ Ft, ItemPart *ipart,
                                               float *rowpart, float *colpart, int *flags,
                                               double *lds) {
    const int RB = td.rb_rows;
    const int row0 = it.rb * RB;
    const int col0 = it.cb * td.tile;
    const int N_t0 = (int)td.N_t0, N_tau = (int)td.N_tau;
    const int N = (int)td.N;
    const uint32_t TA = td.TAtom, dt0 = td.dt0, dtau = td.dtau;
    const StepShape sh = step_shape(RB, td.tile, td.N_tau, dt0, dtau, TA);
    float *sh_rowM = reinterpret_cast<float *>(lds);
    float *sh_rowS = sh_rowM + RB;
    lds += RB;
    const uint32_t T0 = td.t0 + TA / 2 - td.t_min;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    int jb = 0;  // entry in LDS slot 0
    if (LDS) {
        const uint32_t Tr = T0 + (uint32_t)row0 * dt0;
        const uint32_t Tl = T0 + (uint32_t)min(row0 + RB - 1, N_t0 - 1) * dt0;
        const uint32_t xf = td.tau + (uint32_t)col0 * dtau;
        const uint32_t xl = td.tau + (uint32_t)min(col0 + td.tile - 1, N_tau - 1) * dtau;
        uint32_t rem;
        const StepRange range = step_range(Tr, xf, Tl, xl, N,
                                           [&](uint32_t x) { return div_TA(x, td, rem); });
        jb = range.first;
        const int nw = range.count * NC;
        const double *__restrict__ src = P + (int64_t)jb * NC;
        for (int k0 = threadIdx.x; k0 < nw; k0 += 8 * WG) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (k0 + u * WG < nw) v[u] = src[k0 + u * WG];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int k = k0 + u * WG;
                if (k < nw) lds[k + ((k / NC) >> sh.pad)] = v[u];
            }
        }
    }
    int colidx[C], Q[C];
    uint32_t R[C], voff[C];
#pragma unroll
    for (int c = 0; c < C; c++) {
        colidx[c] = col0 + c * 64 + lane;
        const bool valid = colidx[c] < N_tau;
        const uint32_t x = td.tau + (uint32_t)(valid ? colidx[c] : col0) * dtau;
        Q[c] = (int)div_TA(x, td, R[c]) - jb;
        voff[c] = valid ? (uint32_t)colidx[c] * 4u : 0x80000000u;
    }
    const bool cols_full = col0 + 64 * C <= N_tau;
    const uint32_t rowb = (uint32_t)N_tau * (uint32_t)sizeof(float);
    const uint32_t dq = dt0 / TA, dphi = dt0 % TA;
    Reducer<BTSG, C> red;
    red.init();
    bool single = false;
    __syncthreads();
    for (int s = 0; s < RB / 16; s++) {
        const int rl0 = s * 16 + wave * 4;
        const int m0 = row0 + rl0;
        if (m0 >= N_t0) break;
        const int nvr = min(N_t0 - m0, 4);
        uint32_t phi;
        uint32_t q = div_TA(T0 + (uint32_t)m0 * dt0, td, phi);
        float F[4][C];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            // (rows past the map repeat the last one: their entries are staged)
            if (r > 0 && r < nvr) {
                phi += dphi;
                q += dq + (phi >= TA);
                phi -= phi >= TA ? TA : 0;
            }
            const int i = min((int)q, N - 1);
            double Pi[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) Pi[k] = P[(int64_t)i * NC + k];
#pragma unroll
            for (int c = 0; c < C; c++) {
                const int j = min(max((int)q + Q[c] + (R[c] >= TA - phi), 1 - jb), N - jb);
                double w[NC];
                if (LDS) {
                    const double *e = lds + (__umul24(j, NC) + (j >> sh.pad));
#pragma unroll
                    for (int k = 0; k < NC; k++) w[k] = e[k];
                } else {
                    const double *e = P + (int64_t)j * NC;
#pragma unroll
                    for (int k = 0; k < NC; k++) w[k] = e[k];
                }
                F[r][c] = cell_F(w[0] - Pi[0], w[1] - Pi[1], w[2] - Pi[2], w[3] - Pi[3],
                                 w[4] - Pi[4], w[5] - Pi[5], w[6] - Pi[6]);
                // i_t1 == i_t0 (i_t1 = j - 1)
                if (STRICT) single |= j + jb - 1 == i && r < nvr && colidx[c] < N_tau;
            }
        }
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            Ft + (int64_t)m0 * N_tau, (short)0, (int)((uint32_t)nvr * rowb), BUF_RSRC_WORD3);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int c = 0; c < C; c++)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(F[r][c]), rs, (int)voff[c],
                                                      (int)(r * rowb), 0);
        if (!cols_full || nvr < 4) {
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int c = 0; c < C; c++)
                    F[r][c] = r < nvr && colidx[c] < N_tau ? F[r][c] : -INFINITY;
        }
        red.add(F, m0, colidx, N_tau, lane, rl0, sh_rowM, sh_rowS);
    }
    if (STRICT && single) atomicOr(flags + it.t, FLAG_SINGLE_ATOM);
    wave_argmax(red.best, red.bidx);
    __syncthreads();  // the staged range is consumed: the final reduction reuses it
    finish_item(red, wave, lane, td, it, item_id, min(RB, N_t0 - row0), ipart, rowpart, colpart,
                sh_rowM, sh_rowS, *reinterpret_cast<FinShared *>(lds),
                [](int ln, int c) { return c * 64 + ln; });
}

template <bool BTSG, bool STRICT>
__global__ __launch_bounds__(WG) void rect_step_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items, int64_t item0,
    const double *__restrict__ prefix, float *__restrict__ Fout,
    ItemPart *__restrict__ ipart, float *__restrict__ rowpart,
    float *__restrict__ colpart, int *__restrict__ flags) {
    extern __shared__ double lds_raw[];  // one dynamic LDS symbol per file
    const int64_t item_id = item0 + block_slot();
    const ItemDev it = items[item_id];
    const TmplDev td = tds[it.t];
    if (!td.walk) return;  // block-uniform: a rect_generic_kernel item
    const int groups = (min((int)td.tile, (int)td.N_tau - it.cb * td.tile) + 63) / 64;
#define STEP_ITEM(lds, cols)                                                                  \
    rect_step_item<BTSG, STRICT, lds, cols>(td, it, item_id, prefix + td.prefix_off,           \
                                            Fout + td.F_off, ipart, rowpart, colpart, flags, \
                                            lds_raw)
    if (!step_in_lds(step_shape(td.rb_rows, td.tile, td.N_tau, td.dt0, td.dtau, td.TAtom)))
        STEP_ITEM(false, 4);
    else if (groups == 4)
        STEP_ITEM(true, 4);
    else if (groups == 3)
        STEP_ITEM(true, 3);
    else if (groups == 2)
        STEP_ITEM(true, 2);
    else
        STEP_ITEM(true, 1);
#undef STEP_ITEM
}

// ----------------------------------------------------------------------------
// generic per-cell kernels (rect with exact wrap-around semantics; exp)
// ----------------------------------------------------------------------------
//
// Lanes own columns col0 + c*64 + lane (c = 0..3); wave w owns item rows
// w, w+4, w+8, ...  Row quantities are wave-uniform.

struct RowRect {
    uint32_t i0;       // window start index
    uint32_t x0;       // (t0_m + tau - t_min + TAtom/2) mod 2^32 at n = 0
    uint32_t nwrap;    // first n whose x wrapped past 2^32 (N_tau if none)
    uint32_t i1_pre;   // i_t1 just before the wrap (running maximum after it)
};

__device__ __forceinline__ RowRect rect_row(const TmplDev &td, uint32_t m) {
    RowRect rr;
    const uint32_t t0m = td.t0 + m * td.dt0;
    rr.i0 = idx_start(t0m, td.t_min, td.TAtom, td.N);
    rr.x0 = t0m + td.tau - td.t_min + td.TAtom / 2;
    const uint64_t room = (1ull << 32) - (uint64_t)rr.x0;  // n*dtau >= room wraps
    const uint64_t nw = (room + td.dtau - 1) / td.dtau;
    rr.nwrap = nw < (uint64_t)td.N_tau ? (uint32_t)nw : td.N_tau;
    rr.i1_pre = 0;
    if (rr.nwrap < td.N_tau) {
        const uint32_t xp = rr.x0 + (rr.nwrap - 1) * td.dtau;
        rr.i1_pre = idx_end_q(xp / td.TAtom, td.N);
    }
    return rr;
}

template <bool BTSG, bool STRICT>
__global__ __launch_bounds__(WG) void rect_generic_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items, int64_t item0,
    const double *__restrict__ prefix, float *__restrict__ Fout,
    ItemPart *__restrict__ ipart, float *__restrict__ rowpart,
    float *__restrict__ colpart, int *__restrict__ flags) {
    __shared__ float sh_rowM[MAX_RB];
    __shared__ float sh_rowS[MAX_RB];
    __shared__ FinShared sh_fin;
    const int64_t item_id = item0 + block_slot();
    const ItemDev it = items[item_id];
    const TmplDev td = tds[it.t];
    if (td.walk) return;  // block-uniform: a rect_step_kernel item
    const int RB = td.rb_rows;
    const int row0 = it.rb * RB;
    const int col0 = it.cb * TILE_COLS;
    const int N_t0 = (int)td.N_t0, N_tau = (int)td.N_tau;
    const double *__restrict__ P = prefix + td.prefix_off;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    Reducer<BTSG> red;
    red.init();
    bool single = false;
    float *__restrict__ Ft = Fout + td.F_off;
    int colidx[4];
#pragma unroll
    for (int c = 0; c < 4; c++) colidx[c] = col0 + c * 64 + lane;

    for (int rl = wave; rl < RB; rl += 4) {
        const int m = row0 + rl;
        if (m >= N_t0) break;
        const RowRect rr = rect_row(td, (uint32_t)m);
        double Pi[NC];
#pragma unroll
        for (int k = 0; k < NC; k++) Pi[k] = P[(int64_t)rr.i0 * NC + k];
        float F[1][4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const bool valid = colidx[c] < N_tau;
            const uint32_t n = valid ? (uint32_t)colidx[c] : 0u;
            const uint32_t x = rr.x0 + n * td.dtau;
            const uint32_t i1 = idx_end_q(x / td.TAtom, td.N);
            // running maximum of i_t1 over n' <= n (the i_t1_last recursion)
            const uint32_t run = (n >= rr.nwrap) ? max(i1, rr.i1_pre) : i1;
            const uint32_t j = max(rr.i0, run + 1);
            const double *Pj = P + (int64_t)j * NC;
            const float f = cell_F(Pj[0] - Pi[0], Pj[1] - Pi[1], Pj[2] - Pi[2], Pj[3] - Pi[3],
                                   Pj[4] - Pi[4], Pj[5] - Pi[5], Pj[6] - Pi[6]);
            if (STRICT) single |= valid && (i1 == rr.i0);
            if (valid) Ft[(int64_t)m * N_tau + colidx[c]] = f;
            F[0][c] = valid ? f : -INFINITY;
        }
        red.add(F, m, colidx, N_tau, lane, rl, sh_rowM, sh_rowS);
    }
    if (STRICT && single) atomicOr(flags + it.t, FLAG_SINGLE_ATOM);
    __syncthreads();
    wave_argmax(red.best, red.bidx);
    finish_item(red, wave, lane, td, it, item_id, min(RB, N_t0 - row0), ipart, rowpart,
                colpart, sh_rowM, sh_rowS, sh_fin, [](int ln, int c) { return c * 64 + ln; });
}

// Exponential window off the atom grid: the window sum slides with any starts an
// atom or more apart, and any durations.
//
// Row m starts at T = t0 + m dt0 - t_min = TAtom q + phi, column n lasts 3 tau =
// TAtom Q + R.  The cell's atoms (exp.cu:39-102) are lo(m) .. hi(m, n),
//   lo = q + [phi > 0],   hi = q + Q - 1 + [s >= h] + [s >= TAtom + h],
// s = phi + R, h = TAtom - TAtom / 2 (atoms at or past N count as zero), with
// weights w rho^(i - lo), rho = e^(-TAtom/tau).  F does not change with a
// common factor of the weights, so w is left out of the sums, and
//   E(m) = sum_{i = lo}^{hi} rho^(i - lo) x_i   (rho^2 for a^2, b^2, ab)
// goes from row to row by the atoms that enter (the same on every lane) and
// those that leave (dt0 / TAtom or one more, by lane):
//   E(m-1) = rho^(lo - lo') E(m) + sum_{i = lo'}^{lo-1} rho^(i-lo') x_i
//            - sum_{i = hi'+1}^{hi} rho^(i-lo') x_i;
// rho^(hi' + 1 - lo') is one of four values per lane, as that exponent is
// Q - 1 .. Q + 2.  (The numerator and the determinant take their factor w^4
// before they are rounded to float, as they have it in the direct sum, so that F
// is the same float and nearly equal maxima keep their order; 30 instead of 28.5
// us.)  A cell costs O(dt0 / TAtom) instead of O(3 tau / TAtom).
//
// An item is RB rows x 64 columns, one column a lane, and its rows are shared
// out to eight waves from the top down.  The waves share the direct sum at the
// item's top row by atoms (staged in LDS chunk by chunk); then each sums what
// enters and leaves between its own top row and the next wave's (two Horner
// sums, the recurrence over many rows at once), which gives every wave the sum
// at its top row; then each walks its rows.  Entering and leaving atoms come
// from LDS where the item's ranges of them fit.
//
// What the direct sum gives exactly and a sliding sum would not: a window
// whose bins are all zero has E = 0 (the kind column counts bins with data),
// and from the first infinite or NaN atom on, the item's rows are summed
// directly, as are all rows where the steps are longer than the windows.
//
// Bound: latency of the item's phases (one or two workgroups a CU), and for long
// windows the direct sum (16 to 21 instructions an atom and wave).  125 x 125
// cells and 1000 bins: 32 templates 700 us with a direct sum for every cell, 52
// with items of 256 columns whose waves all walked every row, 30 so (13 of them
// the direct sum, 3 the steps between the waves' rows); 256 templates 139, now
// 71.  500 x 500 cells and 4000 bins: 64 templates 577, now 352; one 200, now 57.
constexpr int WALK_WAVES = 8;
constexpr int WALK_WG = 64 * WALK_WAVES;
constexpr int WALK_TILE = 64;        // columns of an item
constexpr int WALK_TAIL_CAP = 1024;  // leaving atoms staged in LDS (32 KB)
constexpr int WALK_HEAD_CAP = 256;   // entering atoms staged in LDS (8 KB)
constexpr int WALK_CHUNK = 1024;     // atoms of the direct sum staged at a time (32 KB)
static_assert(WALK_WAVES * MERGED_STRIDE * 64 * 2 <= WALK_TAIL_CAP * MERGED_STRIDE &&
                  WALK_CHUNK <= WALK_TAIL_CAP,
              "the direct sum's chunk and parts share the leaving atoms' LDS");
// a wave's change of E to the next wave's top row: 7 sums, the kinds, and the
// power of rho that E takes
constexpr int WALK_STEP = NC + 2;
constexpr int walk_rows(int rb) { return (rb + 3) / 4 * 4; }
constexpr int walk_lds(int rb) {
    return ((WALK_TAIL_CAP + WALK_HEAD_CAP) * MERGED_STRIDE + walk_rows(rb) * 2) *
               (int)sizeof(float) +
           (WALK_WAVES - 1) * WALK_STEP * 64 * (int)sizeof(double);
}

struct WalkCol {  // a lane's column, 3 tau = TAtom Q + R
    double rho[2];   // rho^2, rho
    double lead[4];  // rho^(Q - 1 + k)
    double ratau;    // TAtom / tau
    double w4[3];    // w^4 of the row, and its change to the next row without and with a wrap
    int Q;
    uint32_t R;
};

struct WalkRow {  // a row's start, T = TAtom q + phi
    int q;
    uint32_t phi;
    __device__ int lo() const { return q + (phi > 0); }
    // hi - (q + Q - 1) of the lane's column
    __device__ int end(const WalkCol &wc, uint32_t TA) const {
        const uint32_t s = phi + wc.R, h = TA - TA / 2;
        return (s >= h) + (s >= TA + h);
    }
    __device__ int hi(const WalkCol &wc, uint32_t TA) const { return q + wc.Q - 1 + end(wc, TA); }
};

// Copy `count` atoms (at most CAP) of the table to LDS, all loads of a thread
// in flight together; true if one of this thread's atoms is not finite.
template <int CAP>
__device__ __forceinline__ bool walk_stage(float *dst, const float *__restrict__ src, int count) {
    static_assert(MERGED_STRIDE == 8, "two 16-byte words an atom, the kind in the second");
    constexpr int PER = (CAP * 2 + WALK_WG - 1) / WALK_WG;
    f32x4 v[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int k = i * WALK_WG + (int)threadIdx.x;
        if (k < count * 2) v[i] = reinterpret_cast<const f32x4 *>(src)[k];
    }
    bool odd = false;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int k = i * WALK_WG + (int)threadIdx.x;
        if (k < count * 2) {
            reinterpret_cast<f32x4 *>(dst)[k] = v[i];
            odd |= (k & 1) && v[i][3] == BIN_ODD;
        }
    }
    return odd;
}

// E = sum over atoms x[0 .. count) of rho^l x_l, and the sum of their kinds, by
// Horner from the far end.  MASK: atoms l >= L are left out on this lane: the
// sum starts anew at l = L - 1 (the weight of what came before is 0 there,
// which is why every atom has to be finite).
template <bool MASK>
__device__ __forceinline__ void walk_horner(const float *x, int count, int L, const WalkCol &wc,
                                            double (&E)[NC], float &kinds) {
#pragma unroll 2  // (4: more than 128 VGPRs)
    for (int l = count - 1; l >= 0; l--) {
        const float *v = x + l * MERGED_STRIDE;
        double r0 = wc.rho[0], r1 = wc.rho[1];
        if (MASK) {
            r0 = l == L - 1 ? 0.0 : r0;
            r1 = l == L - 1 ? 0.0 : r1;
            kinds = l == L - 1 ? 0.0f : kinds;
        }
#pragma unroll
        for (int c = 0; c < NC; c++) E[c] = fma(c < 3 ? r0 : r1, E[c], (double)v[c]);
        kinds += v[NC];
    }
}

// The direct sum of a row, for any atoms: lo + l for l below the lane's L (at
// most Lmax on any lane; uniform), read from the table X below atom N.
__device__ __forceinline__ void walk_row_sum(const float *__restrict__ X, int N, const WalkCol &wc,
                                             int lo, int L, int Lmax, double (&E)[NC],
                                             float &kinds) {
#pragma unroll
    for (int c = 0; c < NC; c++) E[c] = 0.0;
    kinds = 0.0f;
#pragma unroll 1
    for (int l = min(Lmax, N - lo) - 1; l >= 0; l--) {
        const float *v = X + (int64_t)(lo + l) * MERGED_STRIDE;  // uniform: scalar loads
#pragma unroll
        for (int c = 0; c < NC; c++)
            E[c] = fma(wc.rho[c < 3 ? 0 : 1], E[c], l < L ? (double)v[c] : 0.0);
        kinds += l < L ? v[NC] : 0.0f;
    }
}

template <bool BTSG, bool STRICT>
__global__ __launch_bounds__(WALK_WG) void exp_walk_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items, int64_t item0,
    const float *__restrict__ merged, float *__restrict__ Fout, ItemPart *__restrict__ ipart,
    float *__restrict__ rowpart, float *__restrict__ colpart, int *__restrict__ flags) {
    extern __shared__ double lds_raw[];  // one dynamic LDS symbol per file
    __shared__ float sh_best[WALK_WAVES], sh_M[WALK_WAVES], sh_S[WALK_WAVES];
    __shared__ int sh_bidx[WALK_WAVES];
    __shared__ float sh_col[WALK_WAVES][64];
    const int64_t item_id = item0 + block_slot();
    const ItemDev it = items[item_id];
    const TmplDev td = tds[it.t];
    if (!td.walk) return;  // block-uniform: an exp_direct_kernel item
    float *lds = reinterpret_cast<float *>(lds_raw);
    const float *__restrict__ X = merged + td.merged_off;
    float *__restrict__ Ft = Fout + td.F_off;
    const int RB = td.rb_rows;
    const int row0 = it.rb * RB, col0 = it.cb * WALK_TILE;
    const int N_tau = (int)td.N_tau;
    const int nrows = min(RB, (int)td.N_t0 - row0);
    const int N = (int)td.N;
    const uint32_t TA = td.TAtom;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int n = col0 + lane;
    const bool valid = n < N_tau;
    float *tail = lds;
    double *comb = reinterpret_cast<double *>(lds);
    float *head = tail + WALK_TAIL_CAP * MERGED_STRIDE;
    double *step = reinterpret_cast<double *>(head + WALK_HEAD_CAP * MERGED_STRIDE);
    float *sh_rowM = reinterpret_cast<float *>(step + (WALK_WAVES - 1) * WALK_STEP * 64);
    float *sh_rowS = sh_rowM + walk_rows(RB);
    for (int k = threadIdx.x; k < walk_rows(RB); k += WALK_WG) {
        sh_rowM[k] = -INFINITY;
        sh_rowS[k] = 0.0f;
    }
    // the wave's rows within the item, top .. bot: whole groups of four
    const int groups = (nrows + 3) / 4, per = (groups + WALK_WAVES - 1) / WALK_WAVES;
    auto top_of = [&](int k) { return min(nrows, 4 * (groups - k * per)) - 1; };  // < 0: no rows
    const int top = top_of(wave), next = top_of(wave + 1), bot = max(next + 1, 0);

    WalkCol wc;
    {
        const uint32_t tau = td.tau + (uint32_t)min(n, N_tau - 1) * td.dtau;
        wc.ratau = (double)TA / (double)tau;
        wc.Q = (int)(3u * tau / TA);
        wc.R = 3u * tau % TA;
    }
    wc.rho[1] = exp(-wc.ratau);
    wc.rho[0] = wc.rho[1] * wc.rho[1];
    wc.lead[0] = exp(-(double)(wc.Q - 1) * wc.ratau);
#pragma unroll
    for (int k = 1; k < 4; k++) wc.lead[k] = wc.lead[k - 1] * wc.rho[1];
    // w = e^(-psi/tau): the row's first atom lies psi after its start
    const uint32_t dphi = td.dt0 % TA;
    wc.w4[1] = exp(-4.0 * (double)dphi * wc.ratau / (double)TA);
    wc.w4[2] = exp(4.0 * (double)(TA - dphi) * wc.ratau / (double)TA);
    // the last lane's window is the longest, the first one's the shortest
    const int Q0 = __builtin_amdgcn_readlane(wc.Q, 0), Q63 = __builtin_amdgcn_readlane(wc.Q, 63);

    const int dq = (int)(td.dt0 / TA);
    auto row_at = [&](int rl) {
        const uint32_t T = td.t0 - td.t_min + (uint32_t)(row0 + rl) * td.dt0;
        return WalkRow{(int)(T / TA), T % TA};
    };
    const WalkRow first = row_at(nrows - 1), bottom = row_at(0);
    double E[NC];
    float kinds = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; c++) E[c] = 0.0;
    bool odd = false;  // an infinity or NaN in reach of the block (block-uniform)
    {   // the direct sum at the item's top row, chunk by chunk over its longest
        // window: the waves take equal shares of each chunk
        const int lo = first.lo();
        const int L = first.hi(wc, TA) - lo + 1;
        const int Lmin = __builtin_amdgcn_readlane(L, 0), Lmax = __builtin_amdgcn_readlane(L, 63);
        const int Lblk = min(Lmax, N - lo);
        for (int c0 = 0; c0 < Lblk; c0 += WALK_CHUNK) {  // block-uniform
            const int nc = min(WALK_CHUNK, Lblk - c0);
            odd |= __syncthreads_or(walk_stage<WALK_CHUNK>(
                tail, X + (int64_t)(lo + c0) * MERGED_STRIDE, nc));
            const int share = (nc + WALK_WAVES - 1) / WALK_WAVES;
            const int s0 = wave * share, cnt = min(share, nc - s0);
            if (cnt > 0 && !odd) {  // uniform
                double H[NC];
                float kh = 0.0f;
#pragma unroll
                for (int c = 0; c < NC; c++) H[c] = 0.0;
                if (c0 + s0 + cnt <= Lmin) {
                    walk_horner<false>(tail + s0 * MERGED_STRIDE, cnt, 0, wc, H, kh);
                } else {
                    walk_horner<true>(tail + s0 * MERGED_STRIDE, cnt, L - c0 - s0, wc, H, kh);
                    if (L <= c0 + s0) {  // the lane's window ends before the share
                        kh = 0.0f;
#pragma unroll
                        for (int c = 0; c < NC; c++) H[c] = 0.0;
                    }
                }
                const double w1 = exp(-(double)(c0 + s0) * wc.ratau);
#pragma unroll
                for (int c = 0; c < NC; c++) E[c] = fma(c < 3 ? w1 * w1 : w1, H[c], E[c]);
                kinds += kh;
            }
            __syncthreads();
        }
    }
    {   // add the parts, in one order on all waves
        double *mine = comb + wave * MERGED_STRIDE * 64 + lane;
#pragma unroll
        for (int c = 0; c < NC; c++) mine[c * 64] = E[c];
        mine[NC * 64] = (double)kinds;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NC; c++) E[c] = 0.0;
        kinds = 0.0f;
#pragma unroll 2
        for (int k = 0; k < WALK_WAVES; k++) {
            const double *part = comb + k * MERGED_STRIDE * 64 + lane;
#pragma unroll
            for (int c = 0; c < NC; c++) E[c] += part[c * 64];
            kinds += (float)part[NC * 64];
        }
        __syncthreads();  // comb is staged over
    }
    // atoms that leave and enter between the item's rows: block-uniform ranges below N
    const int tail_lo = bottom.q + Q0;  // hi' + 1 at least
    const int tail_n = min(N, first.q + Q63 + 2) - tail_lo;
    const int head_lo = bottom.lo();
    const int head_n = min(N, first.lo()) - head_lo;
    const bool in_lds = tail_n < WALK_TAIL_CAP && head_n <= WALK_HEAD_CAP;
    bool head_odd = false;
    if (in_lds) {
        // slot 0 holds zeros, for the lanes with no atom to take out
        if (threadIdx.x < MERGED_STRIDE) tail[threadIdx.x] = 0.0f;
        walk_stage<WALK_TAIL_CAP>(tail + MERGED_STRIDE, X + (int64_t)tail_lo * MERGED_STRIDE,
                                  tail_n);
        head_odd = walk_stage<WALK_HEAD_CAP>(head, X + (int64_t)head_lo * MERGED_STRIDE, head_n);
    } else {
        for (int k = threadIdx.x; k < head_n; k += WALK_WG)
            head_odd |= X[(int64_t)(head_lo + k) * MERGED_STRIDE + NC] == BIN_ODD;
    }
    odd |= __syncthreads_or(head_odd);
    // sum every row directly: where an atom is not finite, or the steps are
    // longer than the windows
    const bool direct = odd || dq >= Q63;
    auto load = [&](float (&x)[MERGED_STRIDE], const float *sh, int64_t at, bool some) {
        if (in_lds) {
#pragma unroll
            for (int c = 0; c < MERGED_STRIDE; c++) x[c] = sh[c];
        } else {
#pragma unroll
            for (int c = 0; c < MERGED_STRIDE; c++) x[c] = some ? X[at * MERGED_STRIDE + c] : 0.0f;
        }
    };
    // sum += rho^(l - lo2) x_l for the entering atoms l = lo2 .. lo - 1
    auto enter = [&](int lo, int lo2, double (&sum)[NC], float &k) {
        for (int l = min(lo, N) - 1; l >= lo2; l--) {
            float x[MERGED_STRIDE];
            load(x, head + (l - head_lo) * MERGED_STRIDE, l, true);
            k += x[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) sum[c] = fma(wc.rho[c < 3 ? 0 : 1], sum[c], (double)x[c]);
        }
    };

    WalkRow row = row_at(max(top, 0));
    int hi = row.hi(wc, TA);
    uint32_t psi = row.phi > 0 ? TA - row.phi : 0;
    wc.w4[0] = exp(-4.0 * (double)psi * wc.ratau / (double)TA);
    if (!direct) {  // block-uniform
        if (next >= 0) {
            const WalkRow to = row_at(next);
            const int lo = row.lo(), lo2 = to.lo(), hi2 = to.hi(wc, TA), last = min(hi, N - 1);
            double D[NC], O[NC];
            float kd = 0.0f;
#pragma unroll
            for (int c = 0; c < NC; c++) D[c] = O[c] = 0.0;
            enter(lo, lo2, D, kd);
            for (int i = hi2 + row.q - to.q + 2; i > hi2; i--) {  // (the same count on every lane)
                const bool out = i <= last;
                float x[MERGED_STRIDE];
                load(x, tail + (out ? i - tail_lo + 1 : 0) * MERGED_STRIDE, i, out);
                kd -= x[NC];
#pragma unroll
                for (int c = 0; c < NC; c++) O[c] = fma(wc.rho[c < 3 ? 0 : 1], O[c], (double)x[c]);
            }
            const double w1 = exp(-(double)(hi2 + 1 - lo2) * wc.ratau), w2 = w1 * w1;
            double *mine = step + wave * WALK_STEP * 64 + lane;
#pragma unroll
            for (int c = 0; c < NC; c++) mine[c * 64] = fma(c < 3 ? -w2 : -w1, O[c], D[c]);
            mine[NC * 64] = (double)kd;
            mine[(NC + 1) * 64] = exp(-(double)(lo - lo2) * wc.ratau);
        }
        __syncthreads();
        if (top >= 0) {
#pragma unroll 2
            for (int k = 0; k < wave; k++) {
                const double *part = step + k * WALK_STEP * 64 + lane;
                const double m1 = part[(NC + 1) * 64], m2 = m1 * m1;
                kinds += (float)part[NC * 64];
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    const double e = fma(c < 3 ? m2 : m1, E[c], part[c * 64]);
                    E[c] = kinds == 0.0f ? 0.0 : e;
                }
            }
        }
    } else if (top >= 0) {
        walk_row_sum(X, N, wc, row.lo(), hi - row.lo() + 1, row.q + Q63 + 2 - row.lo(), E, kinds);
    }

    Reducer<BTSG, 1> red;
    red.init();
    bool single = false;
    const int colidx[1] = {n};
    for (int r4 = top >= 0 ? top / 4 * 4 : -1; r4 >= bot; r4 -= 4) {
        float F4[4][1];
#pragma unroll
        for (int j = 3; j >= 0; j--) {
            const int m = row0 + r4 + j;
            F4[j][0] = -INFINITY;
            if (r4 + j >= nrows) continue;  // uniform
            const double num = cell_num(E[0], E[1], E[2], E[3], E[4], E[5], E[6]);
            const double D = cell_D(E[0], E[1], E[2]);
            const float q = (float)(wc.w4[0] * num) * __builtin_amdgcn_rcpf((float)(wc.w4[0] * D));
            const float f = cell_ok(E[0], E[1], E[2]) ? q : 2.0f;
            if (valid) {
                Ft[(int64_t)m * N_tau + n] = f;
                F4[j][0] = f;
            }
            if (STRICT) {
                const int i0 = min(row.q + (row.phi + TA / 2 >= TA), N - 1);
                single |= valid && min(hi, N - 1) == i0;
            }
            if (r4 + j == bot) continue;
            // to row m - 1
            const int lo = row.lo();
            row.q -= dq;
            if (row.phi < dphi) {
                row.phi += TA;
                row.q--;
            }
            row.phi -= dphi;
            psi += dphi;
            const bool wrap = psi >= TA;
            psi -= wrap ? TA : 0;
            wc.w4[0] *= wrap ? wc.w4[2] : wc.w4[1];
            const int lo2 = row.lo(), hi2 = row.hi(wc, TA);
            if (direct) {  // uniform
                walk_row_sum(X, N, wc, lo2, hi2 - lo2 + 1, row.q + Q63 + 2 - lo2, E, kinds);
            } else {
                enter(lo, lo2, E, kinds);
                const int lead = row.end(wc, TA) + (row.phi == 0);
                const double wa = lead & 1 ? wc.lead[1] : wc.lead[0];
                const double wb = lead & 1 ? wc.lead[3] : wc.lead[2];
                double w1 = lead & 2 ? wb : wa;
                double w2 = w1 * w1;
                const int last = min(hi, N - 1);
                for (int i = hi2 + 1, d = 0; d <= dq; d++, i++) {
                    const bool out = i <= last;
                    float x[MERGED_STRIDE];
                    load(x, tail + (out ? i - tail_lo + 1 : 0) * MERGED_STRIDE, i, out);
#pragma unroll
                    for (int c = 0; c < NC; c++)
                        E[c] = fma(c < 3 ? -w2 : -w1, (double)x[c], E[c]);
                    kinds -= x[NC];
                    w1 *= wc.rho[1];
                    w2 *= wc.rho[0];
                }
                if (kinds == 0.0f) {
#pragma unroll
                    for (int c = 0; c < NC; c++) E[c] = 0.0;
                }
            }
            hi = hi2;
        }
        red.add(F4, row0 + r4, colidx, N_tau, lane, r4, sh_rowM, sh_rowS);
    }
    if (STRICT && single) atomicOr(flags + it.t, FLAG_SINGLE_ATOM);
    // combine: a column belongs to all waves, a row to one
    wave_argmax(red.best, red.bidx);
    float stot = 0.0f;
    if (BTSG) stot = wave_sum(red.total());
    if (lane == 0) {
        sh_best[wave] = red.best;
        sh_bidx[wave] = red.bidx;
        sh_M[wave] = red.ML;
        sh_S[wave] = stot;
    }
    if (BTSG) sh_col[wave][lane] = red.Scol[0];
    __syncthreads();
    float M = sh_M[0];
    for (int k = 1; k < WALK_WAVES; k++) M = fmaxf(M, sh_M[k]);
    if (BTSG) {
        if (valid && wave == 0) {
            float S = 0.0f;
            for (int k = 0; k < WALK_WAVES; k++)
                if (sh_M[k] != -INFINITY) S += sh_col[k][lane] * exp2_diff(sh_M[k], M);
            colpart[td.colpart_off + (int64_t)it.rb * N_tau + n] = S;
        }
        for (int rl = threadIdx.x; rl < nrows; rl += WALK_WG)
            rowpart[td.rowpart_off + (int64_t)it.cb * td.N_t0 + row0 + rl] =
                sh_rowM[rl] != -INFINITY ? sh_rowS[rl] * exp2_diff(sh_rowM[rl], M) : 0.0f;
    }
    if (threadIdx.x == 0) {
        float bv = sh_best[0];
        int bi = sh_bidx[0];
        float S = 0.0f;
        for (int k = 0; k < WALK_WAVES; k++) {
            argmax_merge(bv, bi, sh_best[k], sh_bidx[k]);
            if (BTSG && sh_M[k] != -INFINITY) S += sh_S[k] * exp2_diff(sh_M[k], M);
        }
        ipart[item_id] = ItemPart{bv, bi, M, S};
    }
}

// Exponential window, direct weighted sum over the truncated support
// (exp.cu:39-102): atoms i in [i_t0, i_t1] with t0 <= t_i <= t1 = t0 + 3 tau,
// weight w_i = exp(-(t_i - t0)/tau), A/B/C weighted by w^2, Fa/Fb by w.  All
// lanes of a wave share the row (t0) and therefore the atom stream, which is
// read once per wave through uniform loads; each lane carries its own tau.
// The weights are advanced by rho = exp(-TAtom/tau) per atom (FP64, relative
// error ~ k * 1e-16 after k atoms), the sums are FP64.
// Bound: latency of the sums' chains, so the rows and groups of 64 columns of an
// item are dealt to DIRECT_WAVES waves, which leave F in LDS, and four of them
// then reduce whole rows; 64 VGPRs, two workgroups a CU.  Half-atom starts, maps
// us with four waves an item | so: 12 templates of 31 x 23 cells 99 | 56, 32 of 125
// x 125 793 | 369, 64 of 250 x 500 10300 | 7840 (eight waves 67, 511, 8030; the
// unmasked loop unrolled by 2: 57, 396, 13090).
constexpr int DIRECT_WAVES = 16;
constexpr int DIRECT_ROWS = 16;
constexpr int DIRECT_WG = 64 * DIRECT_WAVES;

template <bool BTSG, bool STRICT>
__global__ __launch_bounds__(DIRECT_WG, 8) void exp_direct_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items, int64_t item0,
    const float *__restrict__ merged, float *__restrict__ Fout,
    ItemPart *__restrict__ ipart, float *__restrict__ rowpart,
    float *__restrict__ colpart, int *__restrict__ flags) {
    __shared__ float sh_rowM[MAX_RB];
    __shared__ float sh_rowS[MAX_RB];
    __shared__ FinShared sh_fin;
    __shared__ float sh_F[DIRECT_ROWS][TILE_COLS];
    const int64_t item_id = item0 + block_slot();
    const ItemDev it = items[item_id];
    const TmplDev td = tds[it.t];
    if (td.walk) return;  // block-uniform: an exp_walk_kernel item
    const int RB = td.rb_rows;
    const int row0 = it.rb * RB;
    const int col0 = it.cb * TILE_COLS;
    const int N_t0 = (int)td.N_t0, N_tau = (int)td.N_tau;
    const float *__restrict__ X = merged + td.merged_off;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    Reducer<BTSG> red;
    red.init();
    bool single = false;
    float *__restrict__ Ft = Fout + td.F_off;
    const uint32_t TA = td.TAtom;
    int colidx[4];
#pragma unroll
    for (int c = 0; c < 4; c++) colidx[c] = col0 + c * 64 + lane;

    const int nrows = min(RB, N_t0 - row0);
    const int groups = (min(TILE_COLS, N_tau - col0) + 63) / 64;  // of 64 columns
    for (int r0 = 0; r0 < nrows; r0 += DIRECT_ROWS) {
        const int rows = min(DIRECT_ROWS, nrows - r0);
        // a wave sums one row of one group at a time
        for (int pair = wave; pair < rows * groups; pair += DIRECT_WAVES) {
            const int rl = pair / groups, c = pair % groups;
            const int m = row0 + r0 + rl;
            const uint32_t t0m = td.t0 + (uint32_t)m * td.dt0;
            const uint32_t i0 = idx_start(t0m, td.t_min, TA, td.N);
            // first atom with t_i >= t0m (timestamps t_min + i*TA never wrap)
            uint32_t ilo = 0;
            if (t0m > td.t_min) ilo = (uint32_t)(((uint64_t)(t0m - td.t_min) + TA - 1) / TA);
            const uint32_t lo = max(i0, ilo);
            const int col = col0 + c * 64 + lane;
            const bool valid = col < N_tau;
            const uint32_t n = (uint32_t)min(col, N_tau - 1);
            const uint32_t tau = td.tau + n * td.dtau;
            const uint32_t t1 = t0m + 3u * tau;
            const uint32_t i1 = idx_end_q((uint32_t)(t1 - td.t_min + TA / 2) / TA, td.N);
            if (STRICT) single |= valid && (i1 == i0);
            // last atom with t_i <= t1
            int64_t ihi = -1;
            if (t1 >= td.t_min) ihi = (int64_t)((t1 - td.t_min) / TA);
            const int64_t hi = min((int64_t)i1, ihi);
            double acc[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) acc[k] = 0.0;
            const double rtau = 1.0 / (double)tau;
            const double rho = exp(-(double)TA * rtau);
            double w = exp(-(double)(td.t_min + lo * TA - t0m) * rtau);
            // wave-uniform loop bounds: every lane up to the shortest window's end,
            // then those whose window goes on (a zero weight would let an infinity
            // or NaN past a lane's end in)
            int64_t hi_w = hi, hi_0 = hi;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                hi_w = max(hi_w, (int64_t)__shfl_xor((long long)hi_w, o));
                hi_0 = min(hi_0, (int64_t)__shfl_xor((long long)hi_0, o));
            }
            auto add = [&](int64_t i) {
                const float *xi = X + i * MERGED_STRIDE;
                const double w2 = w * w;
                acc[0] = fma(xi[0], w2, acc[0]);
                acc[1] = fma(xi[1], w2, acc[1]);
                acc[2] = fma(xi[2], w2, acc[2]);
                acc[3] = fma(xi[3], w, acc[3]);
                acc[4] = fma(xi[4], w, acc[4]);
                acc[5] = fma(xi[5], w, acc[5]);
                acc[6] = fma(xi[6], w, acc[6]);
            };
            int64_t i = lo;
#pragma unroll 1  // (unrolled, the loads' scalar registers spill)
            for (; i <= hi_0; i++) {
                add(i);
                w *= rho;
            }
            for (; i <= hi_w; i++) {
                if (i <= hi) add(i);
                w *= rho;
            }
            const float f = cell_F(acc[0], acc[1], acc[2], acc[3], acc[4], acc[5], acc[6]);
            if (valid) Ft[(int64_t)m * N_tau + col] = f;
            sh_F[rl][c * 64 + lane] = valid ? f : -INFINITY;
        }
        __syncthreads();
        for (int rl = wave; wave < 4 && rl < rows; rl += 4) {
            float F[1][4];
#pragma unroll
            for (int c = 0; c < 4; c++) F[0][c] = c < groups ? sh_F[rl][c * 64 + lane] : -INFINITY;
            red.add(F, row0 + r0 + rl, colidx, N_tau, lane, r0 + rl, sh_rowM, sh_rowS);
        }
        __syncthreads();
    }
    if (STRICT && single) atomicOr(flags + it.t, FLAG_SINGLE_ATOM);
    if (wave < 4) {
        wave_argmax(red.best, red.bidx);
        finish_item(red, wave, lane, td, it, item_id, nrows, ipart, rowpart, colpart, sh_rowM,
                    sh_rowS, sh_fin, [](int ln, int c) { return c * 64 + ln; });
    } else {
        __syncthreads();  // finish_item's
    }
}

// ----------------------------------------------------------------------------
// exponential window on the atom grid: sliding recurrence along t0
// ----------------------------------------------------------------------------
//
// When t0 - t0_data, dt0, tau and dtau are whole multiples of TAtom (and
// nothing wraps around 2^32), the window of cell (m, n) covers the atoms
// k(m) = k00 + a*m .. k(m) + L(n) - 1, L(n) = 3*tau_n/TAtom, clipped at the
// data end, and atom k(m) + l has weight rho^l, rho = exp(-TAtom/tau_n)
// (exp.cu:53-90: t1 = t0 + 3 tau, so i_t1 = k + L - 1, and t0 <= t_i <= t1).
// The weighted window sum E(k) = sum_{l < L} rho^l x_{k+l} slides by one atom
// at a time:
//     E(k - 1) = rho E(k) + x_{k-1} - rho^L x_{k-1+L}
// (rho^2 and rho^2L = e^-6 for the a^2, b^2, ab columns; rho^L = e^-3), so a
// cell costs O(1) instead of O(L).  This first-order linear recurrence runs
// down the rows in chunks of RB rows (the map's row blocks), in parallel:
//   exp_init_kernel  E at the top row of the top chunk, by the direct O(L) sum;
//   exp_seg_kernel   Y(s): the recurrence across chunk s started from E = 0;
//   exp_scan_kernel  per tau column, E at every chunk top:
//                    E_top(s-1) = rho^(a RB) E_top(s) + Y(s);
//   exp_fast_kernel  each chunk walks its rows from E_top, evaluating F.
// Chunk s spans rows s*RB .. (s+1)*RB - 1 (rows past N_t0 are walked but not
// output).  Batches with many (template, column block) pairs use one chunk per
// column (RB up to 1024 rows): no exp_seg or exp_scan, and exp_fast adds the
// direct sum's parts itself.  Atoms at or past H (no output window reaches
// them) count as zero everywhere, which keeps the recurrence exact for every
// output row.  Atoms entering and leaving the windows of a chunk are staged
// in LDS, pass by pass; one thread per tau column.

struct ExpCol {
    double rho[2];   // rho^2 (a2, b2, ab), rho (Fa, Fb)
    double rhoL[2];  // rho^(2L) = exp(-6), rho^L = exp(-3)
    int L;
};

__device__ __forceinline__ ExpCol exp_col(const TmplDev &td, int n) {
    ExpCol ec;
    ec.L = td.L0 + td.Ls * n;
    const double tau = (double)td.tau + (double)n * (double)td.dtau;
    const double r1 = exp(-(double)td.TAtom / tau);
    ec.rho[0] = r1 * r1;
    ec.rho[1] = r1;
    ec.rhoL[1] = exp(-3.0);
    ec.rhoL[0] = exp(-6.0);
    return ec;
}

// Rows per work item of the recurrence at most (the walk stages its atoms in
// passes, so this bounds the item's pass bookkeeping, not its LDS).
constexpr int MAX_RB_EXPF = 1024;
// batches with fewer (template, column block) pairs than this walk the rows
// above the map instead of summing the top chunk directly
constexpr int64_t DIRECT_INIT_MIN_BLOCKS = 256;
// Untuned batches with at least DIRECT_INIT_MIN_BLOCKS pairs: row chunks per
// column block so that the map kernel has about this many work items.  When
// the pairs alone reach it, every column is one chunk: the map kernel walks
// it from the direct sum at its top and no chunk walk from zero (exp_seg) or
// chunk scan is needed.
constexpr int64_t EXP_TARGET_ITEMS = 512;
constexpr int INIT_PARTS = 8;  // blocks sharing one column block's direct sum
// exp_init beside exp_seg on a second stream only when the two launches hold
// at least this many blocks together (a fork and join costs ~10 µs)
constexpr int64_t EXP_FORK_MIN_BLOCKS = 1024;

// Atoms a walk stages in LDS, per pass of up to EXPW_PASS rows (dt0 == TAtom).
// Entering (head) atoms are the same on every lane of a row step: atom-major
// [j][8] doubles, read as broadcasts.  Leaving (tail) atoms differ per lane (L
// grows with the column): component planes [c][EXPW_TAIL_CAP] doubles, lanes
// Ls doubles apart (Ls = 3 for dtau = TAtom: 16 lanes hit 32 distinct banks).
// FP64 in LDS spares the walk a conversion per component and step.  Both
// ranges start one atom below the pass's last step, so every row reads the
// next row's atoms ahead (in range) while its own F is evaluated.
// 896 x 7 x 8 + 136 x 64 B = 58.9 KB: two workgroups per CU.
constexpr int EXPW_PASS = 128;
constexpr int EXPW_TAIL_CAP = 896;
constexpr int EXPW_HEAD_CAP = EXPW_PASS + 8;
constexpr int EXPF_LDS_BYTES = (NC * EXPW_TAIL_CAP + EXPW_HEAD_CAP * MERGED_STRIDE) *
                               (int)sizeof(double);
constexpr int EXPW_MAX_PASSES = MAX_RB_EXPF / 16;

// Rows per LDS pass of a walk over `cols` columns, or 0 when its atoms do not
// fit (dt0 > TAtom, or windows spread too far): the walk then reads the
// table directly.  A multiple of 4, at least 16.
__host__ __device__ __forceinline__ int expw_pass_rows(int a, int Ls, int cols) {
    if (a != 1) return 0;
    const int64_t room = (int64_t)EXPW_TAIL_CAP - 1 - (int64_t)Ls * (cols - 1);
    const int64_t pr = (room < EXPW_PASS ? room : (int64_t)EXPW_PASS) & ~(int64_t)3;
    return pr >= 16 ? (int)pr : 0;
}

struct ExpWalk {
    const float *X;   // the template's atom table (float32 merged sums)
    double *tl;       // LDS tail planes [c][EXPW_TAIL_CAP]
    double *hd;       // LDS head atoms [j][MERGED_STRIDE]
    int64_t head_lo;  // atom in head slot 0
    int64_t tail_lo;  // atom in tail slot 0
    int H;
};

__device__ __forceinline__ ExpWalk expw_init(const TmplDev &td, const float *X, double *lds) {
    ExpWalk wk;
    wk.X = X;
    wk.tl = lds;
    wk.hd = lds + NC * EXPW_TAIL_CAP;
    wk.head_lo = 0;
    wk.tail_lo = 0;
    wk.H = td.H;
    return wk;
}

// Staging of one pass: the atoms of the steps at rows sb..st (dt0 == TAtom)
// of columns col0..col_last -- head atoms k(m) - 1 and tail atoms k(m) - 1 +
// L(n), each range with one more atom below (read ahead at row sb); atoms
// outside [0, H) count as zero.  Thread tid moves component tid & 7 of atoms
// (tid >> 3) + 32 k (consecutive threads read consecutive doubles of the
// table), through registers: expw_fetch issues the loads, expw_put writes
// LDS, so the next pass's loads stay in flight during the current walk.
constexpr int EXPW_HEAD_PER = (EXPW_HEAD_CAP + 31) / 32;
constexpr int EXPW_TAIL_PER = EXPW_TAIL_CAP / 32;
static_assert(EXPW_TAIL_CAP % 32 == 0 && WG == 256, "staging decomposition");

struct ExpPass {
    int64_t head_lo, tail_lo;
    int nhead, ntail;
    float h[EXPW_HEAD_PER];  // exact: the table holds float32 sums
    float t[EXPW_TAIL_PER];
};

__device__ __forceinline__ void expw_fetch(const ExpWalk &wk, const TmplDev &td, int st, int sb,
                                           int col0, int col_last, ExpPass &ps) {
    ps.head_lo = (int64_t)td.k00 + sb - 2;
    ps.tail_lo = ps.head_lo + td.L0 + (int64_t)td.Ls * col0;
    ps.nhead = st - sb + 2;
    ps.ntail = ps.nhead + td.Ls * (col_last - col0);
    const int c = threadIdx.x & 7, j0 = threadIdx.x >> 3;
#pragma unroll
    for (int k = 0; k < EXPW_HEAD_PER; k++) {
        const int j = j0 + 32 * k;
        const int64_t atom = ps.head_lo + j;
        ps.h[k] = j < ps.nhead && atom >= 0 && atom < wk.H ? wk.X[atom * MERGED_STRIDE + c] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < EXPW_TAIL_PER; k++) {
        const int j = j0 + 32 * k;
        const int64_t atom = ps.tail_lo + j;
        ps.t[k] = c < NC && j < ps.ntail && atom >= 0 && atom < wk.H
                      ? wk.X[atom * MERGED_STRIDE + c]
                      : 0.0f;
    }
}

// The caller synchronises before the walk reads LDS.
__device__ __forceinline__ void expw_put(ExpWalk &wk, const ExpPass &ps) {
    wk.head_lo = ps.head_lo;
    wk.tail_lo = ps.tail_lo;
    const int c = threadIdx.x & 7, j0 = threadIdx.x >> 3;
#pragma unroll
    for (int k = 0; k < EXPW_HEAD_PER; k++) {
        const int j = j0 + 32 * k;
        if (j < ps.nhead) wk.hd[j * MERGED_STRIDE + c] = (double)ps.h[k];
    }
#pragma unroll
    for (int k = 0; k < EXPW_TAIL_PER; k++) {
        const int j = j0 + 32 * k;
        if (c < NC && j < ps.ntail) wk.tl[c * EXPW_TAIL_CAP + j] = (double)ps.t[k];
    }
}

// Operands of one row step from LDS: head slot jh (wave-uniform), tail slot jt.
__device__ __forceinline__ void expw_load(const ExpWalk &wk, int jh, int jt, double (&xh)[NC],
                                          double (&xt)[NC]) {
    const double *h = wk.hd + jh * MERGED_STRIDE;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        xh[c] = h[c];
        xt[c] = wk.tl[c * EXPW_TAIL_CAP + jt];
    }
}

// E(k - 1) = rho E(k) + (x_{k-1} - rho^L x_{k-1+L})
__device__ __forceinline__ void expw_step(const ExpCol &ec, const double (&xh)[NC],
                                          const double (&xt)[NC], double (&E)[NC]) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int g = c < 3 ? 0 : 1;
        const double d = fma(-ec.rhoL[g], xt[c], xh[c]);
        E[c] = fma(ec.rho[g], E[c], d);
    }
}

// One row step read from the table: k -> k - a (a atom steps).  The entering
// atoms k - l >= 0 for every step a walk takes.
__device__ __forceinline__ void expw_step_table(const ExpWalk &wk, const ExpCol &ec, int a,
                                                int64_t k, double (&E)[NC]) {
    for (int l = 1; l <= a; l++) {
        const int64_t kk = k - l;     // entering atom (wave-uniform)
        const int64_t kt = kk + ec.L;  // leaving atom
        const float *ph = wk.X + min(kk, (int64_t)wk.H - 1) * MERGED_STRIDE;
        const float *pt = wk.X + min(kt, (int64_t)wk.H - 1) * MERGED_STRIDE;
        double xh[NC], xt[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            xh[c] = kk < wk.H ? (double)ph[c] : 0.0;
            xt[c] = kt < wk.H ? (double)pt[c] : 0.0;
        }
        expw_step(ec, xh, xt, E);
    }
}

// Etab layout per template: [segment][component][tau column]
__device__ __forceinline__ double *expf_etab(double *etab, const TmplDev &td, int s, int c) {
    return etab + td.etab_off + ((int64_t)s * NC + c) * td.N_tau;
}

// Y(s), s >= 1: the recurrence across chunk s (from its top row down to the
// top row of chunk s-1) started from zero.  Work items (t, s, cb).
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(2, 2))) void exp_seg_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items,
    const float *__restrict__ merged, double *__restrict__ etab, int lds_ok) {
    extern __shared__ double lds_raw[];  // one dynamic LDS symbol per file
    const ItemDev it = items[block_slot()];
    const TmplDev td = tds[it.t];
    const int RB = td.rb_rows;
    const int col0 = it.cb * TILE_COLS;
    const int n = col0 + threadIdx.x;
    const int N_tau = (int)td.N_tau;
    const bool valid = n < N_tau;
    const int col_last = min(col0 + TILE_COLS, N_tau) - 1;
    // steps at rows r_top .. r_bot + 1
    const int r_top = (it.rb + 1) * RB - 1, r_bot = it.rb * RB - 1;
    const int ncol = valid ? n : col0;  // lanes past the map follow the first column
    const ExpCol ec = exp_col(td, ncol);
    ExpWalk wk = expw_init(td, merged + td.merged_off, lds_raw);
    double E[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) E[c] = 0.0;
    const int pr = lds_ok ? expw_pass_rows(td.a, td.Ls, col_last - col0 + 1) : 0;  // uniform
    if (pr > 0) {
        ExpPass ps;
        expw_fetch(wk, td, r_top, max(r_bot + 1, r_top - pr + 1), col0, col_last, ps);
        for (int st = r_top; st > r_bot; st -= pr) {
            const int sb = max(r_bot + 1, st - pr + 1);
            expw_put(wk, ps);
            __syncthreads();
            if (st - pr > r_bot)  // the next pass's atoms, in flight during this walk
                expw_fetch(wk, td, st - pr, max(r_bot + 1, st - 2 * pr + 1), col0, col_last, ps);
            int jh = st - sb + 1;
            int jt = jh + td.Ls * (ncol - col0);
            double xh[NC], xt[NC];
            expw_load(wk, jh, jt, xh, xt);
#pragma unroll 2
            for (int m = st; m >= sb; m--) {
                double nh[NC], nt[NC];
                expw_load(wk, jh - 1, jt - 1, nh, nt);  // the next row's atoms
                expw_step(ec, xh, xt, E);
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    xh[c] = nh[c];
                    xt[c] = nt[c];
                }
                jh--;
                jt--;
            }
            __syncthreads();  // the next pass restages
        }
    } else {
        int64_t k = (int64_t)td.k00 + (int64_t)td.a * r_top;
        for (int m = r_top; m > r_bot; m--) {
            expw_step_table(wk, ec, td.a, k, E);
            k -= td.a;
        }
    }
    if (valid) {
#pragma unroll
        for (int c = 0; c < NC; c++) expf_etab(etab, td, it.rb, c)[n] = E[c];
    }
}

// E at the top row of the top chunk, r = n_seg*RB - 1, by the direct sum
// E(k) = sum_{l < L} rho^l x_{k+l} (atoms at or past H count as zero, as in
// the walks), split over INIT_PARTS waves per (template, column block): part
// p sums its share of the block's l range into slot n_seg + p; the scan adds
// the parts.  Each lane sums INIT_GROUPS columns (its lane, + 64, + 128, +
// 192 of the block), so every atom, read from LDS as a broadcast, feeds up to
// 4 x 7 FMAs of Horner sums that run from the far end of the share, where the
// windows are longest, to its near end.  The wave stages its atoms in LDS in
// chunks of INIT_CHUNK with coalesced loads, the next chunk in flight in
// registers while the current one is summed.  The l range runs in segments
// that start where a column group's longest window ends (before that the
// group has nothing to sum); within 63 Ls atoms of that end the lanes of the
// group start one by one.
// Bound: FP64 issue (7 FMAs an atom and column) at 55% of it, the heaviest
// waves' shares.  256 templates of 512 columns, windows of 6 to 1540 atoms:
// 65 us with weights advanced beside forward sums (9 instructions an atom and
// column), now 55 (unrolled by 4 instead of 2: 90, spills).
constexpr int INIT_WG = 64;
constexpr int INIT_GROUPS = TILE_COLS / INIT_WG;
constexpr int INIT_CHUNK = 64;                                // atoms per LDS chunk (4 KB)
constexpr int INIT_PER = INIT_CHUNK * MERGED_STRIDE / INIT_WG;  // doubles per lane per chunk

struct InitState {
    double E[INIT_GROUPS][NC];
    double rho[INIT_GROUPS][2];
    int lr[INIT_GROUPS];  // this lane's window end, per group
};

template <bool MASK>
__device__ __forceinline__ void init_add(InitState &S, int i, int l, const double *x) {
    if (!MASK || l < S.lr[i]) {
#pragma unroll
        for (int c = 0; c < NC; c++) S.E[i][c] = fma(S.rho[i][c < 3 ? 0 : 1], S.E[i][c], x[c]);
    }
}

// atoms [a, b) of the chunk starting at atom c0, from b - 1 down, for the column
// groups I0 .. INIT_GROUPS - 1; the lanes of group I0 start at their windows'
// ends when MASK0, the later groups never need to (their shortest window
// reaches past b)
template <int I0, bool MASK0>
__device__ __forceinline__ void init_segment(InitState &S, const double *buf, int c0, int a,
                                             int b) {
#pragma unroll 2
    for (int l = b - 1; l >= a; l--) {
        double x[NC];
        const double *p = buf + (l - c0) * MERGED_STRIDE;  // broadcast
#pragma unroll
        for (int c = 0; c < NC; c++) x[c] = p[c];
        init_add<MASK0>(S, I0, l, x);
#pragma unroll
        for (int i = I0 + 1; i < INIT_GROUPS; i++) init_add<false>(S, i, l, x);
    }
}

__global__ __launch_bounds__(INIT_WG, 4) void exp_init_kernel(const TmplDev *__restrict__ tds,
                                                           const ItemDev *__restrict__ items,
                                                           const float *__restrict__ merged,
                                                           double *__restrict__ etab) {
    __shared__ double buf[INIT_CHUNK * MERGED_STRIDE];
    const ItemDev it = items[blockIdx.x];  // (t, part, column block)
    const int part = it.rb;
    const TmplDev td = tds[it.t];
    const int col0 = it.cb * TILE_COLS;
    const int col_last = min(col0 + TILE_COLS, (int)td.N_tau) - 1;
    const int lane = (int)threadIdx.x;
    const int64_t k0 = (int64_t)td.k00 + (int64_t)td.a * ((int64_t)td.n_seg * td.rb_rows - 1);
    const int64_t room = (int64_t)td.H - k0;
    // (H is an int32)
    auto clip = [&](int64_t L) { return (int)max(min(L, room), (int64_t)0); };
    // longest window of the block (L grows with n), clipped at H: uniform
    const int lr_blk = clip((int64_t)td.L0 + (int64_t)td.Ls * col_last);
    const int q = (lr_blk + INIT_PARTS - 1) / INIT_PARTS;
    const int l0 = min(part * q, lr_blk), l1 = min(lr_blk, l0 + q);
    InitState S;
    double w[INIT_GROUPS];  // rho^l0
    int lo0 = 0, hi[INIT_GROUPS];  // group 0's shortest window, each one's longest (uniform)
#pragma unroll
    for (int i = 0; i < INIT_GROUPS; i++) {
#pragma unroll
        for (int c = 0; c < NC; c++) S.E[i][c] = 0.0;
        const int g0 = col0 + INIT_WG * i;
        const int glast = min(g0 + INIT_WG - 1, col_last);
        const int n = min(g0 + lane, col_last);  // lanes past the map follow the last column
        const bool any = g0 <= col_last;
        S.lr[i] = any ? clip((int64_t)td.L0 + (int64_t)td.Ls * n) : 0;
        if (i == 0) lo0 = any ? clip((int64_t)td.L0 + (int64_t)td.Ls * g0) : 0;
        hi[i] = any ? clip((int64_t)td.L0 + (int64_t)td.Ls * glast) : hi[max(i, 1) - 1];
        const double tau = (double)td.tau + (double)n * (double)td.dtau;
        const double r1 = exp(-(double)td.TAtom / tau);
        S.rho[i][0] = r1 * r1;
        S.rho[i][1] = r1;
        w[i] = exp(-(double)l0 * (double)td.TAtom / tau);
    }
    // Windows grow with the column: group i's shortest window (lo) is at
    // least group i-1's longest (hi).  Atoms below lo[0] lie inside every
    // window; segment I0 = [hi[I0-1], hi[I0]) needs group I0 masked and no
    // group before it.
    const int seg_begin[5] = {0, lo0, hi[0], hi[1], hi[2]};
    // rows k0 + l, l < l1 <= room, lie below H
    const float *__restrict__ X = merged + td.merged_off + k0 * MERGED_STRIDE;
    float r[INIT_PER];  // exact: the table holds float32 sums
    auto fetch = [&](int c1) {  // atoms [max(l0, c1 - INIT_CHUNK), c1)
        const int c0 = max(l0, c1 - INIT_CHUNK);
        const int nq = (c1 - c0) * MERGED_STRIDE;
#pragma unroll
        for (int k = 0; k < INIT_PER; k++) {
            const int qd = k * INIT_WG + lane;
            r[k] = qd < nq ? X[(int64_t)c0 * MERGED_STRIDE + qd] : 0.0f;
        }
    };
    if (l0 < l1) fetch(l1);
    for (int c1 = l1; c1 > l0; c1 -= INIT_CHUNK) {
        const int c0 = max(l0, c1 - INIT_CHUNK);
        __syncthreads();  // the previous chunk is consumed
#pragma unroll
        for (int k = 0; k < INIT_PER; k++) buf[k * INIT_WG + lane] = (double)r[k];
        __syncthreads();
        if (c0 > l0) fetch(c0);  // in flight while this chunk is summed
        int sb = c1;
#pragma unroll
        for (int sgm = 4; sgm >= 0; sgm--) {
            const int sa = max(c0, min(sb, seg_begin[sgm]));
            if (sa < sb) {  // uniform
                if (sgm == 0) init_segment<0, false>(S, buf, c0, sa, sb);
                if (sgm == 1) init_segment<0, true>(S, buf, c0, sa, sb);
                if (sgm == 2) init_segment<1, true>(S, buf, c0, sa, sb);
                if (sgm == 3) init_segment<2, true>(S, buf, c0, sa, sb);
                if (sgm == 4) init_segment<3, true>(S, buf, c0, sa, sb);
            }
            sb = sa;
        }
    }
#pragma unroll
    for (int i = 0; i < INIT_GROUPS; i++) {
        const int n = col0 + INIT_WG * i + lane;
        if (n <= col_last) {
#pragma unroll
            for (int c = 0; c < NC; c++)
                expf_etab(etab, td, td.n_seg + part, c)[n] =
                    (c < 3 ? w[i] * w[i] : w[i]) * S.E[i][c];
        }
    }
}

// Per tau column: E at every chunk top.  Work items (t, -, cb).  With mult the
// weight factor of one chunk of rows, the chunk tops are V(n_seg-1) = the
// direct sum and V(s-1) = mult V(s) + Y(s).  Slot s holds Y(s) on entry and
// V(s) on exit (slot 0 has no Y).  A thread per (column, sum): its loads and
// stores coalesce over the columns, and SCAN_AHEAD slots are loaded together,
// since the loads' latency, not the recurrence, is the bound.
// One map of 2000 x 2000 cells (62 chunks): 13.4 us with a wave per column and a
// lane per chunk (log depth, but every lane on its own cache line), now 7.2
// (8.0 with 16 slots ahead, 9.4 with 8); 32 of 1000 x 1000: the three
// recurrence kernels 415, now 301.
constexpr int SCAN_WG = 64;
constexpr int SCAN_SPLIT = TILE_COLS / SCAN_WG;
constexpr int SCAN_AHEAD = 32;

__global__ __launch_bounds__(SCAN_WG) void exp_scan_kernel(const TmplDev *__restrict__ tds,
                                                           const ItemDev *__restrict__ items,
                                                           double *__restrict__ etab) {
    const ItemDev it = items[blockIdx.x / (SCAN_SPLIT * NC)];
    const TmplDev td = tds[it.t];
    const int part = (int)(blockIdx.x % (SCAN_SPLIT * NC));
    const int c = part / SCAN_SPLIT;
    const int n = it.cb * TILE_COLS + part % SCAN_SPLIT * SCAN_WG + (int)threadIdx.x;
    if (n >= (int)td.N_tau) return;
    const double tau = (double)td.tau + (double)n * (double)td.dtau;
    const double steps = (double)td.a * td.rb_rows;
    const double m1 = exp(-(double)td.TAtom * steps / tau);
    const double mult = c < 3 ? m1 * m1 : m1;
    double E = 0.0;
    if (!td.init_empty) {  // top chunk: the direct sum's parts
        double y[INIT_PARTS];
#pragma unroll
        for (int pp = 0; pp < INIT_PARTS; pp++) y[pp] = expf_etab(etab, td, td.n_seg + pp, c)[n];
#pragma unroll
        for (int pp = 0; pp < INIT_PARTS; pp++) E += y[pp];
    }
    double *slot0 = expf_etab(etab, td, 0, c) + n;
    const int64_t stride = (int64_t)NC * td.N_tau;
    for (int s = td.n_seg - 1; s >= 1; s -= SCAN_AHEAD) {
        double Y[SCAN_AHEAD];
#pragma unroll
        for (int u = 0; u < SCAN_AHEAD; u++)  // (slot 1 again past the end)
            Y[u] = slot0[max(s - u, 1) * stride];
#pragma unroll
        for (int u = 0; u < SCAN_AHEAD; u++)
            if (s - u >= 1) {  // uniform
                slot0[(s - u) * stride] = E;
                E = fma(mult, E, Y[u]);
            }
    }
    slot0[0] = E;
}

// Rows st .. sb of a chunk (one pass) in groups of 4 (the pass's rows are a
// multiple of 4), reduced together.  Rows past the map (m > m_hi, only in a
// template's last chunk) are evaluated but neither stored nor reduced, which
// keeps the loop free of branches.  LDS: the pass's atoms are staged (dt0 ==
// TAtom), jt_off = Ls * (the
// lane's column - the first column); otherwise each step reads the table.
template <bool BTSG, bool STRICT, bool LDS>
__device__ __forceinline__ void expw_rows(const TmplDev &td, const ExpWalk &wk, const ExpCol &ec,
                                          double (&E)[NC], Reducer<BTSG, 1> &red, bool &single,
                                          float *__restrict__ Ft, int st, int sb, int row0,
                                          int m_hi, int n, bool valid, int lane, int jt_off,
                                          float *sh_rowM, float *sh_rowS) {
    const int N_tau = (int)td.N_tau;
    const int colidx[1] = {n};
    int64_t k = (int64_t)td.k00 + (int64_t)td.a * st;  // first window atom of row m
    // stores without a branch: one buffer resource over the pass's rows inside
    // the map, a byte offset per lane that falls outside it for lanes past the
    // last column (2^31 and below it by less than 2^31 minus the resource's
    // size, as the plan bounds N_tau); rows past the map lie beyond it too
    const int nv = min(st, m_hi) - sb + 1;
    const uint32_t rowb = (uint32_t)N_tau * (uint32_t)sizeof(float);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        Ft + (int64_t)sb * N_tau, (short)0, nv > 0 ? (int)((uint32_t)nv * rowb) : 0,
        BUF_RSRC_WORD3);
    uint32_t vo = valid ? (uint32_t)(st - sb) * rowb + (uint32_t)n * (uint32_t)sizeof(float)
                        : 0x80000000u;  // row st
    // LDS path: head and tail slots of the step at the group's first row;
    // the group's rows address slots below them by constants
    int jh = st - sb + 1;
    int jt = jh + jt_off;
    double xh[NC], xt[NC];
    if (LDS) expw_load(wk, jh, jt, xh, xt);
    for (int g = st; g >= sb; g -= 4) {
        const bool last = g - 3 == row0;
        float F4[4][1];  // F4[r] is row g - 3 + r
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int m = g - j;
            double nh[NC], nt[NC];
            if (LDS) expw_load(wk, jh - 1 - j, jt - 1 - j, nh, nt);  // the next row's atoms
            // every lane evaluates F (no branch around it, so the compiler
            // can overlap the rows' evaluations); stores and masks follow
            F4[3 - j][0] = cell_F(E[0], E[1], E[2], E[3], E[4], E[5], E[6]);
            if (STRICT) single |= valid && m <= m_hi && (k >= (int64_t)td.N - 1);
            // the chunk's final row takes no step: from the table it could
            // read below atom 0; from LDS the step reads staged slots and its
            // result is never used, so it runs unconditionally (no branch)
            if (LDS)
                expw_step(ec, xh, xt, E);
            else if (j < 3 || !last)
                expw_step_table(wk, ec, td.a, k, E);
            if (LDS) {
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    xh[c] = nh[c];
                    xt[c] = nt[c];
                }
            }
            k -= td.a;
        }
        jh -= 4;
        jt -= 4;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = g - 3 + r;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(F4[r][0]), rs,
                                                  (int)(vo - (uint32_t)(3 - r) * rowb), 0, 0);
            F4[r][0] = valid && m <= m_hi ? F4[r][0] : -INFINITY;
        }
        vo -= 4 * rowb;
        if (g - 3 <= m_hi)
            red.add(F4, g - 3, colidx, N_tau, lane, g - 3 - sb, sh_rowM, sh_rowS);
    }
}

// The map: chunk rb walks rows (rb+1)*RB - 1 .. rb*RB from E_top(rb), in
// passes.  BTSG row sums: after each pass the 4 waves' sums of its rows are
// combined relative to the pass reference (the waves' largest reference then)
// and written; at the end, the rows of passes whose reference lies below the
// item's are rescaled by the threads that wrote them.
template <bool BTSG, bool STRICT>
// Two workgroups share a CU (LDS): registers for two waves per SIMD.
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(2, 2))) void exp_fast_kernel(
    const TmplDev *__restrict__ tds, const ItemDev *__restrict__ items, int64_t item0,
    const float *__restrict__ merged, const double *__restrict__ etab,
    float *__restrict__ Fout, ItemPart *__restrict__ ipart, float *__restrict__ rowpart,
    float *__restrict__ colpart, int *__restrict__ flags, int lds_ok) {
    extern __shared__ double lds_raw[];  // one dynamic LDS symbol per file
    __shared__ float sh_rowM[4][EXPW_PASS];
    __shared__ float sh_rowS[4][EXPW_PASS];
    __shared__ float sh_passM[EXPW_MAX_PASSES];
    __shared__ float sh_best[4];
    __shared__ int sh_bidx[4];
    __shared__ float sh_M[4];
    __shared__ float sh_S[4];
    const int64_t item_id = item0 + block_slot();
    const ItemDev it = items[item_id];
    const TmplDev td = tds[it.t];
    const int RB = td.rb_rows;
    const int row0 = it.rb * RB;
    const int N_t0 = (int)td.N_t0, N_tau = (int)td.N_tau;
    const int r_top = row0 + RB - 1;
    const int m_hi = min(r_top, N_t0 - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int col0 = it.cb * TILE_COLS;
    const int n = col0 + threadIdx.x;
    const bool valid = n < N_tau;
    const int col_last = min(col0 + TILE_COLS, N_tau) - 1;
    const int ncol = valid ? n : col0;
    const ExpCol ec = exp_col(td, ncol);
    ExpWalk wk = expw_init(td, merged + td.merged_off, lds_raw);
    double E[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) E[c] = 0.0;
    if (valid && td.n_seg > 1) {
#pragma unroll
        for (int c = 0; c < NC; c++) E[c] = expf_etab((double *)etab, td, it.rb, c)[n];
    } else if (valid && !td.init_empty) {  // one chunk: E_top is the direct sum's parts
#pragma unroll
        for (int pp = 0; pp < INIT_PARTS; pp++)
#pragma unroll
            for (int c = 0; c < NC; c++) E[c] += expf_etab((double *)etab, td, 1 + pp, c)[n];
    }

    Reducer<BTSG, 1> red;
    red.init();
    bool single = false;
    float *__restrict__ Ft = Fout + td.F_off;
    float *__restrict__ rp = rowpart + td.rowpart_off + (int64_t)it.cb * td.N_t0;
    const int prl = lds_ok ? expw_pass_rows(td.a, td.Ls, col_last - col0 + 1) : 0;  // uniform
    const int pr = prl > 0 ? prl : EXPW_PASS;
    int npass = 0;
    ExpPass ps;
    if (prl > 0) expw_fetch(wk, td, r_top, max(row0, r_top - pr + 1), col0, col_last, ps);
    for (int st = r_top; st >= row0; st -= pr, npass++) {
        const int sb = max(row0, st - pr + 1);
        if (prl > 0) {
            expw_put(wk, ps);
            __syncthreads();
            if (st - pr >= row0)  // the next pass's atoms, in flight during this walk
                expw_fetch(wk, td, st - pr, max(row0, st - 2 * pr + 1), col0, col_last, ps);
            expw_rows<BTSG, STRICT, true>(td, wk, ec, E, red, single, Ft, st, sb, row0, m_hi, n,
                                          valid, lane, td.Ls * (ncol - col0), sh_rowM[wave],
                                          sh_rowS[wave]);
        } else {
            expw_rows<BTSG, STRICT, false>(td, wk, ec, E, red, single, Ft, st, sb, row0, m_hi, n,
                                           valid, lane, 0, sh_rowM[wave], sh_rowS[wave]);
        }
        const int nv = min(st, m_hi) - sb + 1;  // rows of the pass inside the map
        if (BTSG && nv > 0) {  // block-uniform
            if (lane == 0) sh_M[wave] = red.ML;
            __syncthreads();
            const float Ms = fmaxf(fmaxf(sh_M[0], sh_M[1]), fmaxf(sh_M[2], sh_M[3]));
            for (int rl = threadIdx.x; rl < nv; rl += WG) {
                float S = 0.0f;
#pragma unroll
                for (int w = 0; w < 4; w++)
                    if (sh_M[w] != -INFINITY) S += sh_rowS[w][rl] * exp2_diff(sh_rowM[w][rl], Ms);
                rp[sb + rl] = S;
            }
            if (threadIdx.x == 0) sh_passM[npass] = Ms;
        }
        __syncthreads();  // staging, row sums and sh_M are rewritten by the next pass
    }
    if (STRICT && single) atomicOr(flags + it.t, FLAG_SINGLE_ATOM);
    // combine: each column belongs to one lane; each row to all 4 waves
    wave_argmax(red.best, red.bidx);
    float stot = 0.0f;
    if (BTSG) stot = wave_sum(red.total());
    if (lane == 0) {
        sh_best[wave] = red.best;
        sh_bidx[wave] = red.bidx;
        sh_M[wave] = red.ML;
        sh_S[wave] = stot;
    }
    __syncthreads();
    const float M = fmaxf(fmaxf(sh_M[0], sh_M[1]), fmaxf(sh_M[2], sh_M[3]));
    if (BTSG) {
        if (valid)
            colpart[td.colpart_off + (int64_t)it.rb * td.N_tau + n] =
                red.ML == -INFINITY ? 0.0f : red.Scol[0] * exp2_diff(red.ML, M);
        // rows written relative to an earlier, lower reference: the same
        // threads (same rows) rescale them
        for (int j = 0; j < npass; j++) {
            const int st = r_top - j * pr;
            const int sb = max(row0, st - pr + 1);
            const int nv = min(st, m_hi) - sb + 1;
            if (nv <= 0) continue;
            const float Ms = sh_passM[j];
            if (Ms == M || Ms == -INFINITY) continue;  // block-uniform
            const float sc = exp2_diff(Ms, M);
            for (int rl = threadIdx.x; rl < nv; rl += WG) rp[sb + rl] *= sc;
        }
    }
    if (threadIdx.x == 0) {
        float bv = sh_best[0];
        int bi = sh_bidx[0];
#pragma unroll
        for (int w = 1; w < 4; w++) argmax_merge(bv, bi, sh_best[w], sh_bidx[w]);
        float S = 0.0f;
        if (BTSG) {
#pragma unroll
            for (int w = 0; w < 4; w++)
                if (sh_M[w] != -INFINITY) S += sh_S[w] * exp2_diff(sh_M[w], M);
        }
        ipart[item_id] = ItemPart{bv, bi, M, S};
    }
}

// ----------------------------------------------------------------------------
// finalize: per-template stats from the partials
// ----------------------------------------------------------------------------

constexpr int FIN_SCALE_CAP = 4096;        // per-item scale factors kept in LDS
// Batches smaller than this finalize with 1024 threads (1024 templates with
// 1024 threads each: 125 x 125 cells 17 us, 250-2000 rows and columns 40-46 us;
// with 256 threads 9.5 and 39).
constexpr int64_t FIN_WIDE_MAX_T = 256;
// Partials of a row or column loaded together (1024 templates of 250 to 2000
// rows and columns: 66 us one by one, 50 by 4, 43 by 8, 39 by 12).
constexpr int FIN_AHEAD = 12;

// FP64 values across the wave without LDS, as wave_sum and wave_max do for
// floats: every lane ends with the same bits.
template <typename Op>
__device__ __forceinline__ double wave_reduce_d(double v, Op op) {
    v = op(v, dpp_d<DPP_QUAD_XOR1>(v));
    v = op(v, dpp_d<DPP_QUAD_XOR2>(v));
    v = op(v, dpp_d<DPP_ROW_ROR4>(v));
    v = op(v, dpp_d<DPP_ROW_ROR8>(v));
    auto both = [](unsigned lo, unsigned hi) {
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    };
    {
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        const auto l = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32),
                                                        false, false);
        v = op(both(l[0], h[0]), both(l[1], h[1]));
    }
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false,
                                                    false);
    return op(both(l[0], h[0]), both(l[1], h[1]));
}

__device__ __forceinline__ double wave_sum_d(double v) {
    return wave_reduce_d(v, [](double a, double b) { return a + b; });
}

// Wave argmax of doubles (none NaN), the first index on ties.
__device__ __forceinline__ void wave_argmax_d(double &v, int &i) {
    const double m = wave_reduce_d(v, [](double a, double b) { return a > b ? a : b; });
    i = wave_min_idx(v == m ? i : 0x7fffffff);
    v = m;
}

// The sum, in order, of the partials p[0], p[stride], ... (count of them), each
// times its item's scale, of a row or column; FIN_AHEAD loads in flight.
template <typename Scale>
__device__ __forceinline__ double partial_sum(const float *__restrict__ p, uint32_t count,
                                              uint32_t stride, Scale scale) {
    double sum = 0.0;
    for (uint32_t b = 0; b < count; b += FIN_AHEAD) {
        float x[FIN_AHEAD];
#pragma unroll
        for (uint32_t u = 0; u < FIN_AHEAD; u++)  // (a repeated load past the end, not added)
            x[u] = p[(int64_t)min(b + u, count - 1) * stride];
#pragma unroll
        for (uint32_t u = 0; u < FIN_AHEAD; u++)
            if (b + u < count) sum += (double)(x[u] * scale(b + u));
    }
    return sum;
}

// One workgroup of NT threads per template (NT = 1024 for small batches, whose
// maps are large, 256 otherwise): the argmax of F with the largest item
// reference Mref (log2 units), then the lnBtSG sum and the two posterior
// argmaxes.  Item k's partials are relative to 2^(M_k) (M_k = -inf: no valid
// cell, partials 0), rescaled here by exp((M_k - Mref) / LOG2E) <= 1, so no
// item reference needs maxF; the row and column partials of a thread are read
// in one pass.
//
// Bound: latency -- the descriptor, the items, three barriers, and each
// thread's partials (2000 x 2000 cells at 192 rows an item are 8 passes of 8 +
// 11 loads).  The reductions go through DPP; with pairwise exchanges through
// LDS and partials read one by one: 128 maps of 250 to 1000 rows 16 us, now
// 10; one map of 47 x 46 cells 10, now 5; 1024 maps of 250 to 2000 rows 66, now
// 39.
template <bool BTSG, int NT>
__global__ __launch_bounds__(NT) void finalize_kernel(
    const TmplDev *__restrict__ tds, const ItemPart *__restrict__ ipart,
    const float *__restrict__ rowpart, const float *__restrict__ colpart,
    const int *__restrict__ flags, tcw_stats *__restrict__ stats) {
    constexpr int NW = NT / 64;
    __shared__ float sh_scale[FIN_SCALE_CAP];
    __shared__ float sh_max[NW], sh_M[NW];
    __shared__ int sh_idx[NW];
    __shared__ double sh_sum[NW], sh_row[NW], sh_colv[NW];
    __shared__ int sh_ri[NW], sh_ci[NW];
    constexpr double INV_LOG2E = 1.0 / (double)LOG2E;
    const int t = blockIdx.x;
    const TmplDev td = tds[t];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t nitems = (int64_t)td.n_rowblk * td.n_colblk;
    const ItemPart *ip = ipart + td.item_begin;
    float bv = -INFINITY, Mref = -INFINITY;
    int bi = 0x7fffffff;
    ItemPart first{-INFINITY, 0x7fffffff, -INFINITY, 0.0f};
    for (int64_t k = threadIdx.x; k < nitems; k += NT) {
        const ItemPart q = ip[k];
        if (k < NT) first = q;  // the only one unless the template has over NT items
        argmax_merge(bv, bi, q.maxF, q.idx);
        Mref = fmaxf(Mref, q.M);
    }
    wave_argmax(bv, bi);
    Mref = wave_max(Mref);
    if (lane == 0) {
        sh_max[wave] = bv;
        sh_idx[wave] = bi;
        sh_M[wave] = Mref;
    }
    __syncthreads();
    bv = lane < NW ? sh_max[lane] : -INFINITY;
    bi = lane < NW ? sh_idx[lane] : 0x7fffffff;
    Mref = wave_max(lane < NW ? sh_M[lane] : -INFINITY);
    wave_argmax(bv, bi);
    const float maxF = bv;
    const int64_t m_ML = bi / (int)td.N_tau;
    const int64_t n_ML = bi - m_ML * (int64_t)td.N_tau;

    double lnB = NAN, t0_MP = NAN, tau_MP = NAN;
    int64_t m_MP = -1, n_MP = -1;
    if (BTSG) {
        auto item_scale = [&](float Mk) -> float {
            return Mk == -INFINITY ? 0.0f : __expf((float)((double)(Mk - Mref) * INV_LOG2E));
        };
        double s = 0.0;
        for (int64_t k = threadIdx.x; k < nitems; k += NT) {
            const float Mk = k < NT ? first.M : ip[k].M, Sk = k < NT ? first.S : ip[k].S;
            const float sc = item_scale(Mk);
            if (k < FIN_SCALE_CAP) sh_scale[k] = sc;
            s += (double)Sk * (double)sc;
        }
        s = wave_sum_d(s);
        if (lane == 0) sh_sum[wave] = s;
        __syncthreads();  // sh_scale and sh_sum are complete
        auto scale = [&](uint32_t k) -> float {
            return k < FIN_SCALE_CAP ? sh_scale[k] : item_scale(ip[k].M);
        };
        double rv = -1.0, cv = -1.0;
        int ri = 0x7fffffff, ci = 0x7fffffff;
        const int nmax = max((int)td.N_t0, (int)td.N_tau);
        for (int i = threadIdx.x; i < nmax; i += NT) {
            double R = -1.0, Cs = -1.0;
            if (i < (int)td.N_t0) {  // row i: [colblk][N_t0]
                const uint32_t k0 = (uint32_t)(i / td.rb_rows) * td.n_colblk;
                R = partial_sum(rowpart + td.rowpart_off + i, td.n_colblk, td.N_t0,
                                [&](uint32_t cb) { return scale(k0 + cb); });
            }
            if (i < (int)td.N_tau) {  // column i: [rowblk][N_tau]
                const uint32_t cb = (uint32_t)(i / td.tile);
                Cs = partial_sum(colpart + td.colpart_off + i, td.n_rowblk, td.N_tau,
                                 [&](uint32_t rb) { return scale(rb * td.n_colblk + cb); });
            }
            if (R > rv) {  // i grows within a thread: the first maximum stays
                rv = R;
                ri = i;
            }
            if (Cs > cv) {
                cv = Cs;
                ci = i;
            }
        }
        wave_argmax_d(rv, ri);
        wave_argmax_d(cv, ci);
        if (lane == 0) {
            sh_row[wave] = rv;
            sh_ri[wave] = ri;
            sh_colv[wave] = cv;
            sh_ci[wave] = ci;
        }
        __syncthreads();
        if (wave > 0) return;
        rv = lane < NW ? sh_row[lane] : -1.0;
        ri = lane < NW ? sh_ri[lane] : 0x7fffffff;
        cv = lane < NW ? sh_colv[lane] : -1.0;
        ci = lane < NW ? sh_ci[lane] : 0x7fffffff;
        wave_argmax_d(rv, ri);
        wave_argmax_d(cv, ci);
        s = wave_sum_d(lane < NW ? sh_sum[lane] : 0.0);
        lnB = log(70.0 / ((double)td.N_t0 * (double)td.N_tau)) + (double)Mref * INV_LOG2E + log(s);
        m_MP = ri;
        n_MP = ci;
        t0_MP = (double)td.o_t0 + ((double)m_MP + 0.5) * ((double)td.o_t0Band / (double)td.N_t0);
        tau_MP = (double)td.o_tau + ((double)n_MP + 0.5) * ((double)td.o_tauBand / (double)td.N_tau);
    }
    if (threadIdx.x == 0) {
        tcw_stats st;
        st.maxF = maxF;
        st.single_atom = flags[t] & FLAG_SINGLE_ATOM;
        st.m_ML = m_ML;
        st.n_ML = n_ML;
        st.N_t0 = td.N_t0;
        st.N_tau = td.N_tau;
        st.t0_ML = (int64_t)td.t0 + m_ML * (int64_t)td.dt0;
        st.tau_ML = (int64_t)td.tau + n_ML * (int64_t)td.dtau;
        st.lnBtSG = lnB;
        st.m_MP = m_MP;
        st.n_MP = n_MP;
        st.t0_MP = t0_MP;
        st.tau_MP = tau_MP;
        st.numAtoms = td.N;
        st.t0_data = td.t_min;
        stats[t] = st;
    }
}

// ----------------------------------------------------------------------------
// binned merge for many templates (tcw_merge_batch) and its adjoint
// ----------------------------------------------------------------------------

struct MergeTmpl {
    int64_t seg_begin, seg_end;  // into the SegDev table
    int64_t out_off;             // first merged bin of the template
    uint32_t N, t_min;
};

// A workgroup owns MERGE_BINS consecutive bins of one template.  Per detector
// the block's atoms are bounded; chunk by chunk their bins are
// formed, the first atom of every bin is marked where the bin changes, and each
// thread sums the atoms of its bins, MERGE_WG apart, so that the lanes' reads of
// the columns and the stores are nearly and exactly consecutive.  Float32 sums,
// detectors in order, atoms in order -- the accumulation order of
// mergeMultiFstatAtomsBinned, so the result is bit-identical to the stage
// kernel's merge.  atom_bin[k] = out_off + (ts[k] - t_min) / TA of every atom is
// written by the blocks in equal shares of the atoms.
// Bound: HBM bytes -- 32 an atom in, 28 a bin and 8 an atom out.  512 templates
// of 2 x 1844 atoms: 33 us with a binary search of the timestamps per bin and
// 7 for the atoms' bins in a kernel of its own, 24 together so (4.3 TB/s).
constexpr int MERGE_WG = 256;
constexpr int MERGE_PER = 4;                      // bins and atoms of a thread
constexpr int MERGE_BINS = MERGE_WG * MERGE_PER;  // bins per block, atoms per chunk

__global__ __launch_bounds__(MERGE_WG) void merge_kernel(
    const MergeTmpl *__restrict__ mt, const SegDev *__restrict__ segs, int64_t T,
    const uint32_t *__restrict__ ts, const float *__restrict__ cols, int64_t cstride,
    uint32_t TA, float *__restrict__ out, int64_t ostride, int64_t *__restrict__ atom_bin) {
    __shared__ int s_bin[MERGE_BINS], s_first[MERGE_BINS];
    __shared__ int64_t s_rng[4];
    const int tid = threadIdx.x;
    for (int64_t t = blockIdx.y; t < T; t += gridDim.y) {
        const MergeTmpl m = mt[t];
        const uint32_t B0 = blockIdx.x * (uint32_t)MERGE_BINS;
        if (B0 >= m.N) continue;  // block-uniform
        const int nb = (int)min(m.N - B0, (uint32_t)MERGE_BINS);
        const int64_t blocks = ((int64_t)m.N + MERGE_BINS - 1) / MERGE_BINS;  // of the template
        const uint64_t t_lo = (uint64_t)m.t_min + (uint64_t)B0 * TA;
        const uint64_t t_hi = t_lo + (uint64_t)nb * TA;
        float v[MERGE_PER][NC];
#pragma unroll
        for (int j = 0; j < MERGE_PER; j++)
#pragma unroll
            for (int c = 0; c < NC; c++) v[j][c] = 0.0f;
        for (int64_t s = m.seg_begin; s < m.seg_end; s++) {
            const SegDev sg = segs[s];
            const int two = (int)(s - m.seg_begin) & 1;  // bounded two at a time
            if (two == 0) bound_two(ts, segs, s, m.seg_end, t_lo, t_hi, s_rng);
            const int64_t ka = s_rng[2 * two], kb = s_rng[2 * two + 1];
            for (int64_t c0 = ka; c0 < kb; c0 += MERGE_BINS) {  // block-uniform
                const int na = (int)min((int64_t)MERGE_BINS, kb - c0);
                int bin[MERGE_PER];
#pragma unroll
                for (int j = 0; j < MERGE_PER; j++) {
                    const int i = j * MERGE_WG + tid;
                    bin[j] = i < na ? (int)((ts[c0 + i] - (uint32_t)t_lo) / TA) : MERGE_BINS;
                    s_bin[i] = bin[j];
                    s_first[i] = -1;
                }
                __syncthreads();
#pragma unroll
                for (int j = 0; j < MERGE_PER; j++) {
                    const int i = j * MERGE_WG + tid;
                    if ((unsigned)bin[j] < (unsigned)MERGE_BINS && (i == 0 || s_bin[i - 1] != bin[j]))
                        s_first[bin[j]] = i;
                }
                __syncthreads();
                const float *__restrict__ col = cols + c0;
                int k[MERGE_PER];
                float x[MERGE_PER][NC];  // the bins' first atoms, all loads in flight
#pragma unroll
                for (int j = 0; j < MERGE_PER; j++) {
                    k[j] = s_first[j * MERGE_WG + tid];
#pragma unroll
                    for (int c = 0; c < NC; c++) x[j][c] = col[c * cstride + max(k[j], 0)];
                }
#pragma unroll
                for (int j = 0; j < MERGE_PER; j++) {
                    if (k[j] < 0) continue;
#pragma unroll
                    for (int c = 0; c < NC; c++) v[j][c] += x[j][c];
                    for (int q = k[j] + 1; q < na && s_bin[q] == j * MERGE_WG + tid; q++) {
#pragma unroll
                        for (int c = 0; c < NC; c++) v[j][c] += col[c * cstride + q];
                    }
                }
                __syncthreads();  // bins consumed before the next chunk
            }
            if (atom_bin)  // the block's share of the detector's atoms
                for (int64_t k = sg.begin + B0 + tid; k < sg.end; k += blocks * MERGE_BINS)
#pragma unroll
                    for (int j = 0; j < MERGE_PER; j++)
                        if (k + j * MERGE_WG < sg.end)
                            atom_bin[k + j * MERGE_WG] =
                                m.out_off + (int64_t)((ts[k + j * MERGE_WG] - m.t_min) / TA);
            __syncthreads();  // s_rng is rewritten by the next detector
        }
#pragma unroll
        for (int j = 0; j < MERGE_PER; j++) {
            const int b = j * MERGE_WG + tid;
            if (b < nb) {
#pragma unroll
                for (int c = 0; c < NC; c++) out[c * ostride + m.out_off + B0 + b] = v[j][c];
            }
        }
    }
}

__global__ __launch_bounds__(256) void gather_bins_kernel(const float *__restrict__ in,
                                                          int64_t istride,
                                                          const int64_t *__restrict__ atom_bin,
                                                          int64_t n, float *__restrict__ out,
                                                          int64_t ostride) {
    for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < n;
         j += (int64_t)gridDim.x * 256) {
        const int64_t b = atom_bin[j];
#pragma unroll
        for (int c = 0; c < NC; c++) out[c * ostride + j] = in[c * istride + b];
    }
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------

using tcwc::DevBuf;
using tcwc::fail;
using tcwc::set_device;


}  // namespace

// Host data on its way to the device for one call: gathered in pinned memory and
// sent by one copy into one device buffer, of which the destinations are
// views.  Grow-only up to HOST_STAGE_MAX; the caller waits for the stream
// before the next use.
constexpr size_t HOST_STAGE_MAX = 16u << 20;
struct HostStage {
    char *pin = nullptr;
    size_t cap = 0;
    DevBuf dev;
    int ensure(size_t bytes) {
        const int rc = ensure_pin(bytes);
        return rc ? rc : dev.ensure(bytes);
    }
    int ensure_pin(size_t bytes) {
        if (bytes > cap) {
            if (pin) (void)hipHostFree(pin);
            pin = nullptr;
            cap = 0;
            if (hipHostMalloc((void **)&pin, bytes, hipHostMallocDefault) != hipSuccess) {
                pin = nullptr;
                return fail(TCW_ERR_NOMEM, "hipHostMalloc of " + std::to_string(bytes) + " bytes failed");
            }
            cap = bytes;
        }
        return TCW_OK;
    }
    ~HostStage() {
        if (pin) (void)hipHostFree(pin);
        dev.release();
    }
};
// A batch plan's descriptors go in one pageable copy up to this size (planning 256
// maps of 48 x 48 to 240 x 240 cells: seven allocations and copies 89 us, one of
// each 50); beyond it the bytes count, and gathering them would double those.
constexpr size_t PACKED_TABLES_MAX = 256u << 10;
constexpr size_t stage_align(size_t bytes) { return (bytes + 255) / 256 * 256; }

struct tcw_plan {
    int device = 0;
    uint32_t flags = 0;
    int64_t T = 0;
    std::vector<TmplDev> tmpl;
    std::vector<SegDev> segs;
    std::vector<ItemDev> items;      // grouped by mode
    std::vector<ItemDev> seg_items;  // MODE_EXP_FAST (t, chunk, column block), chunk >= 1
    std::vector<ItemDev> col_items;  // MODE_EXP_FAST (t, -, column block)
    std::vector<ItemDev> init_items;  // exp_init waves (t, part, column block), heaviest first
    std::vector<int32_t> exp_tmpls;  // templates needing the atom table
    // templates needing the prefix table, per stage_kernel class, longest first
    std::vector<int32_t> rect_tmpls[SR_CLASSES];
    // exp_tmpls, then the classes of rect_tmpls (one buffer: a single map fills no more of it)
    std::vector<int32_t> tmpl_list;
    int64_t exp_max_N = 0;
    bool exp_init_needed = false;  // some exp template has a non-empty direct sum
    int64_t mode_begin[MODE_COUNT + 1] = {0, 0, 0, 0, 0};
    int64_t prefix_doubles = 0, merged_floats = 0, rowpart_n = 0, colpart_n = 0;
    int64_t etab_doubles = 0;
    int64_t F_total = 0;
    int max_lds_bytes = 0;  // rect_fast_kernel dynamic LDS
    int max_lds_expf = 0;   // exp_fast_kernel dynamic LDS
    int max_lds_walk = 0;   // exp_walk_kernel dynamic LDS
    int max_lds_step = 0;   // rect_step_kernel dynamic LDS
    int64_t walk_tmpls = 0, direct_tmpls = 0;   // MODE_EXP_DIRECT templates of either kernel
    int64_t step_tmpls = 0, generic_tmpls = 0;  // MODE_RECT_GENERIC templates of either kernel
    DevBuf d_tmpl, d_segs, d_items, d_prefix, d_merged, d_ipart, d_rowpart, d_colpart,
        d_flags, d_seg_items, d_col_items, d_etab, d_tmpl_list, d_init_items;
    hipGraphExec_t graph = nullptr;
    hipStream_t cap_stream = nullptr;  // private stream the graph is captured on
    // exp_init_kernel runs here beside exp_seg_kernel (they are independent)
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    const void *g_ts = nullptr, *g_cols = nullptr, *g_F = nullptr, *g_stats = nullptr;
    int64_t g_cstride = -1;
    // rows per work item requested for each kernel mode (0: built-in choice)
    int32_t rows_req[MODE_COUNT] = {0, 0, 0, 0};
    // when set, the descriptors (and ts / cols, if host_ts) go through it in one copy
    HostStage *stage = nullptr;
    const uint32_t *host_ts = nullptr;  // n_host_atoms timestamps
    const float *host_cols = nullptr;   // [7][n_host_atoms]
    int64_t n_host_atoms = 0;
    DevBuf d_ts, d_cols;                // views of the stage's device buffer
    DevBuf d_tables;  // a batch plan's small descriptors: views of this one
    // when set, device buffers are views into this memory (tcw_map_noalloc)
    char *arena = nullptr;
    size_t arena_bytes = 0;
    bool arena_short = false;  // the last plan needed more than arena_bytes
    // the layout that decides what the arena accepts, so that a faster one
    // neither refuses nor accepts other maps: COMPACT_* rows and, off the grid,
    // the per-cell kernels
    bool compact = false;
    bool dry = false;  // stop once the scratch is sized
    void reset() {
        tmpl.clear();
        segs.clear();
        items.clear();
        seg_items.clear();
        col_items.clear();
        init_items.clear();
        exp_tmpls.clear();
        for (auto &r : rect_tmpls) r.clear();
        exp_max_N = 0;
        exp_init_needed = false;
        prefix_doubles = merged_floats = rowpart_n = colpart_n = F_total = 0;
        etab_doubles = 0;
        max_lds_bytes = 0;
        max_lds_expf = 0;
        max_lds_walk = 0;
        max_lds_step = 0;
        walk_tmpls = direct_tmpls = step_tmpls = generic_tmpls = 0;
        if (graph) (void)hipGraphExecDestroy(graph);
        graph = nullptr;
    }
    ~tcw_plan() {
        if (graph) (void)hipGraphExecDestroy(graph);
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
        if (side) (void)hipStreamDestroy(side);
        if (ev_fork) (void)hipEventDestroy(ev_fork);
        if (ev_join) (void)hipEventDestroy(ev_join);
        d_tmpl.release();
        d_segs.release();
        d_items.release();
        d_prefix.release();
        d_merged.release();
        d_ipart.release();
        d_rowpart.release();
        d_colpart.release();
        d_flags.release();
        d_seg_items.release();
        d_col_items.release();
        d_init_items.release();
        d_etab.release();
        d_tmpl_list.release();
        d_ts.release();
        d_cols.release();
        d_tables.release();
    }
};

// The handle keeps one plan and one stats slot for single-map calls, reused
// (grow-only) across calls so tcw_map allocates nothing in steady state.
struct tcw_handle {
    int device = 0;
    tcw_plan single;
    HostStage single_in;   // the single plan's descriptors and host atoms
    HostStage single_out;  // a small map on its way to the caller (pin only)
    tcw_plan noalloc;  // tcw_map_noalloc: buffers are views into the static scratch
    tcw_stats *h_stats = nullptr;  // pinned, written by the last kernel
    tcw_stats *d_stats = nullptr;  // its device address
    DevBuf d_mtab, d_msegs;  // tcw_merge_batch tables
    ~tcw_handle() {
        if (h_stats) (void)hipHostFree(h_stats);
        d_mtab.release();
        d_msegs.release();
    }
};

int tcwc::handle_device(const tcw_handle *h) { return h->device; }

namespace {

// Per-device address of the static scratch, looked up once per device (with
// that device current) by tcw_create; hipGetSymbolAddress's status is kept,
// so tcw_map_noalloc reports a failed lookup instead of using a bad address.
constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
hipError_t g_scratch_err[NOALLOC_MAX_DEVICES] = {};
bool g_scratch_done[NOALLOC_MAX_DEVICES] = {};

void noalloc_scratch_setup(int device) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_done[device]) return;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    g_scratch_err[device] = e;
    g_scratch_ptr[device] = e == hipSuccess ? ptr : nullptr;
    g_scratch_done[device] = true;
}

int noalloc_scratch_ptr(int device, char **out) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES)
        return fail(TCW_ERR_INVALID, "tcw_map_noalloc: device " + std::to_string(device) +
                                         " beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_done[device])
        return fail(TCW_ERR_INVALID, "tcw_map_noalloc: no handle was created on device " +
                                         std::to_string(device));
    if (g_scratch_err[device] != hipSuccess || !g_scratch_ptr[device])
        return fail(TCW_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") +
                                        hipGetErrorString(g_scratch_err[device]));
    *out = (char *)g_scratch_ptr[device];
    return TCW_OK;
}

}  // namespace

namespace {

// Effective window and shape (tcw_fstat_map_funcs.py:742-780, on a copy).
int effective_window(uint32_t numAtoms, uint32_t TAtom, uint32_t t0_data,
                     const tcw_window &in, tcw_window &w, int64_t &N_t0, int64_t &N_tau) {
    w = in;
    if (w.type >= TCW_TRANSIENT_LAST)
        return fail(TCW_ERR_INVALID, "Unknown window-type (" + std::to_string(w.type) +
                                         ") passed as input. Allowed are [0," +
                                         std::to_string(TCW_TRANSIENT_LAST - 1) + "].");
    if (w.type == TCW_TRANSIENT_NONE) {
        w.type = TCW_TRANSIENT_RECTANGULAR;
        w.t0 = t0_data;
        w.t0Band = 0;
        w.dt0 = TAtom;
        w.tau = numAtoms * TAtom;
        w.tauBand = 0;
        w.dtau = TAtom;
    }
    if (w.dt0 == 0 || w.dtau == 0)
        return fail(TCW_ERR_INVALID, "windowRange.dt0 and windowRange.dtau must be positive.");
    N_t0 = (int64_t)(w.t0Band / w.dt0) + 1;
    N_tau = (int64_t)(w.tauBand / w.dtau) + 1;
    if (N_t0 * N_tau >= (int64_t)0x7fffffff)
        return fail(TCW_ERR_INVALID, "map of " + std::to_string(N_t0) + " x " +
                                         std::to_string(N_tau) + " cells exceeds 2^31-1 cells.");
    return TCW_OK;
}

// Atom-column products an exp_init wave does for (template, column block,
// part): the kernel's l range of the part, each column group counted up to its
// longest window (the order the waves are launched in: heaviest first).
int32_t init_work(const TmplDev &td, uint32_t cb, int part) {
    const int64_t k0 = (int64_t)td.k00 + (int64_t)td.a * ((int64_t)td.n_seg * td.rb_rows - 1);
    const int64_t room = (int64_t)td.H - k0;
    auto clip = [&](int64_t L) { return std::max<int64_t>(std::min<int64_t>(L, room), 0); };
    const int64_t col0 = (int64_t)cb * TILE_COLS;
    const int64_t col_last = std::min<int64_t>(col0 + TILE_COLS, td.N_tau) - 1;
    const int64_t lr_blk = clip((int64_t)td.L0 + (int64_t)td.Ls * col_last);
    const int64_t q = (lr_blk + INIT_PARTS - 1) / INIT_PARTS;
    const int64_t l0 = part * q, l1 = std::min<int64_t>(lr_blk, l0 + q);
    int64_t w = 0;
    for (int i = 0; i < INIT_GROUPS; i++) {
        const int64_t g0 = col0 + (int64_t)INIT_WG * i;
        if (g0 > col_last) break;
        const int64_t glast = std::min<int64_t>(g0 + INIT_WG - 1, col_last);
        const int64_t hi = clip((int64_t)td.L0 + (int64_t)td.Ls * glast);
        w += std::max<int64_t>(0, std::min(l1, hi) - l0);
    }
    return (int32_t)std::min<int64_t>(w, 0x7fffffff);
}

// Build one template's descriptor and items.  seg range and N/t_min precomputed.
int plan_template(tcw_plan &p, int64_t t, const tcw_window &win_in, uint32_t N,
                  uint32_t TAtom, uint32_t t_min, int64_t seg_begin, int64_t seg_end,
                  std::vector<ItemDev> (&items_by_mode)[MODE_COUNT]) {
    tcw_window w;
    int64_t N_t0, N_tau;
    int rc = effective_window(N, TAtom, t_min, win_in, w, N_t0, N_tau);
    if (rc) return rc;
    TmplDev td;
    std::memset(&td, 0, sizeof(td));
    td.seg_begin = seg_begin;
    td.seg_end = seg_end;
    td.N = N;
    td.TAtom = TAtom;
    td.TA_rcp = 0xffffffffu / TAtom;
    td.t_min = t_min;
    td.type = w.type;
    td.t0 = w.t0;
    td.dt0 = w.dt0;
    td.tau = w.tau;
    td.dtau = w.dtau;
    td.N_t0 = (uint32_t)N_t0;
    td.N_tau = (uint32_t)N_tau;
    td.o_t0 = win_in.t0;
    td.o_t0Band = win_in.t0Band;
    td.o_tau = win_in.tau;
    td.o_tauBand = win_in.tauBand;

    int mode;
    if (w.type == TCW_TRANSIENT_EXPONENTIAL) {
        mode = MODE_EXP_DIRECT;
        // on the atom grid and free of uint32 wrap-around: the recurrence path
        const uint64_t end = (uint64_t)w.t0 + w.t0Band + 3ull * ((uint64_t)w.tau + w.tauBand) +
                             TAtom;
        const bool on_grid = w.t0 >= t_min && (w.t0 - t_min) % TAtom == 0 &&
                             w.dt0 % TAtom == 0 && w.tau % TAtom == 0 &&
                             w.dtau % TAtom == 0 && w.tau >= TAtom;
        // (rows of at most 2^20 cells: the map kernel's row stores address a
        // pass of rows by 32-bit byte offsets)
        // off the grid: the sliding sum with any steps.  (Starts that step by
        // part of an atom repeat windows: the posterior's mode is then one of
        // several equal rows, and which one the sums' rounding decides.  They
        // keep the direct sum and with it their answers.)
        td.walk = !(p.flags & TCW_FLAG_GENERIC) && w.t0 >= t_min && end < (1ull << 32) &&
                  w.tau >= TAtom && !p.compact && (w.dt0 >= TAtom || N_t0 == 1);
        if (!(p.flags & TCW_FLAG_GENERIC) && on_grid && end < (1ull << 32) &&
            N_tau <= (int64_t)1 << 20) {
            mode = MODE_EXP_FAST;
            td.k00 = (int32_t)((w.t0 - t_min) / TAtom);
            td.a = (int32_t)(w.dt0 / TAtom);
            td.L0 = (int32_t)(3ull * w.tau / TAtom);
            td.Ls = (int32_t)(3ull * w.dtau / TAtom);
            const int64_t kmax = (int64_t)td.k00 + (int64_t)td.a * (N_t0 - 1);
            const int64_t Lmax = (int64_t)td.L0 + (int64_t)td.Ls * (N_tau - 1);
            td.H = (int32_t)std::min<int64_t>((int64_t)N, kmax + Lmax);
        }
    } else {
        mode = MODE_RECT_GENERIC;
        const uint64_t half = TAtom / 2;
        const bool regular = (w.dt0 % TAtom == 0) && (w.dtau % TAtom == 0) && (w.dt0 == w.dtau);
        const uint64_t x_lo = (uint64_t)w.t0 + half;  // must not be below t_min
        const uint64_t x_hi = (uint64_t)w.t0 + w.t0Band + w.tau + w.tauBand + half;
        // (rows of at most 2^20 cells: partial sub-tiles store by 32-bit byte
        // offsets within their four rows)
        td.walk = !(p.flags & TCW_FLAG_GENERIC) && x_lo >= t_min && x_hi < (1ull << 32) &&
                  N_tau <= (int64_t)1 << 20;
        // the kernel's start indices of a wave's four rows, up to three past the
        // map, are 32 bits wide
        const uint64_t q0 = ((uint64_t)w.t0 - t_min + half) / TAtom;
        const bool starts_fit =
            q0 + (uint64_t)(w.dt0 / TAtom) * (uint64_t)(N_t0 + 2) <= 0x7fffffffu;
        if (td.walk && regular && starts_fit) {
            mode = MODE_RECT_FAST;
            td.a = (int32_t)(w.dt0 / TAtom);
            td.q0 = (int32_t)q0;
            td.q00 = (int32_t)(((uint64_t)w.t0 + w.tau - t_min + half) / TAtom);
        } else if (p.compact || (w.dt0 < TAtom && N_t0 > 1) || (w.dtau < TAtom && N_tau > 1)) {
            td.walk = 0;  // (steps of part of an atom repeat rows or columns, as above)
        }
    }
    td.mode = mode;
    const int req = p.rows_req[mode];  // the plan's tuned rows, 0 = built-in choice
    int rb = req > 0 ? req : RB_DEFAULT[mode];
    if ((mode == MODE_RECT_FAST || (mode == MODE_RECT_GENERIC && td.walk)) && req <= 0) {
        // few or small maps (the single-map call): fewer rows per item, so
        // that the batch's items cover the CUs (about SMALL_BATCH_ITEMS of them
        // if the templates are alike)
        const int most = p.compact                ? COMPACT_RECT_ROWS
                         : mode == MODE_RECT_FAST ? RB_DEFAULT[mode]
                                                  : STEP_RB;
        const double ncb = (double)((N_tau + TILE_COLS - 1) / TILE_COLS);
        const double want = (double)N_t0 * ncb * (double)p.T /
                            (double)(p.compact                ? COMPACT_RECT_ITEMS
                                     : mode == MODE_RECT_FAST ? SMALL_BATCH_ITEMS
                                                              : STEP_ITEMS);
        rb = want >= most ? most : std::max(16, ((int)std::ceil(want) + 15) / 16 * 16);
    }
    if (mode == MODE_EXP_DIRECT && td.walk && req <= 0) {
        // enough items for the chip, and otherwise long ones: each starts with
        // a direct sum
        const double ncb = (double)((N_tau + WALK_TILE - 1) / WALK_TILE);
        const double want = (double)N_t0 * ncb * (double)p.T / (double)WALK_ITEMS;
        rb = std::min(WALK_MAX_ROWS, std::max(32, ((int)std::min(want, 1e6) + 31) / 32 * 32));
    }
    if (mode == MODE_EXP_FAST && req <= 0) {
        const int64_t pairs = p.T * ((N_tau + TILE_COLS - 1) / TILE_COLS);
        if (pairs < DIRECT_INIT_MIN_BLOCKS) {
            const int64_t span = ((int64_t)td.H - td.k00 + td.a - 1) / std::max(td.a, 1);
            const int64_t want = pairs * std::max<int64_t>(span, N_t0) / EXP_SMALL_CHUNKS;
            rb = (int)std::min<int64_t>(EXP_SMALL_MAX_ROWS,
                                        std::max<int64_t>(EXP_SMALL_MIN_ROWS, (want + 15) / 16 * 16));
            if (p.compact) rb = COMPACT_EXP_ROWS;
        } else {
            // about EXP_TARGET_ITEMS work items: one chunk per column when the
            // batch has that many column blocks
            const int64_t chunks = std::max<int64_t>(1, (EXP_TARGET_ITEMS + pairs - 1) / pairs);
            const int64_t per = (N_t0 + chunks - 1) / chunks;
            rb = (int)std::min<int64_t>(MAX_RB_EXPF, (per + 15) / 16 * 16);
        }
    }
    if (mode == MODE_EXP_FAST)  // rows past the map are walked: no longer chunks than the map
        rb = (int)std::min<int64_t>(rb, (N_t0 + 15) / 16 * 16);
    td.rb_rows = rb;
    td.n_rowblk = (uint32_t)((N_t0 + rb - 1) / rb);
    td.tile = mode == MODE_EXP_DIRECT && td.walk ? WALK_TILE : TILE_COLS;
    if (mode == MODE_RECT_GENERIC && td.walk) {
        auto bytes = [&](int tile) {
            return step_bytes(step_shape(rb, tile, td.N_tau, td.dt0, td.dtau, TAtom));
        };
        while (td.tile > 64 && bytes(td.tile) > STEP_LDS_AIM) td.tile /= 2;
        if (bytes(td.tile) > STEP_LDS_MOST) td.tile = TILE_COLS;
    }
    td.n_colblk = (uint32_t)((N_tau + td.tile - 1) / td.tile);
    if (mode == MODE_EXP_DIRECT || mode == MODE_EXP_FAST) {
        td.mode = mode;  // exp_table_bins reads it
        if (mode == MODE_EXP_FAST) {
            // E at the top chunk's top row comes from a direct O(L) sum
            // (exp_init_kernel, slot n_seg of the table).  With enough
            // independent column blocks in the batch the chunks are just the
            // map's row blocks (least total work); otherwise extra chunks above
            // the map reach H, where E = 0 and the direct sum is empty, so that
            // no lane runs a long serial sum.
            int64_t nseg = std::max<int64_t>((int64_t)td.n_rowblk, 1);
            if (p.T * (int64_t)td.n_colblk < DIRECT_INIT_MIN_BLOCKS) {
                const int64_t steps = ((int64_t)td.H - td.k00 + td.a - 1) / td.a;  // rows to H
                nseg = std::max<int64_t>(nseg, (std::max<int64_t>(steps, 0) + rb) / rb);
            }
            td.n_seg = (int32_t)nseg;
            // the top chunk's top row lies at or beyond H: its direct sum is
            // empty, exp_scan starts from 0 and exp_init need not run
            td.init_empty = (int64_t)td.H - ((int64_t)td.k00 + (int64_t)td.a * (nseg * rb - 1)) <= 0;
            if (!td.init_empty) {
                p.exp_init_needed = true;
                for (uint32_t cbk = 0; cbk < td.n_colblk; cbk++)
                    for (int part = 0; part < INIT_PARTS; part++)
                        p.init_items.push_back(ItemDev{(int32_t)t, part, (int32_t)cbk,
                                                       init_work(td, cbk, part)});
            }
            td.etab_off = p.etab_doubles;
            p.etab_doubles += (nseg + INIT_PARTS) * NC * N_tau;
            for (int64_t sg = 1; sg < nseg; sg++)
                for (uint32_t cbk = 0; cbk < td.n_colblk; cbk++)
                    p.seg_items.push_back(ItemDev{(int32_t)t, (int32_t)sg, (int32_t)cbk, 0});
            if (nseg > 1)  // one chunk: the map kernel adds the direct sum's parts
                for (uint32_t cbk = 0; cbk < td.n_colblk; cbk++)
                    p.col_items.push_back(ItemDev{(int32_t)t, 0, (int32_t)cbk, 0});
            if (expw_pass_rows(td.a, td.Ls, (int)std::min<int64_t>(TILE_COLS, N_tau)) > 0)
                p.max_lds_expf = EXPF_LDS_BYTES;  // fixed plane strides
        }
        const int64_t nbins = exp_table_bins(td);
        td.merged_off = p.merged_floats;
        p.merged_floats += nbins * MERGED_STRIDE;
        p.exp_tmpls.push_back((int32_t)t);
        p.exp_max_N = std::max<int64_t>(p.exp_max_N, nbins);
        if (mode == MODE_EXP_DIRECT && td.walk) {
            p.max_lds_walk = std::max(p.max_lds_walk, walk_lds(rb));
            p.walk_tmpls++;
        } else if (mode == MODE_EXP_DIRECT) {
            p.direct_tmpls++;
        }
    } else {
        p.rect_tmpls[stage_class(N)].push_back((int32_t)t);
        td.prefix_off = p.prefix_doubles;
        p.prefix_doubles += ((int64_t)N + 1) * NC;
    }
    td.F_off = p.F_total;
    p.F_total += N_t0 * N_tau;
    td.rowpart_off = p.rowpart_n;
    p.rowpart_n += N_t0 * (int64_t)td.n_colblk;
    td.colpart_off = p.colpart_n;
    p.colpart_n += N_tau * (int64_t)td.n_rowblk;
    // items of a template are contiguous in item-id space; item_begin counts from
    // the mode's first item until plan_finish
    std::vector<ItemDev> &items = items_by_mode[mode];
    td.item_begin = (int64_t)items.size();
    items.resize(items.size() + (size_t)td.n_rowblk * td.n_colblk);
    ItemDev *it = items.data() + td.item_begin;
    for (uint32_t rbk = 0; rbk < td.n_rowblk; rbk++)
        for (uint32_t cbk = 0; cbk < td.n_colblk; cbk++)
            *it++ = ItemDev{(int32_t)t, (int32_t)rbk, (int32_t)cbk, 0};
    if (mode == MODE_RECT_GENERIC && td.walk) {
        p.max_lds_step = std::max(
            p.max_lds_step,
            step_lds(rb, step_shape(rb, td.tile, td.N_tau, td.dt0, td.dtau, TAtom)));
        p.step_tmpls++;
    } else if (mode == MODE_RECT_GENERIC) {
        p.generic_tmpls++;
    }
    if (mode == MODE_RECT_FAST) {
        // the widest column block (the first) and the last one
        const int last = (int)N_tau - (int)(td.n_colblk - 1) * TILE_COLS;
        for (int rem : {(int)std::min<int64_t>(N_tau, TILE_COLS), last})
            p.max_lds_bytes = std::max(p.max_lds_bytes, rect_item_lds(rb, rect_lane_cols(rem)));
    }
    p.tmpl.push_back(td);
    return TCW_OK;
}

// Every device buffer of a plan with the bytes the plan needs in it.
template <typename F>
void plan_buffers(tcw_plan &p, F f) {
    f(p.d_tmpl, sizeof(TmplDev) * std::max<size_t>(p.tmpl.size(), 1));
    f(p.d_segs, sizeof(SegDev) * std::max<size_t>(p.segs.size(), 1));
    f(p.d_items, sizeof(ItemDev) * std::max<size_t>(p.items.size(), 1));
    f(p.d_prefix, sizeof(double) * std::max<int64_t>(p.prefix_doubles, 1));
    f(p.d_merged, sizeof(float) * std::max<int64_t>(p.merged_floats, 1));
    f(p.d_ipart, sizeof(ItemPart) * std::max<size_t>(p.items.size(), 1));
    f(p.d_rowpart, sizeof(float) * std::max<int64_t>(p.rowpart_n, 1));
    f(p.d_colpart, sizeof(float) * std::max<int64_t>(p.colpart_n, 1));
    f(p.d_flags, sizeof(int) * std::max<int64_t>(p.T, 1));
    f(p.d_seg_items, sizeof(ItemDev) * std::max<size_t>(p.seg_items.size(), 1));
    f(p.d_col_items, sizeof(ItemDev) * std::max<size_t>(p.col_items.size(), 1));
    f(p.d_init_items, sizeof(ItemDev) * std::max<size_t>(p.init_items.size(), 1));
    f(p.d_etab, sizeof(double) * std::max<int64_t>(p.etab_doubles, 1));
    f(p.d_tmpl_list, sizeof(int32_t) * std::max<size_t>(p.tmpl_list.size(), 1));
}

// After all templates: lay out items mode by mode, fix item_begin (the items
// of one template stay contiguous, rb-major), size scratch (own buffers, or
// views into p.arena when set), upload descriptors (asynchronously on `st`
// when given, else synchronously).
int plan_finish(tcw_plan &p, std::vector<ItemDev> (&items_by_mode)[MODE_COUNT],
                hipStream_t st, bool async) {
    // exp_init waves heaviest first (work estimate in .pad): the last waves
    // to start are the short ones
    std::stable_sort(p.init_items.begin(), p.init_items.end(),
                     [](const ItemDev &x, const ItemDev &y) { return x.pad > y.pad; });
    p.items.clear();
    for (int md = 0; md < MODE_COUNT; md++) {
        p.mode_begin[md] = (int64_t)p.items.size();
        if (p.items.empty())  // most batches hold one mode
            p.items.swap(items_by_mode[md]);
        else
            p.items.insert(p.items.end(), items_by_mode[md].begin(), items_by_mode[md].end());
    }
    p.mode_begin[MODE_COUNT] = (int64_t)p.items.size();
    for (TmplDev &td : p.tmpl) td.item_begin += p.mode_begin[td.mode];
    p.tmpl_list = p.exp_tmpls;
    for (auto &r : p.rect_tmpls) {
        // the longest templates first: the last workgroups to start are short
        std::stable_sort(r.begin(), r.end(),
                         [&](int32_t x, int32_t y) { return p.tmpl[x].N > p.tmpl[y].N; });
        p.tmpl_list.insert(p.tmpl_list.end(), r.begin(), r.end());
    }
    struct Up {
        DevBuf *buf;
        const void *src;
        size_t bytes;
    };
    std::vector<Up> ups = {
        {&p.d_tmpl, p.tmpl.data(), sizeof(TmplDev) * p.tmpl.size()},
        {&p.d_segs, p.segs.data(), sizeof(SegDev) * p.segs.size()},
        {&p.d_items, p.items.data(), sizeof(ItemDev) * p.items.size()},
        {&p.d_seg_items, p.seg_items.data(), sizeof(ItemDev) * p.seg_items.size()},
        {&p.d_col_items, p.col_items.data(), sizeof(ItemDev) * p.col_items.size()},
        {&p.d_init_items, p.init_items.data(), sizeof(ItemDev) * p.init_items.size()},
        {&p.d_tmpl_list, p.tmpl_list.data(), sizeof(int32_t) * p.tmpl_list.size()},
    };
    if (p.host_ts) {
        ups.push_back({&p.d_ts, p.host_ts, sizeof(uint32_t) * (size_t)p.n_host_atoms});
        ups.push_back({&p.d_cols, p.host_cols, sizeof(float) * NC * (size_t)p.n_host_atoms});
    }
    // one copy instead of one per table (each costs ~4 us of launch and, from
    // pageable memory, ~4 us of a staging kernel on the stream)
    size_t staged = 0;
    for (const Up &u : ups) staged += stage_align(std::max<size_t>(u.bytes, 1));
    const bool one_copy = p.stage && async && staged <= HOST_STAGE_MAX;
    const bool packed = !p.arena && !async && staged <= PACKED_TABLES_MAX;
    int rc = TCW_OK;
    if (one_copy) {
        if ((rc = p.stage->ensure(staged))) return rc;
        size_t off = 0;
        for (const Up &u : ups) {
            const size_t a = stage_align(std::max<size_t>(u.bytes, 1));
            if (u.bytes) std::memcpy(p.stage->pin + off, u.src, u.bytes);
            u.buf->set_view((char *)p.stage->dev.p + off, a);
            off += a;
        }
        TCW_HIP_TRY(hipMemcpyAsync(p.stage->dev.p, p.stage->pin, staged, hipMemcpyHostToDevice, st));
    } else if (packed) {
        if ((rc = p.d_tables.ensure(staged))) return rc;
        const std::unique_ptr<char[]> host(new char[staged]);
        size_t off = 0;
        for (const Up &u : ups) {
            const size_t a = stage_align(std::max<size_t>(u.bytes, 1));
            if (u.bytes) std::memcpy(host.get() + off, u.src, u.bytes);
            u.buf->set_view((char *)p.d_tables.p + off, a);
            off += a;
        }
        TCW_HIP_TRY(hipMemcpy(p.d_tables.p, host.get(), staged, hipMemcpyHostToDevice));
    } else {
        for (const Up &u : ups)  // views of an earlier call
            if (u.buf->view) u.buf->release();
    }
    if (p.arena) {
        // carve every buffer out of the caller-provided arena (no allocation)
        size_t off = 0;
        plan_buffers(p, [&](DevBuf &b, size_t bytes) {
            const size_t a = (bytes + 255) / 256 * 256;
            if (off + a <= p.arena_bytes) b.set_view(p.arena + off, a);
            off += a;
        });
        p.arena_short = off > p.arena_bytes;
        if (p.arena_short)
            return fail(TCW_ERR_INVALID, "this map needs " + std::to_string(off) +
                                             " bytes of scratch; the static scratch holds " +
                                             std::to_string(p.arena_bytes) + " bytes");
        if (p.dry) return TCW_OK;
    } else {
        plan_buffers(p, [&](DevBuf &b, size_t bytes) {
            if (!rc) rc = b.ensure(bytes);
        });
        if (rc) return rc;
    }
    if (one_copy || packed) return TCW_OK;
    for (const Up &u : ups) {
        if (u.bytes == 0) continue;
        if ((rc = u.buf->ensure(u.bytes))) return rc;
        TCW_HIP_TRY(async ? hipMemcpyAsync(u.buf->p, u.src, u.bytes, hipMemcpyHostToDevice, st)
                          : hipMemcpy(u.buf->p, u.src, u.bytes, hipMemcpyHostToDevice));
    }
    return TCW_OK;
}

// Rows per work item a caller may request for kernel mode `mode`.
int check_rows(int mode, int rows) {
    const int maxr = mode == MODE_EXP_FAST ? MAX_RB_EXPF : MAX_RB;
    if (rows != 0 && (rows < 16 || rows > maxr || rows % 16))
        return fail(TCW_ERR_INVALID, "rows per item for mode " + std::to_string(mode) +
                                         " must be 0 or a multiple of 16 in [16, " +
                                         std::to_string(maxr) + "], not " + std::to_string(rows));
    return TCW_OK;
}

// Plan `d` into `p` (buffers reused, grow-only).  rows_by_mode: host [4] or
// null (built-in choices).
int plan_build(tcw_plan &p, int device, const tcw_batch_desc *d, uint32_t flags,
               int64_t *F_off, hipStream_t st, bool async,
               const int32_t *rows_by_mode = nullptr) {
    if (d->T <= 0) return fail(TCW_ERR_INVALID, "no templates");
    if (d->TAtom < 2) return fail(TCW_ERR_INVALID, "TAtom must be at least 2 seconds.");
    for (int md = 0; md < MODE_COUNT; md++) {
        const int r = rows_by_mode ? rows_by_mode[md] : 0;
        int rc = check_rows(md, r);
        if (rc) return rc;
        p.rows_req[md] = r;
    }
    p.reset();
    p.device = device;
    p.flags = flags;
    p.T = d->T;
    std::vector<ItemDev> items_by_mode[MODE_COUNT];
    for (int64_t t = 0; t < d->T; t++) {
        const int64_t s0 = d->seg_begin[t], s1 = d->seg_begin[t + 1];
        if (s1 <= s0 || s1 - s0 > TCW_MAX_DETECTORS)
            return fail(TCW_ERR_INVALID, "template " + std::to_string(t) + ": needs 1.." +
                                             std::to_string(TCW_MAX_DETECTORS) +
                                             " detector segments");
        uint32_t tmin = 0xffffffffu, tmax = 0;
        const int64_t first_seg = (int64_t)p.segs.size();
        for (int64_t s = s0; s < s1; s++) {
            if (d->seg_off[s + 1] <= d->seg_off[s])
                return fail(TCW_ERR_INVALID, "template " + std::to_string(t) + ": empty detector");
            if (d->seg_tlast[s] < d->seg_tfirst[s])
                return fail(TCW_ERR_INVALID, "template " + std::to_string(t) +
                                                 ": timestamps not in ascending order");
            tmin = std::min(tmin, d->seg_tfirst[s]);
            tmax = std::max(tmax, d->seg_tlast[s]);
            p.segs.push_back(SegDev{d->seg_off[s], d->seg_off[s + 1]});
        }
        const uint64_t N = (uint64_t)(tmax - tmin) / d->TAtom + 1;
        if (F_off) F_off[t] = p.F_total;
        int rc = plan_template(p, t, d->windows[t], (uint32_t)N, d->TAtom, tmin, first_seg,
                               (int64_t)p.segs.size(), items_by_mode);
        if (rc) return rc;
    }
    if (F_off) F_off[d->T] = p.F_total;
    return plan_finish(p, items_by_mode, st, async);
}

template <bool BTSG, bool STRICT>
void launch_maps(tcw_plan &p, float *F, hipStream_t st) {
    auto *tds = (const TmplDev *)p.d_tmpl.p;
    auto *items = (const ItemDev *)p.d_items.p;
    auto *prefix = (const double *)p.d_prefix.p;
    auto *merged = (const float *)p.d_merged.p;
    auto *ipart = (ItemPart *)p.d_ipart.p;
    auto *rowpart = (float *)p.d_rowpart.p;
    auto *colpart = (float *)p.d_colpart.p;
    auto *flags = (int *)p.d_flags.p;
    int64_t n;
    if ((n = p.mode_begin[MODE_RECT_FAST + 1] - p.mode_begin[MODE_RECT_FAST]) > 0)
        hipLaunchKernelGGL((rect_fast_kernel<BTSG, STRICT>), dim3((unsigned)n), dim3(WG),
                           p.max_lds_bytes, st, tds, items, p.mode_begin[MODE_RECT_FAST],
                           prefix, F, ipart, rowpart, colpart, flags);
    // the items of a mode lie template by template: where two kernels share a
    // mode, each leaves the other's items at once
    if ((n = p.mode_begin[MODE_RECT_GENERIC + 1] - p.mode_begin[MODE_RECT_GENERIC]) > 0) {
        if (p.step_tmpls > 0)
            hipLaunchKernelGGL((rect_step_kernel<BTSG, STRICT>), dim3((unsigned)n), dim3(WG),
                               p.max_lds_step, st, tds, items, p.mode_begin[MODE_RECT_GENERIC],
                               prefix, F, ipart, rowpart, colpart, flags);
        if (p.generic_tmpls > 0)
            hipLaunchKernelGGL((rect_generic_kernel<BTSG, STRICT>), dim3((unsigned)n), dim3(WG), 0,
                               st, tds, items, p.mode_begin[MODE_RECT_GENERIC], prefix, F, ipart,
                               rowpart, colpart, flags);
    }
    if ((n = p.mode_begin[MODE_EXP_FAST + 1] - p.mode_begin[MODE_EXP_FAST]) > 0)
        hipLaunchKernelGGL((exp_fast_kernel<BTSG, STRICT>), dim3((unsigned)n), dim3(WG),
                           p.max_lds_expf, st, tds, items, p.mode_begin[MODE_EXP_FAST], merged,
                           (const double *)p.d_etab.p, F, ipart, rowpart, colpart, flags,
                           p.max_lds_expf > 0 ? 1 : 0);
    if ((n = p.mode_begin[MODE_EXP_DIRECT + 1] - p.mode_begin[MODE_EXP_DIRECT]) > 0) {
        if (p.walk_tmpls > 0)
            hipLaunchKernelGGL((exp_walk_kernel<BTSG, STRICT>), dim3((unsigned)n), dim3(WALK_WG),
                               p.max_lds_walk, st, tds, items, p.mode_begin[MODE_EXP_DIRECT],
                               merged, F, ipart, rowpart, colpart, flags);
        if (p.direct_tmpls > 0)
            hipLaunchKernelGGL((exp_direct_kernel<BTSG, STRICT>), dim3((unsigned)n),
                               dim3(DIRECT_WG), 0,
                               st, tds, items, p.mode_begin[MODE_EXP_DIRECT], merged, F, ipart,
                               rowpart, colpart, flags);
    }
}

// Optional per-stage event marks: ev[0] before the stage kernel, ev[1] after
// it, ev[2] after the map kernels, ev[3] after finalize.
// check_errors = false while a stream is being captured (hipGetLastError is
// not permitted then; launch errors surface at instantiate/launch instead).
int launch_all(tcw_plan &p, const uint32_t *ts, const float *cols, int64_t cstride,
               float *F, tcw_stats *stats_dev, hipStream_t st, hipEvent_t *ev = nullptr,
               bool check_errors = true) {
    const bool btsg = p.flags & TCW_FLAG_BTSG;
    const bool strict = p.flags & TCW_FLAG_LAL_STRICT;
    auto *flags = (int *)p.d_flags.p;
    if (ev) TCW_HIP_TRY(hipEventRecord(ev[0], st));
    const int32_t *rect = (const int32_t *)p.d_tmpl_list.p + p.exp_tmpls.size();
    for (int k = 0; k < SR_CLASSES; k++) {
        const unsigned n = (unsigned)p.rect_tmpls[k].size();
        if (n == 0) continue;
        const bool wide = k == SR_CLASSES - 1 && n <= SR_WIDE_TMPLS;
        auto *kern = wide     ? stage_kernel<SR_WIDE_THREADS>
                     : k == 0 ? stage_kernel<SR_THREADS[0]>
                              : stage_kernel<SR_THREADS[1]>;
        hipLaunchKernelGGL(kern, dim3(n), dim3(wide ? SR_WIDE_THREADS : SR_THREADS[k]), 0, st,
                           (const TmplDev *)p.d_tmpl.p, rect, (const SegDev *)p.d_segs.p, ts, cols,
                           cstride, (double *)p.d_prefix.p, flags);
        rect += n;
    }
    if (!p.exp_tmpls.empty()) {
        const int64_t n_exp = (int64_t)p.exp_tmpls.size();
        const int64_t wide_blocks = (p.exp_max_N + 1023) / 1024;
        const unsigned gy = (unsigned)std::min<int64_t>(n_exp, 65535);
        if (n_exp > 0 && wide_blocks * n_exp < SX_NARROW_BELOW)
            hipLaunchKernelGGL(stage_exp_kernel<1>, dim3((unsigned)((p.exp_max_N + 255) / 256), gy),
                               dim3(256), 0, st, (const TmplDev *)p.d_tmpl.p,
                               (const int32_t *)p.d_tmpl_list.p, n_exp, (const SegDev *)p.d_segs.p,
                               ts, cols, cstride, (float *)p.d_merged.p, flags);
        else if (n_exp > 0)
            hipLaunchKernelGGL(stage_exp_kernel<4>, dim3((unsigned)wide_blocks, gy), dim3(256), 0,
                               st, (const TmplDev *)p.d_tmpl.p, (const int32_t *)p.d_tmpl_list.p,
                               n_exp, (const SegDev *)p.d_segs.p, ts, cols, cstride,
                               (float *)p.d_merged.p, flags);
    }
    // exp_init and exp_seg read the atom table and write different slots of the
    // E table: with enough blocks for both, exp_init runs on the side stream
    // exp_init runs one wave per item; blocks of 4 waves as the unit here
    const int64_t init_blocks = p.exp_init_needed ? (int64_t)p.init_items.size() / INIT_GROUPS : 0;
    const bool fork = p.side && init_blocks > 0 && !p.seg_items.empty() &&
                      init_blocks + (int64_t)p.seg_items.size() >= EXP_FORK_MIN_BLOCKS;
    if (fork) {
        TCW_HIP_TRY(hipEventRecord(p.ev_fork, st));
        TCW_HIP_TRY(hipStreamWaitEvent(p.side, p.ev_fork, 0));
    }
    if (p.exp_init_needed)
        hipLaunchKernelGGL(exp_init_kernel, dim3((unsigned)p.init_items.size()), dim3(INIT_WG), 0,
                           fork ? p.side : st, (const TmplDev *)p.d_tmpl.p,
                           (const ItemDev *)p.d_init_items.p, (const float *)p.d_merged.p,
                           (double *)p.d_etab.p);
    if (!p.seg_items.empty())
        hipLaunchKernelGGL(exp_seg_kernel, dim3((unsigned)p.seg_items.size()), dim3(WG),
                           p.max_lds_expf, st, (const TmplDev *)p.d_tmpl.p,
                           (const ItemDev *)p.d_seg_items.p, (const float *)p.d_merged.p,
                           (double *)p.d_etab.p, p.max_lds_expf > 0 ? 1 : 0);
    if (fork) {
        TCW_HIP_TRY(hipEventRecord(p.ev_join, p.side));
        TCW_HIP_TRY(hipStreamWaitEvent(st, p.ev_join, 0));
    }
    if (!p.col_items.empty())
        hipLaunchKernelGGL(exp_scan_kernel, dim3((unsigned)(p.col_items.size() * SCAN_SPLIT * NC)),
                           dim3(SCAN_WG), 0, st, (const TmplDev *)p.d_tmpl.p,
                           (const ItemDev *)p.d_col_items.p, (double *)p.d_etab.p);
    if (ev) TCW_HIP_TRY(hipEventRecord(ev[1], st));
    if (btsg) {
        if (strict)
            launch_maps<true, true>(p, F, st);
        else
            launch_maps<true, false>(p, F, st);
        if (ev) TCW_HIP_TRY(hipEventRecord(ev[2], st));
        if (p.T < FIN_WIDE_MAX_T)
            hipLaunchKernelGGL((finalize_kernel<true, 1024>), dim3((unsigned)p.T), dim3(1024), 0, st,
                           (const TmplDev *)p.d_tmpl.p, (const ItemPart *)p.d_ipart.p,
                           (const float *)p.d_rowpart.p, (const float *)p.d_colpart.p,
                           (const int *)p.d_flags.p, stats_dev);
        else
            hipLaunchKernelGGL((finalize_kernel<true, WG>), dim3((unsigned)p.T), dim3(WG), 0, st,
                           (const TmplDev *)p.d_tmpl.p, (const ItemPart *)p.d_ipart.p,
                           (const float *)p.d_rowpart.p, (const float *)p.d_colpart.p,
                           (const int *)p.d_flags.p, stats_dev);
    } else {
        if (strict)
            launch_maps<false, true>(p, F, st);
        else
            launch_maps<false, false>(p, F, st);
        if (ev) TCW_HIP_TRY(hipEventRecord(ev[2], st));
        if (p.T < FIN_WIDE_MAX_T)
            hipLaunchKernelGGL((finalize_kernel<false, 1024>), dim3((unsigned)p.T), dim3(1024), 0, st,
                           (const TmplDev *)p.d_tmpl.p, (const ItemPart *)p.d_ipart.p,
                           (const float *)p.d_rowpart.p, (const float *)p.d_colpart.p,
                           (const int *)p.d_flags.p, stats_dev);
        else
            hipLaunchKernelGGL((finalize_kernel<false, WG>), dim3((unsigned)p.T), dim3(WG), 0, st,
                           (const TmplDev *)p.d_tmpl.p, (const ItemPart *)p.d_ipart.p,
                           (const float *)p.d_rowpart.p, (const float *)p.d_colpart.p,
                           (const int *)p.d_flags.p, stats_dev);
    }
    if (ev) TCW_HIP_TRY(hipEventRecord(ev[3], st));
    if (check_errors) TCW_HIP_TRY(hipGetLastError());
    return TCW_OK;
}

// The exp side stream and its events, made on first use (never while a
// stream is being captured).
int ensure_side(tcw_plan *p) {
    if (p->side || p->col_items.empty() || p->seg_items.empty()) return TCW_OK;
    hipStream_t s = nullptr;
    hipEvent_t a = nullptr, b = nullptr;
    hipError_t e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&a, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b, hipEventDisableTiming);
    if (e != hipSuccess) {
        if (s) (void)hipStreamDestroy(s);
        if (a) (void)hipEventDestroy(a);
        return fail(TCW_ERR_DEVICE, std::string("exp side stream: ") + hipGetErrorString(e));
    }
    p->side = s;
    p->ev_fork = a;
    p->ev_join = b;
    return TCW_OK;
}

}  // namespace

extern "C" {

const char *tcw_version(void) { return "tcw_hip 0.1 (gfx950)"; }

const char *tcw_last_error(void) { return tcwc::g_err.c_str(); }

int tcw_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int tcw_device_name(int device, char *buf, int buflen) {
    if (!buf || buflen <= 0) return fail(TCW_ERR_INVALID, "tcw_device_name: no buffer");
    hipDeviceProp_t prop;
    TCW_HIP_TRY(hipGetDeviceProperties(&prop, device));
    std::snprintf(buf, (size_t)buflen, "%s", prop.name);
    return TCW_OK;
}

int tcw_map_shape(uint32_t numAtoms, uint32_t TAtom, uint32_t t0_data, const tcw_window *win,
                  int64_t *N_t0, int64_t *N_tau) {
    if (!win || !N_t0 || !N_tau) return fail(TCW_ERR_INVALID, "tcw_map_shape: null argument");
    tcw_window w;
    return effective_window(numAtoms, TAtom, t0_data, *win, w, *N_t0, *N_tau);
}

int tcw_create(int device, tcw_handle **out) {
    if (!out) return fail(TCW_ERR_INVALID, "tcw_create: null output");
    int n = tcw_device_count();
    if (device < 0 || device >= n)
        return fail(TCW_ERR_INVALID, "Requested HIP device number " + std::to_string(device) +
                                         " exceeds number of available devices (" +
                                         std::to_string(n) + ").");
    int rc = set_device(device);
    if (rc) return rc;
    auto *h = new tcw_handle;
    h->device = device;
    noalloc_scratch_setup(device);  // with `device` current
    h->single.stage = &h->single_in;
    if (hipHostMalloc(&h->h_stats, sizeof(tcw_stats), hipHostMallocDefault) != hipSuccess ||
        hipHostGetDevicePointer((void **)&h->d_stats, h->h_stats, 0) != hipSuccess) {
        delete h;
        return fail(TCW_ERR_NOMEM, "tcw_create: stats slot allocation failed");
    }
    *out = h;
    return TCW_OK;
}

int tcw_destroy(tcw_handle *h) {
    if (h) (void)set_device(h->device);
    delete h;
    return TCW_OK;
}

int tcw_batch_plan(tcw_handle *h, const tcw_batch_desc *d, uint32_t flags, tcw_plan **out,
                   int64_t *F_off) {
    return tcw_batch_plan_rows(h, d, flags, nullptr, out, F_off);
}

int tcw_batch_plan_rows(tcw_handle *h, const tcw_batch_desc *d, uint32_t flags,
                        const int32_t *rows_by_mode, tcw_plan **out, int64_t *F_off) {
    if (!h || !d || !out) return fail(TCW_ERR_INVALID, "tcw_batch_plan: null argument");
    int rc = set_device(h->device);
    if (rc) return rc;
    auto *p = new tcw_plan;
    rc = plan_build(*p, h->device, d, flags, F_off, nullptr, false, rows_by_mode);
    if (rc) {
        delete p;
        return rc;
    }
    *out = p;
    return TCW_OK;
}

int64_t tcw_plan_scratch_bytes(const tcw_plan *p) {
    if (!p) return 0;
    return (int64_t)(p->d_tmpl.cap + p->d_segs.cap + p->d_items.cap + p->d_prefix.cap +
                     p->d_merged.cap + p->d_ipart.cap + p->d_rowpart.cap + p->d_colpart.cap +
                     p->d_flags.cap + p->d_seg_items.cap + p->d_col_items.cap +
                     p->d_etab.cap + p->d_init_items.cap);
}

int tcw_plan_items(const tcw_plan *p, int64_t *items) {
    if (!p || !items) return fail(TCW_ERR_INVALID, "tcw_plan_items: null argument");
    for (int md = 0; md < MODE_COUNT; md++) items[md] = p->mode_begin[md + 1] - p->mode_begin[md];
    return TCW_OK;
}

int tcw_plan_kernels(const tcw_plan *p, int64_t *templates) {
    if (!p || !templates) return fail(TCW_ERR_INVALID, "tcw_plan_kernels: null argument");
    int64_t n[MODE_COUNT] = {0, 0, 0, 0};
    for (const TmplDev &td : p->tmpl) n[td.mode]++;
    templates[0] = n[MODE_RECT_FAST];
    templates[1] = p->step_tmpls;
    templates[2] = p->generic_tmpls;
    templates[3] = n[MODE_EXP_FAST];
    templates[4] = p->walk_tmpls;
    templates[5] = p->direct_tmpls;
    return TCW_OK;
}

int tcw_batch_run(tcw_handle *h, tcw_plan *p, const uint32_t *ts, const float *cols,
                  int64_t col_stride, float *F_out, tcw_stats *stats_dev, int use_graph,
                  void *stream) {
    if (!h || !p || !ts || !cols || !F_out || !stats_dev)
        return fail(TCW_ERR_INVALID, "tcw_batch_run: null argument");
    int rc = set_device(p->device);
    if (rc) return rc;
    if ((rc = ensure_side(p))) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (!use_graph) return launch_all(*p, ts, cols, col_stride, F_out, stats_dev, st);
    const bool same = p->graph && p->g_ts == ts && p->g_cols == cols && p->g_F == F_out &&
                      p->g_stats == stats_dev && p->g_cstride == col_stride;
    if (!same) {
        if (p->graph) {
            (void)hipGraphExecDestroy(p->graph);
            p->graph = nullptr;
        }
        // Capture on a private stream: the caller's stream may be the legacy
        // default stream, which cannot be captured.  The graph is then
        // launched on the caller's stream.
        if (!p->cap_stream)
            TCW_HIP_TRY(hipStreamCreateWithFlags(&p->cap_stream, hipStreamNonBlocking));
        hipGraph_t g = nullptr;
        TCW_HIP_TRY(hipStreamBeginCapture(p->cap_stream, hipStreamCaptureModeThreadLocal));
        rc = launch_all(*p, ts, cols, col_stride, F_out, stats_dev, p->cap_stream, nullptr,
                        false);
        hipError_t e = hipStreamEndCapture(p->cap_stream, &g);  // always end the capture
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess)
            return fail(TCW_ERR_DEVICE, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
        e = hipGraphInstantiate(&p->graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            p->graph = nullptr;
            return fail(TCW_ERR_DEVICE, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        }
        p->g_ts = ts;
        p->g_cols = cols;
        p->g_F = F_out;
        p->g_stats = stats_dev;
        p->g_cstride = col_stride;
    }
    TCW_HIP_TRY(hipGraphLaunch(p->graph, st));
    return TCW_OK;
}

int tcw_batch_run_timed(tcw_handle *h, tcw_plan *p, const uint32_t *ts, const float *cols,
                        int64_t col_stride, float *F_out, tcw_stats *stats_dev,
                        double *ms_out, void *stream) {
    if (!h || !p || !ts || !cols || !F_out || !stats_dev || !ms_out)
        return fail(TCW_ERR_INVALID, "tcw_batch_run_timed: null argument");
    int rc = set_device(p->device);
    if (rc) return rc;
    if ((rc = ensure_side(p))) return rc;
    hipStream_t st = (hipStream_t)stream;
    hipEvent_t ev[4];
    for (int k = 0; k < 4; k++) TCW_HIP_TRY(hipEventCreate(&ev[k]));
    rc = launch_all(*p, ts, cols, col_stride, F_out, stats_dev, st, ev);
    hipError_t e = hipSuccess;
    if (!rc) e = hipEventSynchronize(ev[3]);
    if (!rc && e == hipSuccess) {
        float a = 0, b = 0, c = 0;
        (void)hipEventElapsedTime(&a, ev[0], ev[1]);
        (void)hipEventElapsedTime(&b, ev[1], ev[2]);
        (void)hipEventElapsedTime(&c, ev[2], ev[3]);
        ms_out[0] = a;
        ms_out[1] = b;
        ms_out[2] = c;
    }
    for (int k = 0; k < 4; k++) (void)hipEventDestroy(ev[k]);
    if (rc) return rc;
    if (e != hipSuccess) return fail(TCW_ERR_DEVICE, std::string("hipEventSynchronize: ") + hipGetErrorString(e));
    return TCW_OK;
}

int tcw_plan_destroy(tcw_plan *p) {
    delete p;
    return TCW_OK;
}

}  // extern "C"

namespace {

// The tables of a batched merge.
struct MergeTables {
    int64_t T = 0, total = 0, maxN = 0, max_end = 0;
    uint32_t TAtom = 0;
    std::vector<MergeTmpl> tmpl;
    std::vector<SegDev> segs;
};

int merge_tables(const tcw_batch_desc *d, MergeTables &tab, int64_t *m_off, uint32_t *t_data) {
    if (d->T <= 0) return fail(TCW_ERR_INVALID, "no templates");
    if (d->TAtom < 2) return fail(TCW_ERR_INVALID, "TAtom must be at least 2 seconds.");
    tab.T = d->T;
    tab.TAtom = d->TAtom;
    tab.tmpl.resize((size_t)d->T);
    int64_t off = 0;
    for (int64_t t = 0; t < d->T; t++) {
        const int64_t s0 = d->seg_begin[t], s1 = d->seg_begin[t + 1];
        if (s1 <= s0 || s1 - s0 > TCW_MAX_DETECTORS)
            return fail(TCW_ERR_INVALID, "template " + std::to_string(t) + ": needs 1.." +
                                             std::to_string(TCW_MAX_DETECTORS) +
                                             " detector segments");
        uint32_t tmin = 0xffffffffu, tmax = 0;
        for (int64_t s = s0; s < s1; s++) {
            if (d->seg_off[s + 1] <= d->seg_off[s])
                return fail(TCW_ERR_INVALID, "template " + std::to_string(t) + ": empty detector");
            if (d->seg_tlast[s] < d->seg_tfirst[s])
                return fail(TCW_ERR_INVALID, "template " + std::to_string(t) +
                                                 ": timestamps not in ascending order");
            tmin = std::min(tmin, d->seg_tfirst[s]);
            tmax = std::max(tmax, d->seg_tlast[s]);
        }
        const int64_t N = (int64_t)((tmax - tmin) / d->TAtom) + 1;
        tab.tmpl[(size_t)t] = MergeTmpl{(int64_t)tab.segs.size(),
                                        (int64_t)tab.segs.size() + (s1 - s0), off, (uint32_t)N, tmin};
        for (int64_t s = s0; s < s1; s++) {
            tab.segs.push_back(SegDev{d->seg_off[s], d->seg_off[s + 1]});
            tab.max_end = std::max(tab.max_end, d->seg_off[s + 1]);
        }
        m_off[t] = off;
        t_data[t] = tmin;
        off += N;
        tab.maxN = std::max(tab.maxN, N);
    }
    m_off[d->T] = tab.total = off;
    return TCW_OK;
}

int merge_check(const MergeTables &tab, int64_t col_stride, int64_t merged_stride) {
    if (merged_stride < tab.total)
        return fail(TCW_ERR_INVALID, "merged_stride " + std::to_string(merged_stride) +
                                         " < merged bins " + std::to_string(tab.total));
    if (col_stride < tab.max_end)
        return fail(TCW_ERR_INVALID, "col_stride smaller than the atom count");
    return TCW_OK;
}

int merge_upload(const MergeTables &tab, DevBuf &d_tab, DevBuf &d_segs) {
    int rc;
    if ((rc = d_tab.ensure(tab.tmpl.size() * sizeof(MergeTmpl))) ||
        (rc = d_segs.ensure(tab.segs.size() * sizeof(SegDev))))
        return rc;
    TCW_HIP_TRY(hipMemcpy(d_tab.p, tab.tmpl.data(), tab.tmpl.size() * sizeof(MergeTmpl),
                          hipMemcpyHostToDevice));
    TCW_HIP_TRY(hipMemcpy(d_segs.p, tab.segs.data(), tab.segs.size() * sizeof(SegDev),
                          hipMemcpyHostToDevice));
    return TCW_OK;
}

int merge_launch(const MergeTables &tab, const DevBuf &d_tab, const DevBuf &d_segs,
                 const uint32_t *ts, const float *cols, int64_t col_stride, float *merged,
                 int64_t merged_stride, int64_t *atom_bin, hipStream_t st) {
    const unsigned gy = (unsigned)std::min<int64_t>(tab.T, 65535);
    hipLaunchKernelGGL(merge_kernel, dim3((unsigned)((tab.maxN + MERGE_BINS - 1) / MERGE_BINS), gy),
                       dim3(MERGE_WG), 0, st, (const MergeTmpl *)d_tab.p, (const SegDev *)d_segs.p,
                       tab.T, ts, cols, col_stride, tab.TAtom, merged, merged_stride, atom_bin);
    TCW_HIP_TRY(hipGetLastError());
    return TCW_OK;
}

}  // namespace

// The tables of a merge that is run many times, on the device.
struct tcw_merge_plan {
    int device = 0;
    MergeTables tab;  // sizes only
    DevBuf d_tab, d_segs;
    ~tcw_merge_plan() {
        d_tab.release();
        d_segs.release();
    }
};

namespace {

// One template as a batch of one (tcw_map and tcw_map_noalloc): checks the
// atoms and plans `p` on `st` (descriptor uploads queued on `st`).
int plan_single(tcw_handle *h, tcw_plan &p, const tcw_atoms *atoms, const tcw_window *win,
                uint32_t flags, hipStream_t st, const char *who) {
    if (atoms->numDet < 1 || atoms->numDet > TCW_MAX_DETECTORS)
        return fail(TCW_ERR_INVALID,
                    std::string(who) + ": numDet must be 1.." + std::to_string(TCW_MAX_DETECTORS));
    if (!atoms->ts || !atoms->cols) return fail(TCW_ERR_INVALID, std::string(who) + ": null atoms");
    if (atoms->t_max < atoms->t_min)
        return fail(TCW_ERR_INVALID, std::string(who) + ": t_max < t_min");
    int rc = set_device(h->device);
    if (rc) return rc;
    int64_t seg_begin[2] = {0, (int64_t)atoms->numDet};
    uint32_t tfirst[TCW_MAX_DETECTORS], tlast[TCW_MAX_DETECTORS];
    // only the overall min/max matter for the binned length
    for (uint32_t X = 0; X < atoms->numDet; X++) {
        tfirst[X] = atoms->t_min;
        tlast[X] = atoms->t_max;
    }
    tcw_batch_desc d;
    d.T = 1;
    d.TAtom = atoms->TAtom;
    d.seg_begin = seg_begin;
    d.seg_off = atoms->det_off;
    d.seg_tfirst = tfirst;
    d.seg_tlast = tlast;
    d.windows = win;
    return plan_build(p, h->device, &d, flags, nullptr, st, true);
}

// An upper bound of the compact layout's scratch lies below `room` (the bound is
// a few times too high; it spares a map that is small anyway a second plan).
bool surely_fits(const tcw_atoms *atoms, const tcw_window *win, size_t room) {
    if (atoms->TAtom < 2 || atoms->t_max < atoms->t_min) return false;  // refused by the plan
    const uint64_t N = (uint64_t)(atoms->t_max - atoms->t_min) / atoms->TAtom + 1;
    tcw_window w;
    int64_t N_t0, N_tau;
    if (effective_window((uint32_t)N, atoms->TAtom, atoms->t_min, *win, w, N_t0, N_tau))
        return false;
    const double n_t0 = (double)N_t0, n_tau = (double)N_tau, n = (double)N;
    const double rowblks = n_t0 / 16 + 1, colblks = n_tau / TILE_COLS + 1;
    const double segs = (n + n_t0) / 16 + 3;  // exp chunks of 16 rows, one atom apart
    const double bytes = 65536 + 56 * (n + 1) + 4 * MERGED_STRIDE * (n + 4096) +
                         rowblks * colblks * (sizeof(ItemDev) + sizeof(ItemPart)) +
                         4 * (colblks * n_t0 + rowblks * n_tau) +
                         sizeof(ItemDev) * colblks * (segs + 1 + INIT_PARTS) +
                         8 * NC * n_tau * (segs + INIT_PARTS);
    return bytes < (double)room;
}

// A map on its way to the host goes through pinned memory up to this size (the
// map's copy then shares the call's one wait); larger ones are copied
// afterwards, straight to the caller's memory.
constexpr size_t HOST_OUT_MAX = 4u << 20;

// tcw_map (host = false) and tcw_map_host (the atoms' ts and cols, and F_host
// if given, in host memory); returns with the stream drained.
int map_single(tcw_handle *h, const tcw_atoms *atoms, const tcw_window *win, float *F_dev,
               float *F_host, tcw_stats *stats, uint32_t flags, hipStream_t st, bool host,
               const char *who) {
    tcw_plan &p = h->single;
    p.host_ts = nullptr;
    if (host && atoms->numDet >= 1 && atoms->numDet <= TCW_MAX_DETECTORS && atoms->ts && atoms->cols) {
        const int64_t n = atoms->det_off[atoms->numDet];
        if (n < 1 || atoms->col_stride != n)
            return fail(TCW_ERR_INVALID, std::string(who) + ": host columns must be [7][atoms]");
        p.host_ts = atoms->ts;
        p.host_cols = atoms->cols;
        p.n_host_atoms = n;
    }
    int rc = plan_single(h, p, atoms, win, flags, st, who);
    if (!rc)
        rc = launch_all(p, host ? (const uint32_t *)p.d_ts.p : atoms->ts,
                        host ? (const float *)p.d_cols.p : atoms->cols, atoms->col_stride, F_dev,
                        h->d_stats, st);
    size_t out = 0;
    if (!rc && F_host) {
        out = sizeof(float) * (size_t)p.F_total;
        if (out > HOST_OUT_MAX) out = 0;
        if (out && !(rc = h->single_out.ensure_pin(out)) &&
            hipMemcpyAsync(h->single_out.pin, F_dev, out, hipMemcpyDeviceToHost, st) != hipSuccess)
            rc = fail(TCW_ERR_DEVICE, std::string(who) + ": copying the map failed");
    }
    // (also after a failure: the staged copy may still be reading)
    const hipError_t e = hipStreamSynchronize(st);
    if (rc) return rc;
    TCW_HIP_TRY(e);
    *stats = *h->h_stats;
    if (out)
        std::memcpy(F_host, h->single_out.pin, out);
    else if (F_host)
        TCW_HIP_TRY(hipMemcpy(F_host, F_dev, sizeof(float) * (size_t)p.F_total,
                              hipMemcpyDeviceToHost));
    if ((flags & TCW_FLAG_LAL_STRICT) && stats->single_atom)
        return fail(TCW_ERR_SINGLE_ATOM,
                    "encountered a single-atom Fstat-calculation. This is degenerate and cannot "
                    "be computed! t0 must stay away *at least* 2*TAtom from the end of the data.");
    return TCW_OK;
}

}  // namespace

extern "C" {

int tcw_map(tcw_handle *h, const tcw_atoms *atoms, const tcw_window *win, float *F_mn_dev,
            tcw_stats *stats, uint32_t flags, void *stream) {
    if (!h || !atoms || !win || !F_mn_dev || !stats)
        return fail(TCW_ERR_INVALID, "tcw_map: null argument");
    return map_single(h, atoms, win, F_mn_dev, nullptr, stats, flags, (hipStream_t)stream, false,
                      "tcw_map");
}

int tcw_map_host(tcw_handle *h, const tcw_atoms *atoms, const tcw_window *win, float *F_mn_dev,
                 float *F_mn_host, tcw_stats *stats, uint32_t flags, void *stream) {
    if (!h || !atoms || !win || !F_mn_dev || !stats)
        return fail(TCW_ERR_INVALID, "tcw_map_host: null argument");
    return map_single(h, atoms, win, F_mn_dev, F_mn_host, stats, flags, (hipStream_t)stream, true,
                      "tcw_map_host");
}

int tcw_map_noalloc(tcw_handle *h, const tcw_atoms *atoms, const tcw_window *win,
                    float *F_mn_dev, tcw_stats *stats_dev, uint32_t flags, void *stream) {
    if (!h || !atoms || !win || !F_mn_dev || !stats_dev)
        return fail(TCW_ERR_INVALID, "tcw_map_noalloc: null argument");
    char *base = nullptr;
    int rc = noalloc_scratch_ptr(h->device, &base);
    if (rc) return rc;
    h->noalloc.arena = base;
    h->noalloc.arena_bytes = TCW_NOALLOC_SCRATCH_BYTES;
    hipStream_t st = (hipStream_t)stream;
    // the plan's buffers become views into the scratch (plan_finish), or the
    // call fails before anything is queued when the map needs more
    tcw_plan &p = h->noalloc;
    p.arena_short = false;
    p.compact = p.dry = !surely_fits(atoms, win, p.arena_bytes);
    if (p.dry) {
        if ((rc = plan_single(h, p, atoms, win, flags, st, "tcw_map_noalloc"))) return rc;
        p.compact = p.dry = false;
    }
    rc = plan_single(h, p, atoms, win, flags, st, "tcw_map_noalloc");
    if (rc && p.arena_short) {
        // narrower items or shorter chunks take more scratch than the compact layout
        p.compact = true;
        rc = plan_single(h, p, atoms, win, flags, st, "tcw_map_noalloc");
    }
    if (rc) return rc;
    // every scratch byte a kernel reads is written earlier in the same call
    // (the stage kernel also clears the single-atom flag), so nothing is cleared
    return launch_all(p, atoms->ts, atoms->cols, atoms->col_stride, F_mn_dev, stats_dev, st);
}

int tcw_merge_plan_create(tcw_handle *h, const tcw_batch_desc *d, tcw_merge_plan **out,
                          int64_t *m_off, uint32_t *t_data) {
    if (!h || !d || !out || !m_off || !t_data)
        return fail(TCW_ERR_INVALID, "tcw_merge_plan_create: null argument");
    MergeTables tab;
    int rc = merge_tables(d, tab, m_off, t_data);
    if (rc) return rc;
    if ((rc = set_device(h->device))) return rc;
    auto *p = new tcw_merge_plan;
    p->device = h->device;
    rc = merge_upload(tab, p->d_tab, p->d_segs);
    if (rc) {
        delete p;
        return rc;
    }
    tab.tmpl.clear();
    tab.segs.clear();
    p->tab = tab;
    *out = p;
    return TCW_OK;
}

int tcw_merge_plan_destroy(tcw_merge_plan *p) {
    if (p) (void)set_device(p->device);
    delete p;
    return TCW_OK;
}

int tcw_merge_run(tcw_merge_plan *p, const uint32_t *ts, const float *cols, int64_t col_stride,
                  float *merged, int64_t merged_stride, int64_t *atom_bin, void *stream) {
    if (!p || !ts || !cols || !merged)
        return fail(TCW_ERR_INVALID, "tcw_merge_run: null argument");
    int rc = merge_check(p->tab, col_stride, merged_stride);
    if (rc || (rc = set_device(p->device))) return rc;
    return merge_launch(p->tab, p->d_tab, p->d_segs, ts, cols, col_stride, merged, merged_stride,
                        atom_bin, (hipStream_t)stream);
}

int tcw_merge_batch(tcw_handle *h, const tcw_batch_desc *d, const uint32_t *ts,
                    const float *cols, int64_t col_stride, float *merged, int64_t merged_stride,
                    int64_t *m_off, uint32_t *t_data, int64_t *atom_bin, void *stream) {
    if (!h || !d || !m_off || !t_data) return fail(TCW_ERR_INVALID, "tcw_merge_batch: null argument");
    MergeTables tab;
    int rc = merge_tables(d, tab, m_off, t_data);
    if (rc) return rc;
    if (!merged) return TCW_OK;
    if (!ts || !cols) return fail(TCW_ERR_INVALID, "tcw_merge_batch: null atoms");
    if ((rc = merge_check(tab, col_stride, merged_stride)) || (rc = set_device(h->device))) return rc;
    hipStream_t st = (hipStream_t)stream;
    // the previous call's kernels may still read the tables
    TCW_HIP_TRY(hipStreamSynchronize(st));
    if ((rc = merge_upload(tab, h->d_mtab, h->d_msegs)) ||
        (rc = merge_launch(tab, h->d_mtab, h->d_msegs, ts, cols, col_stride, merged, merged_stride,
                           atom_bin, st)))
        return rc;
    TCW_HIP_TRY(hipStreamSynchronize(st));
    return TCW_OK;
}

int tcw_gather_bins(const float *in, int64_t in_stride, const int64_t *atom_bin, int64_t n_atoms,
                    float *out, int64_t out_stride, void *stream) {
    if (n_atoms < 0 || out_stride < n_atoms)
        return fail(TCW_ERR_INVALID, "tcw_gather_bins: bad sizes");
    if (n_atoms == 0) return TCW_OK;
    if (!in || !atom_bin || !out) return fail(TCW_ERR_INVALID, "tcw_gather_bins: null argument");
    const unsigned g = (unsigned)std::min<int64_t>((n_atoms + 255) / 256, 65536);
    hipLaunchKernelGGL(gather_bins_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, in,
                       in_stride, atom_bin, n_atoms, out, out_stride);
    TCW_HIP_TRY(hipGetLastError());
    return TCW_OK;
}

}  // extern "C"
