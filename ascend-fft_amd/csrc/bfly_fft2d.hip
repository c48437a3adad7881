// bfly_fft2d.hip -- 2-D C2C transforms of [batch][n1][n2] interleaved
// complex arrays (row-major: n1 rows of n2 points).
//
// X[k1][k2] = sum_{j1, j2} x[j1][j2] W_n1^{j1 k1} W_n2^{j2 k2} is separable:
// the row pass is the C2C kernels over batch * n1 rows of n2 points; the
// column pass takes up to C columns per workgroup, so that every load and
// store is a run of consecutive complex values.  Matrices of C columns and
// their multiples are cut into groups of C; narrower ones go whole into a
// group; the columns of other widths are numbered through the batch, so that
// a group may span two matrices and no lane idles (bfly_columns.hpp).  Two
// kernels:
//
//   k_cols       16 points per thread, up to 256-point columns (and 512- and
//                1024-point ones in few groups): C >= 16;
//   k_cols_wide  32 points per thread (bfly_wide.hpp), 512 to 4096 points in
//                256 / 512 / 1024-thread workgroups (launch_wide).
//
// One pass, so the 2-D transform is two HBM round trips.  Fewer than
// kOnePassCols 4096-point columns are split n1 = P * Q = 64 * 64 instead
// (four-step along the columns, more and shorter workgroups):
//
//   j1 = Q p + q,  k1 = kp + P kq
//   Y[Q kp + q][c] = W_n1^{q kp} * FFT_P over p of x[Q p + q][c]   (k_cols, twiddle)
//   X[kp + P kq][c] = FFT_Q over q of Y[Q kp + q][c]              (k_cols, row map)
//
// with W_n1^e = A[e mod 64] * B[e / 64] from two LDS tables.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "bfly_columns.hpp"
#include "bfly_hip.h"
#include "bfly_kernels.hpp"
#include "bfly_tables.hpp"
#include "bfly_units.hpp"
#include "bfly_wide.hpp"

namespace {

using namespace bfly_dev;
using namespace bfly_cols;

// Addressing of one column pass.  A batch item of `item` elements holds
// `mats` matrices of `ncols` columns; matrix m of item b reads rows at
// in + b*item + m*in_mstride (row pitch in_rstride) and writes at
// out + b*item + m*out_mstride (row pitch out_rstride).  Columns are numbered
// f = (b*mats + m)*ncols + column, `total` of them.
struct ColView {
    uint64_t item;
    uint64_t in_mstride, out_mstride;
    uint32_t in_rstride, out_rstride;
    uint32_t ncols, mats, total;
    uint32_t col_div;  // twiddle pass: q = column / col_div
    int temporal;      // without the streaming hint (line_aligned)
    uint32_t win;      // log2 of the units per XCD window (kAutoWindow: the launcher's choice)
    uint32_t per;      // set by the launcher, as what follows: columns per workgroup
    Divider unit;      // by the groups per matrix if whole, else by its columns
    Divider mat;       // by mats
};

// Rows that start on 128-byte lines: a run of 16 or more columns then covers
// whole lines and takes the streaming hint (512 x 1024 x 32: 48.1 us against
// 52.1 without it, 256 x 1024 x 64 46.7 against 49.0).  Other rows share every
// line with the neighbouring columns' workgroup, which the L2 serves and merges
// only without the hint (256 x 1001 x 48 42.2 us against 73.1 with it, 1024 x
// 1001 x 12 52.1 against 80.0).
bool on_lines(const void* in, const void* out) {
    return (reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) % 128 == 0;
}
bool line_aligned(const void* in, const void* out, uint32_t ncols) { return ncols % 16 == 0 && on_lines(in, out); }

// Units per XCD window (xcd_window) of k_cols.  Sweep 1 / 2 / 4 / 8 / 16 / 32 /
// 64: 256 x 1001 x 48 66.3 / 55.5 / 48.4 / 44.0 / 42.2 / 41.0 / 41.7 us, 64 x
// 1001 x 200 49.8 / 45.4 / 43.0 / 41.8 / 41.1 / 40.5 / 40.4, 256 x 1024 x 64 49.8 /
// 49.4 / 48.3 / 47.0 / 46.6 / 46.7 / 46.9.
constexpr uint32_t kColWindow = 4;  // log2
constexpr uint32_t kAutoWindow = ~0u;

// 4096-point columns from which one pass is used (4096 x 64 x 16, 1024 of
// them: 18.5 us against 27.9 in two passes, 2-D 4096 x 256 x 4 41.0 against
// 45.8; 512 of them: 17.8 against 14.1).
constexpr uint32_t kOnePassCols = 1024;

// One column group per workgroup: C = WG / T columns, 16 points per thread.
// Bound by HBM (run lengths of C columns); columns up to 256 points, and
// 512- and 1024-point ones in few groups (column_pass).
// HINT: streaming accesses (a template argument: both forms in one kernel cost
// a launch 0.1 us more, 256 x 256 x 8 5.04 -> 4.95).
template <int I, int DIR, bool TW, int WG, bool HINT, bool WHOLE, Order ORDER>
__global__ __launch_bounds__(WG) void k_cols(const float2* __restrict__ in, float2* __restrict__ out,
                                              const float2* __restrict__ tw, const float2* __restrict__ wab,
                                              ColView cv) {
    using PL = PlanOf<I>;
    using LT = C2cLdsTw<I>;
    constexpr int L = PL::N, T = PL::T, C = WG / T;
    constexpr int R0 = PL::R0, RL = PL::RL, P = PL::P;
    constexpr int STRIDE = lds_len(L) + 1;
    // the twiddle is read after the transform, whose LDS exchange (two or
    // more passes) orders the table writes before it
    static_assert(!TW || PL::NRAD > 1, "twiddle pass needs a multi-pass column plan");
    __shared__ float2 lds[C * STRIDE];
    __shared__ float2 ltw[LT::LEN];
    __shared__ float2 wt[TW ? 128 : 1];
    const int tid = threadIdx.x;
    constexpr bool FIRST = ORDER == kFirst || ORDER == kFirstGuard, GUARD = ORDER == kFirstGuard || ORDER == kAheadGuard;
    // the column plan's tables: [its pass tables | A | B] as in the local C2C table
    const float2* ab = tw + bfly_plan::stage_twiddle_len(I);
    C2cLdsTwFetch<I, WG> tabs;
    auto stage = [&] {
        if constexpr (FIRST) c2c_lds_tw<I, WG>(ltw, tw, ab, tid);
        else tabs.park(ltw, tid);
        if constexpr (TW)
            for (int i = tid; i < 128; i += WG) wt[i] = wab[i];
    };
    if constexpr (FIRST) stage();
    else tabs.fetch(tw, ab, tid);
    const int c = tid % C, t = tid / C;
    const uint32_t blk = xcd_window_log2(blockIdx.x, gridDim.x, cv.win);
    uint32_t mi, col;  // matrix and column of this lane
    bool active;
    if constexpr (WHOLE) {
        mi = cv.unit.divide(blk, &col);
        col = col * C + c;
        active = !GUARD || col < cv.ncols;
    } else if (cv.ncols % C == 0) {
        // (never at a launch of this form, but with this test in front of them
        // the loads of ragged groups are scheduled better: 32 x 2099 x 57 11.3 ->
        // 10.9 us, 16 x 689 x 378 11.9 -> 11.6)
        mi = cv.unit.divide(blk, &col);
        col = col * C + c;
        active = true;
    } else {
        const uint32_t f0 = blk * cv.per, f = f0 + c;
        active = (uint32_t)c < cv.per && f < cv.total;
        if constexpr (GUARD) {
            mi = cv.unit.divide(f, &col);
        } else {
            const uint32_t last = (cv.per < cv.total - f0 ? f0 + cv.per : cv.total) - 1;
            mi = cv.unit.divide(active ? f : last, &col);  // reads the last column again
        }
    }
    uint32_t b = mi, m = 0;
    if (cv.mats > 1) b = cv.mat.divide(mi, &m);
    const float2* src = in + b * cv.item + m * cv.in_mstride + col;
    float2 v[P];
#pragma unroll
    for (int mm = 0; mm < P / R0; mm++)
#pragma unroll
        for (int r = 0; r < R0; r++) {
            const float2* p = &src[(uint64_t)cv.in_rstride * (t + mm * T + r * (L / R0))];
            v[mm * R0 + r] = !GUARD || active ? ld_io<HINT>(p) : make_float2(0.f, 0.f);
        }
    if constexpr (!FIRST) stage();
    // the transform's first LDS exchange orders the table writes before any read
    run_plan_lt<I, T, DIR, LX_PAD>(v, lds + c * STRIDE, 0, ltw, ltw + LT::NLO, ltw + LT::NLO + LT::NHI, t,
                                   std::make_index_sequence<PL::NRAD>{});
    if (!active) return;
    float2* dst = out + b * cv.item + m * cv.out_mstride + col;
    const uint32_t q = TW ? col / cv.col_div : 0u;
#pragma unroll
    for (int mm = 0; mm < P / RL; mm++)
#pragma unroll
        for (int r = 0; r < RL; r++) {
            const int k = t + mm * T + r * (L / RL);
            float2 x = v[mm * RL + r];
            if constexpr (TW) {
                const uint32_t e = q * (uint32_t)k;  // < n1 <= 4096
                const float2 a = wt[e & 63], w = wt[64 + (e >> 6)];
                x = cmul_tw<DIR>(x, make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x));
            }
            st_io<HINT>(&dst[(uint64_t)cv.out_rstride * k], x);
        }
}

// Plans of the wide column kernel: the second pass's twiddles come from its
// own LDS table, the third pass's from wide_table.
template <int L>
struct ColPlan;
template <> struct ColPlan<512> { static constexpr int R0 = 32, R1 = 16, R2 = 1; };
template <> struct ColPlan<1024> { static constexpr int R0 = 32, R1 = 32, R2 = 1; };
template <> struct ColPlan<2048> { static constexpr int R0 = 16, R1 = 4, R2 = 32; };
template <> struct ColPlan<4096> { static constexpr int R0 = 16, R1 = 8, R2 = 32; };

// W_L^m from the column table of L; 2048 and 4096 points: m a multiple of 32
// (the 4096-point table holds W_4096^j only for j < 64 and multiples of 64).
template <int L>
__device__ __forceinline__ float2 col_root(const float2* __restrict__ tc, int m) {
    if constexpr (L == 512) {  // last pass of 16 16 2: W^k at [256 + 2 k + 1], k < 256
        const float2 w = tc[256 + 2 * (m & 255) + 1];
        return m & 256 ? make_float2(-w.x, -w.y) : w;
    } else if constexpr (L == 1024) {  // 16 16 4: W^k at [256 + 4 k + 1], quarter turns beyond
        const float2 w = tc[256 + 4 * (m & 255) + 1];
        const int q = m >> 8;
        return q == 0 ? w : q == 1 ? make_float2(w.y, -w.x) : q == 2 ? make_float2(-w.x, -w.y) : make_float2(-w.y, w.x);
    } else if constexpr (L == 2048) {  // 16 16 8: W^{4 k} at [256 + 8 k + 4], k < 256
        const float2 w = tc[256 + 8 * ((m & 1023) / 4) + 4];
        return m & 1024 ? make_float2(-w.x, -w.y) : w;
    } else {
        const Wide64 w = root64(m, L);
        return make_float2((float)w.x, (float)w.y);
    }
}

// One group of C = 32 WG / L columns per workgroup, 32 points per thread.
// HBM-bound: one read and one write of every value, in runs of C columns; the
// exchanges hold one component at a time, so 16384 points take 70 KiB of LDS
// and two 512-thread workgroups share a CU, where the 16-point kernel's one
// (139 KiB) loaded, computed and stored in turn.  1024 points take two passes
// (32 32) instead of three, and 4096 points fit one workgroup at all (two
// kernels and a third HBM round trip before).  Measured, 16-point kernels ->
// this one: 1024 x 1024 x 16 59.3 -> 49.0 us (5.5 TB/s), 2048 x 1024 x 8 83.7
// -> 57.7, 4096 x 1024 x 4 112.3 -> 68; rows that do not start on lines
// (windows and hints below included): 512 x 1001 x 24 98.6 -> 47.6, 1024 x
// 1001 x 12 98.4 -> 52.9, 2048 x 999 x 6 120 -> 54, 4096 x 333 x 9 91.5 -> 73.
template <int L, int DIR, int WG>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_cols_wide(
    const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tc, uint32_t ncols,
    Divider cols, uint32_t total, uint32_t per, int stream_in, int stream_out, uint32_t win) {
    using P = ColPlan<L>;
    constexpr int T = L / kWide, C = WG / T;
    // columns lie 32 / C banks apart (mod 64), so that the C columns and the
    // 32 / C consecutive points of a half-wave's access hit 32 banks
    constexpr int SH = C >= 32 ? 1 : 32 / C;
    constexpr int STRIDE = lds_len(L) + (SH - lds_len(L) % 64 + 64) % 64;
    constexpr int T1 = P::R0 * P::R1;
    __shared__ float lds[C * STRIDE];
    __shared__ float2 t1[T1];
    __shared__ Wide64 tab[P::R2 > 1 ? kWideTab<L> : 1];
    const int tid = threadIdx.x;
    const int c = tid % C;
    int t = tid / C;
    // columns are numbered through the batch (f = item * ncols + column), `per`
    // of them to a workgroup
    const uint32_t f0 = xcd_window_log2(blockIdx.x, gridDim.x, win) * per, f = f0 + c;
    const uint32_t end = per < total - f0 ? f0 + per : total;
    const uint32_t fr = f < end ? f : end - 1;  // beyond: reads the last column again
    uint32_t col;
    const uint32_t item = cols.divide(fr, &col);
    const uint64_t at = (uint64_t)item * L * ncols + col;
    const float2* src = in + (at + (uint64_t)t * ncols);
    float2 v[kWide];
    auto load = [&](auto nt) {
#pragma unroll
        for (int m = 0; m < kWide / P::R0; m++)
#pragma unroll
            for (int r = 0; r < P::R0; r++)
                v[m * P::R0 + r] = ld_io<decltype(nt)::value>(src + (uint64_t)(m * T + r * (L / P::R0)) * ncols);
    };
    if (stream_in) load(std::true_type{});
    else load(std::false_type{});
    // the tables, behind the columns' loads (ahead of them they held the
    // loads back: 2048 x 1024 x 4 27.5 -> 30.3 us)
    for (int i = tid; i < T1; i += WG) t1[i] = col_root<L>(tc, (i / P::R0) * (i % P::R0) * (L / T1));
    if constexpr (P::R2 > 1) {
        wide_table<L>(tab, tid);
        stockham_wide<L, T, DIR, P::R0, 1, P::R0, P::R1, P::R2>(v, lds + c * STRIDE, tab, t1, t);
    } else {
        stockham_wide<L, T, DIR, P::R0, 1, P::R0, P::R1>(v, lds + c * STRIDE, tab, t1, t);
    }
    if (f >= end) return;
    constexpr int RL = P::R2 > 1 ? P::R2 : P::R1;
    asm volatile("" : "+v"(t));
    float2* dst = out + (at + (uint64_t)t * ncols);
    auto store = [&](auto nt) {
#pragma unroll
        for (int m = 0; m < kWide / RL; m++)
#pragma unroll
            for (int r = 0; r < RL; r++)
                st_io<decltype(nt)::value>(dst + (uint64_t)(m * T + r * (L / RL)) * ncols, v[m * RL + r]);
    };
    if (stream_out) store(std::true_type{});
    else store(std::false_type{});
}

template <int L, int WG>
hipError_t launch_cols_wide(const float2* in, float2* out, const float2* tc, uint32_t ncols, uint32_t total,
                            bool aligned, bool on_line, int sign, hipStream_t s) {
    const Grid grid = column_grid(WG / (L / kWide), L, ncols, total, false, true);
    const uint32_t per = grid.per, blocks = grid.blocks;
    // Access hints and windows (kColWindow: why windows; line_aligned: why
    // other rows stay without hints).  Whole-line rows take the streaming
    // hint on the input: read into the L2s without it, the lines of a buffer
    // that another kernel writes next (the 2-D transform's workspace) made
    // that kernel's writes slow (2-D 1024 x 256 x 8 18.2 us against 23.2).
    // Outputs of runs under a line (2048 and 4096 points) are merged in the
    // L2 without the hint (4096 x 1024 x 4: 66.7 us against 76), except at
    // 2048 points and 512 threads (2-D 2048 x 256 x 4: 22.5 against 24.1);
    // so are 1024-point ones in one round of workgroups (1024 x 256 x 32:
    // 26.9 against 29.1).
    const int own = grid.own && on_line;
    const int in_hint = aligned || own;
    const int out_hint = (own && !aligned) || (aligned && (L == 512 || (L == 1024 && (WG < 1024 || blocks >= 512)) || (L == 2048 && WG == 512)));
    // Windows (log2): 32 for rows off the lines, the best of 1 .. 64 at 512 x
    // 1001 x 24 (58.9 us at 1, 49.6 at 8, 47.7 at 32, 49.8 at 64), 1024 x 1001 x
    // 12 (68.6, 54.4, 52.2, 53.7), 2048 x 999 x 6 and 4096 x 333 x 9.  On the
    // lines they matter less: 1024-thread groups of narrow 1024-point matrices
    // take 64 (1024 x 256 x 64 52.3 us at 1, 51.4 at 32, 49.8 at 64), 4096
    // points lose 25 % without (4096 x 1024 x 4 89.7 at 1, 66.5 at 16, 71.2 at
    // 32), the others are equal within 2 % from 4.
    const uint32_t win = !aligned ? 5 : WG == 1024 ? (L == 1024 && ncols <= 256 ? 6 : 5) : WG == 512 && L < 2048 ? 5 : 2;
    if (sign < 0)
        hipLaunchKernelGGL((k_cols_wide<L, -1, WG>), dim3(blocks), dim3(WG), 0, s, in, out, tc, ncols, Divider(ncols), total, per,
                           in_hint, out_hint, win);
    else
        hipLaunchKernelGGL((k_cols_wide<L, 1, WG>), dim3(blocks), dim3(WG), 0, s, in, out, tc, ncols, Divider(ncols), total, per,
                           in_hint, out_hint, win);
    return hipGetLastError();
}

// Picks the wide kernel's workgroup.  256, 512 and 1024 threads keep the same
// number of columns resident (four, two and one workgroup to a CU), so the
// smallest that still gives every CU at most one workgroup is the fastest:
// with a few more, some CUs run two while the others wait (whole-line rows,
// the smaller -> the larger workgroup: 2-D 2048 x 256 x 12 53.0 -> 45.0 us,
// 1024 x 1024 x 6 45.4 -> 41.3, 4096 x 256 x 6 67.1 -> 50.0; one size too large:
// 1024 x 1024 x 2 19.5 -> 22.3).  Beyond one to a CU, whole-line rows take
// 1024 threads: longer runs (256 bytes at 1024 points; 1024 x 1024 x 16: 48.7
// us against 55.7 at 512, 2048 x 1024 x 8: 55.0 against 75.9).  The lines below
// are where the measurements leave this rule.
template <int L>
hipError_t launch_wide(const float2* in, float2* out, const float2* tc, uint32_t ncols, uint32_t total, bool aligned,
                       bool on_line, bool rows_behind, int sign, hipStream_t s) {
    constexpr uint32_t kOne = 256 * (16384 / L);  // columns of one 512-thread workgroup per CU
    constexpr uint32_t C512 = 16384 / L;          // columns of a 512-thread workgroup
    // Matrices narrower than a line, once smaller workgroups would give each CU
    // one: the smallest that holds a matrix (bfly_columns.hpp; 1024 x 12 x 400 24.2 ->
    // 17.1 us, 2048 x 7 x 300 24.4 -> 16.7; below, 1024 x 12 x 50 8.2 against 10.0),
    // or two that fill it (1024 x 8 x 1000 26.0 -> 21.6)
    if (ncols < 16) {
        const uint32_t mats = total / ncols;
        if constexpr (L < 4096)
            if (2 * ncols <= C512 && !(2 * ncols == C512 && mats > 768))
                return launch_cols_wide<L, 256>(in, out, tc, ncols, total, aligned, on_line, sign, s);
        if constexpr (L > 512)
            if (ncols > C512 && total > 192 * C512)
                return launch_cols_wide<L, 1024>(in, out, tc, ncols, total, aligned, on_line, sign, s);
        if (ncols <= C512 && total > 96 * C512)
            return launch_cols_wide<L, 512>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    }
    if constexpr (L == 512) {
        // 256 threads: whole-line rows of few columns (512 x 256 x 80 73.0 us
        // against 65.5 at 512 threads, x 128 105 against 99; 512 columns 63.5
        // against 66.5), other rows up to three quarters of the resident
        // columns (512 x 999 x 12 20.1 against 18.0, x 16 25.3 against 26.8)
        if (aligned ? ncols <= 256 : total <= 12288)
            return launch_cols_wide<L, 256>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    } else if constexpr (L == 4096) {
        if (total > kOne) return launch_cols_wide<L, 1024>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    } else if (aligned) {
        // narrow matrices, behind the 2-D transform's row pass or in less than
        // a round, run better at 512 threads (2-D 1024 x 128 x 128 90.4 us
        // against 95.1, where the column pass by itself takes 61.1 against
        // 51.8; 1024 x 128 x 48 39.9 against 41.5)
        const bool narrow = ncols < 256 && (total < 2 * kOne || (L == 1024 && rows_behind));
        if (total > kOne && !narrow)
            return launch_cols_wide<L, 1024>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    } else if (L == 1024 && total <= 6144) {
        // (1024 x 999 x 6 21.4 us against 22.3 at 512 threads, x 7 32.6 against 26.6)
        return launch_cols_wide<L, 256>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    }
    // (2048 points: 512 threads from half a round, 2-D 2048 x 256 x 4 23.2 us
    // against 24.0, x 2 22.2 against 20.2)
    if (L == 4096 || total >= kOne / (L == 2048 && aligned ? 2 : 1))
        return launch_cols_wide<L, 512>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    if constexpr (L < 4096) return launch_cols_wide<L, 256>(in, out, tc, ncols, total, aligned, on_line, sign, s);
    return hipErrorInvalidValue;
}

template <int I, bool TW, int WG = bfly_plan::kBlock>
hipError_t launch_cols(const float2* in, float2* out, const float2* tw, const float2* wab, ColView cv, bool on_line,
                       int sign, hipStream_t s) {
    constexpr uint32_t C = WG / PlanOf<I>::T;
    constexpr int L = PlanOf<I>::N;
    // (a pass of the split reads or writes rows that its matrices share)
    const bool split = TW || cv.mats > 1;
    const Grid grid = column_grid(C, L, cv.ncols, cv.total, true, !split);
    const bool whole = grid.whole;
    const uint32_t blocks = grid.blocks;
    cv.per = grid.per;
    if (grid.own && on_line) cv.temporal = 0;
    // whole-line rows in fewer workgroups: as dealt (the split's first pass at
    // 4096 x 64 x 4 5.4 us against 6.6; 256 x 64 x 256 13.6 against 14.1); 64 and 128 points
    // always (128 x 2048 x 64 46.2 us against 59.0 in windows, other widths equal)
    if (cv.win == kAutoWindow) cv.win = blocks >= 2048 && L != 64 && L != 128 ? kColWindow : 0;
    cv.unit = Divider(whole ? cv.ncols / C : cv.ncols);
    cv.mat = Divider(cv.mats);
    auto go = [&](auto hint, auto w, auto order) {
        constexpr bool H = decltype(hint)::value, W = decltype(w)::value;
        constexpr Order O = decltype(order)::value;
        if (sign < 0)
            hipLaunchKernelGGL((k_cols<I, -1, TW, WG, H, W, O>), dim3(blocks), dim3(WG), 0, s, in, out, tw, wab, cv);
        else
            hipLaunchKernelGGL((k_cols<I, 1, TW, WG, H, W, O>), dim3(blocks), dim3(WG), 0, s, in, out, tw, wab, cv);
    };
    auto pick = [&](auto w, auto order) {
        if (cv.temporal) go(std::false_type{}, w, order);
        else go(std::true_type{}, w, order);
    };
    constexpr std::integral_constant<Order, kFirst> first{};
    constexpr std::integral_constant<Order, kFirstGuard> first_guard{};
    if constexpr (!TW)  // (the split's first pass is 64 ncols wide: whole)
        if (!whole) {
            // the split's second pass: tables first from 16 columns (4096 x 16 x
            // 40 17.6 -> 15.6 us, 4096 x 100 x 7 18.9 -> 17.3), else as the first
            // (4096 x 5 x 200 27.0 -> 25.9)
            if constexpr (L == 64)
                if (split && (cv.ncols >= 16 || blocks > 256)) {
                    if (cv.ncols >= 16 && blocks > 512) pick(std::false_type{}, first_guard);
                    else if (cv.ncols >= 16) pick(std::false_type{}, first);
                    else pick(std::false_type{}, std::integral_constant<Order, kAheadGuard>{});
                    return hipGetLastError();
                }
            // ragged groups: tables ahead, at 16 and 32 points guarded (16 x
            // 1000 x 400 22.5 us against 23.7, 256 x 1001 x 48 44.0 against 42.5
            // at 256); matrices by themselves as whole groups at their counts
            const uint32_t in256 = blocks * (WG / 256);
            if (grid.own && in256 > 512 && in256 <= 1024) pick(std::false_type{}, first_guard);
            else pick(std::false_type{}, std::integral_constant<Order, L <= 32 ? kAheadGuard : kAhead>{});
            return hipGetLastError();
        }
    // (the split's passes: 4096 x 5 x 200 25.9 us against 27.2 tables first, 29.8
    // unguarded; 4096 x 5 x 60 14.9 tables first, 15.2 ahead)
    const Order order = !split ? whole_order(L, blocks * (WG / 256))
                        : blocks > 512 ? kAheadGuard : blocks > 448 ? kAhead : kFirst;
    if constexpr (L <= 128)
        if (order == kAhead) {
            pick(std::true_type{}, std::integral_constant<Order, kAhead>{});
            return hipGetLastError();
        }
    if constexpr (L == 64 || L == 128)
        if (order == kAheadGuard) {
            pick(std::true_type{}, std::integral_constant<Order, kAheadGuard>{});
            return hipGetLastError();
        }
    if (order == kFirstGuard) pick(std::true_type{}, first_guard);
    else pick(std::true_type{}, first);
    return hipGetLastError();
}

// The column pass; `rows_behind`: of a 2-D transform whose row pass has just
// written `in`.
hipError_t column_pass(const float* in, float* out, uint32_t n1, uint32_t ncols, uint32_t batch, int sign,
                              const float* table_cols, void* work, bool rows_behind, hipStream_t s) {
    const float2* i2 = reinterpret_cast<const float2*>(in);
    float2* o2 = reinterpret_cast<float2*>(out);
    const float2* tc = reinterpret_cast<const float2*>(table_cols);
    const bfly_host::Fft2dLayout L = bfly_host::fft2d_layout(n1);
    const uint64_t item = (uint64_t)n1 * ncols, total = (uint64_t)ncols * batch;
    // the guards keep batch * n1 * ncols / 16 below 2^31, so column and
    // workgroup counts fit 32 bits
    if (total == 0 || total > 0x7fffffffull) return hipErrorInvalidValue;
    const uint32_t F = (uint32_t)total;
    const bool on_line = on_lines(in, out), al = line_aligned(in, out, ncols);
    constexpr auto idx = bfly_plan::plan_index;
    // (16 and 32 points, whose runs of 2 and 1 KiB are mostly whole lines
    // however the rows start, past what the last-level cache holds: 16 x 1000
    // x 700 32.6 us with the hint, 34.7 without; 16 x 1000 x 400 20.4 against
    // 17.2, 32 x 167 x 500 11.6 against 9.3)
    const bool hint = al || (n1 <= 32 && item * batch > (1ull << 23));
    const ColView cv{item, 0, 0, ncols, ncols, ncols, 1, F, 1, hint ? 0 : 1, al ? kAutoWindow : kColWindow, 0, {}, {}};
    const float2* t1 = tc + L.p_table;
    switch (n1) {
        case 16: return launch_cols<idx(16), false>(i2, o2, t1, nullptr, cv, on_line, sign, s);
        case 32: return launch_cols<idx(32), false>(i2, o2, t1, nullptr, cv, on_line, sign, s);
        case 64: return launch_cols<idx(64), false>(i2, o2, t1, nullptr, cv, on_line, sign, s);
        case 128: return launch_cols<idx(128), false>(i2, o2, t1, nullptr, cv, on_line, sign, s);
        case 256: return launch_cols<idx(256), false>(i2, o2, t1, nullptr, cv, on_line, sign, s);
        case 512:
            // whole-line rows in fewer column groups than the wide kernel
            // needs to fill the chip: 512 x 64 x 4 5.7 us against 6.3, 512 x
            // 64 x 128 11.6 against 12.7 (512 x 64 x 256: 26.4 against 23.1)
            // (and narrower than a line, while few or in groups that own their
            // lines: 512 x 8 x 1000 11.6 against 12.4; 512 x 1 x 5587 21.5 against 20.4)
            if ((al && F < 12288) || (ncols < 16 && (F <= 4096 || column_grid(16, 512, ncols, F, true, true).own)))
                return launch_cols<idx(512), false, 512>(i2, o2, t1, nullptr, cv, on_line, sign, s);
            return launch_wide<512>(i2, o2, t1, ncols, F, al, on_line, rows_behind, sign, s);
        case 1024:
            // whole-line rows, more columns than 256-thread workgroups take in
            // one per CU and fewer than 512-thread ones: 2-D 1024 x 1024 x 3
            // 24.2 us against 29.6 and 23.9, 1024 x 128 x 24 23.5 against 29.1
            // and 26.1, 1024 x 64 x 40 23.2 against 24.6 and 27.0
            if (al && F > 2048 && F < 4096)
                return launch_cols<idx(1024), false, 1024>(i2, o2, t1, nullptr, cv, on_line, sign, s);
            return launch_wide<1024>(i2, o2, t1, ncols, F, al, on_line, rows_behind, sign, s);
        case 2048: return launch_wide<2048>(i2, o2, t1, ncols, F, al, on_line, rows_behind, sign, s);
        default: break;
    }
    if (F >= kOnePassCols) return launch_wide<4096>(i2, o2, t1, ncols, F, al, on_line, rows_behind, sign, s);
    // P-point pass with the twiddle: in -> ws; Q-point pass with the row map: ws -> out
    float2* ws = reinterpret_cast<float2*>(work);
    const uint32_t qn = L.q * ncols;
    const bool whole = line_aligned(in, ws, qn);
    const ColView a{item, 0, 0, qn, qn, qn, 1, qn * batch, ncols, whole ? 0 : 1, whole ? kAutoWindow : kColWindow, 0, {}, {}};
    hipError_t e = launch_cols<idx(64), true>(i2, ws, t1, tc + L.wab, a, false, sign, s);
    if (e != hipSuccess) return e;
    // (with the hint from 16 columns however the rows start: read without it,
    // the lines of the workspace slow the next call's first pass, as above:
    // 4096 x 60 x 7 14.4 us against 18.5; 4096 x 3 x 214 25.7 against 21.7)
    const bool own = line_aligned(ws, out, ncols);
    const ColView b{item, qn, ncols, ncols, L.p * ncols, ncols, L.p, qn * batch, 1, own || ncols >= 16 ? 0 : 1,
                    own ? kAutoWindow : kColWindow, 0, {}, {}};
    return launch_cols<idx(64), false>(ws, o2, tc + L.q_table, nullptr, b, false, sign, s);
}

}  // namespace

namespace bfly_kern {

hipError_t columns(const float* in, float* out, uint32_t n1, uint32_t ncols, uint32_t batch, int sign,
                   const float* table_cols, void* work, hipStream_t s) {
    return column_pass(in, out, n1, ncols, batch, sign, table_cols, work, false, s);
}

hipError_t fft2d(const float* in, float* out, uint32_t n1, uint32_t n2, uint32_t batch, int sign,
                 const float* table_rows, const float* table_cols, void* work, hipStream_t s) {
    // the row pass takes the C2C kernel the library picks for (n2, batch * n1)
    const int rows = bfly_host::auto_variant(n2, batch * n1);
    if (n1 < 4096 || (uint64_t)n2 * batch >= kOnePassCols) {
        // rows in -> work, columns work -> out
        float* w = static_cast<float*>(work);
        hipError_t e = c2c(in, w, n2, batch * n1, sign, rows, table_rows, nullptr, s);
        return e != hipSuccess ? e : column_pass(w, out, n1, n2, batch, sign, table_cols, nullptr, true, s);
    }
    // rows in -> out, columns out -> work -> out
    hipError_t e = c2c(in, out, n2, batch * n1, sign, rows, table_rows, nullptr, s);
    return e != hipSuccess ? e : column_pass(out, out, n1, n2, batch, sign, table_cols, work, true, s);
}

}  // namespace bfly_kern
