// bfly_columns.hpp -- how the column kernels (bfly_fft2d.hip) share out the
// columns among workgroups.  Host code without HIP.
#pragma once
#include <cstdint>

namespace bfly_cols {

// Columns per workgroup, at most C.  Matrices of up to C columns go whole into
// a group, k at a time: few of them are spread over the CUs, down to `least` a
// group, and the group owns its 128-byte lines (a matrix is a multiple of 16
// values), so that `own` accesses take the streaming hint as whole-line rows
// do.  Numbered through the batch, 256 columns of 1-column matrices ended up in
// one workgroup, and every line was two groups'.  16 x 1 x 256 2.2 us against
// 5.2, 256 x 1 x 120 4.9 against 6.0, 512 x 1 x 120 5.8 against 11.1, 512 x 12 x
// 400 8.9 against 11.6, 2048 x 8 x 200 14.0 against 17.3.  Below 2^20 points
// (8 MB) the hint costs (64 x 5 x 256 4.8 us against 3.5), and where a wave
// stores parts of lines (256 x 5 x 3730 18.5 against 14.8, 64 x 39 x 866 10.2
// against 8.8; the 1024- and 2048-point kernels still gain from two lines on:
// 2048 x 7 x 300 15.1 against 19.6); groups that leave lanes idle then number
// columns through the batch when they are many (16 x 100 x 600 4.6 against 5.3).
struct Share {
    uint32_t per;
    bool own;
};
inline Share column_share(uint32_t C, uint32_t L, uint32_t ncols, uint32_t total) {
    auto up = [](uint32_t a, uint32_t b) { return (a + b - 1) / b; };
    if (ncols > C) {
        // 16 points load and store with nothing between: spread over the CUs
        // (16 x 1000 x 4 2.7 -> 2.3 us; 64 x 300 x 20 would take 4.2 instead of 3.9)
        const uint32_t even = up(total, 256) < 64 ? 64 : up(total, 256);
        return {L == 16 && even < C ? even : C, false};
    }
    const uint32_t mats = total / ncols, fit = C / ncols;
    // 8 matrices of 16 or 32 points, longer ones up to about 768 rows (64 x 1 x
    // 600 in 1 / 4 / 12 matrices 5.2 / 4.2 / 3.9 us, 64 x 8 x 120 6.9 / 4.1 / 3.5),
    // but no more than 64 columns; 2048 rows at 1024 points (1 x 120 7.5 against 10.1)
    uint32_t least = L <= 32 ? 8 : L < 512 ? 768 / L : 1;
    least = L < 512 ? (least < up(C < 64 ? C : 64, ncols) ? least : up(C < 64 ? C : 64, ncols))
                    : L == 1024 && ncols == 1 ? 2 : 1;
    uint32_t k = up(mats, 256);
    k = k < least ? least : k;
    k = k < fit ? k : fit;
    // values that a wave's instruction stores side by side
    const uint32_t run = C < 64 ? 64 / C * ncols : ncols;
    const bool own = (run % 16 == 0 || (L >= 1024 && run >= 32)) && (uint64_t)total * L >= (1u << 20);
    if (!own && 8 * k * ncols < 7 * C && up(mats, k) > 256) return {C, false};
    return {k * ncols, own};
}

// The grid of a column kernel whose workgroups take up to C columns of `total`
// = matrices * ncols ones.
//   whole: workgroup b has columns C (b % g) .. + C - 1 of matrix b / g, where
//          g = ncols / C (k_cols only);
//   else:  columns per b .. per b + per - 1, numbered through the batch, `total`
//          being the end of the last workgroup's.
struct Grid {
    bool whole, own;
    uint32_t per, blocks;
};
inline Grid column_grid(uint32_t C, uint32_t L, uint32_t ncols, uint32_t total, bool can_be_whole, bool may_share) {
    if (can_be_whole && ncols % C == 0) return {true, false, C, total / C};
    const Share s = may_share ? column_share(C, L, ncols, total) : Share{C, false};
    return {false, s.own, s.per, (uint32_t)(((uint64_t)total + s.per - 1) / s.per)};
}

// Forms of k_cols.  WHOLE: every group lies inside one matrix and is full.
// ORDER: the tables are staged before the columns' loads or fetched ahead of
// them and parked behind.  GUARD: the loads lie under a branch, so that the
// first butterflies wait for all of them; without it they start on the first
// arrivals.  Measured on whole groups, by workgroups (four fit a CU):
//   first               up to 512, and 256 points above 1024 (128 x 256 x 32
//                       4.9 -> 4.6 us; 256 x 1024 x 64 48.3 -> 47.2)
//   first, guarded      513 to 1024: the workgroups of a CU no longer load all
//                       at once (32 x 512 x 150 8.9 -> 7.5, 256 x 64 x 192
//                       10.4 -> 8.8)
//   ahead               above 1024 at 16 to 64 points (32 x 1024 x 512 44.5
//                       -> 43.6), 257 to 512 at 64 and 128 (128 x 128 x 128
//                       6.5 -> 6.25)
//   ahead, guarded      above 2560 at 128 points (128 x 2048 x 64 45.6 -> 44.7)
enum Order { kFirst, kFirstGuard, kAhead, kAheadGuard };
inline Order whole_order(int L, uint32_t blocks) {  // blocks: in 256 threads
    if (blocks <= 512) return blocks > 256 && (L == 64 || L == 128) ? kAhead : kFirst;
    if (blocks <= 1024) return kFirstGuard;
    if (L <= 64) return kAhead;
    return L == 128 && blocks > 2560 ? kAheadGuard : kFirst;
}

}  // namespace bfly_cols
