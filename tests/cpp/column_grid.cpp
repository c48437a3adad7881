// Walks the column kernels' grids (csrc/bfly_columns.hpp) the way the kernels
// do and checks that every column of every matrix is one lane's, none lies
// outside, and no workgroup is empty.  Prints the number of grids walked.
#include <cstdio>
#include <vector>

#include "bfly_columns.hpp"

using namespace bfly_cols;

static int fail(const char* what, uint32_t C, uint32_t L, uint32_t ncols, uint32_t mats) {
    std::printf("%s: C %u L %u ncols %u matrices %u\n", what, C, L, ncols, mats);
    return 1;
}

static int walk(uint32_t C, uint32_t L, uint32_t ncols, uint32_t mats, bool can_be_whole, bool may_share) {
    const uint32_t total = ncols * mats;
    const Grid g = column_grid(C, L, ncols, total, can_be_whole, may_share);
    if (g.per < 1 || g.per > C) return fail("columns per workgroup", C, L, ncols, mats);
    if (g.whole && (g.per != C || !can_be_whole)) return fail("whole", C, L, ncols, mats);
    if (g.own && (g.per % ncols || !may_share)) return fail("own", C, L, ncols, mats);
    std::vector<uint8_t> seen(total, 0);
    for (uint32_t b = 0; b < g.blocks; b++) {
        uint32_t lanes = 0;
        for (uint32_t c = 0; c < C; c++) {
            uint32_t m, col;
            if (g.whole) {
                m = b / (ncols / C);
                col = b % (ncols / C) * C + c;
            } else {
                const uint32_t f = b * g.per + c;
                if (c >= g.per || f >= total) continue;
                m = f / ncols;
                col = f % ncols;
            }
            if (m >= mats || col >= ncols) return fail("outside", C, L, ncols, mats);
            if (seen[m * ncols + col]++) return fail("twice", C, L, ncols, mats);
            lanes++;
        }
        if (!lanes) return fail("empty workgroup", C, L, ncols, mats);
    }
    for (uint8_t s : seen)
        if (!s) return fail("missing", C, L, ncols, mats);
    return 0;
}

int main() {
    std::vector<uint32_t> widths, counts;
    for (uint32_t n = 1; n <= 70; n++) widths.push_back(n);
    for (uint32_t n : {96u, 100u, 127u, 128u, 129u, 192u, 255u, 256u, 257u, 333u, 512u, 1000u, 1024u, 4096u}) widths.push_back(n);
    for (uint32_t n = 1; n <= 20; n++) counts.push_back(n);
    for (uint32_t n : {63u, 64u, 100u, 255u, 256u, 257u, 300u, 511u, 513u, 1000u, 1025u, 3000u}) counts.push_back(n);
    long grids = 0;
    for (uint32_t L = 16; L <= 4096; L *= 2)
        for (uint32_t C : {4096 / L, 16u, 8192 / L, 16384 / L, 32768 / L})
            for (uint32_t ncols : widths)
                for (uint32_t mats : counts) {
                    if (!C || C > 512 || (uint64_t)ncols * mats > 100000) continue;
                    for (int f = 0; f < 4; f++, grids++)
                        if (walk(C, L, ncols, mats, f & 1, f & 2)) return 1;
                }
    // the orders a launch asks for are the ones it has kernels of
    for (int L = 16; L <= 1024; L *= 2)
        for (uint32_t blocks = 1; blocks < 6000; blocks++) {
            const Order o = whole_order(L, blocks);
            if ((o == kAhead && L > 128) || (o == kAheadGuard && L != 128)) return fail("order", 0, L, 0, blocks);
        }
    std::printf("%ld grids\n", grids);
    return 0;
}
