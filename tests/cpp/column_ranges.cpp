// The column ranges of a folded product (ttm_amd/csrc/ttm_columns.hpp) on
// random folds: every column of A and of C lies in exactly one range, at the
// offset that range, stride w and slab sizes give it, no range is wider than
// asked for or than widest_range says, and parts of a slab start at a multiple
// of 256 columns.  Host code only.
#include "ttm_columns.hpp"

#include <cstdio>
#include <random>
#include <vector>

using namespace ttm_amd;

int main()
{
    std::mt19937 rg(5);
    int bad = 0, several = 0, parts = 0;
    for (int trial = 0; trial < 4000; ++trial) {
        Fold f;
        f.w = rg() % 3 == 0 ? 1 : 1 + rg() % (rg() % 2 ? 3000 : 40);
        f.outer = 1 + rg() % (rg() % 2 ? 4 : 700);
        f.nq = 1 + rg() % 5;
        f.m = 1 + rg() % 5;
        uint64_t const max_cols = 256 * (1 + rg() % 8);
        std::vector<int> seen_a(f.numel_a()), seen_c(f.numel_c());
        uint64_t widest = 0, count = 0;
        for_columns(f, max_cols, [&](ColumnRange const &r) {
            ++count;
            widest = r.ncols > widest ? r.ncols : widest;
            if (r.ncols == 0 || r.ncols > max_cols) ++bad;
            for (uint64_t n = 0; n < r.ncols; ++n) { // as the kernels place column n of a range
                uint64_t const k = n / f.w, i = n - k * f.w;
                for (uint64_t l = 0; l < f.nq; ++l) {
                    uint64_t const at = r.a + k * f.nq * f.w + l * f.w + i;
                    if (at >= seen_a.size()) ++bad;
                    else ++seen_a[at];
                }
                for (uint64_t j = 0; j < f.m; ++j) {
                    uint64_t const at = r.c + k * f.m * f.w + j * f.w + i;
                    if (at >= seen_c.size()) ++bad;
                    else ++seen_c[at];
                }
            }
            uint64_t const i0 = r.a % (f.nq * f.w); // first column of the range within its slab
            if (i0 % 256 != 0 || (f.w <= max_cols && i0 != 0) || i0 + (f.w > max_cols ? r.ncols : 0) > f.w) ++bad;
            if (i0 != 0) ++parts;
        });
        for (int x : seen_a) bad += x != 1;
        for (int x : seen_c) bad += x != 1;
        bad += widest != widest_range(f, max_cols);
        several += count > 1;
    }
    std::printf("%d violations, %d folds of several ranges, %d parts of slabs\n", bad, several, parts);
    return bad != 0 || several < 500 || parts < 500;
}
