// A folded product in ranges of columns (n = k * w + i, one column of C each),
// so that the converted copy of A that a kernel needs is never larger than a
// range.  A range is the same fold over part of A and C: whole slabs, or, of a
// slab wider than the range, part of its block (rows of A and C keep their
// stride w; n / w stays 0).
#pragma once

#include <algorithm>
#include <cstdint>

#include "ttm_plan.hpp"

namespace ttm_amd
{

struct ColumnRange
{
    uint64_t a, c;  // elements from the start of A and of C
    uint64_t ncols; // columns
};

// Columns of the widest range of for_columns.
inline uint64_t widest_range(const Fold &f, uint64_t max_cols)
{
    uint64_t const total = f.outer * f.w;
    if (total <= max_cols) return total;
    return f.w > max_cols ? max_cols : max_cols / f.w * f.w;
}

// fn(ColumnRange) for consecutive ranges of at most max_cols columns (a
// multiple of 256, so that parts of a block start where vectors do).
template <class Fn>
void for_columns(const Fold &f, uint64_t max_cols, Fn fn)
{
    uint64_t const total = f.outer * f.w;
    if (total <= max_cols) {
        fn(ColumnRange{0, 0, total});
        return;
    }
    if (f.w <= max_cols) {
        uint64_t const slabs = max_cols / f.w;
        for (uint64_t k = 0; k < f.outer; k += slabs)
            fn(ColumnRange{k * f.nq * f.w, k * f.m * f.w, std::min(slabs, f.outer - k) * f.w});
        return;
    }
    for (uint64_t k = 0; k < f.outer; ++k)
        for (uint64_t i = 0; i < f.w; i += max_cols)
            fn(ColumnRange{k * f.nq * f.w + i, k * f.m * f.w + i, std::min(max_cols, f.w - i)});
}

} // namespace ttm_amd
