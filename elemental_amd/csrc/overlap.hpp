// Whether two column-major blocks of device memory share an element.
#pragma once

#include <cstdint>

namespace elemamd {

// X: rx x cx with leading dimension ldx >= rx, Y: ry x cy with ldy >= ry.
// Exact: two blocks of one matrix usually interleave in memory without
// sharing anything (rows 0..127 of every column and the rows below them).
template <typename T>
bool blocks_overlap(const T* X, int64_t ldx, int64_t rx, int64_t cx, const T* Y, int64_t ldy, int64_t ry, int64_t cy) {
    if (rx <= 0 || cx <= 0 || ry <= 0 || cy <= 0) return false;
    const int64_t size = sizeof(T);
    const int64_t d = (int64_t)((uintptr_t)Y - (uintptr_t)X);  // bytes
    if (d >= ((cx - 1) * ldx + rx) * size || d + ((cy - 1) * ldy + ry) * size <= 0) return false;
    if (d % size != 0) return true;  // (elements that are not aligned with each other)
    const int64_t e = d / size;
    if (ldx == ldy) {
        // Y's first element is at row s, column q of X's columns; rows of Y
        // past the leading dimension lie one column further
        int64_t s = e % ldx, q = e / ldx;
        if (s < 0) s += ldx, --q;
        const bool here = s < rx && q < cx && q + cy > 0;
        const bool next = s + ry > ldx && q + 1 < cx && q + 1 + cy > 0;
        return here || next;
    }
    // column by column, both in increasing order
    for (int64_t i = 0, j = 0; i < cx && j < cy;) {
        const int64_t x = i * ldx, y = e + j * ldy;
        if (x + rx <= y) ++i;
        else if (y + ry <= x) ++j;
        else return true;
    }
    return false;
}

}  // namespace elemamd
