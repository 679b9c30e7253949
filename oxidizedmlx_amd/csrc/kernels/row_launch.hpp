// row_launch.hpp — the launches that a row operation takes (rows.hip). Plain
// C++, so that its bounds can be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mlxhip {

// Work-items of a row of `cols` columns, at most (a row of up to 4096 columns
// takes 64 to 256; longer than the registers hold: the streaming kernel's 256).
constexpr int row_threads(int64_t cols) {
    return cols <= 4096 ? 256 : cols <= 8192 ? 512 : cols <= 32768 ? 1024 : 256;
}

// Rows of one launch: a dispatch counts its work-items in 32 bits; 2^30 of
// them here.
constexpr int64_t row_chunk(int64_t cols) { return (int64_t(1) << 30) / row_threads(cols); }

// Rows are independent, so a long batch runs as several launches:
// launch(first row, rows, causal), until one returns nonzero. A causal mask is
// indexed by the row and masks nothing from row `cols` on, so the first
// launch of a causal call takes at least those rows.
template <class Launch>
int for_row_chunks(int64_t rows, int64_t cols, int causal, Launch&& launch) {
    for (int64_t r0 = 0; r0 < rows;) {
        int64_t n = row_chunk(cols);
        if (causal && r0 == 0) n = std::max(n, cols);
        n = std::min(n, rows - r0);
        const int rc = launch(r0, n, r0 == 0 ? causal : 0);
        if (rc != 0) return rc;
        r0 += n;
    }
    return 0;
}

}  // namespace mlxhip
