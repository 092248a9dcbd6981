// Offsets of the bounds-checked result stores: what a buffer store of a sub-tile over the last columns
// addresses, and what its bounds check drops. Plain arithmetic without a device type in it, so that a
// host program can walk every lane of a sub-tile.
//
// A buffer store at byte `offset` of a window of `left` bytes is dropped when offset >= left. The window
// starts at a sub-tile's first element and ends with the matrix' (or the group's) last row, so rows
// behind the end drop by themselves. A lane whose columns lie outside takes WINDOW_OUT, plus up to a few
// hundred bytes: that is out of range only of a window of at most WINDOW_OUT bytes, whatever lies behind
// the sub-tile (an output may be larger than 2 GiB), so the window is cut to that. The cut window still
// holds what the sub-tile stores: its rows are at most WINDOW_MAX_N - 1 elements of four bytes, a group
// of 16 rows is under 2^28 bytes, and of the at most eight groups the last starts after seven of them.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define PT_HD __host__ __device__ __forceinline__
#else
#define PT_HD inline
#endif

namespace pt {

constexpr uint32_t WINDOW_OUT        = 0x80000000u;
constexpr int64_t  WINDOW_MAX_N      = 1 << 22; // columns of the matrix: below this
constexpr int      WINDOW_MAX_GROUPS = 8;       // row groups (of 16) of a sub-tile
static_assert(WINDOW_MAX_GROUPS * (16 * 4 * WINDOW_MAX_N) <= int64_t{WINDOW_OUT}, "the cut window holds every row group");

// bytes of the window of a sub-tile at (wm, wn) of a matrix of `n` columns whose rows end at m_end
PT_HD uint32_t window_bytes(int64_t m_end, int64_t wm, int64_t wn, int64_t n, int elem_bytes) {
    const int64_t bytes = ((m_end - wm) * n - wn) * elem_bytes;
    return bytes < 0 ? 0u : (bytes > int64_t{WINDOW_OUT} ? WINDOW_OUT : static_cast<uint32_t>(bytes));
}
// the window as it is seen from the next row group, `group_bytes` further on
PT_HD uint32_t window_next(uint32_t left, uint32_t group_bytes) {
    return left > group_bytes ? left - group_bytes : 0u;
}
// offset of a lane's piece that starts at column `col` of the sub-tile (`piece` bytes from `lane_offset`);
// `cols` of the sub-tile's columns are inside the matrix
PT_HD uint32_t window_offset(uint32_t lane_offset, int col, int cols, int piece) {
    return (col < cols ? lane_offset : WINDOW_OUT) + static_cast<uint32_t>(piece);
}

} // namespace pt
