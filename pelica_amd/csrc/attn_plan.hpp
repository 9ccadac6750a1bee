// Address rules of the kernels as plain arithmetic: constexpr, so that device
// code and a host test run the same lines.
#pragma once
#include <cstdint>

namespace pelica {

// Byte offset of a tile's first row, row `first` of a sequence's rows in a
// cache.  A tile that is not wanted is placed 64 rows below row 0: a
// sequence's span leaves 128 rows below 4 GiB (the check of every call), so
// modulo 2^32 each lane's piece of such a tile lies past the rows, where a
// load reads nothing.
constexpr uint32_t tile_base(bool wanted, int first, uint32_t stride_b) {
    return (uint32_t)(wanted ? first : -64) * stride_b;
}

// Positions a decode over keys [key_begin, ...) is moved up by, so that its
// first key begins a split (whole 64-key blocks): every block of it then
// starts at a row >= 0 of the range's rows, and it touches no more splits
// than its keys fill.
constexpr int range_shift(int key_begin, int split_keys) {
    return key_begin % split_keys ? split_keys - key_begin % split_keys : 0;
}

// The lane's part of the offset of load j + e of a 64-key block requested
// four loads per M0 setting: the instruction adds 1024 for each load after
// the first, which is taken off here.  Never below zero: b, the block's
// first byte, is that of a row >= 0, and step_b, the bytes from one load to
// the next, is at least 1024.
constexpr uint32_t burst_offset(uint32_t lane_off, uint32_t b, uint32_t step_b, int j, int e) {
    return lane_off + (b + (uint32_t)(j + e) * step_b - 1024u * (uint32_t)e);
}

}  // namespace pelica
