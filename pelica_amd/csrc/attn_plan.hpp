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

}  // namespace pelica
