// attn_plan.hpp for ctypes: the kernels' address rules on the host.
#include "../pelica_amd/csrc/attn_plan.hpp"

extern "C" uint32_t tile_base(int wanted, int first, uint32_t stride_b) {
    return pelica::tile_base(wanted != 0, first, stride_b);
}
extern "C" int range_shift(int key_begin, int split_keys) { return pelica::range_shift(key_begin, split_keys); }
extern "C" uint32_t burst_offset(uint32_t lane_off, uint32_t b, uint32_t step_b, int j, int e) {
    return pelica::burst_offset(lane_off, b, step_b, j, e);
}
