// attn_plan.hpp for ctypes: the kernels' address rules on the host.
#include "../pelica_amd/csrc/attn_plan.hpp"

extern "C" uint32_t tile_base(int wanted, int first, uint32_t stride_b) {
    return pelica::tile_base(wanted != 0, first, stride_b);
}
