// attn_plan.hpp for ctypes: the kernels' address rules and launch choices.
#include "../pelica_amd/csrc/attn_plan.hpp"

extern "C" uint32_t tile_base(int wanted, int first, uint32_t stride_b) {
    return pelica::tile_base(wanted != 0, first, stride_b);
}
extern "C" int range_shift(int key_begin, int split_keys) { return pelica::range_shift(key_begin, split_keys); }
extern "C" uint32_t burst_offset(uint32_t lane_off, uint32_t b, uint32_t step_b, int j, int e) {
    return pelica::burst_offset(lane_off, b, step_b, j, e);
}
extern "C" int prefill_split(int hd, int n_head, int n_kv, int n_seq, int T, int kv_len, int key_begin, int key_end,
                             int window, int f32, int64_t row_stride, int cus) {
    return pelica::prefill_split({hd, n_head / n_kv, n_kv, n_seq, T, kv_len, key_begin, key_end, window, f32 != 0,
                                  row_stride ? row_stride : (int64_t)n_kv * hd}, cus);
}
