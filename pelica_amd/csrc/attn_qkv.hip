// The step before attention, fused: per-head RMS norm of the q and k heads,
// rotary embedding of q and k, q written back, the new k and v rows rounded
// to f16 into the cache (linear or ring rows).  qk_dec
// (src/moe_kernels.rs:304-378) and ROPE_KV_T (src/oss_batch.rs:113-170);
// the f16 rows replace gpt-oss's f32 cache (src/oss.rs:615-616).
//
// Head slots [0, n_head) are q heads, then n_kv k heads, then n_kv v heads;
// a lane holds 4 consecutive elements of its slot (16-byte accesses), a wave
// 64/(hd/4) slots.  The norm is a reduction over the slot's lanes.  Two
// kernels: where every access can be 16 bytes wide (launch_qkv's rule) a wave
// takes one token and one or two such groups of slots, and a rotation partner
// comes from its lane's registers; else a few consecutive tokens, with the
// partners through the slot's LDS row.
// HBM-bound: every byte is touched once.
#include <type_traits>

#include "attn_prof.hpp"
#include "attn_qkv.hpp"

namespace pelica {

// 4 consecutive floats: one 16-byte access (VEC), or four
template <bool VEC>
__device__ __forceinline__ float4v load4(const float* p) {
    if (VEC) return *reinterpret_cast<const float4v*>(p);
    return float4v{p[0], p[1], p[2], p[3]};
}
template <bool VEC>
__device__ __forceinline__ void store4(float* p, const float4v& x) {
    if (VEC) {
        *reinterpret_cast<float4v*>(p) = x;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = x[i];
    }
}

// One lane per 4 consecutive elements of a head: HD/4 lanes per head, 64/(HD/4)
// heads (slots) per wave, TPW tokens per wave.  VEC: 16-byte loads and
// stores (q/k/v rows and strides 16-byte aligned, cache rows 8-byte
// aligned).  Every token's loads (row, norm weights, rotation rows) are
// requested before any is used: a wave keeps TPW x 1 KB of its rows in
// flight, not 1 KB.
template <int HD, bool VEC, int TPW>
__global__ __launch_bounds__(256) void qkv_rope_cache_kernel(QkvParams p) {
    constexpr int LPH = HD / 4;     // lanes per head
    constexpr int HPW = 64 / LPH;   // heads per wave
    __shared__ float row[4][TPW][HPW][HD];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int sub = lane / LPH, hl = lane % LPH, e0 = 4 * hl;
    const int slot = (blockIdx.x * 4 + wave) * HPW + sub;
    const int tb = blockIdx.y * TPW, s = blockIdx.z;
    const int n_slot = p.n_head + 2 * p.n_kv;
    const int len = seq_keys(p.seq_len, s, p.kv_len);
    if (len < p.T || len > p.kv_len) return;  // (attention skips such sequences too)
    // lanes of slots past the end keep to the wave's lane exchanges with
    // harmless values and store nothing
    const bool live = slot < n_slot;
    const int kind = !live ? 2 : slot < p.n_head ? 0 : slot < p.n_head + p.n_kv ? 1 : 2;  // q, k, v
    const int h = !live ? 0 : kind == 0 ? slot : kind == 1 ? slot - p.n_head : slot - p.n_head - p.n_kv;
    const float* src0 = kind == 0 ? p.q + (size_t)h * HD : (kind == 1 ? p.k : p.v) + (size_t)h * HD;
    const int64_t tok_stride = kind == 0 ? p.tok_q : p.tok_kv;

    float4v x[TPW];
#pragma unroll
    for (int ti = 0; ti < TPW; ++ti) {
        const int t = tb + ti;
        x[ti] = live && t < p.T ? load4<VEC>(src0 + ((size_t)s * p.T + t) * tok_stride + e0)
                                : float4v{0.f, 0.f, 0.f, 0.f};
    }

    // the norm weights and the rotation's (cos, sin) of this lane's elements
    // are requested with the rows, not after them
    const float* w = kind == 0 ? p.q_norm : kind == 1 ? p.k_norm : nullptr;
    const float4v wv = w ? load4<false>(w + e0) : float4v{1.f, 1.f, 1.f, 1.f};
    const bool rot = kind < 2 && p.table && e0 < p.rot;
    float2 cssn[TPW][4];
    if (rot) {
        const int half = p.rot / 2;
#pragma unroll
        for (int ti = 0; ti < TPW; ++ti) {
            const int pos = len - p.T + min(tb + ti, p.T - 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = e0 + i;
                const int j = e >= p.rot ? 0 : p.neox ? (e < half ? e : e - half) : e >> 1;
                if (p.table_split <= 0) {
                    cssn[ti][i] = *reinterpret_cast<const float2*>(p.table + ((size_t)pos * half + j) * 2);
                } else {
                    // angle addition of the rows for pos / 256 and pos % 256
                    const float2 c1 =
                        *reinterpret_cast<const float2*>(p.table + ((size_t)(pos >> 8) * half + j) * 2);
                    const float2 c2 = *reinterpret_cast<const float2*>(
                        p.table + ((size_t)(p.table_split + (pos & 255)) * half + j) * 2);
                    cssn[ti][i] = make_float2(c1.x * c2.x - c1.y * c2.y, c1.y * c2.x + c1.x * c2.y);
                }
            }
        }
    }

#pragma unroll
    for (int ti = 0; ti < TPW; ++ti) {
        // per-head RMS norm: the sum of squares over the head's LPH lanes
        float ss = x[ti][0] * x[ti][0] + x[ti][1] * x[ti][1] + x[ti][2] * x[ti][2] + x[ti][3] * x[ti][3];
#pragma unroll
        for (int off = LPH / 2; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
        if (w) {
            const float inv = 1.f / __builtin_sqrtf(ss / (float)HD + p.eps);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[ti][i] = x[ti][i] * inv * wv[i];
        }
        // rotary: element e of the first rot pairs with its partner (e +-
        // rot/2, or e ^ 1 for interleaved pairs), read through the head's
        // LDS row
        if (p.table && e0 < p.rot) *reinterpret_cast<float4v*>(row[wave][ti][sub] + e0) = x[ti];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (rot) {
        const int half = p.rot / 2;
#pragma unroll
        for (int ti = 0; ti < TPW; ++ti) {
            const float* r = row[wave][ti][sub];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = e0 + i;
                if (e >= p.rot) continue;
                int a, b;
                if (p.neox) {
                    a = e < half ? e : e - half;
                    b = a + half;
                } else {
                    a = e & ~1;
                    b = a + 1;
                }
                const float x0 = r[a], x1 = r[b];
                x[ti][i] = e == a ? x0 * cssn[ti][i].x - x1 * cssn[ti][i].y : x0 * cssn[ti][i].y + x1 * cssn[ti][i].x;
            }
        }
    }
    if (!live) return;

#pragma unroll
    for (int ti = 0; ti < TPW; ++ti) {
        const int t = tb + ti;
        if (t >= p.T) break;
        const size_t tok = (size_t)s * p.T + t;
        if (kind == 0) {
            store4<VEC>(p.q + tok * p.tok_q + (size_t)h * HD + e0, x[ti]);
        } else {
            const int pos = len - p.T + t;
            const int64_t base = p.seq_off ? p.seq_off[s] : (int64_t)s * (p.ring_cap ? p.ring_cap : p.kv_len);
            const int64_t rowi = base + (p.ring_cap ? pos % p.ring_cap : pos);
            uint16_t* dst = (kind == 1 ? p.k_cache : p.v_cache) + rowi * p.row_stride + (int64_t)h * HD + e0;
            uint16_t hv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) hv[i] = __builtin_bit_cast(uint16_t, (_Float16)x[ti][i]);
            if (VEC) {
                *reinterpret_cast<u32x2*>(dst) = u32x2{hv[0] | (uint32_t)hv[1] << 16, hv[2] | (uint32_t)hv[3] << 16};
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) dst[i] = hv[i];
            }
        }
    }
}

// The same step where every access can be 16 bytes wide (launch_qkv): a
// wave takes one token and IT groups of 64/(HD/4) consecutive heads; the
// token's rotation is loaded in 16-byte pieces, once for all of its groups,
// and a rotation partner comes from its lane's registers, not through LDS.
// Small steps are one dependent chain of load, exchange and store: fewer
// instructions and more waves shorten it; large ones run at the copy rate.
// TPB tokens a workgroup, 4 / TPB of its waves along the heads (launch_qkv).
template <int HD, int IT, int TPB>
__global__ __launch_bounds__(256) void qkv_rope_cache_wide_kernel(QkvParams p) {
    constexpr int LPH = HD / 4, HPW = 64 / LPH, WX = 4 / TPB;
    const int wave = TPB > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int lane = threadIdx.x & 63, sub = lane / LPH, e0 = 4 * (lane % LPH);
    const int t = blockIdx.y * TPB + (TPB > 1 ? wave / WX : 0), s = blockIdx.z, n_slot = p.n_head + 2 * p.n_kv;
    const int slot0 = (blockIdx.x * WX + (TPB > 1 ? wave % WX : wave)) * (HPW * IT) + sub;
    if (slot0 - sub >= n_slot || (TPB > 1 && t >= p.T)) return;
    const int len = seq_keys(p.seq_len, s, p.kv_len);
    if (len < p.T || len > p.kv_len) return;  // (attention skips such sequences too)
    const size_t tok = (size_t)s * p.T + t;
    const int pos = len - p.T + t, half = p.rot / 2;
    float4v x[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int slot = min(slot0 + HPW * it, n_slot - 1);  // (slots past the end store nothing)
        const int hk = slot - p.n_head, hv = hk - p.n_kv;
        const float* src = hk < 0 ? p.q + tok * p.tok_q + (size_t)slot * HD
                                  : (hv < 0 ? p.k + (size_t)hk * HD : p.v + (size_t)hv * HD) + tok * p.tok_kv;
        x[it] = *reinterpret_cast<const float4v*>(src + e0);
    }
    const float4v wq = p.q_norm ? *reinterpret_cast<const float4v*>(p.q_norm + e0) : float4v{1.f, 1.f, 1.f, 1.f};
    const float4v wk = p.k_norm ? *reinterpret_cast<const float4v*>(p.k_norm + e0) : float4v{1.f, 1.f, 1.f, 1.f};
    // cos, sin of this lane's elements: 4 pairs (NeoX) or 2 (interleaved)
    const bool rot = e0 < p.rot;
    const bool hi = p.neox && e0 >= half;  // the second element of its pairs
    float c[4] = {1.f, 1.f, 1.f, 1.f}, sn[4] = {0.f, 0.f, 0.f, 0.f};
    if (rot) {
        const int j = p.neox ? (hi ? e0 - half : e0) : e0 >> 1;
        auto row = [&](size_t r, float (&cc)[4], float (&ss)[4]) {
            const float4v* q = reinterpret_cast<const float4v*>(p.table + (r * half + j) * 2);
            const float4v a = q[0], b = p.neox ? q[1] : a;
            if (p.neox) {
                cc[0] = a[0], ss[0] = a[1], cc[1] = a[2], ss[1] = a[3];
                cc[2] = b[0], ss[2] = b[1], cc[3] = b[2], ss[3] = b[3];
            } else {
                cc[0] = cc[1] = a[0], ss[0] = ss[1] = a[1], cc[2] = cc[3] = a[2], ss[2] = ss[3] = a[3];
            }
        };
        if (p.table_split <= 0) {
            row(pos, c, sn);
        } else {
            float c1[4], s1[4], c2[4], s2[4];
            row(pos >> 8, c1, s1);
            row(p.table_split + (pos & 255), c2, s2);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                c[i] = c1[i] * c2[i] - s1[i] * s2[i];
                sn[i] = s1[i] * c2[i] + c1[i] * s2[i];
            }
        }
    }
    const int partner = !rot || !p.neox ? lane : hi ? lane - half / 4 : lane + half / 4;
    const int64_t base = p.seq_off ? p.seq_off[s] : (int64_t)s * (p.ring_cap ? p.ring_cap : p.kv_len);
    const int64_t rowi = base + (p.ring_cap ? pos % p.ring_cap : pos);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int slot = slot0 + HPW * it, hk = slot - p.n_head, hv = hk - p.n_kv;
        float4v y = x[it];
        if (p.q_norm || p.k_norm) {
            float ss = y[0] * y[0] + y[1] * y[1] + y[2] * y[2] + y[3] * y[3];
#pragma unroll
            for (int off = LPH / 2; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
            if (hk < 0 ? p.q_norm != nullptr : hv < 0 && p.k_norm) {
                const float inv = 1.f / __builtin_sqrtf(ss / (float)HD + p.eps);
                const float4v w = hk < 0 ? wq : wk;
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = y[i] * inv * w[i];
            }
        }
        if (p.table) {
            float4v z;
#pragma unroll
            for (int i = 0; i < 4; ++i) z[i] = p.neox ? __shfl(y[i], partner, 64) : y[i ^ 1];
            if (rot && hv < 0) {
                float4v r;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool second = p.neox ? hi : (i & 1) != 0;
                    r[i] = second ? z[i] * sn[i] + y[i] * c[i] : y[i] * c[i] - z[i] * sn[i];
                }
                y = r;
            }
        }
        if (slot >= n_slot) break;
        if (hk < 0) {
            *reinterpret_cast<float4v*>(p.q + tok * p.tok_q + (size_t)slot * HD + e0) = y;
        } else {
            uint16_t* dst = (hv < 0 ? p.k_cache + (int64_t)hk * HD : p.v_cache + (int64_t)hv * HD) + rowi * p.row_stride + e0;
            const half4 h = {(_Float16)y[0], (_Float16)y[1], (_Float16)y[2], (_Float16)y[3]};
            *reinterpret_cast<half4*>(dst) = h;
        }
    }
}

// tokens per wave of the general kernel (gpt-oss 4096-token step: 1 token 34.7 us, 2 30.3, 3 30.3,
// 4 30.0-30.8, 5 32.7, 6 33-35, 8 36.5)
constexpr int kQkvTpw = 4;

template <int HD>
static void launch_hd(const QkvParams& p, bool vec, dim3 grid, hipStream_t st) {
    if (vec) hipLaunchKernelGGL((qkv_rope_cache_kernel<HD, true, kQkvTpw>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((qkv_rope_cache_kernel<HD, false, kQkvTpw>), grid, dim3(256), 0, st, p);
}

hipError_t launch_qkv(const QkvParams& p, hipStream_t st) {
    const int n_slot = p.n_head + 2 * p.n_kv;
    const int hpw = 64 / (p.hd / 4);  // heads per wave
    const dim3 grid((n_slot + 4 * hpw - 1) / (4 * hpw), (p.T + kQkvTpw - 1) / kQkvTpw, p.n_seq);
    auto al = [](const void* q, int a) { return (reinterpret_cast<uintptr_t>(q) % a) == 0; };
    const bool vec = al(p.q, 16) && al(p.k, 16) && al(p.v, 16) && p.tok_q % 4 == 0 && p.tok_kv % 4 == 0 &&
                     al(p.k_cache, 8) && al(p.v_cache, 8) && p.row_stride % 4 == 0;
    // the wide kernel: 16-byte table rows and norm weights too, and a
    // rotation whose partners are whole lanes away
    const bool wide = vec && (!p.q_norm || al(p.q_norm, 16)) && (!p.k_norm || al(p.k_norm, 16)) &&
                      (!p.table || (al(p.table, 16) && p.rot % (p.neox ? 8 : 4) == 0));
    ProfScope ps(kProfQkv, st);
    if (wide) {
        // one head group a wave while the call waits for its one round trip
        // (gpt-oss step, ring cache: 1 token 4.5 -> 2.6 us against 3.1 with
        // two groups and 8.5 -> 6.9 against 7.0 at 512), two once the rows'
        // bytes bound it (4096 tokens 32.5 -> 30.1 us, 32.6 with one)
        const int groups = (n_slot + hpw - 1) / hpw;
        const int it = (long long)groups * p.T * p.n_seq <= 10240 ? 1 : 2;
        const int waves = (groups + it - 1) / it;  // of one token
        // Workgroups go round the 8 XCDs in order: with an even number of
        // them along the heads, a last one with idle waves falls to the same
        // XCDs for every token.  The least tokens a workgroup (4, 2 or 1
        // waves along the heads) that leaves none idle, or an odd number
        // (4096 tokens: 24 + 16 heads of 64 19.0 -> 15.7 us, 40 + 16 of 128
        // with norms 42.0 -> 38.5; two tokens where the number is odd already
        // only cost: 64 + 16 of 64 27.0 -> 27.5).
        int tpb = 1;
        while (it == 2 && tpb < 4 && waves % (4 / tpb) != 0 && (waves + 4 / tpb - 1) / (4 / tpb) % 2 == 0) tpb *= 2;
        const dim3 g((waves + 4 / tpb - 1) / (4 / tpb), (p.T + tpb - 1) / tpb, p.n_seq);
        auto go = [&](auto hd) {
            constexpr int HD = decltype(hd)::value;
            if (it == 1) hipLaunchKernelGGL((qkv_rope_cache_wide_kernel<HD, 1, 1>), g, dim3(256), 0, st, p);
            else if (tpb == 1) hipLaunchKernelGGL((qkv_rope_cache_wide_kernel<HD, 2, 1>), g, dim3(256), 0, st, p);
            else if (tpb == 2) hipLaunchKernelGGL((qkv_rope_cache_wide_kernel<HD, 2, 2>), g, dim3(256), 0, st, p);
            else hipLaunchKernelGGL((qkv_rope_cache_wide_kernel<HD, 2, 4>), g, dim3(256), 0, st, p);
            return hipGetLastError();
        };
        switch (p.hd) {
            case 64: return go(std::integral_constant<int, 64>{});
            case 128: return go(std::integral_constant<int, 128>{});
            case 256: return go(std::integral_constant<int, 256>{});
            default: return hipErrorNotSupported;
        }
    }
    switch (p.hd) {
        case 64: launch_hd<64>(p, vec, grid, st); break;
        case 128: launch_hd<128>(p, vec, grid, st); break;
        case 256: launch_hd<256>(p, vec, grid, st); break;
        default: return hipErrorNotSupported;
    }
    return hipGetLastError();
}

}  // namespace pelica
