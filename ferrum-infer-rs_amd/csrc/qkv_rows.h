// Where the rows of a fused q|k|v projection go: queries normed and rotated to token-major rows, keys likewise and values as they are to the paged cache.  Shared by the
// stand-alone launch (rope_kv.hip) and the projection that does it itself (tiled_gemm.hip), so that both leave the same bits.
#pragma once
#include <type_traits>

#include "common.h"
#include "kv_layout.h"
#include "rope_rows.h"

namespace fh {

struct QkvRows {
    const __half *q_norm_w, *k_norm_w;
    const float *cos_t, *sin_t;
    __half *q_out, *cache_k, *cache_v;
    const uint32_t *cu, *pos_offsets;
    const int32_t* block_tables;
    int num_seqs, m_total, q_heads, kv_heads;
    float eps;
    int qk_mode, max_blocks;
};

// f with the mode as a constant: chosen for each number by selects, and worked out for values too, a row's arithmetic was what the launch waited for
// (2048 tokens × (16 + 2·8) heads 12.6 → 11.7 µs, 986 9.1 → 8.4).
template <typename F>
__device__ __forceinline__ void qkv_with_mode(int mode, const F& f) {
    if (mode == 1) f(std::integral_constant<int, 1>{});
    else if (mode == 2) f(std::integral_constant<int, 2>{});
    else if (mode == 3) f(std::integral_constant<int, 3>{});
    else f(std::integral_constant<int, 0>{});
}

// A quarter wave's row of one head; tiles: those of this head in the row's cache block.  quad: the wave's quarters hold four tokens of one sequence whose first position is a
// multiple of four (head_dim 128: a value tile keeps four keys of a dimension together, which the quarters exchange).
template <int HD>
__device__ __forceinline__ void qkv_store_row(const RopeRow<HD>& rr, const QkvRows& p, bool is_q, bool is_k, int local_head, int tok, int pos, long physical, bool act, bool quad,
                                              int q16, int quarter) {
    constexpr int PPL = HD / 32;
    using hv = typename RopeRow<HD>::hv;
    if (is_q) {
        if (!act) return;
        __half* dst = p.q_out + ((long)tok * p.q_heads + local_head) * HD;
        *reinterpret_cast<hv*>(dst + rr.off0) = rr.out0;
        *reinterpret_cast<hv*>(dst + rr.off1) = rr.out1;
        return;
    }
    const int slot = pos % KV_BLOCK;
    _Float16* t16 = reinterpret_cast<_Float16*>((is_k ? p.cache_k : p.cache_v) + (physical * p.kv_heads + local_head) * kv_tile_elems(HD));
    if (is_k) {                                              // (PPL dimensions of a row lie within one chunk of eight)
        if (!act) return;
        *reinterpret_cast<hv*>(t16 + k_tile_off(slot, rr.off0)) = rr.out0;
        *reinterpret_cast<hv*>(t16 + k_tile_off(slot, rr.off1)) = rr.out1;
        return;
    }
    if constexpr (HD == 128) {
        if (quad) {
            // quarter t holds token t's dimensions off0 … + 3 and off1 … + 3, as four pairs; quarter r leaves with pair r of all four tokens
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            const u32x2 lo = __builtin_bit_cast(u32x2, rr.out0), hi = __builtin_bit_cast(u32x2, rr.out1);
            uint32_t from[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int pair = (quarter + i) & 3;          // quarter t sends the pair of quarter t + i
                const uint32_t mine = pair == 0 ? lo[0] : pair == 1 ? lo[1] : pair == 2 ? hi[0] : hi[1];
                from[i] = i == 0 ? mine : (uint32_t)__shfl((int)mine, ((quarter - i) & 3) * 16 + q16, 64);
            }
            uint32_t key[4];                                 // from[i] is of token (quarter − i) mod 4
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int i = (quarter - t) & 3;
                key[t] = i == 0 ? from[0] : i == 1 ? from[1] : i == 2 ? from[2] : from[3];
            }
            const int d = (quarter < 2 ? rr.off0 : rr.off1) + 2 * (quarter & 1);
            *reinterpret_cast<u32x2*>(t16 + v_tile_off(slot & ~3, d)) = (u32x2){(key[0] & 0xffff) | key[1] << 16, (key[2] & 0xffff) | key[3] << 16};
            *reinterpret_cast<u32x2*>(t16 + v_tile_off(slot & ~3, d + 1)) = (u32x2){key[0] >> 16 | (key[1] & 0xffff0000u), key[2] >> 16 | (key[3] & 0xffff0000u)};
            return;
        }
    }
    if (!act) return;
#pragma unroll
    for (int k = 0; k < PPL; k++) {
        t16[v_tile_off(slot, rr.off0 + k)] = rr.out0[k];
        t16[v_tile_off(slot, rr.off1 + k)] = rr.out1[k];
    }
}

}  // namespace fh
