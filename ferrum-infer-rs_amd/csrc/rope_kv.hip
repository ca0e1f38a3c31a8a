// Fused split-QKV + per-head QK-RMSNorm + RoPE + paged-KV write (varlen), and the KV read-back.
//
// Reference: `BackendPagedKv::split_qkv_norm_rope_into_paged_cache_varlen`
// (ferrum-kernels/src/backend/traits.rs:1764; CUDA kernels/split_qkv_norm_rope_into_paged_cache.cu:170;
// CPU maths split_qkv + qk_norm_rope, backend/cpu.rs:1645-1783).  qk_mode: 0 copy, 1 norm + half-split
// RoPE, 2 half-split RoPE, 3 interleaved RoPE; V is always copied; pos = pos_offsets[seq] + local index;
// K/V land in pool block block_tables[seq][pos/16], slot pos%16; Q goes out token-major.
#include "common.h"
#include "kernels.h"
#include "knobs.h"
#include "qkv_rows.h"

namespace fh {

// One quarter wave per (token, head): a wave takes four consecutive tokens of a head (q heads, then k heads, then v heads), a workgroup
// four heads.  Row maths in rope_rows.h.  Bound by bytes (read q|k|v once, write it once); with a workgroup of one wave per token and four
// heads it was bound by the workgroups' starts, 0.8 ns each, and by V's stores of two bytes: a tile keeps four keys of a dimension
// together, which is the four tokens of a wave where their positions are aligned, exchanged between its quarters (head_dim 128).
//   8100 tokens × (32 + 2·8) heads: 80 → 41 µs (200 MB, what a copy takes); 2048 × (16 + 2·8): 16.5 → 10 µs
// Few rows (QUADS false): a wave takes four consecutive heads of one token, a workgroup one wave.  µs by tokens, quads | heads:
//   (32 + 2·8) × 128    8: 3.4 | 2.7    128: 3.9 | 3.7    192: 4.2 | 4.2    256: 4.4 | 4.9    1024:  8.4 | 10.7
//   (32 + 2·8) × 256    8: 4.7 | 3.3    128: 5.6 | 4.8    192: 6.2 | 5.8    256: 6.6 | 7.0    1024: 15.7 | 17.5
//   (8 + 2·2) × 128     8: 3.3 | 2.7    512: 3.8 | 3.8    768: 4.3 | 4.3   1024: 4.3 | 4.9
template <int HD, bool QUADS>
__global__ __launch_bounds__(QUADS ? 256 : 64) void split_qkv_norm_rope_paged_kernel(const __half* __restrict__ qkv, QkvRows p) {
    constexpr int HALF = HD / 2;
    constexpr int TOKENS = QUADS ? 4 : 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q16 = lane & 15, quarter = lane >> 4;
    const int heads = p.q_heads + 2 * p.kv_heads, head_raw = blockIdx.y * 4 + (QUADS ? wave : quarter), head = min(head_raw, heads - 1);
    if (QUADS && head_raw >= heads) return;
    const int tok0 = blockIdx.x * TOKENS, tok = QUADS ? min(tok0 + quarter, p.m_total - 1) : tok0;         // clamped: loads stay unconditional
    const bool act = QUADS ? tok0 + quarter < p.m_total : head_raw < heads;
    const int q_dim = p.q_heads * HD, kv_dim = p.kv_heads * HD;
    const __half* row = qkv + (long)tok * (q_dim + 2 * kv_dim);

    // locate the sequences: the last s with cu_seqlens_q[s] ≤ tok (what the reference kernel's linear scan returns), found
    // 64 sequences per memory round trip — a serial scan costs the tokens of the 32nd prompt 31 dependent loads
    int seq4[4] = {0, 0, 0, 0};
    for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
        const int s = s0 + lane;
        const uint32_t first = s < p.num_seqs ? p.cu[s] : 0xffffffffu;
        unsigned long long le = 0;
#pragma unroll
        for (int j = 0; j < TOKENS; j++) {
            le = __ballot(first <= (uint32_t)min(tok0 + j, p.m_total - 1));
            if (le) seq4[j] = s0 + 63 - __clzll((long long)le);
        }
        if (le != ~0ull) break;                              // (the last token's is the largest set)
    }
    const int seq = !QUADS || quarter == 0 ? seq4[0] : quarter == 1 ? seq4[1] : quarter == 2 ? seq4[2] : seq4[3];
    const int pos = (int)p.pos_offsets[seq] + (tok - (int)p.cu[seq]);

    const bool is_q = head < p.q_heads;
    const bool is_k = !is_q && head < p.q_heads + p.kv_heads;
    const int local_head = is_q ? head : is_k ? head - p.q_heads : head - p.q_heads - p.kv_heads;
    const __half* src = row + (is_q ? 0 : is_k ? q_dim : q_dim + kv_dim) + local_head * HD;
    const int mode = (is_q || is_k) ? p.qk_mode : 0;
    const bool quad = QUADS && tok0 + 3 < p.m_total && seq4[0] == seq4[3] && __builtin_amdgcn_readfirstlane(pos) % 4 == 0;
    const long physical = is_q ? 0 : p.block_tables[(long)seq * p.max_blocks + pos / KV_BLOCK];
    auto row_of = [&](auto m) {
        constexpr int MODE = decltype(m)::value;
        const RopeRow<HD> rr = rope_row16<HD>(src, is_q ? p.q_norm_w : p.k_norm_w, p.cos_t + (long)pos * HALF, p.sin_t + (long)pos * HALF,
                                              MODE, MODE == 1, MODE != 0, p.eps, q16);
        qkv_store_row<HD>(rr, p, is_q, is_k, local_head, tok, pos, physical, act, quad, q16, quarter);
    };
    if (QUADS) qkv_with_mode(mode, row_of);
    else if (mode) qkv_with_mode(p.qk_mode, row_of);         // (heads of a wave differ: queries and keys, then values)
    else row_of(std::integral_constant<int, 0>{});
}

int split_qkv_norm_rope_into_paged_cache_varlen_f16(
    const __half* qkv, const __half* q_norm_w, const __half* k_norm_w, const float* cos_t, const float* sin_t,
    __half* q_out, __half* cache_k, __half* cache_v, const uint32_t* cu_seqlens_q, const uint32_t* pos_offsets,
    const int32_t* block_tables, int num_seqs, int m_total, int q_heads, int kv_heads, int head_dim, float eps,
    int qk_mode, int block_size, int max_blocks_per_seq, hipStream_t s) {
    if (m_total <= 0) return 0;
    FH_REQUIRE(block_size == KV_BLOCK, "paged KV: block_size=%d unsupported (native layout uses 16)", block_size);
    FH_REQUIRE(head_dim == 64 || head_dim == 128 || head_dim == 256, "paged KV: head_dim=%d must be 64, 128 or 256", head_dim);
    FH_REQUIRE(qk_mode >= 0 && qk_mode <= 3, "paged KV: qk_mode=%d out of range", qk_mode);
    const bool quads = (long)m_total * (q_heads + 2 * kv_heads) >= knobs().rope_quad_rows;
    const dim3 grid(quads ? cdiv(m_total, 4) : m_total, cdiv(q_heads + 2 * kv_heads, 4));
    const QkvRows p{q_norm_w, k_norm_w, cos_t, sin_t, q_out, cache_k, cache_v, cu_seqlens_q, pos_offsets, block_tables, num_seqs, m_total, q_heads, kv_heads, eps, qk_mode,
                    max_blocks_per_seq};
#define FH_ROPE(HDV, QUADS) hipLaunchKernelGGL((split_qkv_norm_rope_paged_kernel<HDV, QUADS>), grid, dim3(QUADS ? 256 : 64), 0, s, qkv, p)
    if (quads) { if (head_dim == 64) FH_ROPE(64, true); else if (head_dim == 128) FH_ROPE(128, true); else FH_ROPE(256, true); }
    else { if (head_dim == 64) FH_ROPE(64, false); else if (head_dim == 128) FH_ROPE(128, false); else FH_ROPE(256, false); }
#undef FH_ROPE
    FH_CHECK_LAUNCH();
    return 0;
}

// Gather one sequence's K/V back to token-major [kv_len, kv_heads, hd] (the order ferrum-kv's
// read_kv returns, ferrum-kv/src/managers/paged.rs:528-561).  Used by parity tests and by
// prefix-cache style consumers; not on the decode hot path.
__global__ void paged_kv_read_kernel(const __half* __restrict__ cache_k, const __half* __restrict__ cache_v,
                                     const int32_t* __restrict__ block_table, int kv_heads, int hd,
                                     __half* __restrict__ k_out, __half* __restrict__ v_out) {
    const int pos = blockIdx.x, head = blockIdx.y;
    const long physical = block_table[pos / KV_BLOCK];
    const int slot = pos % KV_BLOCK;
    const long tile = (physical * kv_heads + head) * kv_tile_elems(hd);
    for (int d = threadIdx.x; d < hd; d += blockDim.x) {
        long o = ((long)pos * kv_heads + head) * hd + d;
        k_out[o] = cache_k[tile + k_tile_off(slot, d)];
        v_out[o] = cache_v[tile + v_tile_off(slot, d)];
    }
}

int paged_kv_read_f16(const __half* cache_k, const __half* cache_v, const int32_t* block_table, int kv_len,
                      int kv_heads, int head_dim, int block_size, __half* k_out, __half* v_out, hipStream_t s) {
    if (kv_len <= 0) return 0;
    FH_REQUIRE(block_size == KV_BLOCK, "paged KV: block_size=%d unsupported (native layout uses 16)", block_size);
    hipLaunchKernelGGL(paged_kv_read_kernel, dim3(kv_len, kv_heads), dim3(64), 0, s, cache_k, cache_v, block_table,
                       kv_heads, head_dim, k_out, v_out);
    FH_CHECK_LAUNCH();
    return 0;
}

}  // namespace fh
