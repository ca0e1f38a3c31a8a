// What the attention kernels over paged K/V share.
#pragma once
#include "common.h"
#include "kv_layout.h"

namespace fh {

struct AttnArgs {
    const __half* q;        // [total_q, nq, hd]
    const __half* k_pool;   // [blocks, nkv, tile]
    const __half* v_pool;
    __half* out;            // [total_q, nq, hd]
    const uint32_t* cu_seqlens_q;   // [num_seqs+1] or null (decode: token i ↔ seq i)
    const uint32_t* pos_offsets;    // [num_seqs] kv position of each seq's first q token
    const uint32_t* kv_lens;        // decode form: [num_seqs] kv length incl. the new token (pos = len-1)
    const int32_t* block_tables;    // [num_seqs, max_blocks]
    float* partial;         // [tiles][nsplit][16][hd+2] when nsplit > 1
    int num_seqs, nq, nkv, tiles_per_seq, max_blocks, sliding_window, nsplit, units;
    int compact;            // grid.x enumerates real work units of a ragged batch (see the kernel), not num_seqs × tiles_per_seq
    float scale;
    // fused decode form (FUSED_QKV): q / new K / new V come straight from the qkv projection output
    const __half* qkv;      // [num_seqs, (nq + 2·nkv)·hd]
    const __half* q_norm_w;
    const __half* k_norm_w;
    const float* cos_t;
    const float* sin_t;
    __half* k_pool_w;
    __half* v_pool_w;
    float eps;
    int qk_mode;
    // decode forms: the consumer is an act-order o_proj — channel c of a row is stored at out_scatter[c] (inverse of the
    // projection's row permutation), so no gather launch sits between attention and the GEMM
    const int32_t* out_scatter;
};

// A workgroup's kv head, sequence and unit of `tiles` row tiles of it; false: none is left for it.
struct PrefillUnit { int kvh, seq, unit; };
__device__ __forceinline__ bool prefill_unit(const AttnArgs& p, int tiles, int lane, PrefillUnit* u) {
    // workgroup → (kv head, unit): workgroups go to the XCDs in turn, and a head's units are taken on one XCD (on 8 / nkv of them with fewer
    // heads), whose L2 holds the keys of 8000 tokens.  Dealt over all XCDs every L2 saw every head, and a step waited for the last-level
    // cache (8100 tokens of 32 heads on 8 705 → 590 µs, 2048 76 → 62; 1500 and 548 of 16 on 8 47.6 → 42.5).
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    int kvh, from_last;
    if ((p.nkv & 7) == 0) {
        kvh = xcd + 8 * (slot / p.units);
        from_last = slot % p.units;
    } else if ((8 % p.nkv) == 0) {
        kvh = xcd % p.nkv;
        from_last = slot * (8 / p.nkv) + xcd / p.nkv;
    } else {
        kvh = blockIdx.x / p.units;
        from_last = blockIdx.x % p.units;
    }
    if (from_last >= p.units) return false;
    const int G = p.nq / p.nkv;
    int seq = -1, unit = 0;
    {
        const int w = p.units - 1 - from_last;       // launch order reversed: the longest key ranges (last units of a causal prompt) start first
        int base = 0;
        for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
            const int s = s0 + lane;
            int units = 0;
            if (s < p.num_seqs) {
                const int all = ((int)(p.cu_seqlens_q[s + 1] - p.cu_seqlens_q[s]) * G + 15) >> 4;
                units = (all + tiles - 1) / tiles;
            }
            int incl = units;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int t = __shfl_up(incl, off, 64);
                if (lane >= off) incl += t;
            }
            const int total = __shfl(incl, 63, 64);
            if (w < base + total) {
                const unsigned long long hit = __ballot(w < base + incl);
                const int src = __ffsll((long long)hit) - 1;
                seq = s0 + src;
                unit = w - (base + __shfl(incl - units, src, 64));
                break;
            }
            base += total;
        }
        if (seq < 0) return false;
        seq = __builtin_amdgcn_readfirstlane(seq);          // wave-uniform by construction: scalar table reads below
        unit = __builtin_amdgcn_readfirstlane(unit);
    }
    *u = {kvh, seq, unit};
    return true;
}

int paged_prefill_attn_keys(const AttnArgs& a, bool eight, dim3 grid, hipStream_t s);

}  // namespace fh
