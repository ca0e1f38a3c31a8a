// Prompt attention over paged K/V, each wave of a workgroup on keys of its own.
#include "attention_device.h"
#include "knobs.h"

namespace fh {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A workgroup's 64 query rows are in every one of its waves, and each wave goes through keys of its own: wave w through pairs of blocks w, w + NW, …  The waves'
// maxima, sums and outputs are merged at the end, in the order of the waves.
//  * Bound by what the SIMDs issue: 149 vector instructions (44 % of them the rescaling of the sums) and 16 products of 512 cycles for 32 rows × 32 keys, which
//    add up to 97 % of the cycles.  The form that shares keys through LDS with as many rows takes 32 bytes from there for 8192 products where this one
//    takes 8 (queries only) and has a barrier in each step: 1500 and 548 tokens of 16 heads on 8 42 → 28 µs, 2048 of 32 on 8 68 → 58, 986 at 366 35 → 22.
//  * K and V come from the caches into the registers that the products read, a step ahead, and are used by both tiles of 32 rows: 16 KiB for 1024 cycles of
//    products a wave, 64 B a cycle a CU at the most.  A single page for all keys (no misses) changes the time by 5 %.  Loads into AGPRs and four tiles of 16 rows
//    (twice the maxima and half the products an instruction) took 1.2 times as long, one wave a SIMD with K, V and scores of the next step under way 1.07.
//  * Products of 32 × 32: a lane has 16 keys of one row, so a row's maximum is one exchange between lane n and n + 32.  V's tiles hold four keys of a dimension side
//    by side, which is half of an operand: 8-byte loads put the halves together.
template <int NW_>
struct KeysForm {
    static constexpr int NW = NW_, MT = 2, DT = 4, KS = 8, TILE = 16 * 128, NB = 2;
    static constexpr int PART_LDS = DT * NW * 4096, STAT_LDS = MT * NW * 2 * 32 * 4, LDS = PART_LDS + STAT_LDS;
};
template <int NW_>
__global__ __launch_bounds__(64 * NW_, 2) void paged_prefill_attn_keys_kernel(AttnArgs p) {
    typedef KeysForm<NW_> F;
    constexpr int NW = F::NW, MT = F::MT, DT = F::DT, KS = F::KS, TILE = F::TILE, NB = F::NB, HD = 128;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int h = lane >> 5, n = lane & 31;
    PrefillUnit u;
    if (!prefill_unit(p, 4, lane, &u)) return;
    const int kvh = u.kvh, seq = __builtin_amdgcn_readfirstlane(u.seq), unit = __builtin_amdgcn_readfirstlane(u.unit);
    const int G = p.nq / p.nkv;
    const int tok0 = (int)p.cu_seqlens_q[seq];
    const int q_len = (int)p.cu_seqlens_q[seq + 1] - tok0;
    const int rows_total = q_len * G;
    const int pos0 = (int)p.pos_offsets[seq];

    int row_pos[MT], vis_hi[MT], vis_lo[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int row0 = (unit * MT + mt) * 32, rho = row0 + n;
        vis_hi[mt] = __builtin_amdgcn_readfirstlane(row0 + 31 < rows_total ? pos0 + row0 / G : -1);
        vis_lo[mt] = __builtin_amdgcn_readfirstlane(p.sliding_window > 0 ? pos0 + (row0 + 31) / G + 1 - p.sliding_window : 0);
        row_pos[mt] = rho < rows_total ? pos0 + rho / G : -1;
    }
    const int t_first = (unit * 64) / G, t_last = min(q_len - 1, (unit * 64 + 63) / G);
    const int kv_end = __builtin_amdgcn_readfirstlane(pos0 + t_last + 1);
    const int kv_begin = __builtin_amdgcn_readfirstlane(p.sliding_window > 0 ? max(0, pos0 + t_first + 1 - p.sliding_window) : 0);
    const int nblocks = cdiv_dev(kv_end, KV_BLOCK);
    const int first = kv_begin / (NB * KV_BLOCK) + wave, pairs = (nblocks + NB - 1) / NB;      // steps of two blocks: this wave's are first, first + NW, …

    typedef const int32_t __attribute__((address_space(4))) Table;           // (not written in this launch: scalar loads)
    Table* bt = (Table*)(uintptr_t)(p.block_tables + (long)seq * p.max_blocks);
    int phys[NB];
    auto lookup = [&](int pair) {
#pragma unroll
        for (int i = 0; i < NB; i++) phys[i] = bt[min(NB * pair + i, nblocks - 1)];        // past the end: the last block (finite data), masked below
    };
    half8 k[KS], v[NB][DT];
    const int k_lane = h * 128 + (n & 15) * 8, v_lane = k_lane + (n >> 4) * 4;
    auto issue_k = [&] {
        const long at = ((long)(n >> 4 ? phys[1] : phys[0]) * p.nkv + kvh) * TILE + k_lane;
#pragma unroll
        for (int s = 0; s < KS; s++) k[s] = *reinterpret_cast<const half8*>(p.k_pool + at + s * 256);
    };
    auto issue_v = [&] {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const __half* from = p.v_pool + ((long)phys[i] * p.nkv + kvh) * (long)TILE + v_lane;
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const u32x2 x = *reinterpret_cast<const u32x2*>(from + d * 512), y = *reinterpret_cast<const u32x2*>(from + d * 512 + 256);
                v[i][d] = __builtin_bit_cast(half8, (u32x4){x.x, x.y, y.x, y.y});
            }
        }
    };
    if (first < pairs) {                                              // (requested ahead of the queries)
        lookup(first);
        issue_k();
        issue_v();
        lookup(first + NW);
    }
    half8* q_lds = reinterpret_cast<half8*>(smem);                    // [MT][KS][64]
#pragma unroll
    for (int i = 0; i < MT * KS / NW; i++) {
        const int f = wave * (MT * KS / NW) + i, mt = f / KS, s = f % KS;
        const int rho = min((unit * MT + mt) * 32 + n, rows_total - 1);
        q_lds[f * 64 + lane] = *reinterpret_cast<const half8*>(p.q + ((long)(tok0 + rho / G) * p.nq + kvh * G + rho % G) * HD + 16 * s + 8 * h);
    }
    const float sl2 = p.scale * 1.4426950408889634f;
    float m_run[MT], l_run[MT], one = 1.0f;
    asm("" : "+s"(one));                                              // (a product by a known 1 would become a conversion and an addition)
    float16v o_acc[MT][DT], zero16;
#pragma unroll
    for (int r = 0; r < 16; r++) zero16[r] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        m_run[mt] = -INFINITY;
        l_run[mt] = 0.f;
#pragma unroll
        for (int d = 0; d < DT; d++) o_acc[mt][d] = zero16;
    }
    constexpr int QD = 4;                                             // fragments of the queries under way: a product's time each, and LDS takes four
    half8 qf[QD];
    // 32 rows × 32 keys: Sᵀ = K·Qᵀ, probabilities, Oᵀ += Vᵀ·Pᵀ.  A lane has 16 keys of a row (lane n and n + 32 a row).
    auto tile = [&](int mt, int pair, auto behind_scores) {
        float16v s;
#pragma unroll
        for (int i = 0; i < KS; i++) {
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[i], qf[i % QD], i == 0 ? zero16 : s, 0, 0, 0);
            if (i + QD < KS) qf[i % QD] = q_lds[(mt * KS + i + QD) * 64 + lane];
            __builtin_amdgcn_sched_barrier(0);
        }
        behind_scores();
        if (!(pair * 32 + 31 <= vis_hi[mt] && pair * 32 >= vis_lo[mt])) {                // wave-uniform
            const int from = p.sliding_window > 0 ? row_pos[mt] + 1 - p.sliding_window : 0;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int kp = pair * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                s[r] = kp <= row_pos[mt] && kp >= from ? s[r] : -INFINITY;
            }
        }
        asm volatile("s_nop 15" : "+v"(s));                                // (the last product, before the maxima, which are none of the compiler's)
        float part[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            asm("v_max3_f32 %0, %1, %2, %3" : "=v"(part[i]) : "v"(s[4 * i]), "v"(s[4 * i + 1]), "v"(s[4 * i + 2]));      // (fmaxf would quiet its operands, an instruction each)
            asm("v_max_f32 %0, %0, %1" : "+v"(part[i]) : "v"(s[4 * i + 3]));
        }
        float mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])) * sl2;
        const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
        const float m_new = fmaxf(m_run[mt], mx), m = m_new == -INFINITY ? 0.f : m_new;
        if (__ballot(m_new != m_run[mt]) != 0) {                           // wave-uniform: some row's maximum moved
            const float alpha = __builtin_amdgcn_exp2f(m_run[mt] - m);
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) o_acc[mt][d][r] *= alpha;
            l_run[mt] *= alpha;
            m_run[mt] = m_new;
        }
        float l = 0.f;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < QD; i++) qf[i] = q_lds[((1 - mt) * KS + i) * 64 + lane];         // (of the next tile)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            half8 pf;
#pragma unroll
            for (int r = 0; r < 8; r++) pf[r] = (_Float16)__builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * i + r], sl2, -m));
            asm("" : "+v"(pf));                                            // (rounded once: the sums are of the same numbers)
#pragma unroll
            for (int r = 0; r < 8; r += 2) {
                l_run[mt] = __builtin_fmaf((float)pf[r], one, l_run[mt]);
                l = __builtin_fmaf((float)pf[r + 1], one, l);
            }
#pragma unroll
            for (int d = 0; d < DT; d++) o_acc[mt][d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[i][d], pf, o_acc[mt][d], 0, 0, 0);
        }
        l_run[mt] += l;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < QD; i++) asm volatile("" : "+v"(qf[i]));
    };
    __syncthreads();
    if (first < pairs) {
#pragma unroll
        for (int i = 0; i < QD; i++) qf[i] = q_lds[i * 64 + lane];
        for (int pair = first; pair < pairs; pair += NW) {
            tile(0, pair, [] {});
            tile(1, pair, issue_k);
            issue_v();
            lookup(pair + 2 * NW);
        }
    }
    // Merge, a tile of 32 rows after the other: NW / 4 waves sum the parts of 32 dims
    constexpr int QUADS = 16 / NW;                                    // (of four dims and all rows a wave)
    const int my_d = wave / (NW / 4), my_q = wave % (NW / 4) * QUADS;
    float4v* parts = reinterpret_cast<float4v*>(smem);                // [32 dims][waves][4][64]
    float* stats = reinterpret_cast<float*>(smem + F::PART_LDS);      // [tile][waves][m | l][32]
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run[mt]), __float_as_uint(l_run[mt]), false, false);
        const float l = __uint_as_float(w[0]) + __uint_as_float(w[1]);
        if (h == 0) {
            stats[((mt * NW + wave) * 2) * 32 + n] = m_run[mt];
            stats[((mt * NW + wave) * 2 + 1) * 32 + n] = l;
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        __syncthreads();                                              // (the queries, or the parts of the tile before, have been read)
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                parts[((d * NW + wave) * 4 + q) * 64 + lane] = (float4v){o_acc[mt][d][4 * q], o_acc[mt][d][4 * q + 1], o_acc[mt][d][4 * q + 2], o_acc[mt][d][4 * q + 3]};
        __syncthreads();
        float f[NW], l = 0.f, ref = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            f[w] = stats[((mt * NW + w) * 2) * 32 + n];
            ref = fmaxf(ref, f[w]);
        }
        ref = ref == -INFINITY ? 0.f : ref;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            f[w] = __builtin_amdgcn_exp2f(f[w] - ref);
            l += stats[((mt * NW + w) * 2 + 1) * 32 + n] * f[w];
        }
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        const int rho = (unit * MT + mt) * 32 + n;
        __half* to = p.out + ((long)(tok0 + rho / G) * p.nq + kvh * G + rho % G) * HD + my_d * 32 + 8 * my_q + 4 * h;
#pragma unroll
        for (int q = 0; q < QUADS; q++) {
            float4v o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < NW; w++) o += parts[((my_d * NW + w) * 4 + my_q + q) * 64 + lane] * f[w];
            if (rho < rows_total) *reinterpret_cast<half4*>(to + 8 * q) = __builtin_convertvector(o * inv, half4);
        }
    }
}

template <int NW>
static int launch_keys(const AttnArgs& a, dim3 grid, hipStream_t s) {
    typedef KeysForm<NW> F;
    static bool attr = false;
    if (!attr) {
        FH_CHECK_HIP(hipFuncSetAttribute((const void*)paged_prefill_attn_keys_kernel<NW>, hipFuncAttributeMaxDynamicSharedMemorySize, F::LDS));
        attr = true;
    }
    hipLaunchKernelGGL((paged_prefill_attn_keys_kernel<NW>), grid, dim3(64 * NW), F::LDS, s, a);
    FH_CHECK_LAUNCH();
    form_hit(NW == 8 ? FORM_ATTN_KEYS_WIDE : FORM_ATTN_KEYS);
    return 0;
}
int paged_prefill_attn_keys(const AttnArgs& a, bool eight, dim3 grid, hipStream_t s) { return eight ? launch_keys<8>(a, grid, s) : launch_keys<4>(a, grid, s); }

}  // namespace fh
