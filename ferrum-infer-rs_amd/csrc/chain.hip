// The attention half of a decode layer as ONE launch, and the MLP of a dense layer of few rows with it (gfx950).
//
// A decode step of few rows is a chain of small dependent ops (qwen3_moe_forward_unified_layer.rs:46-455 issues them one
// launch at a time): [tail of the previous layer: combine + add + norm] → q|k|v GEMM → QK-norm + RoPE + paged-KV write +
// attention → o_proj GEMM → add + norm + router + top-k.  As five launches every link pays its own ramp, its first memory
// round trips and its drain (≈ 4–5 µs each even when trivial) on top of the kernel boundary, while HBM idles.  Here the five
// links are ROLES of one grid, laid out in dependency order (blocks of role A first, …): every workgroup requests what does
// not depend on its predecessor — its weights (all of them: a wave's K slice is 1–4 quant groups), its block table and
// first K/V tiles, its norm and router weights — and only then waits for the predecessor's rows.  What is left on the
// critical path of a link is: activations in, arithmetic, result out.  One 512-thread workgroup per CU is resident (the
// attention role holds two K/V fragment sets, 225 – 229 registers): at 32 rows the tail (32 workgroups), the q|k|v projection (80)
// and attention (128) are all there from the start, the o projection's workgroups move in as the tail's and q|k|v's leave
// (long before attention is done) and the router's as attention's leave — each early enough to have its weights on the way.
// Layers that take it: head_dim 128, at most 14 query heads a kv head, no biases, act order, zero points, sandwich norms or tensor parallelism; INT4 of 2048 or 4096
// columns with o_proj of K 4096, experts or dense; unquantised dense layers of 1024 columns with K 2048, or of 2048 with K 2048 or 4096.  Their MLP goes in where its
// width is whole 2048s (INT4) or 1024s (fp16), eight at most.  Others (2560, 3072, 3584, 5120 columns, …) run launches of their own.
//
// Hand-offs: the rows are their own flags.  A row that crosses workgroups inside the launch is all ones on entry (NOT_YET); its producer
// stores it write-through (sc1, 8- or 16-byte stores) and is done; a consumer's wave asks for just what it needs (sc1 loads, the GEMM roles
// straight into LDS) until no 32-bit word of it is NOT_YET any more, whatever the order in which pieces arrive.  What a producer stores is
// never NOT_YET: the NaN that would read so loses its sign.  Nothing lies between a producer's stores and its consumers' loads: no drain, no
// counter, no second round trip for the data behind the one that found the flag set (a counter for each link instead: 1.3 – 2 µs from the end of
// a role's work to its consumer's first product, now 0.6 – 1.0; a launch of one row of 2048 columns 17.0 → 15.05 µs, 8 rows 19.7 → 18.05; a step
// of one sequence through 8 expert layers, 32 steps and the prompt: 13.34 → 12.59 ms, of 12 through 32 layers of 4096 75.6 → 72.3).  No role
// waits before all its predecessors' workgroups have been dispatched (dependency order = dispatch order, and nothing that waits comes before
// something it waits for), so one launch cannot starve itself.  Two at once, on two streams or in two processes, can: every wait is bounded (≈ 20 ms), a
// give-up is counted in a host-visible word, and the runner does the call again in separate launches.  The rows are double-buffered: the q|k|v workgroups, behind their own result, make the OTHER
// half all ones for the next launch, which nobody reads any more (no fill node per layer; the forward's head kernel does it for its first launch).
//
// Dense layers of few rows go on behind role B (decode_chain_mlp_supports): gate_up and its activation (G), then down in K parts (D), as roles in
// the same order and by the same rows.  gate_up's weights (59 MB of a layer of 4096 × 14336) are on their way from when q|k|v's workgroups leave,
// which two launches began with; one G workgroup a CU holds 128 columns of them, all but the last group, so that there is one round of them
// (64 columns and two rounds: the second's loads exposed, 39 µs a launch of one row, now 32 against 16 + 15.7 + 9 and two gaps before).  One row: B done
// after 15 µs, G's rows seen 16.5 – 18.5, done 22 – 25, D's act seen 24 – 29, done 31.  (G workgroups that load D's weights through the XCD's cache under
// their products: those took 2 µs longer, and D began no earlier.)
//
// Arithmetic: in an INT4 expert layer each role is the arithmetic of the stand-alone kernel it replaces, operation for operation —
// moe_combine_add_rmsnorm_kernel, w4_gemm_wgsplit_kernel<MT, 2> (K split over the 8 waves, LDS reduction in wave order),
// paged_attn_kernel<128, true, 8> (fused QK-norm / RoPE / KV write, 8 KV-splitting waves merged in wave order),
// add_rmsnorm_route_part_kernel (Q expert parts per token, in-launch ticket merge) — but for o_proj's two parts of K.  fp16 projections and the MLP's roles have
// the products, roundings and fp32 sums of theirs and add K in another order (over the 8 waves, in parts of their own).
#include "common.h"
#include "handed_off.h"
#include "kernels.h"
#include "knobs.h"
#include "kv_layout.h"
#include "rope_rows.h"
#include "w4_device.h"
#include "route_merge.h"
#include "tiled_gemm.h"

namespace fh {

namespace {

constexpr int CH_W = 8;                 // waves per workgroup
constexpr int CH_MAX_KVH = 16;
constexpr int CH_GRAN = 10;              // granules per (token, router part): 8 candidates + max + Σexp
constexpr int CH_O_KS = 2;                // o_proj: K parts per block, each a workgroup of its own (fp32 partial rows, role B adds them)
constexpr int CH_MAX_SPLITS = 16;          // KV ranges per (sequence, kv head) in the attention role
constexpr int CH_MAX_T = CHAIN_MAX_ROWS;
constexpr int CH_GRAN_WORDS = CH_MAX_T * 4 * CH_GRAN * 2;      // tokens × Q ≤ 4 parts, 8-byte granules
constexpr int CH_SMEM = 8 * 16 * (128 + 4) * 4 + 2 * 8 * 16 * 4 + 16 * 128 * 2 + 2 * 128 * 2;     // the attention role's arena: 73,216 B

constexpr int CH_QKV_NST = 1, CH_O_NST = 1;     // 64-column supertiles per workgroup: one head (128 columns) for q|k|v, 64 columns for o_proj; 16 rows each

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct ChainGemm {
    const void* qw; const __half* sc;           // INT4 pack and its scales, or f16t tiles
    int G, N, K;
};

struct ChainArgs {
    int T, H, nq, nkv;
    int qkv_half;                 // q|k|v in 32-column blocks (one 16-row block only: few rows, every CU gets a block)
    int o_half;                   // o_proj likewise
    // role A: residual' = residual + Σ_k w_k·down_k; norm1 = rms_norm(residual')·ln_in   (absent for the first layer)
    int has_a, top_k;              // has_a: 0 no tail, 1 MoE combine (down / comb_w / top_k), 2 dense (the down projection's split-K slabs)
    const __half* down; const float* comb_w; const __half* res_in; const __half* ln_in;
    const float* a_slabs; int a_S; long a_slab_stride; int a_ld;
    const __half* a_x;              // has_a == 3: the MLP output as fp16 rows [T, H]
    float eps;
    __half* res_a;                // residual' — also what role B adds the o projection to
    __half* norm1;                // [T, H]
    ChainGemm qkv;
    __half* qkv_out;              // [T, (nq + 2 nkv)·128]
    // attention
    __half* k_pool; __half* v_pool;
    const int32_t* block_tables; const uint32_t* kv_lens;
    const __half* q_norm_w; const __half* k_norm_w; const float* cos_t; const float* sin_t;
    int qk_mode, max_blocks, sliding_window;
    float scale;
    __half* attn_out;             // [T, nq·128]
    ChainGemm o;
    // role B
    __half* res_b_out; const __half* post_ln; __half* norm2; const __half* router_w;
    int E, r_top_k, Q, norm_topk, defer_merge;
    RouteCand* cand; float* stats; unsigned* route_arrive; int32_t* ids; float* weights;
    unsigned* cnt; unsigned* cnt_next; unsigned* timeout;
    uint32_t* rows_next; int rows_next_pieces;      // the other half of the handed-off rows: NOT_YET again behind this launch
#ifdef FERRUM_HIP_EXPERIMENTS
    unsigned long long* tl;       // development: per-workgroup wall-clock stamps (tools/exp_timeline_chain.py)
#endif
    float* o_part;                // [CH_O_KS][T][H] fp32: o_proj's K parts
    int qkv_wide;                 // q|k|v in 128-column blocks (one head per workgroup)
    // (behind everything else: the one-range kernel's argument layout is the one it was tuned with)
    int attn_splits;              // KV ranges per (sequence, kv head): > 1 → partial states meet by ticket, the last arriver merges them
    float* attn_partial;          // [T·nkv][splits][16 rows][HD + 4] fp32 (m, l in the pad)
    unsigned* attn_tickets;       // [T·nkv] self-resetting
    // the MLP (dense models): norm2 and act are handed-off rows then, and down's K parts fp32 slabs for the next launch
    ChainGemm gu, dn;             // [2·inter, H] gate columns first, [H, inter]
    __half* act;                  // [T, inter]
    float* slabs;                 // [parts][T][H]
    int gelu;
};
#ifdef FERRUM_HIP_EXPERIMENTS
unsigned long long* g_chain_timeline = nullptr;
#define CH_TL(i) do { if (p.tl && threadIdx.x == 0) p.tl[(long)blockIdx.x * 4 + (i)] = wall_clock64(); } while (0)
#else
#define CH_TL(i) do {} while (0)
#endif

// A wave goes on when `ready` (the same for all its lanes) says so.
template <typename F>
__device__ __forceinline__ void chain_until(const F& ready, unsigned* timeout) {
    const unsigned long long t0 = wall_clock64();
    unsigned spins = 0;
    while (!ready()) {
        __builtin_amdgcn_s_sleep(1);
        if ((++spins & 255u) == 0u && wall_clock64() - t0 > 2000000ull) {
            if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(timeout, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            break;
        }
    }
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ uint32_t most4(u32x4 v) { return max(max(v[0], v[1]), max(v[2], v[3])); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t chain_rsrc(const void* base, long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ half8 load16_sc1(__amdgpu_buffer_rsrc_t r, int byte_off) {
    return __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 16));      // aux 16 = sc1
}
// at most N of the wave's loads and stores are still under way
template <int N>
__device__ __forceinline__ void chain_landed() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((N & 15) | 0xF70 | (N >> 4) << 14);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void store16_sc1(__amdgpu_buffer_rsrc_t r, int byte_off, half8 v) {
    u32x4 w = __builtin_bit_cast(u32x4, v);
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = written2(w[i]);
    __builtin_amdgcn_raw_buffer_store_b128(w, r, byte_off, 0, 16);
}
__device__ __forceinline__ void store16_sc1(__amdgpu_buffer_rsrc_t r, int byte_off, float4v v) {
    u32x4 w = __builtin_bit_cast(u32x4, v);
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = written1(w[i]);
    __builtin_amdgcn_raw_buffer_store_b128(w, r, byte_off, 0, 16);
}

// ── role A: MoE combine + residual add + the next input norm (fused.hip kernel A), one workgroup per token ─────────────
// `last`: behind the last layer, the final norm of the row, which goes there (the residual is at its end)
__device__ __forceinline__ void chain_role_a(const ChainArgs& p, int row, unsigned char* smem, __half* last = nullptr) {
    float* red = reinterpret_cast<float*>(smem);
    CH_TL(0); CH_TL(1);
    const int H = p.H, nvec = H >> 3, top_k = p.top_k;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int CH = 2;                        // H ≤ 8192 with 512 threads
    half8 v[CH], ln[CH];
    float ss = 0.f;
    const __amdgpu_buffer_rsrc_t r_res = chain_rsrc(p.res_a, (long)p.T * H * 2), r_n1 = chain_rsrc(p.norm1, (long)p.T * H * 2);
    // (the norm's weights are on their way with the rows, and no store of the residual row lies ahead of a wait: loads and stores retire in order)
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = threadIdx.x + c * 512;
        ln[c] = *reinterpret_cast<const half8*>(p.ln_in + (i < nvec ? i : 0) * 8);
    }
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = threadIdx.x + c * 512;
        if (i < nvec && p.has_a == 3) {
            // dense model, the MLP's output as fp16 rows (no slabs): residual add, as fused_add_rms_norm
            const half8 xv = *reinterpret_cast<const half8*>(p.a_x + (long)row * H + i * 8);
            half8 rv = *reinterpret_cast<const half8*>(p.res_in + (long)row * H + i * 8);
#pragma unroll
            for (int j = 0; j < 8; j++) rv[j] = (_Float16)((float)rv[j] + (float)xv[j]);
            v[c] = rv;
#pragma unroll
            for (int j = 0; j < 8; j++) ss += (float)rv[j] * (float)rv[j];
        } else if (i < nvec && p.has_a == 2) {
            // dense model: the MLP's down projection arrives as S fp32 split-K slabs — summed in slab order and rounded like the
            // fp16 op output (add_rmsnorm_route_kernel<true>, fused.hip), then the residual add
            float o[8];
            half8 rv = *reinterpret_cast<const half8*>(p.res_in + (long)row * H + i * 8);
            asm volatile("" ::: "memory");                            // (ahead of the slabs: behind them it is a round trip of its own)
            reduce_slabs8(p.a_slabs + (long)row * p.a_ld + i * 8, p.a_slab_stride, p.a_S, o);
#pragma unroll
            for (int j = 0; j < 8; j++) rv[j] = (_Float16)((float)rv[j] + (float)(_Float16)o[j]);
            v[c] = rv;
#pragma unroll
            for (int j = 0; j < 8; j++) ss += (float)rv[j] * (float)rv[j];
        } else if (i < nvec) {
            float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            float wk8[8];
            half8 d8[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {        // the first 8 expert rows and the residual row are requested together
                const int kc = k < top_k ? k : top_k - 1;
                wk8[k] = p.comb_w[(long)row * top_k + kc];
                d8[k] = *reinterpret_cast<const half8*>(p.down + ((long)row * top_k + kc) * H + i * 8);
            }
            half8 rv = *reinterpret_cast<const half8*>(p.res_in + (long)row * H + i * 8);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (k < top_k) {
#pragma unroll
                    for (int j = 0; j < 8; j++) acc[j] += wk8[k] * (float)d8[k][j];
                }
            }
            for (int k = 8; k < top_k; k++) {
                const float wk = p.comb_w[(long)row * top_k + k];
                const half8 d = *reinterpret_cast<const half8*>(p.down + ((long)row * top_k + k) * H + i * 8);
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] += wk * (float)d[j];
            }
#pragma unroll
            for (int j = 0; j < 8; j++) rv[j] = (_Float16)((float)rv[j] + acc[j]);
            v[c] = rv;
#pragma unroll
            for (int j = 0; j < 8; j++) ss += (float)rv[j] * (float)rv[j];
        }
    }
    // the stand-alone kernel sums four wave partials of 256 threads; rows of ≤ 2048 elements live in the first four waves
    // here too, wider rows use all eight (same order: wave 0 … 7)
    ss = wave_reduce_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float total = red[0] + red[1] + red[2] + red[3];
    if (nvec > 256) total += red[4] + red[5] + red[6] + red[7];
    const float inv = 1.0f / sqrtf(total / (float)H + p.eps);
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = threadIdx.x + c * 512;
        if (i < nvec) {
            half8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = (_Float16)((float)v[c][j] * inv * (float)ln[c][j]);
            if (last) {
                *reinterpret_cast<half8*>(last + i * 8) = o;
            } else {
                store16_sc1(r_res, (int)(((long)row * H + i * 8) * 2), v[c]);
                store16_sc1(r_n1, (int)(((long)row * H + i * 8) * 2), o);
            }
        }
    }
    CH_TL(2); CH_TL(3);
}

// ── GEMM roles (q|k|v and o_proj): one 16-row block × NST 64-column supertiles per workgroup, K split over its 8 waves ───
// All GPW quant groups of a wave's K slice are requested before the wait, and as many of them as registers hold become numbers there; the
// rows (sc1) come all at once and in whole lines into the wave's region of LDS, over again until all of them have been written (from 5 rows on
// one word of each is watched first: whole rows asked for in vain hold up their producers); the 8 partial sums meet in LDS (summed in wave
// order) and leave as 16-byte write-through stores.  A workgroup reads rows × K activation bytes after its wait, at the ≈ 70 GB/s a
// workgroup gets for handed-off bytes — so the rows are split over workgroups (16 each) rather than the columns made narrower.
// Behind the wait of 12 rows of 4096, 64 columns: 0.9 µs until the rows are there, 1.0 the products, 0.8 the slowest wave's and the meeting, 0.5
// the result (64-byte pieces of 16 rows, two groups ahead, weights expanded behind the wait: 4.1 in all, now 3.2; 16 rows of 2048 in
// 128 columns 4.2 → 3.3, o_proj's halves of K 2.7 → 2.0).
// F16W: unquantised weights, fp16 fragments of a tile row after row of K, all of a wave's (32 – 128 registers) requested before the wait and
// nothing left to expand; the products go straight into the sums.
// NTL = 16-column tiles of the 64-column supertile a workgroup takes (NST = 1): 4, or 2 — a 32-column block `cb` = supertile cb / 2,
// half cb % 2: half the weight bytes per workgroup, twice the workgroups (the stage is as long as its slowest workgroup's fetch).
// F32OUT: the workgroup covers only the quant groups from g_base on (8·GPW of them) and leaves its fp32 partial sums in `out32`
// ([K part][T][N]) — o_proj split over two workgroups per block: the rows a workgroup reads behind its wait (T·K·2 B through one CU)
// are what its stage takes, and role B adds the two parts
// GLU: the gated MLP's first projection; half of a workgroup's columns are gate's and half the same of up's, and act(gate)·up leaves it: a
// supertile of each (NST = 2, INT4: 4 groups of 128 columns, 128 registers, none expanded before the wait), or two tiles of each (NST = 1, fp16)
template <int NST, int GPW, bool F16W, int NTL = 4, bool F32OUT = false, bool GLU = false>
__device__ __forceinline__ void chain_role_gemm(const ChainGemm& w, int cb, int rb, const __half* x_in, __half* out, int T,
                                                bool handed_off, unsigned char* smem, const ChainArgs& p, int g_base = 0, float* out32 = nullptr) {
    static_assert(NTL == 4 || (NTL == 2 && NST == 1), "half supertiles only for single-supertile blocks");
    static_assert(!GLU || (NTL == 4 && NST == (F16W ? 1 : 2) && !F32OUT), "tiles of both halves");
    constexpr int V = NST * NTL * 4, CPR = NST * NTL * 2;                       // accumulator floats per lane; 16-byte chunks per output row
    float* red = reinterpret_cast<float*>(smem);                     // [8 regions of a wave][V][64]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int a = lane >> 4, b = lane & 15;
    CH_TL(0);
    const int g0 = g_base + wave * GPW;                               // G = 8·GPW (· 2 with F32OUT; checked by the launcher)
    const int nt0 = NTL == 2 ? (cb & 1) * 2 : 0;                      // first tile of the block inside its supertile
    const int up = w.N / 32 - 2;                                      // GLU, fp16: tiles 2 and 3 of the block are this many on (N / 2 is whole supertiles)
    constexpr int FIT = 8 / (NST * NTL), PRE = GLU && !F16W ? 0 : F16W || GPW < FIT ? GPW : FIT;       // (128 registers)
    static_assert(!F16W || GPW <= 8 / (NST * NTL), "16-bit weights: all of a wave's in registers");
    u32x4 wq[F16W ? 1 : GPW][NST][NTL];
    uint2 scv[F16W ? 1 : GPW][NST];
    half8 wx[PRE ? PRE : 1][NST][NTL][4];
    if constexpr (F16W) {
        const half8* w_lane = reinterpret_cast<const half8*>(w.qw) + lane;          // f16t: [N / 16][K / 32][64 lanes]
#pragma unroll
        for (int i = 0; i < GPW; i++)
#pragma unroll
            for (int s = 0; s < NST; s++)
#pragma unroll
                for (int nt = 0; nt < NTL; nt++)
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        wx[i][s][nt][k] = __builtin_nontemporal_load(w_lane + ((GLU ? (long)cb * 2 + nt + (nt & 2 ? up : 0) : (long)(cb * NST + s) * NTL + nt) * (w.K / 32) +
                                                                              (g0 + i) * 4 + k) * 64);
    }
    // (GLU, four groups: the last is asked for behind the rows.  Its workgroups fill the chip when the ones before them leave, memory is still busy
    // with their weights when the rows are there, and loads come back in order: the products of three start a quarter of them earlier.  From 5 rows on, whose rows take longer, two of them: a step of 32
    // layers of 4096, one group | two, µs: 1 row 1259 | 1277, 4 1322 | 1340, 5 1318 | 1293, 8 1376 | 1340, 9 1411 | 1378, 12 of 120 keys 1460 | 1423, 16 1518 | 1488)
    constexpr int LATE = GLU && !F16W ? GPW / 4 : 0;
    const bool two_late = LATE > 0 && T > 4;
    auto ask = [&](auto from, auto to) {
        if constexpr (!F16W) {
#pragma unroll
            for (int i = decltype(from)::value; i < decltype(to)::value; i++)
#pragma unroll
                for (int s = 0; s < NST; s++) {
                    const long st = GLU ? (long)cb + s * (w.N / 128) : NTL == 2 ? (long)(cb >> 1) : (long)cb * NST + s;
                    const u32x4* qw_lane = reinterpret_cast<const u32x4*>(w.qw) + (st * w.G * 4) * 64 + lane;
#pragma unroll
                    for (int nt = 0; nt < NTL; nt++) wq[i][s][nt] = __builtin_nontemporal_load(qw_lane + ((long)(g0 + i) * 4 + nt0 + nt) * 64);
                    scv[i][s] = (reinterpret_cast<const uint2*>(w.sc) + (st * w.G) * 16 + b)[(long)(g0 + i) * 16];
                }
        }
    };
    ask(std::integral_constant<int, 0>{}, std::integral_constant<int, GPW - 2 * LATE>{});
    if constexpr (LATE > 0) {
        if (!two_late) ask(std::integral_constant<int, GPW - 2 * LATE>{}, std::integral_constant<int, GPW - LATE>{});
    }
    // the first PRE groups' INT4 weights become numbers (q − 8) while the predecessor works: their expansion, and the products that take the
    // offset of in-place nibbles back, are not behind the wait
    if constexpr (!F16W && PRE > 0) {
        const uint32_t magic = opaque_vgpr(0x64006400u), magic_hi = opaque_vgpr(0x54005400u);
        const uint32_t m_lo = opaque_sgpr(0x000F000Fu), m_hi = opaque_sgpr(0x00F000F0u);
#pragma unroll
        for (int i = 0; i < PRE; i++)
#pragma unroll
            for (int s = 0; s < NST; s++)
#pragma unroll
                for (int nt = 0; nt < NTL; nt++)
#pragma unroll
                    for (int pr = 0; pr < 2; pr++) {
                        const uint32_t d0 = wq[i][s][nt][2 * pr], d1 = wq[i][s][nt][2 * pr + 1], d0s = d0 >> 8, d1s = d1 >> 8;
                        half8 lo = pack_half8(and_or(d0, m_lo, magic), and_or(d0s, m_lo, magic), and_or(d1, m_lo, magic), and_or(d1s, m_lo, magic));
                        half8 hi = pack_half8(and_or(d0, m_hi, magic_hi), and_or(d0s, m_hi, magic_hi), and_or(d1, m_hi, magic_hi), and_or(d1s, m_hi, magic_hi));
                        lo -= splat_half8(1032.0f);
                        hi -= splat_half8(72.0f);
                        asm volatile("" : "+v"(lo), "+v"(hi));            // (here, not at the use)
                        wx[i][s][nt][2 * pr] = lo;
                        wx[i][s][nt][2 * pr + 1] = hi;
                    }
    }
    __builtin_amdgcn_sched_barrier(0);
    const __amdgpu_buffer_rsrc_t r_x = chain_rsrc(x_in, (long)T * w.K * 2);
    constexpr int REGION = GPW * 4096;                                // a wave's rows: [group][16 rows][16 pieces of 16 bytes, piece xor row]
    static_assert(V * 256 <= REGION, "a wave's partial sums take its rows' place");
    unsigned char* const mine = smem + wave * REGION;
    chain_landed<0>();                                                // the weights: from here on only row copies are counted
    auto request = [&] {
#pragma unroll
        for (int i = 0; i < GPW; i++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = 4 * q + a;                              // (rows past the last lie outside of the buffer: zeros, and no traffic)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r_x, (__attribute__((address_space(3))) void*)(mine + (i * 4 + q) * 1024), 16,
                                                         ((rb * 16 + r) * w.K + (b ^ r) * 8) * 2, (g0 + i) * 256, 0, 16);
            }
    };
    if (handed_off) {
        // several rows: first a word of each, until one of them is there, so that whole rows are not asked for over and over
        if (T > 4) {
            const int at = a == 0 && rb * 16 + b < T ? ((rb * 16 + b) * w.K + g0 * 128 + (int)(blockIdx.x % (2 * GPW)) * 64) * 2 : -1;       // (a line of the wave's, by workgroup)
            chain_until([&] { return __ballot(at >= 0 && __builtin_amdgcn_raw_buffer_load_b32(r_x, at, 0, 16) != NOT_YET) != 0ull; }, p.timeout);
        }
        chain_until([&] {
            request();
            chain_landed<0>();
            uint32_t most = 0;
#pragma unroll
            for (int i = 0; i < GPW * 4; i++) most = max(most, most4(*reinterpret_cast<const u32x4*>(mine + i * 1024 + lane * 16)));
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(most) :: "memory");
            return __ballot(most == NOT_YET) == 0ull;
        }, p.timeout);
    } else {
        request();
    }
    CH_TL(1);
    if constexpr (LATE > 0) {
        if (two_late) ask(std::integral_constant<int, GPW - 2 * LATE>{}, std::integral_constant<int, GPW - LATE>{});
        ask(std::integral_constant<int, GPW - LATE>{}, std::integral_constant<int, GPW>{});
        __builtin_amdgcn_sched_barrier(0);
    }
    float4v acc[NST][1][NTL];
#pragma unroll
    for (int s = 0; s < NST; s++)
#pragma unroll
        for (int nt = 0; nt < NTL; nt++) acc[s][0][nt] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < GPW; i++) {
        if constexpr (GLU) {                                          // (handed-off rows are there)
        } else if (i == GPW - 1) chain_landed<0>();
        else if (i == GPW - 2) chain_landed<4>();
        else if (i == GPW - 3) chain_landed<8>();
        else chain_landed<12>();
        half8 af[1][4];
#pragma unroll
        for (int s = 0; s < 4; s++) af[0][s] = *reinterpret_cast<const half8*>(mine + i * 4096 + b * 256 + ((4 * s + a) ^ b) * 16);
#pragma unroll
        for (int s = 0; s < NST; s++) {
            if constexpr (F16W) {
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int nt = 0; nt < NTL; nt++) acc[s][0][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][k], wx[i][s][nt][k], acc[s][0][nt], 0, 0, 0);
                continue;
            }
            const unsigned long long sb = ((unsigned long long)scv[F16W ? 0 : i][s].y << 32) | scv[F16W ? 0 : i][s].x;
            if (i < PRE) {
                float4v t[NTL];
#pragma unroll
                for (int nt = 0; nt < NTL; nt++) t[nt] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int nt = 0; nt < NTL; nt++) t[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][k], wx[i < PRE ? i : 0][s][nt][k], t[nt], 0, 0, 0);
#pragma unroll
                for (int nt = 0; nt < NTL; nt++) {
                    const float s_f = (float)__builtin_bit_cast(_Float16, (uint16_t)(sb >> 16 * (nt0 + nt)));
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[s][0][nt][r] = __builtin_fmaf(s_f, t[nt][r], acc[s][0][nt][r]);
                }
            } else
                w4_consume_group<1, NTL, false, false>(wq[F16W ? 0 : i][s], sb, 0ull, nt0, af, acc[s]);
        }
    }
    // cross-wave reduction through LDS: red[wave][v][lane], v = (supertile·4 + tile)·4 + r
#pragma unroll
    for (int s = 0; s < NST; s++)
#pragma unroll
        for (int nt = 0; nt < NTL; nt++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[wave * (REGION / 4) + ((s * NTL + nt) * 4 + r) * 64 + lane] = acc[s][0][nt][r];
    __syncthreads();
    if constexpr (GLU) {
        // thread → (row, 4 columns of gate and of up): one 8-byte write-through store
        constexpr int COLS = NST * NTL * 8;
        if (threadIdx.x < 16 * (COLS / 4)) {
            const int row = threadIdx.x / (COLS / 4), c4 = (threadIdx.x % (COLS / 4)) * 4;
            const int v = (c4 >> 4) * 4 + (row & 3), ln = (row >> 2) * 16 + (c4 & 15);
            float4v sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int ww = 0; ww < CH_W; ww++)
#pragma unroll
                for (int h = 0; h < 2; h++) sum[h] += *reinterpret_cast<const float4v*>(&red[ww * (REGION / 4) + (v + V / 2 * h) * 64 + ln]);
            union { _Float16 h[4]; uint32_t u[2]; } o;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float g = sum[0][j], u = sum[1][j];
                if constexpr (F16W) {                                 // as gemm_glu
                    o.h[j] = (_Float16)((p.gelu ? gelu_tanh_f32<_Float16>(g) : g * ActMath<_Float16>::sigmoid(g)) * u);
                } else {
                    g = (float)(_Float16)g;
                    u = (float)(_Float16)u;
                    o.h[j] = p.gelu ? gated_act<true>(g, u) : gated_act<false>(g, u);
                }
            }
            const int r_out = rb * 16 + row, n = w.N / 2;
            if (r_out < T)
                __builtin_amdgcn_raw_buffer_store_b64((u32x2){written2(o.u[0]), written2(o.u[1])}, chain_rsrc(out, (long)T * n * 2), (r_out * n + cb * COLS + c4) * 2, 0, 16);
        }
        CH_TL(2); CH_TL(3);
        return;
    }
    // thread → (row, 8 consecutive columns): one 16-byte write-through store
    if (threadIdx.x < 16 * CPR) {
        const int row = threadIdx.x / CPR, c8 = (threadIdx.x % CPR) * 8;
        const int aa = row >> 2, r = row & 3;
        // the row's 8 columns c8 … c8+7 lie in one tile (8 | 16): lanes aa·16 + bb … + 7 of accumulator slot v — 32 contiguous bytes
        const int tile = c8 >> 4, bb = c8 & 15;                               // tile = supertile·4 + nt
        const int v = tile * 4 + r, ln = aa * 16 + bb;
        float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ww = 0; ww < CH_W; ww++) {
            const float4v lo = *reinterpret_cast<const float4v*>(&red[ww * (REGION / 4) + v * 64 + ln]);
            const float4v hi = *reinterpret_cast<const float4v*>(&red[ww * (REGION / 4) + v * 64 + ln + 4]);
#pragma unroll
            for (int j = 0; j < 4; j++) { sum[j] += lo[j]; sum[4 + j] += hi[j]; }
        }
        const int r_out = rb * 16 + row;
        if constexpr (F32OUT) {
            if (r_out < T) {
                const __amdgpu_buffer_rsrc_t r_o = chain_rsrc(out32, (long)T * w.N * 4);
                const int off = (r_out * w.N + cb * 16 * NTL * NST + c8) * 4;
                store16_sc1(r_o, off, (float4v){sum[0], sum[1], sum[2], sum[3]});
                store16_sc1(r_o, off + 16, (float4v){sum[4], sum[5], sum[6], sum[7]});
            }
        } else {
            half8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = (_Float16)sum[j];
            if (r_out < T) {
                const __amdgpu_buffer_rsrc_t r_o = chain_rsrc(out, (long)T * w.N * 2);
                store16_sc1(r_o, (r_out * w.N + cb * 16 * NTL * NST + c8) * 2, o);
            }
        }
    }
    CH_TL(2); CH_TL(3);
}

// ── attention role: paged_attn_kernel<128, true, 8> (decode, one new token per sequence) ────────────────────────────────
template <bool KVS>
__device__ __forceinline__ void chain_role_attn(const ChainArgs& p, int wg, unsigned char* smem) {
    constexpr int HD = 128, NW = CH_W, DT = HD / 16, KS = HD / 32, OSTRIDE = HD + 4;
    float* lds_o = reinterpret_cast<float*>(smem);                    // [NW·16][OSTRIDE]
    float* lds_m = lds_o + NW * 16 * OSTRIDE;
    float* lds_l = lds_m + NW * 16;
    __half* lds_q = reinterpret_cast<__half*>(lds_l + NW * 16);       // [16][HD]
    __half* lds_kv = lds_q + 16 * HD;                                 // [2][HD]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int a = lane >> 4, b = lane & 15;
    // (the ranges of a (sequence, kv head) are neighbours; one range: no divisions on the way to the first K/V request — the role's
    // later workgroups enter when the q|k|v blocks leave their CUs, with the projection already done)
    const int NS = KVS ? p.attn_splits : 1;                          // (a kernel of its own: the one-range form stays as lean as it was)
    const int unit = NS == 1 ? wg : (int)((unsigned)wg / (unsigned)NS), split = NS == 1 ? 0 : wg - unit * NS;
    const int seq = unit % p.T, kvh = unit / p.T;
    CH_TL(0);
    const int G = p.nq / p.nkv;
    const int pos0 = (int)p.kv_lens[seq] - 1;
    const bool row_ok = b < G;
    const int row_pos = pos0;
    const int win_lo = p.sliding_window > 0 ? max(0, row_pos + 1 - p.sliding_window) : 0;
    const int kv_end = pos0 + 1;
    const int kv_begin = p.sliding_window > 0 ? max(0, pos0 + 1 - p.sliding_window) : 0;
    const int all_lo = (kv_begin / KV_BLOCK) / 2;
    const int all_hi = (cdiv_dev(kv_end, KV_BLOCK) + 1) / 2;         // exclusive: block pairs of the whole context
    // this split's share of the pairs (the last split owns the pair with the new token: it patches and writes its K / V)
    const unsigned np_all = (unsigned)max(0, all_hi - all_lo);       // (≤ 2^16 pairs × ≤ 16 ranges: 32-bit)
    const int my_lo = NS == 1 ? all_lo : all_lo + (int)(np_all * (unsigned)split / (unsigned)NS);
    const int my_hi = NS == 1 ? all_hi : all_lo + (int)(np_all * (unsigned)(split + 1) / (unsigned)NS);
    const int first = my_lo + wave;
    const int nblocks = cdiv_dev(kv_end, KV_BLOCK);
    const int32_t* bt = p.block_tables + (long)seq * p.max_blocks;
    const long tile_elems = kv_tile_elems(HD);
    int bt_lo = 2 * my_lo;
    int btv = bt[min(bt_lo + lane, p.max_blocks - 1)];
    struct Frags { half8 k0[KS], k1[KS], v0[KS], v1[KS]; };
    auto issue = [&](int pr, Frags& f) {
        const int blk0 = 2 * pr, blk1 = 2 * pr + 1;
        const bool has1 = blk1 < nblocks;
        if (blk1 - bt_lo >= 64) {
            bt_lo = blk0;
            btv = bt[min(bt_lo + lane, p.max_blocks - 1)];
        }
        const long phys0 = __builtin_amdgcn_readlane(btv, blk0 - bt_lo);
        const long phys1 = has1 ? __builtin_amdgcn_readlane(btv, blk1 - bt_lo) : phys0;
        const __half* k0 = p.k_pool + (phys0 * p.nkv + kvh) * tile_elems + lane * 8;
        const __half* k1 = p.k_pool + (phys1 * p.nkv + kvh) * tile_elems + lane * 8;
        const __half* v0 = p.v_pool + (phys0 * p.nkv + kvh) * tile_elems + lane * 8;
        const __half* v1 = p.v_pool + (phys1 * p.nkv + kvh) * tile_elems + lane * 8;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            f.k0[s] = __builtin_nontemporal_load(reinterpret_cast<const half8*>(k0 + s * 512));
            f.k1[s] = __builtin_nontemporal_load(reinterpret_cast<const half8*>(k1 + s * 512));
        }
#pragma unroll
        for (int s = 0; s < KS; s++) {
            f.v0[s] = __builtin_nontemporal_load(reinterpret_cast<const half8*>(v0 + s * 512));
            f.v1[s] = __builtin_nontemporal_load(reinterpret_cast<const half8*>(v1 + s * 512));
        }
    };
    Frags cur, nxt;
    if (first < my_hi) issue(first, cur);
    if (first + NW < my_hi) issue(first + NW, nxt);
    const int last_blk = pos0 / KV_BLOCK, slot_new = pos0 % KV_BLOCK;
    // norm weights, the RoPE row of this position and the new token's block do not depend on the projection either
    constexpr int HALF = HD / 2;
    const int r16 = threadIdx.x >> 4, q16 = threadIdx.x & 15;
    const int rc = r16 < G + 2 ? r16 : G + 1, rope_mode = rc <= G ? p.qk_mode : 0;
    const RopeCoef<HD> coef = rope_coef16<HD>(rc < G ? p.q_norm_w : p.k_norm_w, p.cos_t + (long)pos0 * HALF, p.sin_t + (long)pos0 * HALF,
                                              rope_mode, p.qk_mode == 1, p.qk_mode != 0, q16);
    const int phys_new = bt[last_blk];
    __builtin_amdgcn_sched_barrier(0);
    half8 qf[KS];
    {
        const int q_dim = p.nq * HD, kv_dim = p.nkv * HD;
        const __half* qrow = p.qkv_out + (long)seq * (q_dim + 2 * kv_dim);
        const __half* src = rc < G ? qrow + (kvh * G + rc) * HD
                                   : rc == G ? qrow + q_dim + kvh * HD : qrow + q_dim + kv_dim + kvh * HD;
        RopeSource<HD> source;
        chain_until([&] {
            source = rope_source16_sc1<HD, true>(src, rope_mode, q16);
            const uint2 c0 = __builtin_bit_cast(uint2, source.c0), c1 = __builtin_bit_cast(uint2, source.c1);
            return __ballot(max(max(c0.x, c0.y), max(c1.x, c1.y)) == NOT_YET) == 0ull;
        }, p.timeout);
        CH_TL(1);
        const RopeRow<HD> rr = rope_row16<HD>(source, coef, rope_mode, p.eps, q16);
        using hv = typename RopeRow<HD>::hv;
        hv z0, z1;
#pragma unroll
        for (int k = 0; k < HD / 32; k++) { z0[k] = (_Float16)0.f; z1[k] = (_Float16)0.f; }
        _Float16* lq = reinterpret_cast<_Float16*>(lds_q) + r16 * HD;
        if (r16 < 16) {
            *reinterpret_cast<hv*>(lq + rr.off0) = r16 < G ? rr.out0 : z0;
            *reinterpret_cast<hv*>(lq + rr.off1) = r16 < G ? rr.out1 : z1;
        }
        if (r16 == G || r16 == G + 1) {
            _Float16* lk = reinterpret_cast<_Float16*>(lds_kv) + (r16 - G) * HD;
            *reinterpret_cast<hv*>(lk + rr.off0) = rr.out0;
            *reinterpret_cast<hv*>(lk + rr.off1) = rr.out1;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KS; s++) qf[s] = *reinterpret_cast<const half8*>(lds_q + b * HD + 32 * s + 8 * a);
    }
    // the new token's K (wave 0) and V (wave 1) go to the cache, read by later launches only: last of all
    auto keep_new = [&]() {
        if (wave < 2 && split == NS - 1) {
            const long toff = ((long)phys_new * p.nkv + kvh) * kv_tile_elems(HD);
            for (int d = lane; d < HD; d += 64) {
                if (wave == 0) p.k_pool[toff + k_tile_off(slot_new, d)] = lds_kv[d];
                else p.v_pool[toff + v_tile_off(slot_new, d)] = lds_kv[HD + d];
            }
        }
    };
    float m_run = -INFINITY, l_run = 0.f;
    float4v o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o_acc[dt] = (float4v){0.f, 0.f, 0.f, 0.f};
    // Two pairs of blocks a wave are on their way before the wait (512 keys a workgroup; one pair, the second asked for behind the wait, left
    // its round trip to memory there), a third takes the place of the first as soon as that is used.  The new token's key and value replace what
    // the fragments hold of its slot by masks (a select for each half and block of the pair: 0.5 µs of the slowest wave's time).  256 keys: 3.9 →
    // 3.3 µs from the rows to the role's result; a step of 8 expert layers, 1 row of 400 keys 386 → 380 µs, 32 of 256 726 → 718; of 32 layers of
    // 4096 columns, 12 rows of 120 keys 1607 → 1596, 4 of 450 1579 → 1527, 1 of 8100 (16 ranges) 1640 → 1586.
    const uint32_t keep_at = (slot_new & 1) ? 0x0000FFFFu : 0xFFFF0000u;
    const uint32_t keep0 = a == slot_new >> 2 && !(slot_new & 2) ? keep_at : ~0u, keep1 = a == slot_new >> 2 && (slot_new & 2) ? keep_at : ~0u;
    auto put_new = [&](half8 (&kf)[KS], half8 (&vf)[KS]) {
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const half8 nk = *reinterpret_cast<const half8*>(lds_kv + 32 * s + 8 * a);
            if (b == slot_new) kf[s] = nk;
        }
#pragma unroll
        for (int ld = 0; ld < KS; ld++) {
            u32x4 w = __builtin_bit_cast(u32x4, vf[ld]);
#pragma unroll
            for (int sub = 0; sub < 2; sub++) {
                const uint32_t one = *reinterpret_cast<const uint16_t*>(lds_kv + HD + 32 * ld + 16 * sub + b), nv = one | one << 16;
                w[2 * sub] = (w[2 * sub] & keep0) | (nv & ~keep0);
                w[2 * sub + 1] = (w[2 * sub + 1] & keep1) | (nv & ~keep1);
            }
            vf[ld] = __builtin_bit_cast(half8, w);
        }
    };
    auto attend = [&](int pr, Frags& f) {
        const int blk0 = 2 * pr, blk1 = 2 * pr + 1;
        const bool has1 = blk1 < nblocks;
        half8 (&kf0)[KS] = f.k0, (&kf1)[KS] = f.k1, (&vf0)[KS] = f.v0, (&vf1)[KS] = f.v1;
        // the new token's key and value take the place of what the fragments hold of its slot
        if (blk0 == last_blk) put_new(f.k0, f.v0);
        if (blk1 == last_blk) put_new(f.k1, f.v1);
        float4v s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; s++) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf0[s], qf[s], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf1[s], qf[s], s1, 0, 0, 0);
        }
        float sc[8];
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int kp0 = blk0 * KV_BLOCK + 4 * a + r, kp1 = blk1 * KV_BLOCK + 4 * a + r;
            const bool ok0 = row_ok && kp0 <= row_pos && kp0 >= win_lo;
            const bool ok1 = row_ok && has1 && kp1 <= row_pos && kp1 >= win_lo;
            sc[r] = ok0 ? s0[r] * p.scale : -INFINITY;
            sc[4 + r] = ok1 ? s1[r] * p.scale : -INFINITY;
            mx = fmaxf(mx, fmaxf(sc[r], sc[4 + r]));
        }
        mx = rows_reduce_max(mx);
        const float m_new = fmaxf(m_run, mx);
        const float m_safe = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __expf(m_run - m_safe);
        float psum = 0.f;
        half8 pf;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float pv = __expf(sc[j] - m_safe);
            psum += pv;
            pf[j] = (_Float16)pv;
        }
        psum = rows_reduce_sum(psum);
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const int ld = dt >> 1, sub = (dt & 1) * 2;
            const u32x4 w0 = __builtin_bit_cast(u32x4, vf0[ld]), w1 = __builtin_bit_cast(u32x4, vf1[ld]);
            const half8 vfrag = __builtin_bit_cast(half8, (u32x4){w0[sub], w0[sub + 1], w1[sub], w1[sub + 1]});
#pragma unroll
            for (int r = 0; r < 4; r++) o_acc[dt][r] *= alpha;
            o_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vfrag, pf, o_acc[dt], 0, 0, 0);
        }
        if (pr + 2 * NW < my_hi) issue(pr + 2 * NW, f);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int pr = first; pr < my_hi; pr += 2 * NW) {
        attend(pr, cur);
        if (pr + NW < my_hi) attend(pr + NW, nxt);
    }
    // merge the 8 waves' partial states through LDS (wave order)
    if (a == 0) {
        lds_m[wave * 16 + b] = m_run;
        lds_l[wave * 16 + b] = l_run;
    }
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
        if (row_ok) *reinterpret_cast<float4v*>(&lds_o[(wave * 16 + b) * OSTRIDE + dt * 16 + 4 * a]) = o_acc[dt];       // (rows past the group are not read)
    __syncthreads();
    constexpr int TPR = NW * 4;                                       // threads per row: 32 → 4 dims each
    const int row = threadIdx.x / TPR, dl = threadIdx.x % TPR;
    float mw[NW], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; w++) { mw[w] = lds_m[w * 16 + row]; M = fmaxf(M, mw[w]); }
    const float Ms = M == -INFINITY ? 0.f : M;
    float fw[NW], L = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) { fw[w] = __expf(mw[w] - Ms); L += lds_l[w * 16 + row] * fw[w]; }
    constexpr int DPT = HD / TPR;
    float ov[DPT];
#pragma unroll
    for (int i = 0; i < DPT; i++) {
        const int d = dl * DPT + i;
        float acc = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) acc += lds_o[(w * 16 + row) * OSTRIDE + d] * fw[w];
        ov[i] = acc;
    }
    float Lm = L, Mm = M;
    if (NS > 1) {
        // several KV ranges per (sequence, kv head): every split leaves its state (m, l, unnormalised o) write-through and takes a
        // ticket; the LAST to arrive reads all of them back (sc1) and merges them in split order — whoever it is, the same bits
        static_assert(DPT == 4, "one 16-byte piece per thread");
        constexpr int PST = HD + 4;
        float* mine = p.attn_partial + ((long)unit * NS + split) * 16 * PST + row * PST;
        const __amdgpu_buffer_rsrc_t pr_ = chain_rsrc(p.attn_partial, (long)p.T * p.nkv * NS * 16 * PST * 4);
        const int my_off = (int)((mine - p.attn_partial) * 4);
        if (row < G) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, (float4v){ov[0], ov[1], ov[2], ov[3]}), pr_, my_off + dl * 16, 0, 16);
            if (dl == 0) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, (float4v){M, L, 0.f, 0.f}), pr_, my_off + HD * 4, 0, 16);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int* s_tk = reinterpret_cast<int*>(lds_m);                     // (the merge above is done with lds_m)
        if (threadIdx.x == 0) *s_tk = (int)__hip_atomic_fetch_add(p.attn_tickets + unit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*s_tk != NS - 1) { keep_new(); CH_TL(2); CH_TL(3); return; }           // not the last: the merge (and the signal) is someone else's
        if (threadIdx.x == 0) __hip_atomic_store(p.attn_tickets + unit, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (row < G) {
            const int base = (int)(((long)unit * NS * 16 * PST + row * PST) * 4);
            // (no branch around a load: all of them are under way together)
            auto merge = [&](auto most) {
                constexpr int N = decltype(most)::value;
                float4v ml[N], os[N];
#pragma unroll
                for (int sp = 0; sp < N; sp++) {
                    const int at = base + min(sp, NS - 1) * 16 * PST * 4;
                    ml[sp] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(pr_, at + HD * 4, 0, 16));
                    os[sp] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(pr_, at + dl * 16, 0, 16));
                }
                Mm = -INFINITY;
#pragma unroll
                for (int sp = 0; sp < N; sp++) Mm = fmaxf(Mm, ml[sp][0]);          // (repeats of the last range change no maximum)
                const float Msafe = Mm == -INFINITY ? 0.f : Mm;
                Lm = 0.f;
#pragma unroll
                for (int i = 0; i < DPT; i++) ov[i] = 0.f;
#pragma unroll
                for (int sp = 0; sp < N; sp++) {
                    const float f = sp < NS ? __expf(ml[sp][0] - Msafe) : 0.f;
                    if (sp < NS) {
                        Lm += ml[sp][1] * f;
#pragma unroll
                        for (int i = 0; i < DPT; i++) ov[i] += os[sp][i] * f;
                    }
                }
            };
            if (NS <= 8) merge(std::integral_constant<int, 8>{});
            else merge(std::integral_constant<int, CH_MAX_SPLITS>{});
        }
    }
    if (row < G) {
        const float inv = Lm > 0.f ? 1.0f / Lm : 0.f;
        union { _Float16 h[4]; unsigned long long u; } o;
#pragma unroll
        for (int i = 0; i < DPT; i++) o.h[i] = (_Float16)(ov[i] * inv);
        __half* dst = p.attn_out + ((long)seq * p.nq + kvh * G + row) * HD + dl * DPT;
        o.u = (unsigned long long)written2((uint32_t)(o.u >> 32)) << 32 | written2((uint32_t)o.u);
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(dst), o.u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);     // 8-byte sc1 store
    }
    CH_TL(2);
    keep_new();
    CH_TL(3);
}

// ── role B: residual += o; post-attention norm; router logits of this part's experts; candidates; in-launch merge ─────────
// (add_rmsnorm_route_part_kernel<false> with arrive: grid (token, part) → wg = token·Q + part)
template <bool MLP>
__device__ __forceinline__ void chain_role_b(const ChainArgs& p, int wg, unsigned char* smem) {
    const int H = p.H, Q = p.Q, num_experts = p.E, top_k = p.r_top_k;
    const long row = wg / Q;
    const int q = wg % Q;
    CH_TL(0);
    __half* xs = reinterpret_cast<__half*>(smem);
    float* part = reinterpret_cast<float*>(smem + (size_t)H * 2);
    const int nvec = H >> 3;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int CH = 2;
    // requested before the wait: the norm weights and this wave's router weights (its whole share: 16 k-steps × 1 KiB)
    half8 wv_pre[CH];
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = threadIdx.x + c * 512;
        wv_pre[c] = *reinterpret_cast<const half8*>(p.post_ln + (i < nvec ? i : 0) * 8);
    }
    constexpr int U = 16;
    const int tiles = (num_experts + 15) >> 4;
    const int tiles_q = num_experts > 0 ? tiles / Q : 0;              // (dense model: no router, Q = 1)
    const int ksplit = (tiles_q >= 8 || tiles_q == 0) ? 1 : 8 / tiles_q;
    const int ksteps = H >> 5;
    half8 bw_pre[U];
    bool pre = false;
    if (wave < tiles_q * ksplit) {
        const int tl = wave / ksplit, ks = wave % ksplit;
        const int s0 = ksteps * ks / ksplit, s1 = ksteps * (ks + 1) / ksplit;
        if (s0 + U <= s1) {
            const __half* wrow = p.router_w + ((long)(q * tiles_q + tl) * ksteps * 64 + lane) * 8;
#pragma unroll
            for (int kk = 0; kk < U; kk++) bw_pre[kk] = *reinterpret_cast<const half8*>(wrow + (long)(s0 + kk) * 512);
            pre = true;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    float* red = part + tiles_q * 16 * (ksplit + 1);                  // [8] behind the logits
    unsigned long long* cand_s = reinterpret_cast<unsigned long long*>(red + 8);     // [8]
    const __amdgpu_buffer_rsrc_t r_x = chain_rsrc(p.o_part, (long)CH_O_KS * p.T * H * 4), r_res = chain_rsrc(p.res_a, (long)p.T * H * 2);
    half8 v[CH];
    float ss = 0.f;
    // o_proj's row: its K parts (fp32) added in part order, rounded to the fp16 the projection's output is.  First one word of it, until it is there.
    u32x4 parts[CH][CH_O_KS][2], res[CH];
    if (wave * 64 < nvec) {
        const int at = (int)((row * H + wave * 512) * 4);
        chain_until([&] { return (uint32_t)__builtin_amdgcn_readfirstlane(__builtin_amdgcn_raw_buffer_load_b32(r_x, at, 0, 16)) != NOT_YET; }, p.timeout);
    }
    chain_until([&] {
        uint32_t most = 0;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int i = threadIdx.x + c * 512;
            if (i < nvec) {
#pragma unroll
                for (int ks = 0; ks < CH_O_KS; ks++) {
                    const int o32 = (int)((((long)ks * p.T + row) * H + i * 8) * 4);
                    parts[c][ks][0] = __builtin_amdgcn_raw_buffer_load_b128(r_x, o32, 0, 16);
                    parts[c][ks][1] = __builtin_amdgcn_raw_buffer_load_b128(r_x, o32 + 16, 0, 16);
                }
                res[c] = __builtin_amdgcn_raw_buffer_load_b128(r_res, (int)((row * H + i * 8) * 2), 0, 16);
            }
        }
#pragma unroll
        for (int c = 0; c < CH; c++)
            if ((int)threadIdx.x + c * 512 < nvec) {
#pragma unroll
                for (int ks = 0; ks < CH_O_KS; ks++) most = max(most, max(most4(parts[c][ks][0]), most4(parts[c][ks][1])));
                if (p.has_a) most = max(most, most4(res[c]));         // (else it is an earlier launch's)
            }
        return __ballot(most == NOT_YET) == 0ull;
    }, p.timeout);
    CH_TL(1);
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = threadIdx.x + c * 512;
        if (i < nvec) {
            float xs32[8];
#pragma unroll
            for (int ks = 0; ks < CH_O_KS; ks++) {
                const float4v lo = __builtin_bit_cast(float4v, parts[c][ks][0]), hi = __builtin_bit_cast(float4v, parts[c][ks][1]);
#pragma unroll
                for (int j = 0; j < 4; j++) { xs32[j] = ks ? xs32[j] + lo[j] : lo[j]; xs32[4 + j] = ks ? xs32[4 + j] + hi[j] : hi[j]; }
            }
            half8 xv;
#pragma unroll
            for (int j = 0; j < 8; j++) xv[j] = (_Float16)xs32[j];
            half8 rv = __builtin_bit_cast(half8, res[c]);
#pragma unroll
            for (int j = 0; j < 8; j++) rv[j] = (_Float16)((float)rv[j] + (float)xv[j]);
            v[c] = rv;
#pragma unroll
            for (int j = 0; j < 8; j++) ss += (float)rv[j] * (float)rv[j];
        }
    }
    ss = wave_reduce_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    const float total = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
    const float inv = 1.0f / sqrtf(total / (float)H + p.eps);
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = threadIdx.x + c * 512;
        if (i < nvec) {
            const half8 wv = wv_pre[c];
            half8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = (_Float16)((float)v[c][j] * inv * (float)wv[j]);
            if constexpr (MLP) store16_sc1(chain_rsrc(p.norm2, (long)p.T * H * 2), (int)((row * H + i * 8) * 2), o);
            *reinterpret_cast<half8*>(xs + i * 8) = o;
            if (MLP) {
                *reinterpret_cast<half8*>(p.res_b_out + row * H + i * 8) = v[c];
            } else if (q == 0) {
                *reinterpret_cast<half8*>(p.norm2 + row * H + i * 8) = o;
                *reinterpret_cast<half8*>(p.res_b_out + row * H + i * 8) = v[c];
            }
        }
    }
    if (MLP || num_experts <= 0) { CH_TL(2); CH_TL(3); return; }           // dense model: add + norm only (norm2 / res_b_out written above)
    __syncthreads();
    const int a = lane >> 4, b = lane & 15;
    // (all sixteen rows of a product are the token's: a row of zeros would need a branch at every read)
    for (int u = wave; u < tiles_q * ksplit; u += 8) {
        const int tl = u / ksplit, ks = u % ksplit;
        const int tile = q * tiles_q + tl;
        const int s0 = ksteps * ks / ksplit, s1 = ksteps * (ks + 1) / ksplit;
        const __half* wrow = p.router_w + ((long)tile * ksteps * 64 + lane) * 8;
        float4v acc = {0.f, 0.f, 0.f, 0.f};
        int s = s0;
        if (u == wave && pre) {
#pragma unroll
            for (int kk = 0; kk < U; kk++) {
                const half8 av = *reinterpret_cast<const half8*>(xs + (s + kk) * 32 + 8 * a);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bw_pre[kk], acc, 0, 0, 0);
            }
            s += U;
        }
        for (; s + U <= s1; s += U) {
            half8 bw[U];
#pragma unroll
            for (int k = 0; k < U; k++) bw[k] = *reinterpret_cast<const half8*>(wrow + (long)(s + k) * 512);
#pragma unroll
            for (int k = 0; k < U; k++) {
                const half8 av = *reinterpret_cast<const half8*>(xs + (s + k) * 32 + 8 * a);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bw[k], acc, 0, 0, 0);
            }
        }
        for (; s < s1; s++) {
            const half8 bwv = *reinterpret_cast<const half8*>(wrow + (long)s * 512);
            const half8 av = *reinterpret_cast<const half8*>(xs + s * 32 + 8 * a);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bwv, acc, 0, 0, 0);
        }
        if (a == 0) part[ks * tiles_q * 16 + tl * 16 + b] = acc[0];
    }
    __syncthreads();
    const int EQ = tiles_q * 16;
    float* lgs = part + ksplit * EQ;
    const int t = threadIdx.x;
    const int e_glob = q * EQ + t;
    float l = -INFINITY;
    if (t < EQ && e_glob < num_experts) {
        l = 0.f;
        float lp[8];
#pragma unroll
        for (int ks = 0; ks < 8; ks++) lp[ks] = part[(ks < ksplit ? ks : 0) * EQ + t];
#pragma unroll
        for (int ks = 0; ks < 8; ks++) if (ks < ksplit) l += lp[ks];
    }
    const int keep = top_k < EQ ? top_k : EQ;
    const float lc = route_logit(l);
    float mx = wave_reduce_max(l), sm;
    int rank = 0;
    if (EQ <= 64) {
        // one wave has them all
        if (wave != 0) return;
        sm = wave_reduce_sum((t < EQ && e_glob < num_experts) ? expf(l - mx) : 0.f);
        rank = route_rank(route_key(lc, t), EQ);
        if (t < EQ && rank < keep) cand_s[rank] = ((unsigned long long)(unsigned)e_glob << 32) | __float_as_uint(lc);
        if (t >= keep && t < 8) cand_s[t] = (0x7fffffffull << 32) | __float_as_uint(-INFINITY);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
    } else {
        if (t < EQ) lgs[t] = lc;
        if (lane == 0) red[wave] = mx;
        __syncthreads();
        mx = fmaxf(red[0], red[1]);
        __syncthreads();
        const float ex = (t < EQ && e_glob < num_experts) ? expf(l - mx) : 0.f;
        sm = wave_reduce_sum(ex);
        if (lane == 0) red[wave] = sm;
        if (t < EQ) {
            for (int j = 0; j < EQ; j++) {
                const float lj = lgs[j];
                rank += (lj > lc || (lj == lc && j < t)) ? 1 : 0;
            }
            if (rank < keep) cand_s[rank] = ((unsigned long long)(unsigned)e_glob << 32) | __float_as_uint(lc);
        }
        if (t >= keep && t < 8) cand_s[t] = (0x7fffffffull << 32) | __float_as_uint(-INFINITY);
        __syncthreads();
        sm = red[0] + red[1];
    }
    CH_TL(2);
    if (wave != 0) return;
    if (p.defer_merge) {
        // the consumer is the NEXT launch (the grouped gate_up GEMM merges the Q lists of every token in its prologue, under its
        // first weight loads): plain stores, no meeting of the parts here — the ≈ 3.7 µs merge leaves the layer's critical path
        unsigned long long* cand_g = reinterpret_cast<unsigned long long*>(p.cand) + (row * Q + q) * 8;
        if (lane < 8) cand_g[lane] = cand_s[lane];
        if (lane == 8) reinterpret_cast<unsigned long long*>(p.stats)[row * Q + q] =
            ((unsigned long long)__float_as_uint(sm) << 32) | __float_as_uint(mx);
        CH_TL(3);
        return;
    }
    // The Q parts of a token meet without a counter: every part but the first publishes its 8 candidates and its two softmax
    // statistics as TAGGED 8-byte granules (one write-through store each — the data is the flag, Guideline 16 R2), and part 0
    // sweeps the (Q − 1)·10 granules of its token until every tag is there, merges, and clears them for the launch after the
    // next (the granules live in the double-buffered counter block: zero on entry).  One store → load latency instead of
    // store → drain → returning ticket → loads: 3.4–3.8 µs → ≈ 1.5 µs on the layer's critical path.
    //   candidate granule: [tag 1 : 16][expert id : 16][logit bits : 32]      statistic granule: [tag 1 : 32][value bits : 32]
    unsigned long long* gran = reinterpret_cast<unsigned long long*>(p.cnt) + (row * Q) * CH_GRAN;
    if (q != 0) {
        unsigned long long g = 0;
        if (lane < 8) g = (1ull << 48) | ((cand_s[lane] >> 32 & 0xffffull) << 32) | (cand_s[lane] & 0xffffffffull);
        else if (lane == 8) g = (1ull << 32) | __float_as_uint(mx);
        else if (lane == 9) g = (1ull << 32) | __float_as_uint(sm);
        if (lane < CH_GRAN) __hip_atomic_store(gran + q * CH_GRAN + lane, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    unsigned long long* gr = cand_s + 8;                               // LDS [Q][CH_GRAN] behind this part's own list
    {
        const int n = (Q - 1) * CH_GRAN;
        unsigned long long* src = gran + CH_GRAN + lane;
        const bool is_stat = (lane % CH_GRAN) >= 8;
        unsigned long long g = 0;
        const unsigned long long t0 = wall_clock64();
        unsigned spins = 0;
        for (;;) {
            if (lane < n) g = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool have = lane >= n || (is_stat ? (g >> 32) == 1ull : (g >> 48) == 1ull);
            if (__ballot(!have) == 0ull) break;
            __builtin_amdgcn_s_sleep(1);
            if ((++spins & 1023u) == 0u && wall_clock64() - t0 > 2000000ull) {
                if (lane == 0) __hip_atomic_fetch_add(p.timeout, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                break;
            }
        }
        if (lane < n) {
            gr[CH_GRAN + lane] = g;
            __hip_atomic_store(src, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // (also cleared with the half by a later launch)
        }
        if (lane < 8) gr[lane] = (1ull << 48) | ((cand_s[lane] >> 32 & 0xffffull) << 32) | (cand_s[lane] & 0xffffffffull);
        else if (lane == 8) gr[8] = (1ull << 32) | __float_as_uint(mx);
        else if (lane == 9) gr[9] = (1ull << 32) | __float_as_uint(sm);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");       // one wave: its own LDS writes, in order
        __builtin_amdgcn_wave_barrier();
    }
    const int ncand = Q * 8;
    unsigned long long c = (0x7fffffffull << 32) | __float_as_uint(-INFINITY);
    if (lane < ncand) {
        const unsigned long long g = gr[(lane >> 3) * CH_GRAN + (lane & 7)];
        const unsigned id16 = (unsigned)(g >> 32) & 0xffffu;
        c = ((unsigned long long)(id16 == 0xffffu ? 0x7fffffffu : id16) << 32) | (g & 0xffffffffull);
    }
    float pmx = -INFINITY, psum = 0.f;
    if (lane < Q) {
        pmx = __uint_as_float((unsigned)gr[lane * CH_GRAN + 8]);
        psum = __uint_as_float((unsigned)gr[lane * CH_GRAN + 9]);
    }
    float ww = 0.f;
    const int place = route_merge_token(c, ncand, pmx, psum, Q, top_k, p.norm_topk, true, &ww);
    if (place < top_k) {
        p.ids[row * top_k + place] = (int)(c >> 32);
        p.weights[row * top_k + place] = ww;
    }
    CH_TL(3);
}

// KVS / WIDE are kernels of their own, not branches: the one-range, 64-column kernel keeps the instruction layout it was tuned
// with (with either compiled in as a runtime branch it lost ≈ 1 % at every batch size — roles entering late have their first
// instructions on the critical path)
// GPW_D: quant groups of a wave in the MLP's second projection (dense models); 0: the launch ends with role B
template <int GPW_QKV, int GPW_O, bool F16W, bool KVS = false, bool WIDE = false, int GPW_D = 0>
__global__ __launch_bounds__(512, 2) void decode_chain_kernel(ChainArgs p) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[CH_SMEM > CH_W * GPW_QKV * 4096 ? CH_SMEM : CH_W * GPW_QKV * 4096];
    static_assert(CH_W * GPW_D * 4096 <= (int)sizeof(smem) && CH_W * GPW_O / CH_O_KS * 4096 <= (int)sizeof(smem), "every role's rows");
    const int RH = (p.T + 15) >> 4;                                   // 16-row blocks
    const int QB = WIDE ? 128 : (p.qkv_half ? 32 : 64);             // q|k|v block width
    const int n_a = p.has_a ? p.T : 0, n_qkv = p.qkv.N / QB * RH, n_attn = p.T * p.nkv * (KVS ? p.attn_splits : 1), n_o = p.o.N / (p.o_half ? 32 : 64 * CH_O_NST) * RH * CH_O_KS;
    int wg = blockIdx.x;
    if (wg == 0) {                                                    // re-arm the other half of the route granules
        for (int i = threadIdx.x; i < (p.E > 0 ? p.T * p.Q * CH_GRAN * 2 : 0); i += 512) p.cnt_next[i] = 0u;
    }
    if (wg < n_a) { chain_role_a(p, wg, smem); return; }
    wg -= n_a;
    if (wg < n_qkv) {
        const int cb = wg / RH;
        if constexpr (WIDE) {
            // one head (128 columns) per workgroup: half as many workgroups of twice the bytes — taken where the narrow blocks and the
            // attention role together exceed the workgroups the chip holds at once (decode_chain_f16)
            chain_role_gemm<2, GPW_QKV, F16W>(p.qkv, cb, wg % RH, p.norm1, p.qkv_out, p.T, p.has_a != 0, smem, p);
        } else if (p.qkv_half)
            chain_role_gemm<1, GPW_QKV, F16W, 2>(p.qkv, cb, wg % RH, p.norm1, p.qkv_out, p.T, p.has_a != 0, smem, p);
        else
            chain_role_gemm<CH_QKV_NST, GPW_QKV, F16W>(p.qkv, cb, wg % RH, p.norm1, p.qkv_out, p.T, p.has_a != 0, smem, p);
        // (behind its own result; read by the launch after this one)
        const __amdgpu_buffer_rsrc_t r_n = chain_rsrc(p.rows_next, (long)p.rows_next_pieces * 16);
        for (int i = wg * 512 + threadIdx.x; i < p.rows_next_pieces; i += n_qkv * 512)
            __builtin_amdgcn_raw_buffer_store_b128((u32x4){NOT_YET, NOT_YET, NOT_YET, NOT_YET}, r_n, i * 16, 0, 16);
        return;
    }
    wg -= n_qkv;
    if (wg < n_attn) { chain_role_attn<KVS>(p, wg, smem); return; }
    wg -= n_attn;
    if (wg < n_o) {
        // (K part fastest: the two workgroups of a block are neighbours)
        static_assert(GPW_O % CH_O_KS == 0, "o_proj's quant groups per wave divide over its K parts");
        const int ks = wg % CH_O_KS, blk = wg / CH_O_KS;
        float* part = p.o_part + (long)ks * p.T * p.o.N;
        if (p.o_half)
            chain_role_gemm<1, GPW_O / CH_O_KS, F16W, 2, true>(p.o, blk / RH, blk % RH, p.attn_out, nullptr, p.T, true, smem, p, ks * (p.o.G / CH_O_KS), part);
        else
            chain_role_gemm<CH_O_NST, GPW_O / CH_O_KS, F16W, 4, true>(p.o, blk / RH, blk % RH, p.attn_out, nullptr, p.T, true, smem, p, ks * (p.o.G / CH_O_KS), part);
        return;
    }
    wg -= n_o;
    if constexpr (GPW_D == 0) {
        chain_role_b<false>(p, wg, smem);
    } else {
        if (wg < p.T) { chain_role_b<true>(p, wg, smem); return; }
        wg -= p.T;
        constexpr int GU = F16W ? 1 : 2;
        const int n_gu = p.gu.N / (64 * GU) * RH;
        if (wg < n_gu) { chain_role_gemm<GU, GPW_QKV, F16W, 4, false, true>(p.gu, wg / RH, wg % RH, p.norm2, p.act, p.T, true, smem, p); return; }
        wg -= n_gu;
        const int parts = p.dn.G / (8 * GPW_D), ks = wg % parts, blk = wg / parts;
        float* slab = p.slabs + (long)ks * p.T * p.dn.N;
        if constexpr (F16W)
            chain_role_gemm<1, GPW_D, true, 2, true>(p.dn, blk / RH, blk % RH, p.act, nullptr, p.T, true, smem, p, ks * 8 * GPW_D, slab);
        else
            chain_role_gemm<2, GPW_D, false, 4, true>(p.dn, blk / RH, blk % RH, p.act, nullptr, p.T, true, smem, p, ks * 8 * GPW_D, slab);
    }
}

void chain_tail_args(const DecodeChainDesc& d, ChainArgs& a) {
    a.T = d.T; a.H = d.H;
    a.has_a = d.has_a ? (d.E > 0 ? 1 : (d.a_x ? 3 : 2)) : 0; a.top_k = d.top_k;
    a.a_x = d.a_x;
    a.a_slabs = d.a_slabs; a.a_S = d.a_S; a.a_slab_stride = d.a_slab_stride; a.a_ld = d.a_ld; a.down = d.down; a.comb_w = d.comb_w; a.res_in = d.res_in; a.ln_in = d.ln_in;
    a.eps = d.eps;
}
// Behind the last layer the tail's rows go through the final norm, the sampled ones alone: one launch of a few µs where the tail, a copy of the
// residual (dense models) and the norm were three (a step of 14 fp16 layers of 1024 columns,
// 8 rows: 328.5 → 324.6 µs; of 8 expert layers, 1 row: 361.5 → 359.8).
__global__ __launch_bounds__(512) void decode_tail_kernel(ChainArgs p, const int32_t* __restrict__ rows, __half* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[8 * sizeof(float)];
    chain_role_a(p, rows[blockIdx.x], smem, out + (long)blockIdx.x * p.H);
}

}  // namespace

int decode_tail_norm_f16(const DecodeChainDesc& d, const int32_t* rows, const __half* w, __half* out, int n, hipStream_t stream) {
    if (n <= 0) return 0;
    FH_REQUIRE(d.has_a && d.H % 8 == 0 && d.H <= 8192, "decode_tail_norm: hidden=%d", d.H);
    ChainArgs a{};
    chain_tail_args(d, a);
    a.ln_in = w;
    hipLaunchKernelGGL(decode_tail_kernel, dim3(n), dim3(512), 0, stream, a, rows, out);
    FH_CHECK_LAUNCH();
    return 0;
}

#ifdef FERRUM_HIP_EXPERIMENTS
extern "C" __attribute__((visibility("default"))) void ferrum_hip_debug_set_chain_timeline(void* p) { g_chain_timeline = (unsigned long long*)p; }
#endif

int decode_chain_counter_words() { return CH_GRAN_WORDS; }
// handed-off rows of a token: role A's two, q|k|v's, attention's, o_proj's K parts; with an MLP in the launch (inter > 0) its input's and act's
size_t decode_chain_row_bytes(int H, int nq, int nkv, int inter) {
    return (size_t)4 * H + ((size_t)nq + 2 * nkv) * 256 + (size_t)nq * 256 + (size_t)CH_O_KS * 4 * H + (inter > 0 ? (size_t)2 * (H + inter) : 0);
}
static int chain_mlp_groups(bool f16w) { return f16w ? 1 : 2; }       // GPW_D
bool decode_chain_mlp_supports(const W4Device& qkv, const W4Device& gu, const W4Device& dn, int inter, int rows, size_t slab_bytes) {
    const bool f16w = qkv.f16t != nullptr;
    for (const W4Device* w : {&gu, &dn})
        if ((f16w ? !w->f16t || w->k != w->G * 128 : !w->qw || w->f16t) || w->zp || w->perm || w->bias || w->n % 128 != 0 ||
            (long)CH_MAX_T * std::max(w->n, w->k) * 4 >= (1L << 31)) return false;
    const int per = 8 * chain_mlp_groups(f16w);
    return inter % 128 == 0 && gu.k == qkv.k && gu.n == 2 * inter && dn.k == inter && dn.n == qkv.k && dn.G % per == 0 && dn.G / per <= 8 &&
           (size_t)(dn.G / per) * rows * dn.n * 4 <= slab_bytes;
}
// Rows up to which the launch takes the MLP: one block of them, and two of the smallest layers.  µs of a step without its vocabulary, the MLP's two launches behind the
// chain | in it.  32 INT4 layers of 4096, inter 14336: 1 row 1228 | 1091, 4 rows 1293 | 1145, 8 1312 | 1181, 12 of 120 keys 1453 | 1282, 16 1454 | 1289, 1 of 8000 keys
// 1417 | 1267.  8 of 4096, 12288, GELU: 1 332 | 282, 8 357 | 310, 16 390 | 337.  8 of 2048, 8192: 1 222 | 186, 8 247 | 205, 16 292 | 228.  14 fp16 layers of 1024, 3072:
// 1 307 | 233, 8 339 | 260, 16 368 | 279, 17 418 | 369, 32 450 | 400.  8 of 2048, 6144: 1 272 | 227, 8 297 | 262, 16 325 | 276.
// Past the line, when it was drawn (vocabularies included): 17 rows of those layers 2096 | 2333, 550 | 557, 407 | 404 (32: 428 | 428), fp16 of 2048 420 | 457, of 1024 64 rows 707 | 751.
int decode_chain_mlp_max_rows(const W4Device& qkv) { return qkv.f16t && qkv.G == 8 ? 32 : 16; }
// Rows up to which a dense layer takes the launch: beyond 64 the 64-row GEMM tiles win (INT4 of 4096 × 14336, 96 rows: 5.56 ms a step against 5.61), and through
// fp16 layers of 2048 columns the fourth block of rows costs more than the launches of their own (µs of a step of 6 layers, those | this one: 32 heads on 8, 48 rows
// 460 | 461, 52 464 | 517, 64 515 | 569; 32 on 4, 48 rows 412 | 410, 52 418 | 459, 64 445 | 495; 16 on 8, 48 rows 432 | 409, 52 438 | 449, 64 486 | 496; of 1024 columns,
// 16 on 8: 52 rows 319 | 303, 64 365 | 341).
int decode_chain_dense_max_rows(const W4Device& qkv) { return qkv.f16t && qkv.G > 8 ? 48 : 64; }
int decode_chain_mlp_parts(const W4Device& dn) { return dn.G / (8 * chain_mlp_groups(dn.f16t != nullptr)); }

bool decode_chain_supports(const DecodeChainDesc& d) {
    if (!d.qkv || !d.o) return false;
    const bool f16w = d.qkv->f16t != nullptr;
    const auto gemm_ok = [&](const W4Device& w) {
        return (f16w ? w.f16t && w.k == w.G * 128 : w.qw && !w.f16t) && !w.zp && !w.perm && !w.bias && w.G % 8 == 0 && w.n % 128 == 0 &&
               (long)CH_MAX_T * std::max(w.n, w.k) * 2 < (1L << 31);
    };
    if (!gemm_ok(*d.qkv) || !gemm_ok(*d.o)) return false;
    // the instantiated forms: a wave's K slices
    const int gq = d.qkv->G / 8, go = d.o->G / 8;
    if (f16w ? d.E > 0 || !((gq == 1 && go == 2) || (gq == 2 && (go == 2 || go == 4))) : !((gq == 2 || gq == 4) && go == 4)) return false;
    if (CH_MAX_T * decode_chain_row_bytes(d.H, d.nq, d.nkv, d.rows_inter) >= (1UL << 31)) return false;
    if (d.gate_up && (d.E > 0 || !d.down_proj || !d.slabs || d.rows_inter != d.down_proj->k ||
                      !decode_chain_mlp_supports(*d.qkv, *d.gate_up, *d.down_proj, d.rows_inter, d.T, ~(size_t)0))) return false;
    if (d.attn_splits > CH_MAX_SPLITS || (d.attn_splits > 1 && (!d.attn_partial || !d.attn_tickets))) return false;
    if (d.T < 1 || d.T > CH_MAX_T || d.head_dim != 128 || d.nkv < 1 || d.nq % d.nkv != 0 || d.nq / d.nkv > 14 || d.nkv > CH_MAX_KVH) return false;
    if (d.H % 32 != 0 || d.H > 8192 || d.qkv->k != d.H || d.qkv->n != (d.nq + 2 * d.nkv) * 128 || d.o->k != d.nq * 128 || d.o->n != d.H) return false;
    if (d.E <= 0) {       // dense model: role B is add + norm, role A sums the down projection's slabs (or adds its fp16 rows)
        if (d.Q != 1 || (d.has_a && !d.a_x && (!d.a_slabs || d.a_S < 1 || d.a_ld < d.H))) return false;
        return (size_t)d.H * 2 + 64 * 4 <= (size_t)CH_SMEM;
    }
    const int tiles = (d.E + 15) / 16;
    if (d.E > 0xfff0 || d.Q < 1 || d.Q > 4 || tiles % d.Q != 0 || tiles / d.Q > 8 || d.r_top_k < 1 || d.r_top_k > 8) return false;
    if (d.has_a && (d.top_k < 1)) return false;
    // LDS of role B: the row + the part logits
    const int tiles_q = tiles / d.Q, ksplit = tiles_q >= 8 ? 1 : 8 / tiles_q;
    if ((size_t)d.H * 2 + (size_t)tiles_q * 16 * (ksplit + 1) * 4 + 8 * 4 + (8 + 4 * CH_GRAN) * 8 + 16 > (size_t)CH_SMEM) return false;
    return true;
}

int decode_chain_f16(const DecodeChainDesc& d, hipStream_t stream) {
    FH_REQUIRE(d.rows && d.rows_next && decode_chain_supports(d), "decode_chain: shapes not taken by the merged form");
    ChainArgs a{};
    chain_tail_args(d, a);
    a.nq = d.nq; a.nkv = d.nkv;
    unsigned char* rows = d.rows;
    auto take = [&](size_t bytes) { unsigned char* at = rows; rows += bytes * d.T; return at; };
    a.norm1 = reinterpret_cast<__half*>(take((size_t)2 * d.H));
    a.res_a = reinterpret_cast<__half*>(take((size_t)2 * d.H));
    if (!d.has_a) { a.norm1 = d.norm1; a.res_a = d.res_a; }
    a.qkv_out = reinterpret_cast<__half*>(take(((size_t)d.nq + 2 * d.nkv) * 256));
    a.attn_out = reinterpret_cast<__half*>(take((size_t)d.nq * 256));
    a.o_part = reinterpret_cast<float*>(take((size_t)CH_O_KS * 4 * d.H));
    if (d.rows_inter > 0) {
        a.norm2 = reinterpret_cast<__half*>(take((size_t)2 * d.H));
        a.act = reinterpret_cast<__half*>(take((size_t)2 * d.rows_inter));
    }
    a.rows_next = reinterpret_cast<uint32_t*>(d.rows_next); a.rows_next_pieces = (int)((rows - d.rows) / 16);
    const bool mlp = d.gate_up != nullptr;
    const bool f16w = d.qkv->f16t != nullptr;
    const auto gemm = [&](const W4Device& w) { return ChainGemm{f16w ? (const void*)w.f16t : w.qw, w.sc, w.G, w.n, w.k}; };
    a.qkv = gemm(*d.qkv);
    a.k_pool = d.k_pool; a.v_pool = d.v_pool; a.block_tables = d.block_tables; a.kv_lens = d.kv_lens;
    a.q_norm_w = d.q_norm_w; a.k_norm_w = d.k_norm_w; a.cos_t = d.cos_t; a.sin_t = d.sin_t;
    a.qk_mode = d.qk_mode; a.max_blocks = d.max_blocks; a.sliding_window = d.sliding_window;
    a.scale = 1.0f / sqrtf((float)d.head_dim);
    a.o = gemm(*d.o);
    if (mlp) { a.gu = gemm(*d.gate_up); a.dn = gemm(*d.down_proj); a.slabs = d.slabs; a.gelu = d.gelu; }
    else a.norm2 = d.norm2;
    a.res_b_out = d.res_b_out; a.post_ln = d.post_ln; a.router_w = d.router_w;
    a.E = d.E; a.r_top_k = d.r_top_k; a.Q = d.Q; a.norm_topk = d.norm_topk; a.defer_merge = d.defer_merge ? 1 : 0;
    a.cand = d.cand; a.stats = d.stats; a.route_arrive = d.route_arrive; a.ids = d.ids; a.weights = d.weights;
    a.cnt = d.cnt; a.cnt_next = d.cnt_next; a.timeout = d.timeout;
#ifdef FERRUM_HIP_EXPERIMENTS
    a.tl = g_chain_timeline;
#endif
    const int rh = (d.T + 15) / 16;
    a.attn_splits = std::max(1, d.attn_splits); a.attn_partial = d.attn_partial; a.attn_tickets = d.attn_tickets;
    // 32-column q|k|v blocks for up to 16 rows, as long as they and the attention role are resident together: beyond, the role's last
    // workgroups enter behind the projection
    a.qkv_half = (knobs().chain_qkv_half && d.T <= 16 && d.qkv->n / 32 + d.T * d.nkv * a.attn_splits <= knobs().chain_slots) ? 1 : 0;
    // (narrow o_proj only: 2048 columns → 64 blocks; Llama-3.1-8B's 4096 columns are 64 blocks of 64 already: c=8 1.908 → 1.930 ms with 32)
    // (and of 1024 columns up to 32 rows: a step of 32 through 14 unquantised layers 540 → 527 µs)
    a.o_half = (knobs().chain_o_half && rh * d.o->n <= 2048) ? 1 : 0;
    // 128-column q|k|v blocks (hidden 2048 only: the two-group weight ring): where the 64-column blocks + the attention role do not fit
    // the chip's resident workgroups, the role's last workgroups enter behind the projection (≈ 2.7 µs of K/V round trips on the
    // critical path, profiles/r03_decode_chain_timeline.txt) — c=32 4.025 → 3.995 ms per step, c=64 4.83 → 4.69; c=20–24 (where they fit) 3 % slower
    a.qkv_wide = 0;
    if (!f16w && !mlp && !a.qkv_half && d.qkv->G / 8 == 2 && a.attn_splits == 1) {
        const int wide = knobs().chain_qkv_wide;
        const int n64 = d.qkv->n / 64 * rh, n_at = d.T * d.nkv * a.attn_splits;
        a.qkv_wide = wide >= 0 ? (wide > 0) : (n64 + n_at > knobs().chain_slots);
    }
    const int blocks = (d.has_a ? d.T : 0) + d.qkv->n / (a.qkv_half ? 32 : (a.qkv_wide ? 128 : 64)) * rh + d.T * d.nkv * a.attn_splits + d.o->n / (a.o_half ? 32 : 64 * CH_O_NST) * rh * CH_O_KS + d.T * d.Q +
                       (mlp ? d.gate_up->n / (f16w ? 64 : 128) * rh + d.H / (f16w ? 32 : 128) * rh * decode_chain_mlp_parts(*d.down_proj) : 0);
    form_hit(FORM_DECODE_CHAIN);
    if (a.attn_splits > 1) form_hit(FORM_CHAIN_ATTN_KV_SPLITS);
    if (a.qkv_wide) form_hit(FORM_CHAIN_QKV_WIDE);
    if (mlp) form_hit(FORM_CHAIN_MLP);
    // Unquantised layers (dense ones of 1024 – 2048 columns; a wave's weights of 4096 columns do not fit its registers, and such
    // layers are streaming, not waiting).  A step of 14 layers of 1024 columns, the launches of their own | this one, µs: 1 row of 60 keys
    // 470 | 380, 8 rows 505 | 424, 16 542 | 450, 17 538 | 491, 32 583 | 527, 33 655 | 572, 48 696 | 643, 64 735 | 723; 1 of 1500 keys 592 | 419, 8 of 900
    // 622 | 538, 32 of 500 732 | 643, 64 of 300 857 | 826.
    if (f16w) {
        const int gq = d.qkv->G / 8, go = d.o->G / 8;
        const bool kvs = a.attn_splits > 1;
#define FH_CHAIN_F16(GQ, GO)                                                                                                                    \
        do {                                                                                                                                    \
            if (mlp && kvs) hipLaunchKernelGGL((decode_chain_kernel<GQ, GO, true, true, false, 1>), dim3(blocks), dim3(512), 0, stream, a);     \
            else if (mlp) hipLaunchKernelGGL((decode_chain_kernel<GQ, GO, true, false, false, 1>), dim3(blocks), dim3(512), 0, stream, a);      \
            else if (kvs) hipLaunchKernelGGL((decode_chain_kernel<GQ, GO, true, true>), dim3(blocks), dim3(512), 0, stream, a);                 \
            else hipLaunchKernelGGL((decode_chain_kernel<GQ, GO, true>), dim3(blocks), dim3(512), 0, stream, a);                                \
        } while (0)
        if (gq == 1) FH_CHAIN_F16(1, 2); else if (go == 2) FH_CHAIN_F16(2, 2); else FH_CHAIN_F16(2, 4);
#undef FH_CHAIN_F16
    } else if (mlp) {
#define FH_CHAIN_MLP(GQ)                                                                                                                        \
        do {                                                                                                                                    \
            if (a.attn_splits > 1) hipLaunchKernelGGL((decode_chain_kernel<GQ, 4, false, true, false, 2>), dim3(blocks), dim3(512), 0, stream, a); \
            else hipLaunchKernelGGL((decode_chain_kernel<GQ, 4, false, false, false, 2>), dim3(blocks), dim3(512), 0, stream, a);               \
        } while (0)
        if (d.qkv->G / 8 == 2) FH_CHAIN_MLP(2); else FH_CHAIN_MLP(4);
#undef FH_CHAIN_MLP
    } else if (a.attn_splits > 1) {
        if (d.qkv->G / 8 == 2) hipLaunchKernelGGL((decode_chain_kernel<2, 4, false, true>), dim3(blocks), dim3(512), 0, stream, a);
        else hipLaunchKernelGGL((decode_chain_kernel<4, 4, false, true>), dim3(blocks), dim3(512), 0, stream, a);
    } else if (a.qkv_wide) hipLaunchKernelGGL((decode_chain_kernel<2, 4, false, false, true>), dim3(blocks), dim3(512), 0, stream, a);
    else if (d.qkv->G / 8 == 2) hipLaunchKernelGGL((decode_chain_kernel<2, 4, false>), dim3(blocks), dim3(512), 0, stream, a);
    else hipLaunchKernelGGL((decode_chain_kernel<4, 4, false>), dim3(blocks), dim3(512), 0, stream, a);
    FH_CHECK_LAUNCH();
    return 0;
}

}  // namespace fh
