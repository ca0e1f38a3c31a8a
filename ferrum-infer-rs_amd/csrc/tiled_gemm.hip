// Dense projections of the layered models (tiled_gemm.h): one kernel for few rows (K split over the waves of a workgroup, summed in
// LDS, no second launch) and one for prompts (tiles of up to 128 × 256, both operands copied to LDS by the load unit itself).
// Every activation, bias and per-row factor of a projection is applied to the fp32 accumulator in the epilogue.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "knobs.h"
#include "tiled_gemm.h"

namespace fh {

template <typename E, bool RARE = false>
__device__ __forceinline__ float gemm_act(const GemmSection& sec, float v) {
    if (sec.act == GEMM_ACT_SIGMOID) return ActMath<E>::sigmoid(v);
    if (sec.act == GEMM_ACT_GELU_TANH) return gelu_tanh_f32<E>(v);
    if (sec.act == GEMM_ACT_XIELU) return xielu_f32<E>(v, sec.p, sec.q);
    if (sec.act == GEMM_ACT_RELU2) { v = fmaxf(v, 0.f); return v * v; }
    if (sec.act == GEMM_ACT_SILU) return v * ActMath<E>::sigmoid(v);
    if (RARE && sec.act == GEMM_ACT_SOFTPLUS) return softplus_f32<E>(v);
    if (RARE && sec.act == GEMM_ACT_LOG_SIGMOID) return sec.p * log_sigmoid_f32<E>(v);
    if (RARE && sec.act == GEMM_ACT_SOFTCAP) return sec.p * ActMath<E>::tanh(v / sec.p);
    return v;
}
// output row of place r, −1: none
template <typename E>
__device__ __forceinline__ int gemm_out_row(const TiledGemm<E>& p, int r) {
    if (p.rows.id) r = p.rows.id[r];
    return r < p.m ? r : -1;
}
template <typename E>
__device__ __forceinline__ void gemm_store(const TiledGemm<E>& p, int g, int row, int col, float v) {
    if (p.row_scale) v *= (float)p.row_scale[row * p.ld_scale + g];
    if (p.col_scale) v *= (float)p.col_scale[p.col_scale_row[row] * p.ld_col_scale + col];
    const long o = row * p.ldo + (p.rows.id ? 0 : g * p.out_group) + col;
    if (p.out_f32) p.out_f32[o] = v; else p.out[o] = (E)v;
}
template <typename E, bool RARE>
__device__ __forceinline__ void gemm_epilogue(const TiledGemm<E>& p, const GemmSection& sec, int g, int place, int col, float v) {
    const int row = gemm_out_row(p, place);
    if (row < 0 || col >= p.n_store) return;
    v *= sec.mul;
    if (p.bias) v += p.bias[(long)g * p.n + col];
    gemm_store(p, g, row, col, gemm_act<E, RARE>(sec, v));
}
template <typename E>
__device__ __forceinline__ float gemm_glu(const GemmSection& sec, float gate, float up) {
    if (sec.act == GEMM_ACT_SILU_GLU) return gate * ActMath<E>::sigmoid(gate) * up;
    if (sec.act == GEMM_ACT_GELU_GLU) return gelu_tanh_f32<E>(gate) * up;
    return clamped_glu_f32<E>(gate, up, sec.p, sec.q);
}
// accumulators of a (gate, up) pair of tiles; col: the gate's column
template <typename E>
__device__ __forceinline__ float gemm_gated(const TiledGemm<E>& p, const GemmSection& sec, int col, float gate, float up) {
    gate *= sec.mul;
    up *= sec.mul;
    if (p.bias) { gate += p.bias[col]; up += p.bias[col + 16]; }
    return gemm_glu<E>(sec, gate, up);
}
__device__ __forceinline__ int gemm_gated_col(const GemmSection& sec, int col) { return sec.begin + ((col - sec.begin) >> 5) * 16 + (col & 15); }
template <typename E>
__device__ __forceinline__ GemmSection gemm_section(const TiledGemm<E>& p, int col) {
    GemmSection s = {0, GEMM_ACT_NONE, 0.f, 0.f, 1.f};
#pragma unroll
    for (int i = 0; i < GEMM_MAX_SECTIONS; i++)
        if (i < p.nsec && col >= p.sec[i].begin) s = p.sec[i];
    return s;
}

// address of lane (a, b)'s 8 values of row tile t at k-step 0, and the distance between k-steps
template <typename E>
__device__ __forceinline__ const E* gemm_row(const TiledGemm<E>& p, int t, int g, int a, int b) {
    if (p.x_blocks) {
        const int tiles = (p.m + 15) >> 4;
        return p.x + (long)p.x_blocks[t < tiles ? t : tiles - 1] * p.x_block_elems + (a * 16 + b) * 8;
    }
    int r = t * 16 + b;
    if (p.rows.id) {
        r = p.rows.id[r];
        return p.x + (long)((unsigned)(r < p.m ? r : p.m - 1) / (unsigned)p.rows.div) * p.ldx + 8 * a;
    }
    return p.x + (long)(r < p.m ? r : p.m - 1) * p.ldx + g * p.x_group + 8 * a;
}
template <typename E>
__device__ __forceinline__ int gemm_row_step(const TiledGemm<E>& p) { return p.x_blocks ? 512 : 32; }

// models whose gate tiles all lie ahead of the up tiles (elsewhere the distance of a pair's tiles stays a constant: 5 % of a gated launch of few rows)
template <typename E> constexpr bool PAIRED = std::is_same_v<E, _Float16>;

// grid (column blocks, row blocks, groups or K slabs); NW waves = (NW / kw) column groups × kw parts of K.  Two register buffers of U
// k-steps: the next one is requested before the current one is multiplied; loads past the part's end repeat its last k-step.
// EXT: with sorted rows, column factors, gated sections or rare activations (each is a branch on the latency-bound path of the launches without).
template <typename E, int MT, int J, bool EXT>
__global__ __launch_bounds__(512) void tiled_gemm_kernel(TiledGemm<E> p, int kw) {
    typedef typename Frag<E>::v8 v8;
    if (!EXT) { p.rows.id = nullptr; p.col_scale = nullptr; p.pair = 0; }
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    floatx4* red = reinterpret_cast<floatx4*>(smem);            // [NW][MT·J][64]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int a = lane >> 4, b = lane & 15;
    const int cw = (blockDim.x >> 6) / kw, part = wave % kw, cg = wave / kw;
    const int n0 = (blockIdx.x * cw + cg) * 16 * J, rb = blockIdx.y;
    const int z = p.slabs > 1 ? blockIdx.z : 0;
    int g = p.slabs > 1 ? 0 : blockIdx.z;
    if (p.rows.id) {
        if (rb * 16 * MT >= *p.rows.total) return;
        g = p.rows.group[rb];
    }
    const int ksteps = p.k >> 5, parts = kw * p.slabs, mine = z * kw + part;
    const bool live = n0 < p.n;
    const int s0 = live ? ksteps * mine / parts : 0, s1 = live ? ksteps * (mine + 1) / parts : 0;
    const E* xrow[MT];
    const int xs = gemm_row_step(p);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) xrow[mt] = gemm_row(p, rb * MT + mt, g, a, b);
    const bool halves = PAIRED<E> && J == 2 && p.pair;
    const E* wt = p.w + ((long)g * (p.n >> 4) + (!live ? 0 : halves ? n0 >> 5 : n0 >> 4)) * ksteps * 512 + lane * 8;
    const int next_tile = halves ? p.pair : 1;
    floatx4 acc[MT][J];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int j = 0; j < J; j++) acc[mt][j] = (floatx4){0.f, 0.f, 0.f, 0.f};
    // (four row tiles by two: two k-steps, 150 registers; four spilled, which cost 13 %: 60 × 8192 × 2048 16.9 → 14.7 µs, 100 × 6144 × 2048
    // 25.6 → 21.4)
    constexpr int U = sizeof(E) == 2 ? (MT * J == 1 ? 8 : MT * J == 8 ? 2 : 4) : 1;
    v8 bw[2][U][J], ax[2][U][MT];
    auto load = [&](v8 (&bq)[U][J], v8 (&aq)[U][MT], int s) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int ss = min(s + u, s1 - 1);
#pragma unroll
            for (int j = 0; j < J; j++) bq[u][j] = __builtin_nontemporal_load(reinterpret_cast<const v8*>(wt + ((long)j * next_tile * ksteps + ss) * 512));
#pragma unroll
            for (int mt = 0; mt < MT; mt++) aq[u][mt] = *reinterpret_cast<const v8*>(xrow[mt] + (long)ss * xs);
        }
    };
    auto mul = [&](v8 (&bq)[U][J], v8 (&aq)[U][MT], int s) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < s1) {
#pragma unroll
                for (int j = 0; j < J; j++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) acc[mt][j] = Frag<E>::mma(aq[u][mt], bq[u][j], acc[mt][j]);
            }
    };
    // every buffer is requested in the block that multiplies the other one, so each wait counts exactly the loads it needs
    if (s0 < s1) {
        int s = s0;
        load(bw[0], ax[0], s);
        while (true) {
            if (s + U >= s1) { mul(bw[0], ax[0], s); break; }
            load(bw[1], ax[1], s + U);
            mul(bw[0], ax[0], s);
            s += U;
            if (s + U >= s1) { mul(bw[1], ax[1], s); break; }
            load(bw[0], ax[0], s + U);
            mul(bw[1], ax[1], s);
            s += U;
        }
    }
    if (p.slabs > 1) p.out_f32 += z * p.slab_stride;
    const GemmSection sec = gemm_section(p, n0);
    const bool gated = EXT && J == 2 && gemm_gated_act(sec.act);
    if (kw == 1) {
        if (!live) return;
        if constexpr (J == 2)
            if (gated) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int row = gemm_out_row(p, (rb * MT + mt) * 16 + 4 * a + r);
                        if (row >= 0) gemm_store(p, g, row, gemm_gated_col(sec, n0 + b), gemm_gated(p, sec, n0 + b, acc[mt][0][r], acc[mt][J - 1][r]));
                    }
                return;
            }
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) gemm_epilogue<E, EXT>(p, sec, g, (rb * MT + mt) * 16 + 4 * a + r, n0 + 16 * j + b, acc[mt][j][r]);
        return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int j = 0; j < J; j++) red[(wave * MT * J + mt * J + j) * 64 + lane] = acc[mt][j];
    __syncthreads();
    if (!live) return;
    auto summed = [&](int t) {
        floatx4 v = red[(cg * kw * MT * J + t) * 64 + lane];
        for (int q = 1; q < kw; q++) v += red[((cg * kw + q) * MT * J + t) * 64 + lane];
        return v;
    };
    if (gated) {
        for (int mt = part; mt < MT; mt += kw) {
            const floatx4 gate = summed(mt * J), up = summed(mt * J + 1);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = gemm_out_row(p, (rb * MT + mt) * 16 + 4 * a + r);
                if (row >= 0) gemm_store(p, g, row, gemm_gated_col(sec, n0 + b), gemm_gated(p, sec, n0 + b, gate[r], up[r]));
            }
        }
        return;
    }
    // tile t of the column group is summed (in the order of the K parts) and finished by part t mod kw
    for (int t = part; t < MT * J; t += kw) {
        const floatx4 v = summed(t);
        const int mt = t / J, j = t % J;
#pragma unroll
        for (int r = 0; r < 4; r++) gemm_epilogue<E, EXT>(p, sec, g, (rb * MT + mt) * 16 + 4 * a + r, n0 + 16 * j + b, v[r]);
    }
}

// Prompts: 2 × 2 waves hold MI × NJ tiles of 16 × 16 each.  Both operands go through LDS, copied there by the load unit itself:
//  * weights in stages of one k-step, a ring of 2G − 1: 16 bytes of every lane of a fragment.  In 16 bits that is 32 of K, one 1-KiB load in
//    lane order; in 32 bits half of a fragment, 16 of K (the first or the last four of every lane's eight);
//  * rows in granules of two steps, a ring of G; a load takes 128 bytes (a cache line) of each of 8 rows, and the 16-byte pieces of row r lie
//    in the order 0 … 7 xor r, so that the 16 lanes that read one piece of 16 rows touch every bank alike.
__device__ const uint16_t zero_fragment[512] = {};
template <int MI, int NJ, int G>
struct BigTile {
    static constexpr int RT = 2 * MI, CT = 2 * NJ, ROWS = 16 * RT, COLS = 16 * CT, STAGES = 2 * G - 1;
    static constexpr int GRANULE = RT * 2048, STAGE = CT * 1024;        // bytes
    static constexpr size_t LDS = (size_t)G * GRANULE + STAGES * STAGE;
    static_assert(MI % 2 == 0 && (NJ == 2 || NJ == 4 || NJ == 8), "every wave copies whole fragments");
    static_assert(LDS >= (size_t)4 * 32 * (16 * NJ + 4) * 4, "the epilogue's rows fit the stages");
};
template <typename E, int MI, int NJ, int G, int PER_CU>
__global__ __launch_bounds__(256, PER_CU) void tiled_gemm_big_kernel(TiledGemm<E> p, int mtiles, int ntiles) {
    typedef BigTile<MI, NJ, G> T;
    typedef typename Frag<E>::v8 v8;
    constexpr bool HALVES = sizeof(E) == 4;
    constexpr int EP = 16 / sizeof(E), SK = 4 * EP;                     // elements of 16 bytes, K of a step
    typedef std::conditional_t<HALVES, typename Frag<E>::v4, v8> operand;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *const rows_lds = smem, *const w_lds = rows_lds + G * T::GRANULE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int a = lane >> 4, b = lane & 15;
    // workgroups go round-robin over 8 XCDs: give each XCD a contiguous run of tiles, and walk 8 row tiles per column tile
    if (p.rows.id) mtiles = *p.rows.total / T::ROWS;
    const int total = mtiles * ntiles, l = blockIdx.x;
    if (l >= total) return;
    const int q8 = total / 8, r8 = total % 8, xcd = l % 8;
    const int id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + l / 8;
    const int band = id / (8 * ntiles), rows_in = min(8, mtiles - band * 8), in_band = id - band * 8 * ntiles;
    const int mt = band * 8 + in_band % rows_in, m0 = mt * T::ROWS, n0 = (in_band / rows_in) * T::COLS;
    const int n = p.k / SK, ntl = p.n >> 4, g = p.rows.id ? p.rows.group[m0 / p.rows.block] : blockIdx.z;
    const int wm = wave >> 1, wn = wave & 1;
    // this wave's loads: MI of a granule (8 rows each), NJ / 2 of a weight stage
    const E *ap[MI], *bp[NJ / 2];
    const int piece = (lane & 7) ^ (lane >> 3);
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int r = (MI * wave + i) * 8 + (lane >> 3);
        ap[i] = HALVES ? gemm_row(p, (m0 + r) >> 4, g, piece >> 1, r & 15) + 4 * (piece & 1) : gemm_row(p, (m0 + r) >> 4, g, piece, r & 15);
    }
#pragma unroll
    for (int i = 0; i < NJ / 2; i++) {
        const int t = min((n0 >> 4) + NJ / 2 * wave + i, ntl - 1);
        bp[i] = p.w + ((long)g * ntl + (p.pair ? (t >> 1) + (t & 1) * p.pair : t)) * (p.k >> 5) * 512 + lane * 8;
    }
    const int xs = (HALVES ? 1 : 2) * gemm_row_step(p);
    const E* none = reinterpret_cast<const E*>(zero_fragment) + lane * EP;       // (past the end of K)
#define BIG_COPY(src, dst) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src), (__attribute__((address_space(3))) void*)(dst), 16, 0, 0)
    auto issue_rows = [&](int i, int place, bool in) {
        BIG_COPY(in ? ap[i] : none, rows_lds + place * T::GRANULE + (MI * wave + i) * 1024);
        ap[i] += xs;
    };
    auto issue_w = [&](int i, int place, bool in, bool second) {        // (second: of a fragment's halves)
        BIG_COPY(in ? bp[i] : none, w_lds + place * T::STAGE + (NJ / 2 * wave + i) * 1024);
        bp[i] += !HALVES ? 512 : second ? 508 : 4;
    };
#undef BIG_COPY
    floatx4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = (floatx4){0.f, 0.f, 0.f, 0.f};
    // 32 bits: sums of 128 products, then sums of those, as short as the few-row kernel's parts of K ever are.  Relative error against 64 bits
    // at K = 512 / 2048 / 6144: 2.1 / 2.2 / 2.4e-7, with sums of 512 4.0 / 4.0 / 4.1e-7 and 2 % faster, the few-row kernel 2.1 / 4.0 / 7.0e-7.
    floatx4 sum[HALVES ? MI : 1][HALVES ? NJ : 1] = {};
    struct Operands { operand x[MI], w[NJ]; };
    constexpr int READS = MI + NJ;
    const unsigned char* my_w = w_lds + wn * NJ * 1024 + lane * 16;
    const unsigned char* my_rows[2];
#pragma unroll
    for (int h = 0; h < 2; h++) my_rows[h] = rows_lds + wm * MI * 2048 + b * 128 + ((HALVES ? 2 * a + h : 4 * h + a) ^ (b & 7)) * 16;
    // fragment f of a k-step: half h of the granule at `gran`, the weight stage at `stage`
    auto read = [&](Operands& o, int f, int h, int gran, int stage) {
        if (f < NJ) o.w[f] = *reinterpret_cast<const operand*>(my_w + stage * T::STAGE + f * 1024);
        else o.x[f - NJ] = *reinterpret_cast<const operand*>(my_rows[h] + gran * T::GRANULE + (f - NJ) * 2048);
    };
    // every load but this wave's last `left` has arrived, for all waves
#define BIG_WAIT(left)                                                          \
    do {                                                                        \
        constexpr int vm = (left);                                              \
        asm volatile("" ::: "memory");                                          \
        __builtin_amdgcn_s_waitcnt((vm & 15) | 0x70 | (vm >> 4) << 14);         \
        __builtin_amdgcn_s_barrier();                                           \
        asm volatile("" ::: "memory");                                          \
        __builtin_amdgcn_sched_barrier(0);                                      \
    } while (0)
    // Step t multiplies the operands that step t − 1 read and meanwhile reads those of t + 1.  At its start all that was requested up to step
    // t − (2G − 2) has arrived: weight stage t + 1, and the granule of t + 1.  Stage t is free then, its operands being in registers, and
    // t + 2G − 1 takes its place; so is, at odd t, the granule of t.  The weights are the first operand: a lane holds four neighbouring columns
    // of one row.
    auto stage_after = [](int i) { return i + 1 < T::STAGES ? i + 1 : 0; };
    auto granule_after = [](int i) { return i + 1 < G ? i + 1 : 0; };
    auto step = [&](const Operands& now, Operands& then, auto odd, int t, int stage, int gran) {
        constexpr bool ODD = decltype(odd)::value;
        constexpr int LOADS = NJ / 2 + (ODD ? MI : 0), PER = MI * NJ / (READS + READS / 4);
        BIG_WAIT((T::STAGES - 2) * (NJ / 2) + (ODD ? G - 2 : G - 1) * MI);
        const bool in = t + T::STAGES < n, rows_in_k = SK * (t + T::STAGES) + EP * piece < p.k;
        const int to = stage_after(stage), from = ODD ? granule_after(gran) : gran;
#pragma unroll
        for (int q = 0; q <= READS; q++) {
            if (q < READS) read(then, q, ODD ? 0 : 1, from, to);
            if (q < NJ / 2) issue_w(q, stage, in, !ODD);          // (2G − 1 steps on: the other half)
            else if (ODD && q < LOADS) issue_rows(q - NJ / 2, gran, rows_in_k);
#pragma unroll
            for (int m = q * PER; m < (q < READS ? (q + 1) * PER : MI * NJ); m++) acc[m / NJ][m % NJ] = Frag<E>::mma(now.w[m % NJ], now.x[m / NJ], acc[m / NJ][m % NJ]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // (as the steps before the first would have requested it)
#pragma unroll
    for (int i = 0; i < T::STAGES; i++) {
#pragma unroll
        for (int f = 0; f < NJ / 2; f++) issue_w(f, i, i < n, i % 2 == 1);
        if (i % 2 == 0) {
#pragma unroll
            for (int f = 0; f < MI; f++) issue_rows(f, i / 2, SK * i + EP * piece < p.k);
        }
    }
    Operands even, odd;
    BIG_WAIT((T::STAGES - 1) * (NJ / 2) + (G - 1) * MI);
#pragma unroll
    for (int f = 0; f < READS; f++) read(even, f, 0, 0, 0);
    int stage = 0, gran = 0;
    for (int t = 0; t < n; t += 2) {
        step(even, odd, std::false_type{}, t, stage, gran);
        stage = stage_after(stage);
        step(odd, even, std::true_type{}, t + 1, stage, gran);
        stage = stage_after(stage);
        gran = granule_after(gran);
        if (HALVES && ((t & 6) == 6 || t + 2 >= n))
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    sum[i][j] += acc[i][j];
                    acc[i][j] = t + 2 >= n ? sum[i][j] : (floatx4){0.f, 0.f, 0.f, 0.f};
                }
    }
#undef BIG_WAIT
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                    // (the requests past the end have landed: the epilogue reuses the ring)
    // epilogue: 32 rows of a wave's accumulators at a time through LDS (the stages are free, the rows its own, LDS operations of a wave
    // complete in order), then a lane finishes 8 columns of a row: bias, activation and factors, and rows leave in 16-byte pieces.  In a
    // gated section the lanes of the up tiles have nothing to do, those of the gate tiles read both.
    __syncthreads();
    // Where the whole launch is one gated section, a row takes half as many lanes, none of them idle: an
    // expert model's up-projections 286 → 272 µs a launch, 2048 rows of a 0.6B model's gate_up 48 → 41.
    constexpr int LD = 16 * NJ + 4;
    float* lf = reinterpret_cast<float*>(smem) + wave * 32 * LD;
    const bool pairs = p.nsec == 1 && p.sec[0].begin == 0 && gemm_gated_act(p.sec[0].act);
    const int lanes = pairs ? NJ : 2 * NJ, place = lane & (lanes - 1), row_in = lane >> __builtin_ctz(lanes), rounds = lanes / 2;      // (rounds of 64 / lanes rows)
    const int cl = pairs ? (place >> 1) * 32 + (place & 1) * 8 : place * 8, col = n0 + wn * 16 * NJ + cl;
    const GemmSection sec = gemm_section(p, min(col, p.n - 1));
    const bool gated = gemm_gated_act(sec.act), vec = p.n_store % 8 == 0 && p.ldo % 8 == 0 && p.out_group % 8 == 0 && ((uintptr_t)p.out & 15) == 0 && ((uintptr_t)p.out_f32 & 15) == 0;
    const bool active = gated ? col < p.n && !(col & 16) : col < p.n_store;
    const int oc = gated ? gemm_gated_col(sec, col) : col;
    float bias[8], bias_up[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        bias[e] = p.bias && active ? p.bias[(long)g * p.n + col + e] : 0.f;
        bias_up[e] = p.bias && active && gated ? p.bias[(long)g * p.n + col + 16 + e] : 0.f;
    }
#pragma unroll
    for (int ch = 0; ch < MI / 2; ch++) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) *reinterpret_cast<floatx4*>(lf + (i * 16 + b) * LD + j * 16 + 4 * a) = acc[2 * ch + i][j];
        const int row0 = m0 + (wm * MI + 2 * ch) * 16;
#pragma unroll 1
        for (int q = 0; q < rounds; q++) {
            const int row = q * (32 / rounds) + row_in, gr = gemm_out_row(p, row0 + row);
            if (gr < 0 || !active) continue;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = lf[row * LD + cl + e] * sec.mul + bias[e];
            if (gated) {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = gemm_glu<E>(sec, v[e], lf[row * LD + cl + 16 + e] * sec.mul + bias_up[e]);
            } else if (sec.act != GEMM_ACT_NONE) {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = gemm_act<E, true>(sec, v[e]);
            }
            if (!vec) {
                for (int e = 0; e < 8; e++)
                    if (gated || col + e < p.n_store) gemm_store(p, g, gr, oc + e, v[e]);
                continue;
            }
            if (p.row_scale) {
                const float f = (float)p.row_scale[gr * p.ld_scale + g];
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= f;
            }
            if (p.col_scale) {
                const v8 f = *reinterpret_cast<const v8*>(p.col_scale + p.col_scale_row[gr] * p.ld_col_scale + oc);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= (float)f[e];
            }
            const long o = gr * p.ldo + (p.rows.id ? 0 : g * p.out_group) + oc;
            if (p.out_f32) {
                *reinterpret_cast<floatx4*>(p.out_f32 + o) = (floatx4){v[0], v[1], v[2], v[3]};
                *reinterpret_cast<floatx4*>(p.out_f32 + o + 4) = (floatx4){v[4], v[5], v[6], v[7]};
            } else {
                v8 y;
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] = (E)v[e];
                *reinterpret_cast<v8*>(p.out + o) = y;
            }
        }
    }
}

template <typename E, int MI, int NJ, int G, int PER_CU>
static int launch_big(const TiledGemm<E>& g, hipStream_t s) {
    typedef BigTile<MI, NJ, G> T;
    static bool attr = false;
    if (!attr) {
        FH_CHECK_HIP(hipFuncSetAttribute((const void*)tiled_gemm_big_kernel<E, MI, NJ, G, PER_CU>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)T::LDS));
        attr = true;
    }
    const int mtiles = g.rows.id ? g.rows.max_blocks * (g.rows.block / T::ROWS) : cdiv(g.m, T::ROWS), ntiles = cdiv(g.n, T::COLS);
    form_hit(g.rows.id ? FORM_TILED_GEMM_GROUPED_BIG : FORM_TILED_GEMM_BIG);
    form_hit(T::ROWS == 64 ? FORM_TILED_GEMM_64X64 : T::COLS == 256 ? FORM_TILED_GEMM_128X256 : T::COLS == 128 ? FORM_TILED_GEMM_128X128 : FORM_TILED_GEMM_128X64);
    hipLaunchKernelGGL((tiled_gemm_big_kernel<E, MI, NJ, G, PER_CU>), dim3(mtiles * ntiles, 1, g.groups), dim3(256), T::LDS, s, g, mtiles, ntiles);
    FH_CHECK_LAUNCH();
    return 0;
}
// Tile sizes, µs of bf16 launches (rows × columns × K):
//                          128 × 256   128 × 128   128 × 64   64 × 64   before (64 of K a stage, the rows' lines fetched by halves)
//   8192 × 10240 × 2048        277         326        396        500      322
//   8192 × 8192 × 8192         831         980       1255       1486      933
//   4096 × 6144 × 2048          91         104        119        148      119
//   4002 × 2048 × 2048          39          36         46         55       49
//   2048 × 4096 × 1024          26          23         28         33       28
//   256 × 8192 × 2048           34          24         17         19       20
//   2048 × 1024 × 2048          34          24         16         18       20
//   300 × 2048 × 2048           34          21         16         12       25
//   128 × 6144 × 2048           34          21         16         12       28
// Two workgroups of the largest tile share a CU, so that one's stores run under the other's products; below a tile per CU the smaller tiles
// cover the chip.  The lines between them, µs on both sides (tiles of the size whose round of 256 or 512 workgroups ends there):
//   128 × 256 → 128 × 128     256 tiles: 456 × 16384 × 2048   39.5 → 39.0     260: 456 × 16640 × 2048   53.9 → 56.3
//   128 × 64 → 128 × 128      256 of 128 × 128: 200 × 16384 × 6144   72 → 81, 968 × 4096 × 2048   26 → 29     264: 200 × 16896 × 6144   100 → 90
//   64 × 64 → 128 × 64        256: 253 × 4096 × 2048   14.5 → 17.3, 125 × 8192 × 4096   26 → 31     288: 253 × 4608 × 2048   19.8 → 17.5
//   few rows → 64 × 64        112: 253 × 1792 × 2048   13.9 → 14.2     128: 253 × 2048 × 2048   14.0 → 14.2, 125 × 4096 × 1024   9.9 → 9.6
//                             144: 253 × 2304 × 2048   22.5 → 14.3
template <typename E>
static int launch_big(const TiledGemm<E>& g, hipStream_t s) {
    auto tiles = [&](int r, int c) { return (long)(g.rows.id ? g.rows.max_blocks * (g.rows.block / r) : cdiv(g.m, r)) * cdiv(g.n, c) * g.groups; };
    if constexpr (sizeof(E) == 4) {
        // 32 bits: bound by the products alone, so the tile whose rounds over the CUs take least (µs of a round below, K = 2048; the few-row
        // kernel, which reads both operands from L2 for every 64 × 32 outputs, is left at 75 TFLOP/s of the 154 of a large product):
        //                        128 × 128   128 × 64   64 × 64   few-row kernel
        //   2048 × 2048 × 2048      142         147                  222
        //   1000 × 6144 × 2048      266         215                  330
        //   1000 × 2048 × 2048      140          83                  115
        //   500 × 2048 × 2048       139                    50         62
        //   1000 × 1024 × 512        41                    17         19
        //   128 × 8192 × 2048       139                    50         63
        //   256 × 2048 × 2048       138                    47         39      (128 tiles: too few; 253 × 2304 × 2048, 144 tiles: 46 and 60)
        const long full = cdiv(tiles(128, 128), 256) * 133L, half = cdiv(tiles(128, 64), 256) * 72L, small = cdiv(tiles(64, 64), 256) * 42L;
        if ((g.rows.id && g.rows.block < 128) || small < std::min(full, half)) return launch_big<E, 2, 2, 3, 3>(g, s);
        return half < full ? launch_big<E, 4, 2, 3, 2>(g, s) : launch_big<E, 4, 4, 2, 2>(g, s);
    } else {
        if (tiles(128, 256) >= knobs().tiled_wide_min_tiles) return launch_big<E, 4, 8, 2, 2>(g, s);
        if (tiles(128, 128) > knobs().tiled_half_max_tiles) return launch_big<E, 4, 4, 2, 2>(g, s);
        return tiles(64, 64) > knobs().tiled_small_max_tiles ? launch_big<E, 4, 2, 3, 2>(g, s) : launch_big<E, 2, 2, 3, 3>(g, s);
    }
}

int tiled_gemm_slabs(int m, int n, int k) {
    if (m > 64) return 1;
    // narrow outputs: enough (column group, K part) workgroups to cover the chip, two k-steps or more per wave
    int S = 1;
    while (S < GEMM_MAX_SLABS && (n / 32) * S < 256 && k / 32 >= 2 * 8 * 2 * S) S *= 2;
    return S;
}

template <typename E, int MT, int J, bool EXT>
static int launch_small(const TiledGemm<E>& g, dim3 grid, int nw, int kw, hipStream_t s) {
    const size_t lds = kw == 1 ? 0 : (size_t)nw * MT * J * 1024;
    hipLaunchKernelGGL((tiled_gemm_kernel<E, MT, J, EXT>), grid, dim3(64 * nw), lds, s, g, kw);
    FH_CHECK_LAUNCH();
    return 0;
}

template <typename E>
int tiled_gemm(const TiledGemm<E>& gin, hipStream_t s) {
    TiledGemm<E> g = gin;
    if (g.m <= 0) return 0;
    if (!g.n_store) g.n_store = g.n;
    FH_REQUIRE(g.n > 0 && g.k > 0 && g.n % 32 == 0 && g.k % 32 == 0, "tiled_gemm: n=%d k=%d must be multiples of 32", g.n, g.k);
    FH_REQUIRE(g.ldx % 8 == 0 && g.x_group % 8 == 0 && g.n_store <= g.n && g.groups >= 1, "tiled_gemm: ldx=%ld group stride=%ld", g.ldx, g.x_group);
    FH_REQUIRE((g.out != nullptr) != (g.out_f32 != nullptr), "tiled_gemm: exactly one output");
    FH_REQUIRE(g.slabs == 1 || (g.groups == 1 && g.out_f32 && !g.bias && !g.nsec && !g.row_scale), "tiled_gemm: slabs are plain fp32 partial sums");
    bool gated = false, rare = false;
    for (int i = 0; i < g.nsec; i++) {
        gated |= gemm_gated_act(g.sec[i].act);
        rare |= gemm_rare_act(g.sec[i].act);
        FH_REQUIRE(g.sec[i].begin % 32 == 0, "tiled_gemm: section at column %d", g.sec[i].begin);
    }
    FH_REQUIRE(!gated || (g.groups == 1 && !g.col_scale), "tiled_gemm: gated sections take one group and no column factors");
    FH_REQUIRE(!g.col_scale || (g.out && g.ld_col_scale % 8 == 0), "tiled_gemm: column factors with rows of %ld", g.ld_col_scale);
    FH_REQUIRE(!g.pair || (PAIRED<E> && gated && g.nsec == 1 && g.sec[0].begin == 0 && g.n == 32 * g.pair), "tiled_gemm: %d tiles of a half, n=%d", g.pair, g.n);
    const GemmRows& rows = g.rows;
    if (rows.id) {
        FH_REQUIRE(g.slabs == 1 && !g.bias && !g.x_blocks && !g.row_scale && rows.div > 0 && rows.max_blocks > 0 && rows.group && rows.total,
                   "tiled_gemm: sorted rows take plain sections");
        FH_REQUIRE(rows.block == 16 || rows.block == 32 || rows.block == 64 || ((rows.block == 128 || rows.block == 256) && sizeof(E) == 2), "tiled_gemm: blocks of %d rows", rows.block);
    }
    constexpr bool F32 = sizeof(E) == 4;
    const long tiles = (rows.id ? (long)rows.max_blocks * (rows.block / 64) : cdiv(g.m, 64)) * cdiv(g.n, 64) * g.groups;
    const bool enough_tiles = tiles >= knobs().tiled_big_min_tiles + F32;
    if (rows.id ? (F32 ? rows.block >= 64 && g.n >= 64 && enough_tiles : rows.block >= 128) : g.m > 64 && g.n >= 64 && g.slabs == 1 && enough_tiles) return launch_big(g, s);
    // rows per workgroup: as many as there are, fewer where narrow outputs would leave CUs idle: in 16 bits as long as a round of 256 workgroups
    // holds the launch (64 × 2048 × 4096, four row tiles | two: 20.6 | 12.8 µs; 65 × 1024 × 4096, two | one: 20.2 | 12.6; past the round, 24 × 3072 ×
    // 2048, two | one: 7.7 | 8.4)
    int mt = rows.id ? rows.block / 16 : g.m <= 16 ? 1 : (g.m <= 32 ? 2 : 4);
    auto row_tiles = [&](int t) { return (long)cdiv(g.m, 16 * t) * (g.n / 16) * g.groups * g.slabs; };
    while (!rows.id && mt > 1 && (F32 ? row_tiles(mt) < knobs().tiled_min_tiles : row_tiles(mt / 2) <= 2 * knobs().tiled_min_tiles)) mt /= 2;
    const int rbs = rows.id ? rows.max_blocks : cdiv(g.m, 16 * mt), ksteps = g.k / 32, zs = rows.id ? 1 : g.groups * g.slabs;
    // Columns and K parts of a wave.  Several row tiles, whose fragments a wave reads again for every column group: 16 columns as long as a
    // round of 256 workgroups holds all of them with K in four parts, else 32, and as many parts as make rounds / parts least (a tie: fewer
    // parts where they are long, so that less is summed through LDS).  µs, bf16, weights from HBM, K in 4 / 2 parts of a workgroup's four waves:
    //                            workgroups     16 columns      32 columns
    //   64 × 4096 × 2048          256 | 128    12.9 | 20.4     14.5 | 22.9
    //   64 × 5120 × 2048          320 | 160    21.1 | 20.4     14.6 | 23.1
    //   64 × 8256 × 2048          516 | 258    28.8 | 35.2     23.6 | 23.4
    //   64 × 8256 × 6144          516 | 258    82.7 | 97.4     66.1 | 59.1
    //   64 × 5120 × 256                                         6.5 |  8.5      (two k-steps a part; 16 columns in two parts 6.9)
    //   32 × 2560 × 6144 in four slabs                         14.7 | 13.4      (16 columns in two parts 16.7)
    // One row tile: four parts up to a round of workgroups, two up to the next; 32 columns where 16 would be more than a round in two parts (8 × 8192 ×
    // 2048: 16 columns 8.2, 32 8.6; 8256 columns: 11.3 and 10.9).  µs (four waves a workgroup, K split over kw of them):
    //                            32 columns      16 columns      before
    //                            kw 4   kw 2     kw 4   kw 2
    //   8 × 4096 × 1024           5.2             4.9    5.3     5.6 (16, eight waves, kw 8)
    //   8 × 6144 × 1024           5.6                    5.6     8.6 (16, eight waves, kw 8)
    //   8 × 5120 × 2048           7.0             8.1    7.3
    //   8 × 8192 × 2048           8.8                    8.3     10.4 (16, eight waves, kw 8)
    //   16 × 10240 × 2048        12.7   12.0            14.2     12.8 (32, eight waves, kw 8)
    //   8 × 1024 × 3072           8.0             6.5            7.4 (16, eight waves, kw 8)
    // Fewer waves a workgroup wait for each other less.  Slabs of a long K want every wave they can get (1 × 2048 × 8192 in four: eight waves 8.1,
    // four 8.4), and so do wide outputs that stream a long K: 8 × 24576 × 4096 in four parts of four waves 39.7, in eight of eight 36.8; 8 × 65536 × 2048
    // in two parts 50, in four 43, in eight 42.  Of a short one rounds decide again: 8 × 49152 × 1024 in two parts 19.3, in eight 21.2.
    // Sorted rows: K is split below 8192 column groups (24 blocks of 16 rows, 4096 × 2048: four parts 68, one 75; 64 blocks: 161 and 137).
    const bool long_slabs = g.slabs > 1 && ksteps / g.slabs >= 64, narrow = sizeof(E) == 4 || long_slabs;
    const long groups16 = (long)rbs * (g.n / 16) * zs;
    const bool plain = !narrow && !rows.id, wide = plain && g.slabs == 1 && groups16 >= 896, several = plain && mt > 1 && !wide && !(g.n <= 96 && g.m > 64);
    int J = several ? (groups16 <= 256 ? 1 : 2)
            : narrow ? (groups16 / 2 < (g.slabs > 1 ? 256 : 257) ? 1 : 2)
                     : (long)rbs * (g.n / 32) * g.groups < (g.n <= 96 && g.m > 64 ? 513 : mt == 1 ? 257 : 160) ? 1 : 2;       // (narrow outputs of prompts: two workgroups per CU)
    if (knobs().tiled_j > 0) J = knobs().tiled_j == 1 ? 1 : 2;
    if (gated) J = 2;
    const long cols = g.n / (16 * J);
    int nw = mt == 1 && (narrow || (wide && ksteps >= 128)) ? 8 : 4, kw = 1;
    if (knobs().tiled_nw > 0) nw = std::min(8, knobs().tiled_nw);
    if (several || (wide && mt == 1 && ksteps < 64)) {
        const int steps = ksteps / g.slabs;
        long least = 0;
        for (int k : {4, 2, 1}) {
            if (k > 1 && steps < 2 * k) continue;
            const long rounds = cdiv((long)rbs * cdiv(cols, 4 / k) * zs, 256);
            const bool tie = least && rounds * kw == least * k;
            if (!least || rounds * kw < least * k || (tie && (k > 1 || steps >= 128) && (steps >= 32 || steps < 4 * kw))) { kw = k; least = rounds; }
        }
    } else if (wide && mt == 1) {
        kw = nw;
    } else {
        const long enough = rows.id ? 8192 : J == 1 && plain ? 513 : 4096;
        while (kw < nw && (long)rbs * cols * zs * kw < enough && ksteps >= 8 * kw * g.slabs) kw *= 2;
    }
    if (knobs().tiled_kw > 0) kw = std::min(nw, knobs().tiled_kw);
    const dim3 grid(cdiv(cols, nw / kw), rbs, zs);
    form_hit(rows.id ? FORM_TILED_GEMM_GROUPED : FORM_TILED_GEMM);
#define SMALL(J_, EXT_) \
    (mt == 1 ? launch_small<E, 1, J_, EXT_>(g, grid, nw, kw, s) : mt == 2 ? launch_small<E, 2, J_, EXT_>(g, grid, nw, kw, s) : launch_small<E, 4, J_, EXT_>(g, grid, nw, kw, s))
    if (rows.id || g.col_scale || gated || rare) return J == 1 ? SMALL(1, true) : SMALL(2, true);
    return J == 1 ? SMALL(1, false) : SMALL(2, false);
#undef SMALL
}
template int tiled_gemm<bf16>(const TiledGemm<bf16>&, hipStream_t);
template int tiled_gemm<float>(const TiledGemm<float>&, hipStream_t);
template int tiled_gemm<_Float16>(const TiledGemm<_Float16>&, hipStream_t);

}  // namespace fh
