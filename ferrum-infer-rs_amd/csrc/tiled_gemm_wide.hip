// Dense projections of prompts over tiles of 256 × 256 (16-bit models; smaller tiles and the other forms: tiled_gemm.hip).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "knobs.h"
#include "tiled_gemm_device.h"

namespace fh {

// Accumulators stay in AGPRs, in place: left to itself the compiler turns a loop over 256 of them into three-address products and copies them all back at its
// end (8192 × 8192 × 8192 1086 µs, this way 809), and the epilogue would move them all to VGPRs at once.
__device__ __forceinline__ void mma_into(floatx4& c, const bf16x8& a, const bf16x8& b) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
__device__ __forceinline__ void mma_into(floatx4& c, const f16x8& a, const f16x8& b) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
__device__ __forceinline__ floatx4 acc_get(const floatx4& c) {
    floatx4 v;
    asm volatile("v_accvgpr_read_b32 %0, %4\n\tv_accvgpr_read_b32 %1, %5\n\tv_accvgpr_read_b32 %2, %6\n\tv_accvgpr_read_b32 %3, %7"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "a"(c[0]), "a"(c[1]), "a"(c[2]), "a"(c[3]));
    return v;
}
typedef uint32_t u32x2w __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4w __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wide_rsrc(const void* p, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000); }
// 16 bytes a lane to LDS; I KiB are added to both addresses
template <int I>
__device__ __forceinline__ void wide_copy(__amdgpu_buffer_rsrc_t r, unsigned char* to, uint32_t v, int at) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 16, v, at, I * 1024, 0);
}
__device__ __forceinline__ void wide_store(__amdgpu_buffer_rsrc_t r, const u32x4w& v, uint32_t at) { __builtin_amdgcn_raw_buffer_store_b128(v, r, at, 0, 0); }
// Eight neighbouring columns a lane, in 16 bits, from the four each of two tiles: lane (a, b) gets columns 16 · (a & 1) + 8 · (a >> 1) … of row b of the pair
template <typename E>
__device__ __forceinline__ u32x4w wide_pair(const floatx4& v0, const floatx4& v1) {
    const u32x2w y0 = __builtin_bit_cast(u32x2w, __builtin_convertvector(v0, typename Frag<E>::v4)), y1 = __builtin_bit_cast(u32x2w, __builtin_convertvector(v1, typename Frag<E>::v4));
    const auto l = __builtin_amdgcn_permlane16_swap(y0.x, y1.x, false, false), h = __builtin_amdgcn_permlane16_swap(y0.y, y1.y, false, false);
    return (u32x4w){l[0], h[0], l[1], h[1]};
}
// 64 bytes of 16 rows in `lo`, the 64 behind them in `hi` → 128 bytes of rows 0 – 7 in `lo`, of rows 8 – 15 in `hi`: lanes of row b + 8 change places with those of row b
__device__ __forceinline__ void wide_lines(u32x4w& lo, u32x4w& hi) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t p = lo[e], q = hi[e];
        lo[e] = __builtin_amdgcn_update_dpp(p, q, 0x128, 0xF, 0xC, false);
        hi[e] = __builtin_amdgcn_update_dpp(q, p, 0x128, 0xF, 0x3, false);
    }
}
template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, const F& f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(const F& f) { each_of(std::make_integer_sequence<int, N>{}, f); }

// 2 × 2 waves of 128 × 128 each, one wave per SIMD; a workgroup per CU works through its tiles one after the other.
//  * Both operands come to LDS by the load unit as in tiled_gemm_big_kernel (rows in granules of two k-steps, two of them; weights in stages of one, four
//    of them), so that the places of four steps are constants.  The addresses are a buffer's: an offset a lane that is the same for a whole tile, a scalar one
//    for the place in K, a constant one that counts in memory and in LDS alike.  A step has 64 products, 16 reads, 8 loads and no vector instruction beside
//    them (64-bit addresses, chosen for each load: 74 of them, and the matrix cores idled a third of the time).
//  * Bound by the power limit of the card (8192 × 8192 × 8192: matrix cores busy for 80 % of the time, at 1.67 GHz), so by what a product costs beside itself: 256 columns
//    take least from LDS (16 KiB a wave for 64 products; 64 × 128 a wave: 24 KiB) and from the caches.  Tiles of 192 and 128 columns for outputs that fill half
//    a round (4096 × 6144 × 2048 by itself 91 → 84 µs) made the prompts that have them no faster: the clock fell by as much, for everything around them.
//  * The last four steps of a tile request the first of the next one, so that nothing is waited for between tiles but the epilogue, which needs no LDS: rows
//    leave in whole lines, put together by lane exchanges.  µs of bf16 launches, tiles of 128 × 256 → these one after the other, epilogue through
//    LDS → so: 8192 × 8192 × 8192 842 → 747 → 730, 8192 × 10240 × 2048 301 → 272 → 253, 8192 × 16384 × 2048 gated 456 → 436 → 404.
struct WideTile {
    static constexpr int ROWS = 256, COLS = 256, GRANULE = 32768, STAGE = 16384, LDS = 2 * GRANULE + 4 * STAGE;
};
template <typename E>
__global__ __launch_bounds__(256, 1) void tiled_gemm_wide_kernel(TiledGemm<E> p, int mtiles, int ntiles) {
    typedef WideTile W;
    typedef typename Frag<E>::v8 v8;
    constexpr int MI = 8, NJ = 8, WL = NJ / 2;                      // (loads of a wave for a stage)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int a = lane >> 4, b = lane & 15, wm = wave >> 1, wn = wave & 1;
    // workgroups go round-robin over 8 XCDs: each XCD has a contiguous run of tiles, in bands of 8 row tiles, which its workgroups take in turn
    if (p.rows.id) mtiles = *p.rows.total / W::ROWS;
    const int total = mtiles * ntiles, xcd = blockIdx.x & 7, first = blockIdx.x >> 3;
    const int mine0 = xcd * (total >> 3) + min(xcd, total & 7), mine = (total >> 3) + (xcd < (total & 7)), per = ((int)gridDim.x - xcd + 7) >> 3;
    if (first >= mine) return;
    const int n = p.k >> 5, ntl = p.n >> 4;
    struct Tile { int m0, n0, g; };
    constexpr int BAND = 8;
    auto tile = [&](int i) {                                // (past the last one: the last one again)
        const int id = mine0 + min(i, mine - 1), band = id / (BAND * ntiles), rows_in = min(BAND, mtiles - band * BAND), in_band = id - band * BAND * ntiles;
        Tile t;
        t.m0 = (band * BAND + in_band % rows_in) * W::ROWS;
        t.n0 = (in_band / rows_in) * W::COLS;
        t.g = p.rows.id ? p.rows.group[t.m0 / p.rows.block] : 0;
        return t;
    };
    // This wave's loads, 8 of a granule and WL of a stage: offsets from 3 KiB below the operands, less what the load's constant adds
    const int piece = (lane & 7) ^ (lane >> 3);
    const uint32_t row_bytes = (uint32_t)p.ldx * sizeof(E);
    struct From { uint32_t x[MI], w[WL]; const char* w0; };
    auto from = [&](const Tile& t) {
        From f;
        f.w0 = reinterpret_cast<const char*>(p.w) + (long)t.g * ntl * n * 1024 - 3072;
#pragma unroll
        for (int i = 0; i < MI; i++) {
            int r = t.m0 + (MI * wave + i) * 8 + (lane >> 3);
            if (p.rows.id) r = p.rows.id[r];
            r = min(r, p.m - 1);
            if (p.rows.id) r = (unsigned)r / (unsigned)p.rows.div;
            f.x[i] = (uint32_t)r * row_bytes + piece * 16 + 3072 - (i & 3) * 1024;
        }
#pragma unroll
        for (int i = 0; i < WL; i++) {
            const int c = min((t.n0 >> 4) + WL * wave + i, ntl - 1);
            f.w[i] = (uint32_t)(p.pair ? (c >> 1) + (c & 1) * p.pair : c) * (uint32_t)(n * 1024) + lane * 16 + 3072 - i * 1024;
        }
        return f;
    };
    const __amdgpu_buffer_rsrc_t rx = wide_rsrc(reinterpret_cast<const char*>(p.x) - 3072, ~0u);
    unsigned char *const my_x_lds = smem + wave * 8192, *const my_w_lds = smem + 2 * W::GRANULE + wave * WL * 1024;
    int at_w = 0, at_x = 0;                                 // the next stage's and granule's place in K
    From now_from = from(tile(first)), next_from;
    auto load_x = [&](auto I, int slot) {
        constexpr int i = decltype(I)::value;
        wide_copy<i & 3>(rx, my_x_lds + slot * W::GRANULE + (i >> 2) * 4096, now_from.x[i], at_x);
        if (i == MI - 1) at_x += 128;
    };
    auto load_w = [&](auto I, int slot) {
        constexpr int i = decltype(I)::value;
        wide_copy<i>(wide_rsrc(now_from.w0, ~0u), my_w_lds + slot * W::STAGE, now_from.w[i], at_w);
        if (i == WL - 1) at_w += 1024;
    };
    floatx4 acc[MI][NJ];
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = (floatx4){0.f, 0.f, 0.f, 0.f};
    };
    struct Operands { v8 x[MI], w[NJ]; };
    constexpr int READS = MI + NJ;
    const unsigned char* my_w = smem + 2 * W::GRANULE + wn * NJ * 1024 + lane * 16;
    const unsigned char* my_rows[2];
#pragma unroll
    for (int h = 0; h < 2; h++) my_rows[h] = smem + wm * MI * 2048 + b * 128 + ((4 * h + a) ^ (b & 7)) * 16;
    auto read = [&](Operands& o, int f, int half, int slot, int stage) {
        if (f < NJ) o.w[f] = *reinterpret_cast<const v8*>(my_w + stage * W::STAGE + f * 1024);
        else o.x[f - NJ] = *reinterpret_cast<const v8*>(my_rows[half] + slot * W::GRANULE + (f - NJ) * 2048);
    };
    // every load but this wave's last `left` has arrived, for all waves, and what was read from LDS
#define WIDE_WAIT(left)                                                                \
    do {                                                                               \
        asm volatile("" ::: "memory");                                                 \
        __builtin_amdgcn_s_waitcnt(((left) & 15) | 0x70 | ((left) >> 4) << 14);        \
        __builtin_amdgcn_s_barrier();                                                  \
        asm volatile("" ::: "memory");                                                 \
        __builtin_amdgcn_sched_barrier(0);                                             \
    } while (0)
    // Step t, T = t mod 4, multiplies the operands that step t − 1 read and meanwhile reads those of t + 1.  At even t it requests weight stages t + 3 and t + 4, whose
    // places are free: that of t − 1, and that of t, whose operands are in registers; at odd t the granule of t + 3, in the place of that of t.  So at its start
    // everything has to have arrived but what step t − 1 requested.  Of the last four steps these requests are the next tile's first.  `fresh`: all
    // requests have arrived (the epilogue waited for them ahead of its stores, which are not to be waited for here).
    auto step = [&](const Operands& now, Operands& then, auto P, bool fresh, bool last) {
        constexpr int T = decltype(P)::value, M = MI * NJ, READ_EVERY = M / (READS + 4), LOAD_EVERY = M / 10;
        constexpr bool ODD = T & 1;
        asm volatile("" ::: "memory");
        if (T >= 2 || !fresh) __builtin_amdgcn_s_waitcnt(0xF70 | (ODD ? NJ : MI));
        WIDE_WAIT(63);
        each<M>([&](auto IM) {
            constexpr int m = decltype(IM)::value, q = (m - 1) / LOAD_EVERY;
            if constexpr (m % READ_EVERY == 0 && m / READ_EVERY < READS) read(then, m / READ_EVERY, (T + 1) & 1, ((T + 1) >> 1) & 1, (T + 1) & 3);
            if constexpr (m % LOAD_EVERY == 1 && q < (ODD ? MI : NJ)) {
                if constexpr (T == 1 && q == 0) {
#pragma unroll
                    for (int i = 0; i < MI; i++) now_from.x[i] = last ? next_from.x[i] : now_from.x[i];
                    at_x = last ? 0 : at_x;
                }
                if constexpr (T == 0 && q == WL) {
#pragma unroll
                    for (int i = 0; i < WL; i++) now_from.w[i] = last ? next_from.w[i] : now_from.w[i];
                    now_from.w0 = last ? next_from.w0 : now_from.w0;
                    at_w = last ? 0 : at_w;
                }
                if constexpr (ODD) load_x(std::integral_constant<int, q>{}, ((T + 3) >> 1) & 1);
                else load_w(std::integral_constant<int, q % WL>{}, q < WL ? (T + 3) & 3 : T);
            }
            mma_into(acc[m / NJ][m % NJ], now.w[m % NJ], now.x[m / NJ]);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    each<WL>([&](auto I) { load_w(I, 0); });
    each<MI>([&](auto I) { load_x(I, 0); });
    each<WL>([&](auto I) { load_w(I, 1); });
    each<WL>([&](auto I) { load_w(I, 2); });
    each<MI>([&](auto I) { load_x(I, 1); });
    next_from = from(tile(first + per));
    Operands even, odd;
    clear();
    WIDE_WAIT(NJ + MI);
#pragma unroll
    for (int f = 0; f < READS; f++) read(even, f, 0, 0, 0);
    bool fresh = false;
    for (int at = first;; at += per) {
        const Tile t = tile(at);
        for (int left = n; left > 0; left -= 4) {
            const bool last = left == 4;
            step(even, odd, std::integral_constant<int, 0>{}, fresh, last);
            step(odd, even, std::integral_constant<int, 1>{}, fresh, last);
            step(even, odd, std::integral_constant<int, 2>{}, fresh, last);
            step(odd, even, std::integral_constant<int, 3>{}, fresh, last);
            fresh = false;
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");                  // (the last products, before anything else reads them)
        next_from = from(tile(at + 2 * per));
        const int col0 = t.n0 + wn * 16 * NJ;
        const GemmSection sec = gemm_section(p, min(col0, p.n - 1));
        const int act = __builtin_amdgcn_readfirstlane(sec.act), row0 = t.m0 + wm * 128;
        const int rows0 = gemm_out_row(p, row0 + lane), rows1 = gemm_out_row(p, row0 + 64 + lane);       // output rows, one a lane
        floatx4 bias[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = col0 + 16 * j + 4 * a;
            bias[j] = (floatx4){0.f, 0.f, 0.f, 0.f};
            if (p.bias && c < p.n) bias[j] = *reinterpret_cast<const floatx4*>(p.bias + c);
        }
        // what the next tile's first two steps need, too
#pragma unroll
        for (int j = 0; j < NJ; j++) asm volatile("s_waitcnt vmcnt(0)" : "+v"(bias[j]) :: "memory");
        const bool glu = gemm_gated_act(act);
        const int oc = (glu ? sec.begin + ((col0 - sec.begin) >> 1) : col0), limit = glu ? sec.begin + ((p.n - sec.begin) >> 1) : p.n_store;
        auto row_of = [&](int i, int r) { return __shfl(i < 4 ? rows0 : rows1, (i & 3) * 16 + r); };
        auto finish = [&](auto kind, auto f32) {
            constexpr int KIND = decltype(kind)::value;
            constexpr bool F32_OUT = decltype(f32)::value, GLU = KIND >= GEMM_ACT_CLAMPED_GLU && KIND <= GEMM_ACT_GELU_GLU;
            constexpr int SIZE = F32_OUT ? 4 : 2, TILES = GLU ? NJ / 2 : NJ, LINE = F32_OUT ? 2 : 4;
            // (a store at `nowhere` is past the end of the output and dropped: rows and columns that are not there)
            const uint32_t out_bytes = (uint32_t)p.ldo * SIZE, nowhere = 0xF0000000u;
            const int cl = (b >> 3) * 8 * LINE + (F32_OUT ? 4 * a : (a & 1) * 16 + (a >> 1) * 8);
            const __amdgpu_buffer_rsrc_t ro = wide_rsrc(F32_OUT ? (const void*)p.out_f32 : (const void*)p.out, 0xE0000000u);
            each<MI>([&](auto I) {
                constexpr int i = decltype(I)::value;
                const int row0 = row_of(i, b & 7), row1 = row_of(i, (b & 7) + 8);
                const uint32_t at_column = (uint32_t)((oc + cl) * SIZE), o0 = row0 < 0 ? nowhere : (uint32_t)row0 * out_bytes + at_column, o1 = row1 < 0 ? nowhere : (uint32_t)row1 * out_bytes + at_column;
                auto value = [&](auto J) { return acc_get(acc[i][decltype(J)::value]) * sec.mul + bias[decltype(J)::value]; };
                auto tile_value = [&](auto J) {
                    constexpr int j = decltype(J)::value * (GLU ? 2 : 1);
                    floatx4 v = value(std::integral_constant<int, j>{});
                    if constexpr (GLU) gemm_glu<E, 4>(sec, KIND, v, value(std::integral_constant<int, j + 1>{}));
                    else gemm_act<E, false, 4>(sec, KIND, v);
                    return v;
                };
                auto half = [&](auto J) {                   // 64 bytes of 16 rows
                    constexpr int j = decltype(J)::value;
                    if constexpr (F32_OUT) return __builtin_bit_cast(u32x4w, tile_value(J));
                    else return wide_pair<E>(tile_value(J), tile_value(std::integral_constant<int, j + 1>{}));
                };
                each<TILES / LINE>([&](auto B) {
                    constexpr int j = LINE * decltype(B)::value;
                    u32x4w lo = half(std::integral_constant<int, j>{}), hi = half(std::integral_constant<int, j + LINE / 2>{});
                    wide_lines(lo, hi);
                    const bool in = oc + cl + 16 * j < limit;
                    wide_store(ro, lo, (in ? o0 : nowhere) + 16 * j * SIZE);
                    wide_store(ro, hi, (in ? o1 : nowhere) + 16 * j * SIZE);
                });
            });
        };
        // columns of several kinds, rare activations: two tiles of 16 rows at a time
        auto finish_any = [&] {
#pragma unroll 1
            for (int q = 0; q < MI * NJ / 2; q++) {
                const int i = q / (NJ / 2), j = q % (NJ / 2) * 2, col = col0 + 16 * j + 4 * a, row = row_of(i, b);
                const GemmSection s = gemm_section(p, min(col0 + 16 * j, p.n - 1));
                floatx4 v[2];
#pragma unroll
                for (int c = 0; c < MI * NJ / 2; c++)
                    if (c == q)
#pragma unroll
                        for (int h = 0; h < 2; h++) v[h] = acc_get(acc[c / (NJ / 2)][c % (NJ / 2) * 2 + h]) * s.mul + bias[c % (NJ / 2) * 2 + h];
                const int kind = __builtin_amdgcn_readfirstlane(s.act);
                const bool gated = gemm_gated_act(kind);
                if (gated) gemm_glu<E, 4>(s, kind, v[0], v[1]);
                else
#pragma unroll
                    for (int h = 0; h < 2; h++) gemm_act<E, true, 4>(s, kind, v[h]);
                if (row < 0) continue;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if (gated ? h > 0 || col >= p.n : col + 16 * h >= p.n_store) continue;
                    const long o = row * p.ldo + (gated ? gemm_gated_col(s, col) : col + 16 * h);
                    if (p.out_f32) *reinterpret_cast<floatx4*>(p.out_f32 + o) = v[h];
                    else *reinterpret_cast<typename Frag<E>::v4*>(p.out + o) = __builtin_convertvector(v[h], typename Frag<E>::v4);
                }
            }
        };
        const bool one_kind = gemm_section(p, min(col0 + 16 * NJ - 1, p.n - 1)).begin == sec.begin && (p.out || act == GEMM_ACT_NONE);
#define KIND(K) if (act == K) finish(std::integral_constant<int, K>{}, std::false_type{}); else
        if (!__builtin_amdgcn_readfirstlane(one_kind) || gemm_rare_act(act)) finish_any();
        else if (p.out_f32) finish(std::integral_constant<int, GEMM_ACT_NONE>{}, std::true_type{});
        else KIND(GEMM_ACT_NONE) KIND(GEMM_ACT_SILU_GLU) KIND(GEMM_ACT_GELU_GLU) KIND(GEMM_ACT_CLAMPED_GLU) KIND(GEMM_ACT_SIGMOID) KIND(GEMM_ACT_GELU_TANH) KIND(GEMM_ACT_XIELU) KIND(GEMM_ACT_RELU2)
            finish(std::integral_constant<int, GEMM_ACT_SILU>{}, std::false_type{});
#undef KIND
        if (at + per >= mine) break;
        clear();
        fresh = true;
    }
#undef WIDE_WAIT
}
// K of whole rounds of four steps; offsets of 32 bits; rows of 16-byte pieces; columns that need no factors
template <typename E>
bool tiled_gemm_wide_supports(const TiledGemm<E>& g) {
    const uint64_t most = 0xE0000000u, rows = g.rows.id ? cdiv(g.m, g.rows.div) : g.m;
    if (g.k % 128 || g.groups != 1 || g.slabs != 1 || g.x_blocks || g.row_scale || g.col_scale || (g.rows.id && g.rows.block % 256)) return false;
    if (rows * g.ldx * sizeof(E) >= most || (uint64_t)(g.n + 32) * g.k * sizeof(E) >= most || (uint64_t)g.m * g.ldo * (g.out ? sizeof(E) : 4) >= most) return false;
    if (g.n_store % 8 || g.ldo % 8 || ((uintptr_t)g.x | (uintptr_t)g.w | (uintptr_t)g.out | (uintptr_t)g.out_f32) & 15) return false;
    for (int i = 0; i < g.nsec; i++)                        // (rare activations are finished slowly)
        if (gemm_rare_act(g.sec[i].act) && (i + 1 < g.nsec ? g.sec[i + 1].begin : g.n) - g.sec[i].begin > 256) return false;
    return !(g.out_f32 && g.nsec && g.sec[0].act != GEMM_ACT_NONE);
}
template <typename E>
int tiled_gemm_wide(const TiledGemm<E>& g, hipStream_t s) {
    typedef WideTile W;
    static bool attr = false;
    if (!attr) {
        FH_CHECK_HIP(hipFuncSetAttribute((const void*)tiled_gemm_wide_kernel<E>, hipFuncAttributeMaxDynamicSharedMemorySize, W::LDS));
        attr = true;
    }
    const int mtiles = g.rows.id ? g.rows.max_blocks * (g.rows.block / W::ROWS) : cdiv(g.m, W::ROWS), ntiles = cdiv(g.n, W::COLS);
    form_hit(g.rows.id ? FORM_TILED_GEMM_GROUPED_BIG : FORM_TILED_GEMM_BIG);
    form_hit(FORM_TILED_GEMM_256X256);
    hipLaunchKernelGGL((tiled_gemm_wide_kernel<E>), dim3(std::min(256, mtiles * ntiles)), dim3(256), W::LDS, s, g, mtiles, ntiles);
    FH_CHECK_LAUNCH();
    return 0;
}
template bool tiled_gemm_wide_supports<bf16>(const TiledGemm<bf16>&);
template bool tiled_gemm_wide_supports<_Float16>(const TiledGemm<_Float16>&);
template int tiled_gemm_wide<bf16>(const TiledGemm<bf16>&, hipStream_t);
template int tiled_gemm_wide<_Float16>(const TiledGemm<_Float16>&, hipStream_t);

}  // namespace fh
