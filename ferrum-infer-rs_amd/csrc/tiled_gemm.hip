// Dense projections of the layered models (tiled_gemm.h): one kernel for few rows (K split over the waves of a workgroup, summed in
// LDS, no second launch) and one for prompts (tiles of up to 128 × 256, both operands copied to LDS by the load unit itself).
// Every activation, bias and per-row factor of a projection is applied to the fp32 accumulator in the epilogue.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "knobs.h"
#include "qkv_rows.h"
#include "tiled_gemm.h"
#include "tiled_gemm_device.h"

namespace fh {

template <typename E>
__device__ __forceinline__ void gemm_store(const TiledGemm<E>& p, int g, int row, int col, float v) {
    if (p.row_scale) v *= (float)p.row_scale[row * p.ld_scale + g];
    if (p.col_scale) v *= (float)p.col_scale[p.col_scale_row[row] * p.ld_col_scale + col];
    const long o = row * p.ldo + (p.rows.id ? 0 : g * p.out_group) + col;
    if (p.out_f32) p.out_f32[o] = v; else p.out[o] = (E)v;
}
// address of the 16-byte piece a of row b of row tile t, and the distance between the steps of four pieces
template <typename E>
__device__ __forceinline__ const E* gemm_row(const TiledGemm<E>& p, int t, int g, int a, int b) {
    constexpr int EP = 16 / sizeof(E);
    if (p.x_blocks) {
        const int tiles = (p.m + 15) >> 4;
        return p.x + (long)p.x_blocks[t < tiles ? t : tiles - 1] * p.x_block_elems + (a * 16 + b) * EP;
    }
    int r = t * 16 + b;
    if (p.rows.id) {
        r = p.rows.id[r];
        return p.x + (long)((unsigned)(r < p.m ? r : p.m - 1) / (unsigned)p.rows.div) * p.ldx + EP * a;
    }
    return p.x + (long)(r < p.m ? r : p.m - 1) * p.ldx + g * p.x_group + EP * a;
}
template <typename E>
__device__ __forceinline__ int gemm_row_step(const TiledGemm<E>& p) { return (p.x_blocks ? 1024 : 64) / sizeof(E); }
// models whose gate tiles all lie ahead of the up tiles (elsewhere the distance of a pair's tiles stays a constant: 5 % of a gated launch of few rows)
template <typename E> constexpr bool PAIRED = std::is_same_v<E, _Float16>;

// Few rows.  grid (column blocks, row blocks, groups or K slabs); a workgroup's waves are cw column groups × kw parts of K, and a part is taken in
// chunks of U loads (16 bytes a lane: 32 of K, in 32 bits 16), the next chunk requested before the current one is multiplied; loads past the
// part's end repeat its last one.
//  * Weights go to registers, a contiguous KiB a load.
//  * Rows go to LDS, a region of its own per wave: a load of 16 bytes a lane takes 64 · U bytes of 16 / U rows, whole cache lines, and the pieces
//    of row r lie in the order 0 … xor (r & 7), so that the 16 lanes that read one piece of 16 rows touch every bank alike.
// Bound by the weights' bytes and, below 30 MB, by the launch and the way to the first of them.  Fragments of the rows read from global memory, 64
// bytes of 16 rows at a time, kept the load units busy for longer than the weights did: 32 × 4608 × 2048 10.0 → 7.4 µs, 8 × 4096 × 1024 4.8 →
// 3.8, 8 × 1024 × 3072 6.5 → 5.3, 64 × 4096 × 2048 12.8 → 8.0, 32 × 32768 × 2048 31 → 26, in 32 bits 4 × 10240 × 2048 27.7 → 17.1 (a fragment is one
// KiB there too); a read of the same weights and nothing else: 4.8, 2.7, 2.5, 4.0, 20.7, 14.2.
// EXT: with sorted rows, rows from a cache, column factors, gated sections or rare activations (each is a branch on the latency-bound path of the
// launches without).
constexpr int FEW_LOADS = 4;
struct FewRows { int kw_log2, cw, rows, chunk; uint32_t ldx16; };       // (rows of x in a region; loads of a part; pieces between rows of x)
template <typename E, int MT, int J, bool EXT>
__global__ __launch_bounds__(512) void tiled_gemm_kernel(FewRows f, TiledGemm<E> p) {
    constexpr int U = FEW_LOADS, EP = 16 / sizeof(E), PIECES = 4 * U, RPL = 64 / PIECES;       // numbers of a piece (16 bytes), pieces and rows of a load
    typedef E piece_t __attribute__((ext_vector_type(EP)));
    if (!EXT) { p.rows.id = nullptr; p.x_blocks = nullptr; p.col_scale = nullptr; p.pair = 0; }
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int a = lane >> 4, b = lane & 15, kw = 1 << f.kw_log2;
    const int part = wave & (kw - 1), cg = wave >> f.kw_log2;
    const int n0 = (blockIdx.x * f.cw + cg) * 16 * J, rb = blockIdx.y;
    const int z = p.slabs > 1 ? blockIdx.z : 0;
    int g = p.slabs > 1 ? 0 : blockIdx.z;
    const int loads = (unsigned)p.k / (4 * EP);
    const bool live = n0 < p.n;
    const int s0 = min(((z << f.kw_log2) + part) * f.chunk, loads), s1 = live ? min(s0 + f.chunk, loads) : 0;
    // the rows that this lane copies, in pieces from p.x; places without a row repeat the last one
    typedef std::conditional_t<EXT, uint64_t, uint32_t> place_t;        // (a cache may be larger than 2^32 pieces)
    place_t at[MT * U];
    const int row_in = lane / PIECES;
    int id = 0;
    if (EXT && p.rows.id) {
        const int first = rb * 16 * MT, total = *p.rows.total;
        id = p.rows.id[first + (lane & (16 * MT - 1))];
        g = p.rows.group[rb];
        if (first >= total) return;
        const int row = (int)((unsigned)min(id, p.m - 1) / (unsigned)p.rows.div);
#pragma unroll
        for (int l = 0; l < MT * U; l++) at[l] = (place_t)__shfl(row, l * RPL + row_in) * f.ldx16;
    } else if (EXT && p.x_blocks) {
#pragma unroll
        for (int l = 0; l < MT * U; l++) {
            const int r = min(rb * 16 * MT + l * RPL + row_in, p.m - 1);
            at[l] = (place_t)(p.x_blocks[r >> 4] * (p.x_block_elems / EP) + (r & 15));
        }
    } else {
#pragma unroll
        for (int l = 0; l < MT * U; l++) at[l] = (place_t)min(rb * 16 * MT + l * RPL + row_in, p.m - 1) * f.ldx16 + (place_t)g * (place_t)(p.x_group / EP);
    }
    const int spread = EXT && p.x_blocks ? 4 : 0;               // (log2 of the pieces between a row's pieces)
    const bool halves = PAIRED<E> && J == 2 && EXT && p.pair;
    const int tile0 = !live ? 0 : halves ? n0 >> 5 : n0 >> 4;
    const unsigned char* wt = reinterpret_cast<const unsigned char*>(p.w) + ((long)g * (p.n >> 4) + tile0) * loads * 1024 + lane * 16;
    const long next_tile = (long)(halves ? p.pair : 1) * loads * 1024;
    // (past the last column of more than two tiles: the last once more)
    auto tile = [&](int j) { return (J > 2 ? min(j, (p.n >> 4) - 1 - tile0) : j) * next_tile; };
    const int buffer = f.rows * PIECES * 16, region = max(2 * buffer, MT * J * 1024);
    unsigned char* const rows_buf = smem + wave * region;
    piece_t bw[2][U][J];
    auto load = [&](piece_t (&bq)[U][J], int buf, int s) {
#pragma unroll
        for (int l = 0; l < MT * U; l++)
            if (l * RPL < f.rows) {
                const int piece = min(4 * s + ((lane & (PIECES - 1)) ^ ((l * RPL + row_in) & 7)), 4 * s1 - 1);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p.x + (uint64_t)(at[l] + ((place_t)piece << spread)) * EP),
                                                 (__attribute__((address_space(3))) void*)(rows_buf + buf * buffer + l * 1024), 16, 0, 0);
            }
        // (rows ahead of weights: the wait of mul counts the latter)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < J; j++) bq[u][j] = __builtin_nontemporal_load(reinterpret_cast<const piece_t*>(wt + tile(j) + (long)min(s + u, s1 - 1) * 1024));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // The part's loads are taken from a chunk of its own on, in a circle.  Where K is a multiple of a high power of two all waves' weights begin at the same
    // address modulo that power, and waves that go on in step ask the same few channels of the memory (µs from the first chunk on → so:
    // 8 × 4096 × 8192 16.1 → 12.9, 8 × 8192 × 4096 16.4 → 14.2, 1 × 2048 × 16384 in four slabs 16.1 → 14.3; K that are no such multiple ± 1 %).
    const int len = s1 - s0, chunks = len > 0 && len % U == 0 ? len / U : 1;
    const int turn = ((blockIdx.x * f.cw + cg + part + z) & ((chunks & -chunks) - 1)) * U;
    auto place = [&](int i) { i += turn; return s0 + (i < len ? i : i - len); };
    if (len > 0) load(bw[0], 0, place(0));
    const GemmSection first = gemm_section(p, n0);
    floatx4 bias[J], acc[MT][J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        bias[j] = (floatx4){0.f, 0.f, 0.f, 0.f};
        if (p.bias && live) bias[j] = *reinterpret_cast<const floatx4*>(p.bias + (long)g * p.n + (J > 2 ? min(n0 + 16 * j, p.n - 16) : n0 + 16 * j) + 4 * a);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[mt][j] = (floatx4){0.f, 0.f, 0.f, 0.f};
    }
    int my_row[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) my_row[mt] = min(16 * mt + b, f.rows - 1);
    // multiplies a chunk of `steps` loads (0: all U); its rows have landed when at most `later` loads, the weights of the chunk behind it, are under way
    auto mul = [&](piece_t (&bq)[U][J], int buf, auto later, int steps) {
        constexpr int vm = decltype(later)::value;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt((vm & 15) | 0xF70 | (vm >> 4) << 14);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (vm == 0 && u >= steps) break;
            piece_t x[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                x[mt] = *reinterpret_cast<const piece_t*>(rows_buf + buf * buffer + (my_row[mt] * PIECES + ((4 * u + a) ^ (my_row[mt] & 7))) * 16);
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[mt][j] = Frag<E>::mma(bq[u][j], x[mt], acc[mt][j]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");              // (the buffer is read before it is written again)
    };
    typedef std::integral_constant<int, U * J> behind;
    typedef std::integral_constant<int, 0> last;
    // 32 bits: sums of 128 products, then sums of those (relative error at K = 2048 / 8736: 2.1 / 2.2e-7, parts summed whole 2.9 / 3.8e-7; no slower)
    constexpr bool F32 = sizeof(E) == 4;
    floatx4 sums[F32 ? MT : 1][F32 ? J : 1] = {};
    if (len > 0) {
        int i = 0;
        for (; i + 2 * U < len; i += 2 * U) {
            load(bw[1], 1, place(i + U));
            mul(bw[0], 0, behind{}, U);
            load(bw[0], 0, place(i + 2 * U));
            mul(bw[1], 1, behind{}, U);
            if constexpr (F32)
#pragma unroll
                for (int t = 0; t < MT * J; t++) {
                    sums[t / J][t % J] += acc[t / J][t % J];
                    acc[t / J][t % J] = (floatx4){0.f, 0.f, 0.f, 0.f};
                }
        }
        if (i + U < len) {
            load(bw[1], 1, place(i + U));
            mul(bw[0], 0, behind{}, U);
            mul(bw[1], 1, last{}, len - i - U);
        } else {
            mul(bw[0], 0, last{}, len - i);
        }
        if constexpr (F32)
#pragma unroll
            for (int t = 0; t < MT * J; t++) acc[t / J][t % J] += sums[t / J][t % J];
    }
    // the parts' sums, in their order, through the waves' regions (their rows are used up); tile t of a column group is finished by part t mod kw.
    // The weights are the first operand: a lane holds four neighbouring columns of one row.
    floatx4* const red = reinterpret_cast<floatx4*>(rows_buf);
#pragma unroll
    for (int t = 0; t < MT * J; t++) red[t * 64 + lane] = acc[t / J][t % J];
    if (kw > 1) __syncthreads();
    if (!live) return;
    auto summed = [&](int t) {
        const unsigned char* v = smem + (size_t)cg * kw * region + (t * 64 + lane) * 16;
        floatx4 sum = *reinterpret_cast<const floatx4*>(v);
#pragma unroll 1
        for (int q = 1; q < kw; q++) sum += *reinterpret_cast<const floatx4*>(v += region);
        return sum;
    };
    if (p.slabs > 1) p.out_f32 += z * p.slab_stride;
    const bool gated = EXT && J == 2 && gemm_gated_act(first.act);
    const bool vec = p.n_store % 4 == 0 && p.ldo % 4 == 0 && p.out_group % 4 == 0 && p.ld_col_scale % 4 == 0 && ((uintptr_t)p.out & 7) == 0 && ((uintptr_t)p.out_f32 & 15) == 0;
    const int tiles = gated ? J : 1;
#pragma unroll 1
    for (int t = part * tiles; t < MT * J; t += kw * tiles) {
        const int mt = t / J, j = t % J;
        const GemmSection sec = J > 2 ? gemm_section(p, min(n0 + 16 * j, p.n - 1)) : first;       // (sections begin at whole 32s)
        floatx4 v = bias[0];
#pragma unroll
        for (int i = 1; i < J; i++) v = j == i ? bias[i] : v;
        v += summed(t) * sec.mul;
        int col = n0 + 16 * j + 4 * a, row = (rb * MT + mt) * 16 + b;
        if (EXT && p.rows.id) row = __shfl(id, 16 * mt + b);
        if (row >= p.m) row = -1;
        if (gated) {
            const floatx4 up = summed(t + J - 1) * sec.mul + bias[J - 1];
            gemm_glu<E, 4>(sec, sec.act, v, up);
            col = gemm_gated_col(sec, col);
        } else gemm_act<E, EXT, 4>(sec, sec.act, v);
        if (row < 0) continue;
        if (!vec) {
#pragma unroll 1
            for (int r = 0; r < 4; r++)
                if (gated || col + r < p.n_store) gemm_store(p, g, row, col + r, r == 0 ? v[0] : r == 1 ? v[1] : r == 2 ? v[2] : v[3]);
            continue;
        }
        if (!gated && col >= p.n_store) continue;
        if (p.row_scale) v *= (float)p.row_scale[row * p.ld_scale + g];
        typedef typename Frag<E>::v4 v4;
        if (p.col_scale) {
            const v4 c = *reinterpret_cast<const v4*>(p.col_scale + p.col_scale_row[row] * p.ld_col_scale + col);
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] *= (float)c[r];
        }
        const long o = row * p.ldo + (p.rows.id ? 0 : g * p.out_group) + col;
        if (p.out_f32) *reinterpret_cast<floatx4*>(p.out_f32 + o) = v;
        else {
            v4 y;
#pragma unroll
            for (int r = 0; r < 4; r++) y[r] = (E)v[r];
            *reinterpret_cast<v4*>(p.out + o) = y;
        }
    }
}

// Prompts: 2 × 2 waves hold MI × NJ tiles of 16 × 16 each.  Both operands go through LDS, copied there by the load unit itself:
//  * weights in stages of one k-step, a ring of 2G − 1: one 1-KiB load per fragment, 32 of K, in 32 bits 16;
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
// Rows: what the launch does with its rows besides (RowsAsTheyAre: nothing; QkvRows: the q|k|v of heads of 128 columns, normed, rotated and stored).
struct RowsAsTheyAre {};
template <typename E, int MI, int NJ, int G, int PER_CU, typename Rows>
__global__ __launch_bounds__(256, PER_CU) void tiled_gemm_big_kernel(TiledGemm<E> p, int mtiles, int ntiles, Rows to) {
    typedef BigTile<MI, NJ, G> T;
    typedef typename Frag<E>::v8 v8;
    constexpr bool F32 = sizeof(E) == 4;
    constexpr int EP = 16 / sizeof(E), SK = 4 * EP;                     // elements of 16 bytes, K of a step
    typedef E operand __attribute__((ext_vector_type(EP)));
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
        ap[i] = gemm_row(p, (m0 + r) >> 4, g, piece, r & 15);
    }
#pragma unroll
    for (int i = 0; i < NJ / 2; i++) {
        const int t = min((n0 >> 4) + NJ / 2 * wave + i, ntl - 1);
        bp[i] = p.w + ((long)g * ntl + (p.pair ? (t >> 1) + (t & 1) * p.pair : t)) * n * (64 * EP) + lane * EP;
    }
    const int xs = 2 * gemm_row_step(p);
    const E* none = reinterpret_cast<const E*>(zero_fragment) + lane * EP;       // (past the end of K)
#define BIG_COPY(src, dst) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src), (__attribute__((address_space(3))) void*)(dst), 16, 0, 0)
    auto issue_rows = [&](int i, int place, bool in) {
        BIG_COPY(in ? ap[i] : none, rows_lds + place * T::GRANULE + (MI * wave + i) * 1024);
        ap[i] += xs;
    };
    auto issue_w = [&](int i, int place, bool in) {
        BIG_COPY(in ? bp[i] : none, w_lds + place * T::STAGE + (NJ / 2 * wave + i) * 1024);
        bp[i] += 64 * EP;
    };
#undef BIG_COPY
    floatx4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = (floatx4){0.f, 0.f, 0.f, 0.f};
    // 32 bits: sums of 128 products, then sums of those, as in the few-row kernel.  Relative error against 64 bits at K = 512 / 2048 / 6144:
    // 2.1 / 2.2 / 2.4e-7, with sums of 512 4.0 / 4.0 / 4.1e-7 and 2 % faster.
    floatx4 sum[F32 ? MI : 1][F32 ? NJ : 1] = {};
    struct Operands { operand x[MI], w[NJ]; };
    constexpr int READS = MI + NJ;
    const unsigned char* my_w = w_lds + wn * NJ * 1024 + lane * 16;
    const unsigned char* my_rows[2];
#pragma unroll
    for (int h = 0; h < 2; h++) my_rows[h] = rows_lds + wm * MI * 2048 + b * 128 + ((4 * h + a) ^ (b & 7)) * 16;
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
            if (q < NJ / 2) issue_w(q, stage, in);
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
        for (int f = 0; f < NJ / 2; f++) issue_w(f, i, i < n);
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
        if (F32 && ((t & 6) == 6 || t + 2 >= n))
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
    if constexpr (std::is_same<Rows, QkvRows>::value) {
        // The tile as fp16, which is what a launch of its own would read, in LDS, whole heads of it; where a row goes is found out once for all heads.  Four tokens of a head a
        // wave and turn, as there.
        constexpr int PITCH = T::COLS + 8, TURNS = T::ROWS / 16;
        static_assert(!F32 && T::COLS % 128 == 0 && (size_t)T::ROWS * (PITCH * 2 + 12) <= T::LDS, "whole heads, and their rows fit the stages");
        _Float16* tile = reinterpret_cast<_Float16*>(smem);
        int *pos_of = reinterpret_cast<int*>(tile + T::ROWS * PITCH), *block_of = pos_of + T::ROWS, *seq_of = block_of + T::ROWS;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) *reinterpret_cast<f16x4*>(tile + ((wm * MI + i) * 16 + b) * PITCH + (wn * NJ + j) * 16 + 4 * a) = __builtin_convertvector(acc[i][j] + 0.f, f16x4);      // (− 0 → 0, as the sum with a bias that is none)
        if ((int)threadIdx.x < T::ROWS) {                                // (whole waves)
            const int tok = min(m0 + (int)threadIdx.x, to.m_total - 1);
            // The last sequence that begins no later than a row's token: of 64 sequences at a time, from the 64 on that hold the tile's first token, one ballot for all rows and a step
            // for each that begins among the wave's (a step for each of all sequences: 8192 × 4096 × 1024 with 512 of them 43 µs longer)
            const uint32_t from = (uint32_t)min(m0 + wave * 64, to.m_total - 1), upto = (uint32_t)min(m0 + wave * 64 + 63, to.m_total - 1);
            int seq = 0, s0 = 0;
            if (to.num_seqs > 64) s0 = 64 * (63 - __clzll((long long)__ballot(lane * 64 < to.num_seqs && to.cu[min(lane * 64, to.num_seqs - 1)] <= from)));
            for (; s0 < to.num_seqs; s0 += 64) {
                const uint32_t first = s0 + lane < to.num_seqs ? to.cu[s0 + lane] : 0xffffffffu;
                const unsigned long long before = __ballot(first <= from), among = __ballot(first <= upto);
                if (before) seq = s0 + 63 - __clzll((long long)before);
                for (unsigned long long rest = among & ~before; rest; rest &= rest - 1) {
                    const int j = __builtin_ctzll(rest);
                    if (__builtin_amdgcn_readlane((int)first, j) <= tok) seq = s0 + j;
                }
                if (among != ~0ull) break;
            }
            const int pos = (int)to.pos_offsets[seq] + (tok - (int)to.cu[seq]);
            pos_of[threadIdx.x] = pos;
            seq_of[threadIdx.x] = seq;
            block_of[threadIdx.x] = to.block_tables[(long)seq * to.max_blocks + pos / KV_BLOCK];
        }
        __syncthreads();
        const int row0 = wave * (T::ROWS / 4) + a;                       // a quarter's first row
#pragma unroll 1
        for (int h = 0; h < T::COLS / 128; h++) {
            const int head = n0 / 128 + h;
            if (head >= to.q_heads + 2 * to.kv_heads) break;
            const bool is_q = head < to.q_heads, is_k = !is_q && head < to.q_heads + to.kv_heads;
            const int local = is_q ? head : is_k ? head - to.q_heads : head - to.q_heads - to.kv_heads, mode = is_q || is_k ? to.qk_mode : 0;
            qkv_with_mode(mode, [&](auto m) {
                constexpr int MODE = decltype(m)::value;
                RopeCoef<128> coef[TURNS];
#pragma unroll
                for (int u = 0; u < TURNS; u++) {
                    const long at = (long)pos_of[row0 + 4 * u] * 64;
                    coef[u] = rope_coef16<128>(is_q ? to.q_norm_w : to.k_norm_w, to.cos_t + at, to.sin_t + at, MODE, MODE == 1, MODE != 0, b);
                }
#pragma unroll
                for (int u = 0; u < TURNS; u++) {
                    const int r = row0 + 4 * u, r0 = __builtin_amdgcn_readfirstlane(r), tok = m0 + r;
                    const RopeRow<128> rr = rope_row16<128>(rope_source16<128>(reinterpret_cast<const __half*>(tile + r * PITCH + h * 128), MODE, b), coef[u], MODE, to.eps, b);
                    const int pos = pos_of[r];
                    const bool quad = m0 + r0 + 3 < to.m_total && seq_of[r0] == seq_of[r0 + 3] && __builtin_amdgcn_readfirstlane(pos) % 4 == 0;
                    qkv_store_row<128>(rr, to, is_q, is_k, local, tok, pos, block_of[r], tok < to.m_total, quad, b, a);
                }
            });
        }
        return;
    }
    // Where the whole launch is one gated section, a row takes half as many lanes, none of them idle: an
    // expert model's up-projections 286 → 272 µs a launch.
    constexpr int LD = 16 * NJ + 4;
    float* lf = reinterpret_cast<float*>(smem) + wave * 32 * LD;
    const bool pairs = p.nsec == 1 && p.sec[0].begin == 0 && gemm_gated_act(p.sec[0].act);
    const int lanes = pairs ? NJ : 2 * NJ, place = lane & (lanes - 1), row_in = lane >> __builtin_ctz(lanes), rounds = lanes / 2;      // (rounds of 64 / lanes rows)
    const int cl = pairs ? (place >> 1) * 32 + (place & 1) * 8 : place * 8, col = n0 + wn * 16 * NJ + cl;
    const GemmSection sec = gemm_section(p, min(col, p.n - 1));
    const bool gated = gemm_gated_act(sec.act), vec = p.n_store % 8 == 0 && p.ldo % 8 == 0 && p.out_group % 8 == 0 && ((uintptr_t)p.out & 15) == 0 && ((uintptr_t)p.out_f32 & 15) == 0;
    const bool active = gated ? col < p.n && !(col & 16) : col < p.n_store;
    const int oc = gated ? gemm_gated_col(sec, col) : col;
    floatx8 bias = {}, bias_up = {};
    if (p.bias && active) {
        bias = *reinterpret_cast<const floatx8*>(p.bias + (long)g * p.n + col);
        if (gated) bias_up = *reinterpret_cast<const floatx8*>(p.bias + (long)g * p.n + col + 16);
    }
    // (here and not at the first use in a loop: there the wait would be for the stores of the round before, too)
    asm volatile("" : "+v"(bias), "+v"(bias_up));
    // A wave's columns are of one kind unless a section begins within them: then the kind is a scalar, chosen ahead of the rounds, and a round is
    // without branches.  With a chain of them for each of the 8 numbers, ids from memory and waits for stores a tile of 128 × 256 took 8 – 9 µs from its
    // last product to its last store, as long as half of a K of 1024; now 4 – 5, of which 0.6 are the stores' (µs of a launch, plain | bias and sigmoid
    // | SiLU-gated: 4096 × 6144 × 2048 96 | 121 | 99 → 93 | 95 | 91, 2048 × 6144 × 1024 38 | 53 | 42 → 35 | 37 | 34).  Stores from the registers, without LDS
    // but 64 bytes of a row at a time: 8192 × 16384 × 2048 536 µs, and 474 this way.
    const int act = __builtin_amdgcn_readfirstlane(sec.act);
    const bool one_kind = vec && __all(sec.act == act) && !p.row_scale && !p.col_scale;
    const long base = (p.rows.id ? 0 : g * p.out_group) + oc;
    const uint32_t ldo = (uint32_t)p.ldo;
    const int round_rows = 32 / rounds;
    const float* from = lf + row_in * LD + cl;
#pragma unroll 1
    for (int ch = 0; ch < MI / 2; ch++) {
        // the output rows of these, one a lane, −1: none; ids in memory would be a wait for every round
        const int own_row = gemm_out_row(p, m0 + (wm * MI + 2 * ch) * 16 + (lane & 31));
#pragma unroll
        for (int c = 0; c < MI / 2; c++)
            if (c == ch)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) *reinterpret_cast<floatx4*>(lf + (i * 16 + b) * LD + j * 16 + 4 * a) = acc[2 * c + i][j];
        auto round = [&](auto glu, auto f32, auto finish) {
            constexpr bool GLU = decltype(glu)::value, F32_OUT = decltype(f32)::value;
            floatx4 next[GLU ? 4 : 2];
            int next_row;
            auto fetch = [&](int q) {
                const floatx4* at = reinterpret_cast<const floatx4*>(from + q * round_rows * LD);
                next[0] = at[0]; next[1] = at[1];
                if constexpr (GLU) { next[2] = at[4]; next[3] = at[5]; }
                next_row = __shfl(own_row, q * round_rows + row_in);
            };
            fetch(0);
#pragma unroll 1
            for (int q = 0; q < rounds; q++) {
                const int row = next_row;
                floatx8 v, up;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    v[e] = next[e >> 2][e & 3] * sec.mul + bias[e];
                    if constexpr (GLU) up[e] = next[2 + (e >> 2)][e & 3] * sec.mul + bias_up[e];
                }
                fetch(min(q + 1, rounds - 1));
                finish(v, up);
                if (row >= 0 && active) {
                    const uint64_t o = (uint64_t)(uint32_t)row * ldo + base;
                    if constexpr (F32_OUT) *reinterpret_cast<floatx8*>(p.out_f32 + o) = v;
                    else *reinterpret_cast<v8*>(p.out + o) = __builtin_convertvector(v, v8);
                }
            }
        };
        typedef std::true_type yes;
        typedef std::false_type no;
#define KIND(GLU, ACT) round(GLU{}, no{}, [&](floatx8& v, const floatx8& up) { if constexpr (GLU::value) gemm_glu<E, 8>(sec, ACT, v, up); else gemm_act<E, true, 8>(sec, ACT, v); })
        if (one_kind && p.out_f32 && act == GEMM_ACT_NONE) round(no{}, yes{}, [](floatx8&, const floatx8&) {});
        else if (one_kind && p.out && act == GEMM_ACT_NONE) KIND(no, GEMM_ACT_NONE);
        else if (one_kind && p.out && act == GEMM_ACT_SILU_GLU) KIND(yes, GEMM_ACT_SILU_GLU);
        else if (one_kind && p.out && act == GEMM_ACT_GELU_GLU) KIND(yes, GEMM_ACT_GELU_GLU);
        else if (one_kind && p.out && act == GEMM_ACT_CLAMPED_GLU) KIND(yes, GEMM_ACT_CLAMPED_GLU);
        else if (one_kind && p.out && act == GEMM_ACT_SIGMOID) KIND(no, GEMM_ACT_SIGMOID);
        else if (one_kind && p.out && act == GEMM_ACT_GELU_TANH) KIND(no, GEMM_ACT_GELU_TANH);
        else if (one_kind && p.out && act == GEMM_ACT_XIELU) KIND(no, GEMM_ACT_XIELU);
        else if (one_kind && p.out && act == GEMM_ACT_RELU2) KIND(no, GEMM_ACT_RELU2);
        else if (one_kind && p.out && act == GEMM_ACT_SILU) KIND(no, GEMM_ACT_SILU);
        else {
            // several kinds, one after the other, factors, and rows or columns that no 16-byte piece begins at
#pragma unroll 1
            for (int q = 0; q < rounds; q++) {
                const int row = __shfl(own_row, q * round_rows + row_in);
                const floatx4* at = reinterpret_cast<const floatx4*>(from + q * round_rows * LD);
                floatx8 v, up = {};
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = at[e >> 2][e & 3] * sec.mul + bias[e];
                if (gated)
#pragma unroll
                    for (int e = 0; e < 8; e++) up[e] = at[4 + (e >> 2)][e & 3] * sec.mul + bias_up[e];
                for (uint64_t todo = __ballot(true); todo;) {
                    const int kind = __builtin_amdgcn_readlane(sec.act, __builtin_ctzll(todo));
                    const bool mine = sec.act == kind;
                    if (mine) {
                        if (gemm_gated_act(kind)) gemm_glu<E, 8>(sec, kind, v, up);
                        else gemm_act<E, true, 8>(sec, kind, v);
                    }
                    todo &= ~__ballot(mine);
                }
                if (row < 0 || !active) continue;
                if (!vec) {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (gated || col + e < p.n_store) gemm_store(p, g, row, oc + e, v[e]);
                    continue;
                }
                if (p.row_scale) v *= (float)p.row_scale[row * p.ld_scale + g];
                if (p.col_scale) {
                    const v8 f = *reinterpret_cast<const v8*>(p.col_scale + p.col_scale_row[row] * p.ld_col_scale + oc);
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] *= (float)f[e];
                }
                const uint64_t o = (uint64_t)(uint32_t)row * ldo + base;
                if (p.out_f32) *reinterpret_cast<floatx8*>(p.out_f32 + o) = v;
                else *reinterpret_cast<v8*>(p.out + o) = __builtin_convertvector(v, v8);
            }
        }
#undef KIND
    }
}

template <typename E, int MI, int NJ, int G, int PER_CU, typename Rows = RowsAsTheyAre>
static int launch_big(const TiledGemm<E>& g, hipStream_t s, const Rows& to = {}) {
    typedef BigTile<MI, NJ, G> T;
    static bool attr = false;
    if (!attr) {
        FH_CHECK_HIP(hipFuncSetAttribute((const void*)tiled_gemm_big_kernel<E, MI, NJ, G, PER_CU, Rows>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)T::LDS));
        attr = true;
    }
    const int mtiles = g.rows.id ? g.rows.max_blocks * (g.rows.block / T::ROWS) : cdiv(g.m, T::ROWS), ntiles = cdiv(g.n, T::COLS);
    form_hit(g.rows.id ? FORM_TILED_GEMM_GROUPED_BIG : FORM_TILED_GEMM_BIG);
    form_hit(T::ROWS == 64 ? FORM_TILED_GEMM_64X64 : T::COLS == 256 ? FORM_TILED_GEMM_128X256 : T::COLS == 128 ? FORM_TILED_GEMM_128X128 : FORM_TILED_GEMM_128X64);
    hipLaunchKernelGGL((tiled_gemm_big_kernel<E, MI, NJ, G, PER_CU, Rows>), dim3(mtiles * ntiles, 1, g.groups), dim3(256), T::LDS, s, g, mtiles, ntiles, to);
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
//   few rows → 64 × 64        128: 253 × 2048 × 2048   9.0 → 14.3     192: 128 × 6144 × 2048   14.5 → 15.1, 65 × 6144 × 4096   27.1 → 26.0
//                             224: 400 × 2048 × 1024   8.9 → 8.8      256: 65 × 8192 × 4096   30.3 → 28.6      288: 192 × 6144 × 2048   24.1 → 17.2
// 256 × 256 (tiled_gemm_wide.hip): a round of 256 tiles, one per CU, takes 11.6 µs + K · 0.0201, a round of 256 of 128 × 256, of which two share a CU, 5.5 + K · 0.01185.
// 150 shapes, 500 – 8192 rows × 1024 – 16384 × 512 – 4096, µs of the latter (rounds) | of the former (rounds):
//   2001 × 8192 × 1024  35.6 (2) | 34.3 (1)     3500 × 8192 × 2048    110 (4) | 100 (2)      8192 × 10240 × 4096  539 (10) | 463 (5)
//   4096 × 4096 × 4096   112 (2) | 98.8 (1)     4096 × 10240 × 2048   148 (5) | 146 (3)      7000 × 8192 × 1024   109 (7) | 111 (4)
//   3000 × 8192 × 4096   164 (3) | 173 (2)      4096 × 6144 × 1024    57 (3) | 67 (2)        5000 × 3072 × 512    22.9 (2) | 23.4 (1)
// so wherever its rounds are half as many as the other's, but for short K: up to 1024 not in two or three rounds, which save the launch 3 µs and cost its neighbours, whose
// clock falls, more (four layers of 1024 columns, ms of a prompt in 128 × 256 | in these: one of 2300 tokens 0.89 | 0.87, of 7000 2.41 | 2.49, of 8192 2.78 | 2.89, 64 of 256
// 3.05 | 2.85).
// A wave with columns of several kinds, or rare ones, finishes its tile 20 – 26 µs later, which four rounds make up for (K = 2048, µs of the latter | of the former: 9472 columns
// with several sections, 1000 rows 55 | 75, 3000 108 | 125, 5000 163 | 176, 8192 281 | 277, 12000 380 | 372; 20224 columns, 600 rows 62 | 75, 3000 219 | 209, 8192 563 | 485).
static long big_tiles(const GemmRows& rows, int m, int n, int groups, int r, int c) { return (long)(rows.id ? rows.max_blocks * (rows.block / r) : cdiv(m, r)) * cdiv(n, c) * groups; }
// rounds of 128 × 256 and of 256 × 256, and the time of either
struct BigRounds { long halves, wholes; float half_us, whole_us; };
template <typename E>
static BigRounds big_rounds(const TiledGemm<E>& g) {
    const long halves = cdiv(big_tiles(g.rows, g.m, g.n, g.groups, 128, 256), 256), wholes = cdiv(big_tiles(g.rows, g.m, g.n, g.groups, 256, 256), 256);
    return {halves, wholes, halves * (5.5f + 0.01185f * g.k), wholes * (11.6f + 0.0201f * g.k)};
}
template <typename E>
bool tiled_gemm_takes_256(const TiledGemm<E>& g) {
    if constexpr (sizeof(E) == 4) {
        return false;
    } else {
        if (knobs().tiled_256 < 0 || (g.rows.id && g.rows.block % 256)) return false;
        if (knobs().tiled_256 == 0) {
            if (knobs().tiled_wide_min_tiles >= 0) return false;        // (a forced size of the tiles below stays what it is)
            const BigRounds r = big_rounds(g);
            bool mixed = false;
            for (int i = 0; i < g.nsec; i++) mixed |= gemm_rare_act(g.sec[i].act) || g.sec[i].begin % 128;
            if (r.halves <= 1 || (mixed && r.wholes < 4) || (g.k <= 1024 && (r.wholes == 2 || r.wholes == 3)) || r.whole_us >= (g.k > 512 ? 0.97f : 0.93f) * r.half_us) return false;
        }
        return tiled_gemm_wide_supports(g);
    }
}
template <typename E>
static int launch_big(const TiledGemm<E>& g, hipStream_t s) {
    auto tiles = [&](int r, int c) { return big_tiles(g.rows, g.m, g.n, g.groups, r, c); };
    if constexpr (sizeof(E) == 4) {
        // 32 bits: bound by the products alone, so the tile whose rounds over the CUs take least (µs of a round below, K = 2048):
        //                        128 × 128   128 × 64   64 × 64   few-row kernel
        //   2048 × 2048 × 2048      142         147
        //   1000 × 6144 × 2048      266         215
        //   1000 × 2048 × 2048      140          83
        //   500 × 2048 × 2048       139                    50
        //   1000 × 1024 × 512        41                    17
        //   128 × 8192 × 2048       139                    47         47
        //   253 × 2048 × 2048       138                    46         25      (128 tiles of 64 × 64: too few)
        //   128 × 6144 × 2048                              47         45      (192)
        const long full = cdiv(tiles(128, 128), 256) * 133L, half = cdiv(tiles(128, 64), 256) * 72L, small = cdiv(tiles(64, 64), 256) * 42L;
        if ((g.rows.id && g.rows.block < 128) || small < std::min(full, half)) return launch_big<E, 2, 2, 3, 3>(g, s);
        return half < full ? launch_big<E, 4, 2, 3, 2>(g, s) : launch_big<E, 4, 4, 2, 2>(g, s);
    } else {
        if (tiled_gemm_takes_256(g)) return tiled_gemm_wide(g, s);
        if (tiles(128, 256) >= (knobs().tiled_wide_min_tiles >= 0 ? knobs().tiled_wide_min_tiles : 257)) return launch_big<E, 4, 8, 2, 2>(g, s);
        if (tiles(128, 128) > knobs().tiled_half_max_tiles) return launch_big<E, 4, 4, 2, 2>(g, s);
        return tiles(64, 64) > knobs().tiled_small_max_tiles ? launch_big<E, 4, 2, 3, 2>(g, s) : launch_big<E, 2, 2, 3, 3>(g, s);
    }
}

// The rows of a q|k|v projection by its own launch: 5.7 µs more of it at 2048 × 4096 × 1024 (23.8 → 29.5) for a launch of 11.7 that reads and writes them once more.  From a
// tile of 128 × 128 for each CU on; µs of a prompt through 14 layers, launch of its own | this: 488 tokens (128 tiles) 1087 | 1149, 700 (192) 1566 | 1570, 986 (256) 1433 | 1408,
// 1500 (384) 1998 | 1936, 2048 (512) 2034 | 1941, 4096 4146 | 4009, 8192 5932 | 5572.
// Where the projection alone would run in tiles of 256 × 256, only if these are faster by less than what the launch saves, 0.65 µs for a million numbers.  µs that a layer takes
// longer with this (four layers of it, 128 tokens a sequence and more):
//   tiles of 256 × 256:    K = 1024, 4096 columns   3000 tokens − 3, 4096 − 8            2048, 4096    3000 + 0, 4096 − 7, 8192 − 10     2048, 5120    2048 + 2, 3000 − 3
//                             3072, 5120            2048 + 10, 3000 + 5                  4096, 6144    1400 + 10, 2048 + 13, 8192 + 6
//   smaller ones:             1024, 4096            1024 − 2, 2048 − 6, 8192 − 26        2048, 5120    1024 − 3, 4096 − 8, 8192 − 28
//                             3072, 5120            1024 − 5, 4096 − 6, 8192 − 37        4096, 6144    700 − 3, 3000 − 10, 4096 − 17
bool tiled_gemm_qkv_supports(const TiledGemm<_Float16>& g, const QkvRows& to) {
    if (big_tiles(g.rows, g.m, g.n, 1, 128, 128) < knobs().qkv_min_tiles || g.m != to.m_total || g.n != (to.q_heads + 2 * to.kv_heads) * 128 || g.bias || g.nsec) return false;
    const BigRounds r = big_rounds(g);
    return !tiled_gemm_takes_256(g) || r.half_us - r.whole_us + 2.f <= 0.65e-6f * g.m * g.n;
}
int tiled_gemm_qkv(const TiledGemm<_Float16>& g, const QkvRows& to, hipStream_t s) {
    FH_REQUIRE(tiled_gemm_qkv_supports(g, to), "tiled_gemm_qkv: %d rows of %d + 2 × %d heads", g.m, to.q_heads, to.kv_heads);
    form_hit(FORM_F16_QKV);
    return big_tiles(g.rows, g.m, g.n, 1, 128, 256) >= (knobs().tiled_wide_min_tiles >= 0 ? knobs().tiled_wide_min_tiles : 257) ? launch_big<_Float16, 4, 8, 2, 2>(g, s, to) : launch_big<_Float16, 4, 4, 2, 2>(g, s, to);
}

int tiled_gemm_slabs(int m, int n, int k) {
    if (m > 64) return 1;
    // Narrow outputs: slabs until 32 columns of one of them for each CU, 1024 of K in two.  µs of the launch and the norm that sums its slabs, bf16, one slab | two |
    // four | eight:
    //   1 × 1024 × 4096    7.7 |  6.9 |  6.3 |  7.3      8 × 1536 × 4096    9.3 |  8.3 |  8.1 | 10.4      64 × 1024 × 2048    7.4 |  7.3 |  7.7 |  9.4
    //   8 × 2048 × 8192   12.9 | 10.9 | 10.9 | 12.2     16 × 2048 × 12288  20.5 | 14.6 | 14.1 | 16.4      64 × 2048 × 8192   18.4 | 16.9 | 14.9 | 17.2
    //   1 × 2048 × 1024    5.9 |  6.0 |  6.0 |  7.1      8 × 3072 × 4096   10.1 | 10.3 | 10.0 | 11.5      32 × 4096 × 4096   14.0 | 13.3 | 13.9 | 17.4
    int S = 1;
    while (S < GEMM_MAX_SLABS && (n / 32) * S < 256 && k >= 1024 * S) S *= 2;
    return S;
}

template <typename E, int MT, int J, bool EXT>
static int launch_small(const TiledGemm<E>& g, dim3 grid, int nw, int kw, hipStream_t s) {
    FewRows f;
    f.kw_log2 = kw >= 8 ? 3 : kw >= 4 ? 2 : kw >= 2 ? 1 : 0;
    f.cw = nw >> f.kw_log2;
    f.rows = g.rows.id ? 16 * MT : std::min(16 * MT, (g.m + 3) / 4 * 4);
    f.chunk = cdiv(g.k / (64 / (int)sizeof(E)), g.slabs << f.kw_log2);
    f.ldx16 = (uint32_t)(g.ldx * sizeof(E) / 16);
    const size_t lds = (size_t)nw * std::max(2 * f.rows * 64 * FEW_LOADS, MT * J * 1024);
    if (lds > 64 * 1024) {
        static bool attr = false;
        if (!attr) {
            FH_CHECK_HIP(hipFuncSetAttribute((const void*)tiled_gemm_kernel<E, MT, J, EXT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            attr = true;
        }
    }
    hipLaunchKernelGGL((tiled_gemm_kernel<E, MT, J, EXT>), grid, dim3(64 * nw), lds, s, f, g);
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
    FH_REQUIRE(!g.x_blocks || sizeof(E) == 2, "tiled_gemm: rows from a cache are 16-bit");
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
    const bool enough_tiles = tiles >= (knobs().tiled_big_min_tiles >= 0 ? knobs().tiled_big_min_tiles + F32 : F32 ? 129 : 193);
    if (rows.id ? (F32 ? rows.block >= 64 && g.n >= 64 && enough_tiles : rows.block >= 128) : g.m > 64 && g.n >= 64 && g.slabs == 1 && enough_tiles) return launch_big(g, s);
    // Rows of a workgroup: as many as there are, fewer where narrow outputs would leave CUs idle: in 16 bits as long as a round of 256 workgroups
    // holds the launch.
    int mt = rows.id ? rows.block / 16 : g.m <= 16 ? 1 : (g.m <= 32 ? 2 : 4);
    auto row_tiles = [&](int t) { return (long)cdiv(g.m, 16 * t) * (g.n / 16) * g.groups * g.slabs; };
    while (!rows.id && mt > 1 && (F32 ? row_tiles(mt) < knobs().tiled_min_tiles : row_tiles(mt / 2) <= 2 * knobs().tiled_min_tiles)) mt /= 2;
    // Columns of a wave (16 · J), waves of a workgroup, K parts among them; µs, bf16, weights from HBM, inside a graph:
    //                             16 columns of a wave,                     32 columns                a read of the weights
    //                             K in 4     K in 2     8 waves, K in 8     K in 4     8, K in 8      and nothing else
    //   8 × 4096 × 1024            3.84       4.3        4.25                4.6                       2.7
    //   8 × 1024 × 3072            5.35                  5.28                6.7        6.9            2.5
    //   3 × 128 × 8128             8.88                  7.53               12.0       11.9            2.0
    //   8 × 6144 × 1024            4.83       4.58       4.90                4.79                      3.7
    //   7 × 6528 × 6912           17.3       18.8                           16.4       16.9           14.8
    //   8 × 2048 × 7680, 4 slabs   7.74       7.68       7.94                7.86       8.03
    //   8 × 2048 × 8192, 4 slabs   7.74       8.12       8.04                7.98       8.20           6.5
    //   8 × 2048 × 9216, 4 slabs   8.54       8.49       9.57                8.70       9.43
    //   8 × 4096 × 3072, 2 slabs   6.59       6.52       7.15                6.84       7.13
    //   8 × 4096 × 4096, 2 slabs   7.72       9.40       8.16                8.10       8.35
    //   8 × 5120 × 1024            4.74       4.88       5.21                4.61       4.83
    //   8 × 5120 × 1536            5.99       5.67       6.43                5.56       6.02
    //   16 × 6144 × 2048           7.96       7.95       8.31                7.50       7.62
    //   8 × 8192 × 2048            7.83       7.84       8.29                8.21       8.27
    //   8 × 8192 × 3072           10.29      10.32      10.58               10.75      10.77
    //   16 × 8192 × 3072          11.46      11.64      11.76               11.18      11.49
    //   8 × 8192 × 5120           15.34      15.79      15.75               15.90      16.12
    //   8 × 12288 × 1024           6.35       6.70       6.65                                          5.3
    //   1 × 10240 × 2048           9.34       9.39       8.93               10.3                       7.8
    //   8 × 20032 × 2048          15.4                  14.97               16.3       15.7           13.6
    //   32 × 4608 × 2048           9.0        8.6       10.6                 7.42       7.60           4.8
    //   32 × 2048 × 2048, 4 slabs  4.87       4.50                           4.79       5.12           2.7
    //   60 × 8192 × 2048                     12.5                           10.6                       6.5
    //   43 × 9600 × 1920          18.0                                      16.5 (K in 2: 14.1)        7.3
    // One row tile: 16 columns, since a wave then has half as much under way before its first sum; K in four up to a round of 256 workgroups
    // and past two, in two between, where that saves a round, until parts of a half get too long: 32 columns in four parts save the round too, and take
    // over at 48 loads of a wave with all of K where the second round is less than three quarters full, at 80 where it is fuller, at 64 of a
    // slab's; eight waves where a wave of four would read 16 loads and more.  Several row tiles: their rows are read again for every column group, so 32 columns
    // past one round.  Four row tiles leave room for one workgroup per CU, two with 64 columns for two: the parts that make rounds / parts least.
    // A vocabulary, many rounds of workgroups (those of 17 – 32 rows on more than 139000 columns do not come here: f16t_gemm): the rows' share grows with rows
    // and K, so wider blocks; eight waves, each with whole chunks, else four.  µs:
    //                             16 columns, 8 waves   32 columns, 8 waves   32 columns, 4 waves   64 columns, K in parts by the rule
    //   8 × 128256 × 4096             154                    156                   167
    //   12 × 128256 × 4096            167                    159                   173
    //   12 × 151936 × 2048            105                     95                    93
    //   12 × 262208 × 5376            498                    437                   431
    //   16 × 262208 × 5376            554                    463                   448
    //   32 × 49152 × 8192                                    143                   138                   159
    //   24 × 65536 × 2048                                     54                    45                    48
    //   32 × 65536 × 2048                                     56                    47                    48
    //   17 × 98304 × 3072                                    103                    94                    95
    //   32 × 98304 × 3072                                    121                   110                   101
    //   32 × 131072 × 1536                                   104                    84                    74
    //   32 × 131072 × 5376                                   295                   273                   232
    //   64 × 151936 × 1024, 32 columns, K in four parts 97, in one 79; 49 × 16992 × 1376: 20.8 and 19.5
    const int rbs = rows.id ? rows.max_blocks : cdiv(g.m, 16 * mt), zs = rows.id ? 1 : g.groups * g.slabs;
    const int loads = g.k / (F32 ? 16 : 32) / g.slabs;                  // (of a wave that has all of a slab's K)
    const long tiles16 = (long)rbs * (g.n / 16) * zs;
    const bool two_rounds = !rows.id && tiles16 > 256 && tiles16 <= 512;
    const bool ext = rows.id || g.x_blocks || g.col_scale || gated || rare, wide = !rows.id && tiles16 > 2048;
    int J = rows.id ? 2 : mt == 1 ? ((two_rounds && loads >= (tiles16 < 448 ? 48 : g.slabs > 1 ? 64 : 80)) || (wide && (g.m > 12 || (g.m > 8 && loads >= 48) || loads > 128)) ? 2 : 1) : tiles16 <= 256 || (two_rounds && loads <= (g.slabs > 1 ? 32 : 8)) ? 1 : 2;
    // Two row tiles, 32 columns and a little more than a workgroup for each CU: the CUs with two are what the launch waits for, at the 29 bytes a clock that a CU's loads
    // get, half of them the rows once more.  48 columns bring it back to one, then 64, where the rows are many bytes and parts not too long (a step of
    // segetar, 32 rows: 598 → 586 µs, of nerenex in 32 bits 363 → 345).  µs, 16 bits, 32 | 48 | 64 columns:
    //                        K = 1024              2048                  4096                  8192
    //   32 × 8192        6.7 |  7.2 |  7.7     9.1 | 10.2 | 11.0    15.1 | 16.8 | 19.1    25.4 | 29.5 | 35.4
    //   32 × 8224        7.7 |  6.9 |  7.7    12.0 | 10.1 | 11.0    21.4 | 16.7 | 19.1    39.5 | 30.2 | 35.7
    //   20 × 9280        7.8 |  7.3 |  7.8    11.9 |  9.9 | 10.7    20.9 | 16.3 | 18.4    37.2 | 28.2 | 34.5
    //   32 × 12288       8.6 |  8.4 |  8.6    13.2 | 11.9 | 12.3    23.5 | 19.6 | 21.2    43.5 | 34.4 | 41.9
    //   32 × 12320       8.6 | 10.0 |  8.6    13.2 | 16.3 | 12.3    23.5 | 28.9 | 21.1    43.6 | 52.5 | 41.8
    //   32 × 14336       8.8 | 10.6 |  9.2    13.6 | 17.1 | 13.2    24.4 | 30.1 | 22.6    44.5 | 55.6 | 47.1
    //   32 × 16384       9.3 | 10.8 |  9.8    14.5 | 17.3 | 14.5    26.4 | 30.6 | 24.9    46.3 | 57.1 | 53.7
    // Slabs of K gain by 48 columns as one slab does, by 64 nothing; groups, the heads' own short columns, by neither.  32 rows, 32 | 48 | 64 columns:
    //   2112 × 8192 in 4 slabs  10.8 |  9.1 |  9.5     3072, 4  11.6 | 11.2 | 12.1     3584, 4  12.3 | 14.5 | 12.8     5120, 2  18.0 | 15.6 | 17.1     7168, 2  21.0 | 25.1 | 21.4
    //   23 groups of 512 × 128   4.0 |  4.8 |  5.9     24 of 512 × 128  4.4 | 5.3 | 7.0     72 of 128 × 512  6.8 | 6.8 | 6.8     96 of 128 × 512  7.0 | 8.2 | 7.2
    // A short K is over before workgroups are waited for, and what a wave does behind it for three tiles counts (32 | 48 columns):
    //   17 × 8224 × 64   4.4 | 5.7     32 × 9280 × 128  4.3 | 5.1     17 × 12288 × 256  4.8 | 5.0     17 × 8224 × 512  5.0 | 5.3     32 × 9280 × 512  5.8 | 5.6     17 × 8224 × 768  6.3 | 6.1
    if (mt == 2 && !ext && g.groups == 1 && tiles16 > 512 && tiles16 <= 768 && loads > 16) J = 3;
    if (mt == 2 && !ext && zs == 1 && tiles16 > 768 && tiles16 <= 896 && loads >= 64 && loads <= 128) J = 4;
    if (mt == 2 && !ext && tiles16 >= 4096 && loads >= (g.m > 24 ? 48 : 96) && g.n % 64 == 0) J = 4;       // (a vocabulary)
    if (knobs().tiled_j > 0) J = knobs().tiled_j == 1 ? 1 : (knobs().tiled_j == 3 || knobs().tiled_j == 4) && mt == 2 && !ext ? knobs().tiled_j : 2;
    if (gated) J = 2;
    const long cols = cdiv(g.n, 16 * J), blocks = (long)rbs * cols * zs;
    int nw = mt == 1 && !rows.id && ((blocks > 512 && loads >= 64 && (!wide || loads % 32 == 0)) || (blocks <= 256 && J == 1 && loads >= 96)) ? 8 : 4, kw = nw;
    if (J == 1 && two_rounds) kw = 2;
    // Sorted rows, 32 columns: K in as many parts as there are waves, until workgroups are so many that the parts' sums and their waits only add.  µs in
    // 4 | 2 | 1 part, tokens of 8 experts each × columns × K (blocks of 32 columns):
    //   16 rows a block    8 of 8: 4 of 64 × 4096 × 1536 (4096)   54 |  53 |  56       160 of 128 × 4096 × 1536 (26624)  257 | 248 | 249
    //                      in 8:   16 of 24 × 8192 × 4096 (8192) 258 | 246 | 244, 240   48 of 64 × 4096 × 4096 (11264)   341 | 333 | 326, 323
    //   32 rows            16 of 8 × 2048 × 512 (768)            6.8 | 7.0 | 8.6        100 of 64 × 2048 × 512 (5696)   38.5 | 29.3 | 27.0
    //                      200 of 128 × 2048 × 512 (11392)        72 |  56 |  52        200 of 128 × 4096 × 1536 (22784) 273 | 250 | 251
    //                      200 of 64 × 1536 × 2048 (5472)         73 |  88 |  84
    //   64 rows            32 of 8 × 1024 × 2048 (384)          11.1 | 15.1 | 24.3      64 of 24 × 2048 × 2048 (2048)      55 | 48 | 49
    //                      600 of 128 × 4096 × 1536 (25984)      466 | 402 | 373
    if (rows.id && mt == 1 && loads >= 96) nw = kw = 8;
    else if (rows.id) kw = mt == 1 ? (blocks < 20000 ? 4 : 1) : mt == 2 ? (blocks < 4096 ? 4 : 1) : blocks < 512 ? 4 : blocks < 3000 ? 2 : 1;
    else if (mt == 4 && (long)rbs * cdiv(cols, 4) * zs > 128) kw = 1;
    else if (mt == 4 || (J == 4 && tiles16 > 1024))
        for (int k : {2, 1}) {
            const int slots = mt == 4 ? 256 : 512;
            if (cdiv((long)rbs * cdiv(cols, 4 / k) * zs, slots) * kw <= cdiv((long)rbs * cdiv(cols, 4 / kw) * zs, slots) * k) kw = k;
        }
    while (kw > 1 && loads < 2 * kw) kw /= 2;
    auto power_of_two = [](int v) { return v >= 8 ? 8 : v >= 4 ? 4 : v >= 2 ? 2 : 1; };
    if (knobs().tiled_nw > 0) nw = std::min(mt == 4 ? 4 : 8, power_of_two(knobs().tiled_nw));
    if (knobs().tiled_kw > 0 || kw > nw) kw = std::min(nw, power_of_two(knobs().tiled_kw > 0 ? knobs().tiled_kw : kw));
    const dim3 grid(cdiv(cols, nw / kw), rbs, zs);
    form_hit(rows.id ? FORM_TILED_GEMM_GROUPED : FORM_TILED_GEMM);
#define SMALL(J_, EXT_) \
    (mt == 1 ? launch_small<E, 1, J_, EXT_>(g, grid, nw, kw, s) : mt == 2 ? launch_small<E, 2, J_, EXT_>(g, grid, nw, kw, s) : launch_small<E, 4, J_, EXT_>(g, grid, nw, kw, s))
    if (ext) return J == 1 ? SMALL(1, true) : SMALL(2, true);
    if (J == 3) {
        form_hit(FORM_TILED_GEMM_COLS48);
        return launch_small<E, 2, 3, false>(g, grid, nw, kw, s);
    }
    if (J == 4) {
        form_hit(FORM_TILED_GEMM_COLS64);
        return launch_small<E, 2, 4, false>(g, grid, nw, kw, s);
    }
    return J == 1 ? SMALL(1, false) : SMALL(2, false);
#undef SMALL
}
template bool tiled_gemm_takes_256<bf16>(const TiledGemm<bf16>&);
template bool tiled_gemm_takes_256<float>(const TiledGemm<float>&);
template int tiled_gemm<bf16>(const TiledGemm<bf16>&, hipStream_t);
template int tiled_gemm<float>(const TiledGemm<float>&, hipStream_t);
template int tiled_gemm<_Float16>(const TiledGemm<_Float16>&, hipStream_t);

}  // namespace fh
