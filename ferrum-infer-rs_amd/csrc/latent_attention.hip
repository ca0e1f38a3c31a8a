// Attention over a compressed cache (multi-head latent attention): a token caches its normed latent c and a single rotated key
// part that every head uses; head h's key is (W_uk,h c | shared part) and its value W_uv,h c.
//
// One token per sequence and short portions never expand keys or values: the query's plain part arrives already multiplied by W_uk,hᵀ (q_lat), so a score is
// q_lat · c + rot(q) · k_rot, and the output is left in latent space (o_lat = Σ p c) for the value projection that follows.  All heads
// of a token share one cache entry, so a 16-row MFMA tile is 16 (token, head) pairs of one sequence and the cache is read once for them.
//
// Cache tiles are K-fragment shaped ([chunk of 8 dims][16 keys][8]): a wave's K fragment is one contiguous 1-KiB load and feeds the
// matrix pipe directly.  The same registers are parked in LDS and come back transposed (ds_read_b64_tr_b16) as the Vᵀ operand of
// Oᵀ += Vᵀ·Pᵀ — the latent is read from memory once for both products.
//
// Prompt portions of many tokens are compute-bound, and the latent form costs 2·kv_rank + rot per (query, key) where keys and values
// cost dim + rot + vdim: for those the projections of the visible cache blocks are expanded once per layer (a GEMM that reads the
// cache's fragments in place) and a flash kernel runs over them.
#include <math.h>

#include <algorithm>

#include "common.h"
#include "knobs.h"
#include "layer_ops.h"
#include "seq_tiles.h"

namespace fh {

// A row's statistics (maximum m, sum l of e^(score − m)) closed by its head's sink: factor of the row's Σ e^(score − m)·value
template <typename E>
__device__ __forceinline__ float softmax_factor(float m, float l, const float* __restrict__ sink, int h) {
    if (!sink) return l > 0.f ? 1.0f / l : 0.f;
    const float z = sink[h], top = fmaxf(m, z), f = attn_exp<E>(m - top);
    return f / (l * f + attn_exp<E>(z - top));
}

// one wave per token: norm of the query latent, norm of the kv latent, rotation of the shared key part, cache write
template <typename E>
__global__ __launch_bounds__(256) void latent_prepare_kernel(const E* __restrict__ dq, const E* __restrict__ dkv, long ld,
                                                             const float* __restrict__ dq_norm, const float* __restrict__ dkv_norm,
                                                             float eps, LatentDims d, LatentBuffers<E> b, BatchView v, E* __restrict__ cq) {
    typedef typename Frag<E>::v8 v8;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= v.T) return;
    const int seq = v.tok_seq[t];
    const long pos = (long)v.pos[seq] + t - v.cu[seq];
    const E *qr = dq + t * ld, *kr = dkv ? dkv + t * ld : nullptr;
    float sq = 0.f, sk = 0.f;
    for (int i = lane * 8; i < d.qp; i += 512) {
        const v8 x = *reinterpret_cast<const v8*>(qr + i);
#pragma unroll
        for (int j = 0; j < 8; j++) sq += (float)x[j] * (float)x[j];      // (padded columns are zero)
    }
    for (int i = lane * 8; dkv && i < d.kp; i += 512) {
        const v8 x = *reinterpret_cast<const v8*>(kr + i);
#pragma unroll
        for (int j = 0; j < 8; j++) sk += (float)x[j] * (float)x[j];
    }
    const float iq = 1.0f / sqrtf(wave_reduce_sum(sq) / (float)(d.q_rank ? d.q_rank : 1) + eps), ik = 1.0f / sqrtf(wave_reduce_sum(sk) / (float)d.kv_rank + eps);
    for (int i = lane * 8; i < d.qp; i += 512) {
        v8 x = *reinterpret_cast<const v8*>(qr + i);
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = (E)((float)x[j] * iq * dq_norm[i + j]);
        *reinterpret_cast<v8*>(cq + (long)t * d.qp + i) = x;
    }
    if (!dkv) return;                                    // (the layer reads another one's cache)
    E* tile = b.pool + (long)v.bt[(long)seq * v.max_blocks + pos / 16] * 16 * (d.kp + d.rp) + (pos % 16) * 8;
    for (int i = lane * 8; i < d.kp + d.rp; i += 512) {
        v8 x = *reinterpret_cast<const v8*>(kr + i);
        if (i < d.kp) {
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = (E)((float)x[j] * ik * dkv_norm[i + j]);
        } else {
            x = rot_apply(x, rot_load(i - d.kp, d.rot_dims, b.cos_t, b.sin_t, pos));
        }
        *reinterpret_cast<v8*>(tile + i * 16) = x;
    }
    const int clear = slots_to_clear(v, seq, t, pos);
    for (int i = lane; i < clear * (d.kp >> 3); i += 64) *reinterpret_cast<v8*>(tile + (i / clear) * 128 + (i % clear + 1) * 8) = v8{};
}

template <typename E>
int latent_prepare(const E* dq, const E* dkv, long ld, const float* dq_norm, const float* dkv_norm, float eps, const LatentDims& d,
                   const LatentBuffers<E>& b, const BatchView& v, E* cq, hipStream_t s) {
    hipLaunchKernelGGL(latent_prepare_kernel<E>, dim3(cdiv(v.T, 4)), dim3(256), 0, s, dq, dkv, ld, dq_norm, dkv_norm, eps, d, b, v, cq);
    FH_CHECK_LAUNCH();
    return 0;
}

// ── plain form: one workgroup per (token, head), 256 keys at a time; any size, both number formats ──
template <typename E>
__global__ __launch_bounds__(256) void latent_attn_plain_kernel(LatentDims d, LatentBuffers<E> b, BatchView v) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, kd = d.kp + d.rp;
    float *q = lds, *pr = lds + kd, *red = pr + 256, *o = red + 8;         // [kd] query, [256] weights, [8], [kp] output
    const int seq = v.tok_seq[t];
    const int pos = v.pos[seq] + t - v.cu[seq];
    for (int i = tid; i < d.kp; i += 256) { q[i] = (float)b.q_lat[((long)t * d.heads + h) * d.kp + i]; o[i] = 0.f; }
    const E* qr = b.q + (long)t * b.ldq + h * (d.dp + d.rp) + d.dp;
    const int half = d.rot_dims >> 1;
    for (int i = tid; i < d.rp; i += 256) {
        float x = (float)qr[i];
        if (i < d.rot_dims) {
            const float c = b.cos_t[(long)pos * half + i / 2], s = b.sin_t[(long)pos * half + i / 2], y = (float)qr[i ^ 1];
            x = i & 1 ? x * c + y * s : x * c - y * s;
        }
        q[d.kp + i] = x;
    }
    const int lo = max(0, pos + 1 - d.window), hi = pos + 1;
    const int32_t* bt = v.bt + (long)seq * v.max_blocks;
    float m_run = -INFINITY, l_run = 0.f;
    __syncthreads();
    for (int k0 = lo; k0 < hi; k0 += 256) {
        const int key = k0 + tid;
        float sc = -INFINITY;
        if (key < hi) {
            const E* kt = b.pool + (long)bt[key / 16] * 16 * kd + (key % 16) * 8;
            float acc = 0.f;
            for (int i = 0; i < kd; i += 8) {
                const typename Frag<E>::v8 x = *reinterpret_cast<const typename Frag<E>::v8*>(kt + i * 16);
#pragma unroll
                for (int j = 0; j < 8; j++) acc += q[i + j] * (float)x[j];
            }
            sc = acc * d.scale;
        }
        float mx = wave_reduce_max(sc);
        if ((tid & 63) == 0) red[wave] = mx;
        __syncthreads();
        const float m_new = fmaxf(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), m_run);
        const float pv = expf(sc - m_new), alpha = expf(m_run - m_new);       // (key lo is visible: m_new is finite)
        pr[tid] = pv;
        const float ps = wave_reduce_sum(pv);
        if ((tid & 63) == 0) red[4 + wave] = ps;
        __syncthreads();
        l_run = l_run * alpha + red[4] + red[5] + red[6] + red[7];
        m_run = m_new;
        const int n = min(256, hi - k0);
        for (int i = tid; i < d.kp; i += 256) {
            float acc = o[i] * alpha;
            for (int k = 0; k < n; k++) {
                const int kk = k0 + k;
                acc += pr[k] * (float)b.pool[(long)bt[kk / 16] * 16 * kd + ((i >> 3) * 16 + kk % 16) * 8 + (i & 7)];
            }
            o[i] = acc;
        }
        __syncthreads();
    }
    float f = 1.0f / l_run;
    if (b.sink) {
        const float z = b.sink[h], top = fmaxf(m_run, z), e = expf(m_run - top);
        f = e / (l_run * e + expf(z - top));
    }
    for (int i = tid; i < d.kp; i += 256) b.o_lat[((long)t * d.heads + h) * d.kp + i] = (E)(o[i] * f);
}

// ── matrix-core form ──
constexpr int LATENT_PARTIAL_PAD = 4;  // floats behind a partial row's outputs: maximum, sum
// offset of lane's 4 values in a transposed read: lane i of a 16-lane group names 4 dims of key 4a + i / 4 (of a 16-key block, 16 dims =
// two chunks) and receives dim i of keys 4a … 4a + 3
__device__ __forceinline__ int tr_offset(int lane) {
    return ((((lane & 3) >> 1) * 16) + 4 * (lane >> 4) + ((lane & 15) >> 2)) * 8 + (lane & 1) * 4;
}
__device__ __forceinline__ shortx4 read_tr(const bf16* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4*)p);
}

// KS, RS: 32-wide steps of the latent and of the rotated part; MT: 16-row tiles per workgroup (two share every key they load where a
// token has more than 16 heads).  grid (tiles × KV splits); a step is 64 keys: wave w scores block w of them for all rows, the row
// maxima meet in LDS, P and the parked latents are shared, and each wave accumulates its own quarter of the output dimensions — so
// nothing is merged at the end and the latents of the next step are in flight during softmax and P·V.
template <int KS, int RS, int MT>
__global__ __launch_bounds__(256, MT == 1 ? 2 : 1) void latent_attn_kernel(LatentDims d, LatentBuffers<bf16> p, BatchView v, int nsplit) {
    constexpr int DT = KS < 2 ? 1 : KS / 2;                                    // 16-dim output tiles per wave
    constexpr int STAGE = KS * 512, PSTR = 72, kd = 32 * (KS + RS), ROWS = 16 * MT;
    __shared__ __attribute__((aligned(16))) bf16 stage[4 * STAGE];
    __shared__ __attribute__((aligned(16))) bf16 lds_p[ROWS * PSTR];
    __shared__ float lds_m[4 * ROWS], lds_l[4 * ROWS];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, a = lane >> 4, b = lane & 15;
    const int split = blockIdx.x % nsplit, tile_id = blockIdx.x / nsplit;
    SeqTile w;
    if (!find_seq_tile(v, d.heads, ROWS, tile_id, &w)) return;
    const int rows = w.q_len * d.heads;
    int row_pos[MT], win_lo[MT], head[MT];
    long qrow[MT], qtok[MT];
    bool ok[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int rho = w.tile * ROWS + mt * 16 + b;
        ok[mt] = rho < rows;
        const int tl = ok[mt] ? rho / d.heads : 0;
        row_pos[mt] = w.pos0 + tl;
        win_lo[mt] = max(0, row_pos[mt] + 1 - d.window);
        qrow[mt] = (long)w.tok0 * d.heads + (ok[mt] ? rho : 0);
        head[mt] = ok[mt] ? rho - tl * d.heads : 0;
        qtok[mt] = (w.tok0 + tl) * p.ldq + head[mt] * (d.dp + d.rp) + d.dp;
    }
    const int t_first = w.tile * ROWS / d.heads, t_last = min(w.q_len - 1, (w.tile * ROWS + ROWS - 1) / d.heads);
    const int kv_end = w.pos0 + t_last + 1, kv_lo = max(0, w.pos0 + t_first + 1 - d.window);
    const int blk_lo = kv_lo / 16, blk_hi = (kv_end + 15) / 16, nstep = (blk_hi - blk_lo + 3) / 4;
    const int st_lo = nstep * split / nsplit, st_hi = nstep * (split + 1) / nsplit;
    const int32_t* bt = v.bt + (long)w.seq * v.max_blocks;

    // block-table entries of this wave's blocks, 64 steps per load; then nothing of the step loop waits for the table
    bf16x8 kf[KS + RS], qf[MT][KS + RS];
    auto table = [&](int st) { return bt[min(blk_lo + 4 * (st + lane) + wave, blk_hi - 1)]; };
    int bt_st = st_lo, btv = table(st_lo);
    auto load = [&](int st) {                                                  // (past the last block: a copy of it, masked below)
        const bf16* t = p.pool + (long)__builtin_amdgcn_readlane(btv, st - bt_st) * 16 * kd + lane * 8;
#pragma unroll
        for (int s = 0; s < KS + RS; s++) kf[s] = *reinterpret_cast<const bf16x8*>(t + s * 512);
    };
    {
        // the rotated part first: its values and angles travel together with the table entries, in front of the latents
        Rot4 rot[MT][RS];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int s = 0; s < RS; s++) {
                qf[mt][KS + s] = *reinterpret_cast<const bf16x8*>(p.q + qtok[mt] + 32 * s + 8 * a);
                rot[mt][s] = rot_load(32 * s + 8 * a, d.rot_dims, p.cos_t, p.sin_t, row_pos[mt]);
            }
        load(st_lo);                                                           // (no load under a condition: it would drain the others)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int s = 0; s < KS; s++) qf[mt][s] = *reinterpret_cast<const bf16x8*>(p.q_lat + qrow[mt] * (32 * KS) + 32 * s + 8 * a);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int s = 0; s < RS; s++) qf[mt][KS + s] = rot_apply(qf[mt][KS + s], rot[mt][s]);
    }
    const int tr_off = tr_offset(lane);
    float m_run[MT], l_run[MT];
    floatx4 o[MT][DT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        m_run[mt] = -INFINITY;
        l_run[mt] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; t++) o[mt][t] = (floatx4){0.f, 0.f, 0.f, 0.f};
    }
    for (int st = st_lo; st < st_hi; st++) {
        floatx4 sc[MT];
        float mx[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            floatx4 s2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};     // two chains: half the dependent MFMA latency
#pragma unroll
            for (int s = 0; s < KS + RS; s++) s2[s & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s], qf[mt][s], s2[s & 1], 0, 0, 0);
            mx[mt] = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = (blk_lo + 4 * st + wave) * 16 + 4 * a + r;
                sc[mt][r] = ok[mt] && key <= row_pos[mt] && key >= win_lo[mt] ? (s2[0][r] + s2[1][r]) * d.scale : -INFINITY;
                mx[mt] = fmaxf(mx[mt], sc[mt][r]);
            }
            mx[mt] = rows_reduce_max(mx[mt]);
        }
        __syncthreads();                                                       // the previous step's P·V has read stage and lds_p
#pragma unroll
        for (int s = 0; s < KS; s++) *reinterpret_cast<bf16x8*>(stage + wave * STAGE + s * 512 + lane * 8) = kf[s];
        if (a == 0) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) lds_m[wave * ROWS + mt * 16 + b] = mx[mt];
        }
        if (st + 1 - bt_st == 64) { bt_st = st + 1; btv = table(bt_st); }
        load(st + 1);
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const float* lm = lds_m + mt * 16 + b;
            const float m_new = fmaxf(m_run[mt], fmaxf(fmaxf(lm[0], lm[ROWS]), fmaxf(lm[2 * ROWS], lm[3 * ROWS])));
            const float m_safe = m_new == -INFINITY ? 0.f : m_new, alpha = __expf(m_run[mt] - m_safe);
            bf16x4 pf;
            float ps = 0.f;
#pragma unroll
            for (int r = 0; r < 4; r++) { const float e = __expf(sc[mt][r] - m_safe); ps += e; pf[r] = (bf16)e; }
            l_run[mt] = l_run[mt] * alpha + ps;                                // (this lane's keys; lanes and waves meet at the end)
            m_run[mt] = m_new;
            *reinterpret_cast<bf16x4*>(lds_p + (mt * 16 + b) * PSTR + wave * 16 + 4 * a) = pf;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[mt][t][r] *= alpha;
        }
        __syncthreads();
        // Oᵀ[d][row] += Vᵀ[d][key]·Pᵀ[key][row], 32 keys (two blocks) at a time: contraction index (a, j < 4) = key 4a + j of the first
        // block, (a, j ≥ 4) = key 4a + j − 4 of the second — a transposed read then covers 512 contiguous bytes
#pragma unroll
        for (int c = 0; c < 2; c++) {
            bf16x8 pv[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const bf16* lp = lds_p + (mt * 16 + b) * PSTR + c * 32 + 4 * a;
                const bf16x4 p0 = *reinterpret_cast<const bf16x4*>(lp), p1 = *reinterpret_cast<const bf16x4*>(lp + 16);
                pv[mt] = (bf16x8){p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
            }
            const bf16* vb = stage + 2 * c * STAGE + tr_off;
#pragma unroll
            for (int t = 0; t < DT; t++)
                if (KS >= 2 || wave < 2 * KS) {
                    const shortx4 v0 = read_tr(vb + (wave + 4 * t) * 256), v1 = read_tr(vb + STAGE + (wave + 4 * t) * 256);
                    typedef short shortx8 __attribute__((ext_vector_type(8)));
                    const shortx8 vt = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        o[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt), pv[mt], o[mt][t], 0, 0, 0);
                }
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const float l = rows_reduce_sum(l_run[mt]);
        if (a == 0) lds_l[wave * ROWS + mt * 16 + b] = l;
    }
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const float* ll = lds_l + mt * 16 + b;
        const float L = ll[0] + ll[ROWS] + ll[2 * ROWS] + ll[3 * ROWS];
        if (nsplit > 1) {
            float* dst = p.partial + ((long)blockIdx.x * ROWS + mt * 16 + b) * (32 * KS + LATENT_PARTIAL_PAD);
#pragma unroll
            for (int t = 0; t < DT; t++)
                if (KS >= 2 || wave < 2 * KS) *reinterpret_cast<floatx4*>(dst + (wave + 4 * t) * 16 + 4 * a) = o[mt][t];
            if (threadIdx.x < 16) { dst[32 * KS] = m_run[mt]; dst[32 * KS + 1] = L; }
        } else if (ok[mt]) {
            const float inv = softmax_factor<bf16>(m_run[mt], L, p.sink, head[mt]);
            bf16* dst = p.o_lat + qrow[mt] * (32 * KS);
#pragma unroll
            for (int t = 0; t < DT; t++)
                if (KS >= 2 || wave < 2 * KS) {
                    bf16x4 y;
#pragma unroll
                    for (int r = 0; r < 4; r++) y[r] = (bf16)(o[mt][t][r] * inv);
                    *reinterpret_cast<bf16x4*>(dst + (wave + 4 * t) * 16 + 4 * a) = y;
                }
        }
    }
}
// grid (tiles, quads of output dimensions / 256): one thread per (row, 4 dimensions); every load is in flight at once
template <typename E, int NS>
__global__ __launch_bounds__(256) void latent_attn_reduce_kernel(LatentDims d, LatentBuffers<E> p, BatchView v, int rows) {
    SeqTile w;
    if (!find_seq_tile(v, d.heads, rows, blockIdx.x, &w)) return;
    const int quads = d.kp >> 2, id = blockIdx.y * 256 + threadIdx.x, row = id / quads, c = (id % quads) * 4, ro = w.tile * rows + row;
    if (row >= rows || ro >= w.q_len * d.heads) return;
    const long ld = d.kp + LATENT_PARTIAL_PAD, zs = rows * ld;
    const float* src = p.partial + ((long)blockIdx.x * NS * rows + row) * ld;
    float m[NS], l[NS], M = -INFINITY, L = 0.f;
    floatx4 o[NS], acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int z = 0; z < NS; z++) {
        m[z] = src[z * zs + d.kp];
        l[z] = src[z * zs + d.kp + 1];
        o[z] = *reinterpret_cast<const floatx4*>(src + z * zs + c);
    }
#pragma unroll
    for (int z = 0; z < NS; z++) M = fmaxf(M, m[z]);
#pragma unroll
    for (int z = 0; z < NS; z++) {
        const float f = attn_exp<E>(m[z] - M);
        L += l[z] * f;
        acc += o[z] * f;
    }
    const float inv = softmax_factor<E>(M, L, p.sink, ro % d.heads);
    typename Frag<E>::v4 y;
#pragma unroll
    for (int r = 0; r < 4; r++) y[r] = (E)(acc[r] * inv);
    *reinterpret_cast<typename Frag<E>::v4*>(p.o_lat + ((long)w.tok0 * d.heads + ro) * d.kp + c) = y;
}


// ── 32-bit models on the matrix cores ──
// grid (tiles of 16 (token, head) rows × KV splits), 64 keys per step.  Scores: every wave takes a quarter of the dimensions for all keys, the four
// partial sums meet in LDS.  Values: wave w takes 128 output dimensions (of latents of 256 and fewer also a part of the keys, summed at the end).
// v_mfma_f32_16x16x4 takes four keys at a time; product j of eight works on dimensions 8b + j, so that the eight dimensions 8b … 8b + 7 of a key,
// which lie together in the cache, are one lane's operands of the eight, and the keys 4a + r of a lane's scores are its weights as they are.
// Bound by the fp32 matrix rate: 2·kv_rank + rot products a (row, key), and the cache is read once for 16 rows where the plain form reads it for
// each.  kv_rank 512, 16 heads, a prompt of 1000 tokens and 8 decoded: plain 4.68 ms, this 0.60 ms; 20 sequences of 50
// tokens and what they decode 1.64 -> 0.86 ms.  Keys dealt out to the waves were slower in decode: at few keys most waves have none.
template <int KS, int RS>
__global__ __launch_bounds__(256) void latent_attn_f32_kernel(LatentDims d, LatentBuffers<float> p, BatchView v, int nsplit) {
    constexpr int KP = 32 * KS, kd = KP + 32 * RS, NG = (KP + 127) / 128, PARTS = NG > 2 ? 1 : 4 / NG, SW = (KS + RS + 3) / 4, LD = KP + 4;
    __shared__ floatx4 lds_s[4][4][64];
    __shared__ __attribute__((aligned(16))) float lds_o[PARTS > 1 ? 16 * LD : 4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, a = lane >> 4, b = lane & 15;
    const int split = blockIdx.x % nsplit, tile_id = blockIdx.x / nsplit, g = wave % NG, part = wave / NG;
    SeqTile w;
    if (!find_seq_tile(v, d.heads, 16, tile_id, &w)) return;
    const int rows = w.q_len * d.heads, rho = w.tile * 16 + b;
    const bool ok = rho < rows, weighs = part < PARTS;
    const int tl = ok ? rho / d.heads : 0, head = ok ? rho - tl * d.heads : 0, row_pos = w.pos0 + tl, win_lo = max(0, row_pos + 1 - d.window);
    const int t_first = w.tile * 16 / d.heads, t_last = min(w.q_len - 1, (w.tile * 16 + 15) / d.heads);
    const int blk_lo = max(0, w.pos0 + t_first + 1 - d.window) / 16, blk_hi = (w.pos0 + t_last + 16) / 16, nstep = (blk_hi - blk_lo + 3) / 4;
    const int st_lo = nstep * split / nsplit, st_hi = nstep * (split + 1) / nsplit;
    const int32_t* bt = v.bt + (long)w.seq * v.max_blocks;
    // 32-wide pieces wave, wave + 4, … of the query (past the last one: zeros)
    floatx8 qf[SW];
#pragma unroll
    for (int i = 0; i < SW; i++) {
        const int s = wave + 4 * i;
        if (s < KS) {
            qf[i] = *reinterpret_cast<const floatx8*>(p.q_lat + ((long)w.tok0 * d.heads + (ok ? rho : 0)) * KP + 32 * s + 8 * a);
        } else if (s < KS + RS) {
            const float* q = p.q + (w.tok0 + tl) * p.ldq + head * (d.dp + d.rp) + d.dp + 32 * (s - KS) + 8 * a;
            qf[i] = rot_apply(*reinterpret_cast<const floatx8*>(q), rot_load(32 * (s - KS) + 8 * a, d.rot_dims, p.cos_t, p.sin_t, row_pos));
        } else {
            qf[i] = (floatx8){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        }
    }
    float m_run = -INFINITY, l_run = 0.f;
    floatx4 o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = (floatx4){0.f, 0.f, 0.f, 0.f};
    for (int st = st_lo; st < st_hi; st++) {
        const float* blk[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {                                          // (past the end: a copy of the last block, masked)
            blk[i] = p.pool + (long)__builtin_amdgcn_readfirstlane(bt[min(blk_lo + 4 * st + i, blk_hi - 1)]) * 16 * kd;
        }
        floatx4 s4[4];
#pragma unroll
        for (int i = 0; i < 4; i++) s4[i] = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < SW; q++) {
            const int s = min(wave + 4 * q, KS + RS - 1);
            floatx8 k[4];
#pragma unroll
            for (int i = 0; i < 4; i++) k[i] = *reinterpret_cast<const floatx8*>(blk[i] + s * 512 + lane * 8);
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) s4[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][j], qf[q][j], s4[i], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) lds_s[wave][i][lane] = s4[i];
        __syncthreads();
        float sc[16], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const floatx4 z = (lds_s[0][i][lane] + lds_s[1][i][lane]) + (lds_s[2][i][lane] + lds_s[3][i][lane]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = (blk_lo + 4 * st + i) * 16 + 4 * a + r;
                sc[4 * i + r] = ok && key <= row_pos && key >= win_lo ? z[r] * d.scale : -INFINITY;
                mx = fmaxf(mx, sc[4 * i + r]);
            }
        }
        __syncthreads();                                                       // (the sums of the next step take their place)
        const float m_new = fmaxf(m_run, rows_reduce_max(mx)), m_safe = m_new == -INFINITY ? 0.f : m_new, alpha = expf(m_run - m_safe);
        float ps = 0.f;
#pragma unroll
        for (int j = 0; j < 16; j++) { sc[j] = expf(sc[j] - m_safe); ps += sc[j]; }
        l_run = l_run * alpha + ps;                                            // (this lane's keys; the four lane groups meet at the end)
        m_run = m_new;
        if (!weighs) continue;
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[j][r] *= alpha;
        const int chunk = min(16 * g + b, KP / 8 - 1);                         // (dimensions past the latent: not written)
#pragma unroll
        for (int q = 0; q < 4 / PARTS; q++) {
            const float* block = blk[q];
            float pr[4] = {sc[4 * q], sc[4 * q + 1], sc[4 * q + 2], sc[4 * q + 3]};
            if (PARTS == 4) {
#pragma unroll
                for (int i = 1; i < 4; i++)
                    if (part == i) {
                        block = blk[i];
#pragma unroll
                        for (int r = 0; r < 4; r++) pr[r] = sc[4 * i + r];
                    }
            } else if (PARTS == 2 && part == 1) {
                block = blk[2 + q];
#pragma unroll
                for (int r = 0; r < 4; r++) pr[r] = sc[8 + 4 * q + r];
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const floatx8 x = *reinterpret_cast<const floatx8*>(block + (chunk * 16 + 4 * a + r) * 8);
#pragma unroll
                for (int j = 0; j < 8; j++) o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], pr[r], o[j], 0, 0, 0);
            }
        }
    }
    const float l = rows_reduce_sum(l_run);
    if (PARTS > 1) {
        for (int turn = 1; turn < PARTS; turn++) {
            if (part == turn) {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (128 * g + 8 * (4 * a + r) < KP)
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            float* x = lds_o + b * LD + 128 * g + 8 * (4 * a + r) + j;
                            *x = turn > 1 ? *x + o[j][r] : o[j][r];
                        }
            }
            __syncthreads();
        }
        if (part == 0) {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (128 * g + 8 * (4 * a + r) < KP)
#pragma unroll
                    for (int j = 0; j < 8; j++) o[j][r] += lds_o[b * LD + 128 * g + 8 * (4 * a + r) + j];
        }
    }
    if (part > 0) return;
    const float f = nsplit > 1 ? 1.f : softmax_factor<float>(m_run, l, p.sink, head);
    float* dst = nsplit > 1 ? p.partial + ((long)blockIdx.x * 16 + b) * (KP + LATENT_PARTIAL_PAD) : p.o_lat + ((long)w.tok0 * d.heads + rho) * KP;
    if (nsplit == 1 && !ok) return;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int c = 128 * g + 8 * (4 * a + r);
        if (c >= KP) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            floatx4 x;
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = o[4 * h + j][r] * f;
            *reinterpret_cast<floatx4*>(dst + c + 4 * h) = x;
        }
    }
    if (nsplit > 1 && g == 0 && a == 0) { dst[KP] = m_run; dst[KP + 1] = l; }
}

// ── portions over expanded keys and values ──
// A workgroup owns 128 tokens of one sequence and head: 4 waves × 2 row tiles of 16.  64 keys per step: wave w copies 16-key block w of
// the step — expanded key rows, the shared rotated part straight from the cache, expanded value rows — as fragments into LDS with the
// load unit, double-buffered; Sᵀ = K·Qᵀ keeps a row's statistics lane-local, values are read back transposed for Oᵀ += Vᵀ·Pᵀ.
// DS: 32-wide steps of the plain query / key dimensions and of the values (padded alike), RS: of the rotated part.
template <int DS, int RS>
__global__ __launch_bounds__(256, 2) void latent_expanded_kernel(LatentDims d, LatentBuffers<bf16> p, BatchView v, LatentExpanded x) {
    constexpr int MT = 2, BLK = (2 * DS + RS) * 512, DT = 2 * DS;
    extern __shared__ __attribute__((aligned(16))) bf16 lds_x[];               // [2][4 blocks][BLK]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, a = lane >> 4, b = lane & 15;
    const int h = blockIdx.y;
    const int32_t* un = x.units + 4 * (gridDim.x - 1 - blockIdx.x);            // the longest key ranges start first
    const int seq = un[0], tile0 = un[1], base = un[2], first_blk = un[3];
    const int tok0 = (int)v.cu[seq], q_len = (int)v.cu[seq + 1] - tok0, pos0 = (int)v.pos[seq];
    const int kd = d.kp + d.rp;
    const float sl2 = d.scale * 1.4426950408889634f;

    bf16x8 qf[MT][DS + RS];
    int row_pos[MT], win_lo[MT], vis_lo[MT], vis_hi[MT];
    bool ok[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int t0 = tile0 + (wave * MT + mt) * 16, t = t0 + b;
        ok[mt] = t < q_len;
        row_pos[mt] = pos0 + min(t, q_len - 1);
        win_lo[mt] = max(0, row_pos[mt] + 1 - d.window);
        vis_hi[mt] = t0 + 15 < q_len ? pos0 + t0 : -1;                         // keys in [vis_lo, vis_hi] are seen by every row of the tile
        vis_lo[mt] = max(0, pos0 + t0 + 16 - d.window);
        const bf16* q = p.q + (long)(tok0 + min(t, q_len - 1)) * p.ldq + h * (d.dp + d.rp) + 8 * a;
#pragma unroll
        for (int s = 0; s < DS; s++)
            qf[mt][s] = *reinterpret_cast<const bf16x8*>(q + 32 * s);
#pragma unroll
        for (int s = 0; s < RS; s++)
            qf[mt][DS + s] = rot_apply(*reinterpret_cast<const bf16x8*>(q + d.dp + 32 * s), rot_load(32 * s + 8 * a, d.rot_dims, p.cos_t, p.sin_t, row_pos[mt]));
    }
    const int t_hi = min(q_len, tile0 + LATENT_TILE_TOKENS);
    const int blk_lo = max(0, pos0 + tile0 + 1 - d.window) / 16, blk_hi = (pos0 + t_hi + 15) / 16, nstep = (blk_hi - blk_lo + 3) / 4;
    auto issue = [&](int st, int buf) {
        const int i = base + min(blk_lo + 4 * st + wave, blk_hi - 1) - first_blk;      // (past the end: a copy of the last block, masked)
        bf16* dst = lds_x + (buf * 4 + wave) * BLK;
        const bf16 *k = x.ke + (long)(i * 16 + b) * x.ldk + h * d.dp + 8 * a, *vr = x.ve + (long)(i * 16 + b) * x.ldv + h * d.vp + 8 * a;
        const bf16* r = p.pool + (long)x.blocks[i] * 16 * kd + d.kp * 16 + lane * 8;
#define LX_COPY(src, slot) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src), (__attribute__((address_space(3))) void*)(dst + (slot) * 512), 16, 0, 0)
#pragma unroll
        for (int s = 0; s < DS; s++)
            LX_COPY(k + 32 * s, s);
#pragma unroll
        for (int s = 0; s < RS; s++)
            LX_COPY(r + s * 512, DS + s);
#pragma unroll
        for (int s = 0; s < DS; s++)
            LX_COPY(vr + 32 * s, DS + RS + s);
#undef LX_COPY
    };
    const int tr_off = tr_offset(lane);
    float m_run[MT], l_run[MT];
    floatx4 o[MT][DT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        m_run[mt] = -INFINITY; l_run[mt] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; t++) o[mt][t] = (floatx4){0.f, 0.f, 0.f, 0.f};
    }
    issue(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int st = 0; st < nstep; st++) {
        const int buf = st & 1;
        if (st + 1 < nstep) issue(st + 1, buf ^ 1);
        const bf16* kb = lds_x + buf * 4 * BLK;
        floatx4 sv[MT][4];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) sv[mt][i] = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < DS + RS; s++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const bf16x8 k = *reinterpret_cast<const bf16x8*>(kb + i * BLK + s * 512 + lane * 8);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) sv[mt][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[mt][s], sv[mt][i], 0, 0, 0);
                }
        }
        bf16x8 pf[MT][2];
        const int key0 = (blk_lo + 4 * st) * 16;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            if (!(key0 + 63 <= vis_hi[mt] && key0 >= vis_lo[mt])) {
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int key = key0 + i * 16 + 4 * a + r;
                        if (!(ok[mt] && key <= row_pos[mt] && key >= win_lo[mt])) sv[mt][i][r] = -INFINITY;
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; i++) mx = fmaxf(mx, fmaxf(fmaxf(sv[mt][i][0], sv[mt][i][1]), fmaxf(sv[mt][i][2], sv[mt][i][3])));
            mx = rows_reduce_max(mx * sl2);                                    // (scale > 0, checked by the caller: the maximum commutes)
            const float m_new = fmaxf(m_run[mt], mx), m_safe = m_new == -INFINITY ? 0.f : m_new;
            if (__ballot(m_new != m_run[mt]) != 0) {
                const float alpha = __builtin_amdgcn_exp2f(m_run[mt] - m_safe);
#pragma unroll
                for (int t = 0; t < DT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) o[mt][t][r] *= alpha;
                l_run[mt] *= alpha;
                m_run[mt] = m_new;
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[mt][i][r], sl2, -m_safe));
                    l_run[mt] += e;
                    pf[mt][i >> 1][(i & 1) * 4 + r] = (bf16)e;
                }
        }
        // contraction index of a 32-key pair: (a, j < 4) = key 4a + j of its first block, (a, j ≥ 4) = key 4a + j − 4 of its second
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const bf16* vb = kb + 2 * c * BLK + (DS + RS) * 512 + tr_off;
#pragma unroll
            for (int t = 0; t < DT; t++) {
                    const shortx4 v0 = read_tr(vb + t * 256), v1 = read_tr(vb + BLK + t * 256);
                    typedef short shortx8 __attribute__((ext_vector_type(8)));
                    const shortx8 vt = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        o[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt), pf[mt][c], o[mt][t], 0, 0, 0);
                }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const float l = rows_reduce_sum(l_run[mt]);
        if (!ok[mt]) continue;
        const long tok = tok0 + tile0 + (wave * MT + mt) * 16 + b;
        float f = softmax_factor<bf16>(m_run[mt] * 0.6931471805599453f, l, p.sink, h);      // (the maximum is kept in base 2)
        if (x.gate) f *= (float)x.gate[tok * x.ld_gate + h];
        bf16* dst = x.out + tok * x.ldo + h * d.vp + 4 * a;
#pragma unroll
        for (int t = 0; t < DT; t++) {
                bf16x4 y;
#pragma unroll
                for (int r = 0; r < 4; r++) y[r] = (bf16)(o[mt][t][r] * f);
                *reinterpret_cast<bf16x4*>(dst + t * 16) = y;
            }
    }
}
bool latent_expanded_supports(const LatentDims& d) { return d.dp == d.vp && d.dp <= 128 && d.rp <= 64 && d.scale > 0.f; }
template <int DS, int RS>
static int launch_expanded(const LatentDims& d, const LatentBuffers<bf16>& b, const BatchView& v, const LatentExpanded& x, hipStream_t s) {
    constexpr size_t lds = (size_t)2 * 4 * (2 * DS + RS) * 512 * sizeof(bf16);
    static bool attr = false;
    if (!attr) { FH_CHECK_HIP(hipFuncSetAttribute((const void*)latent_expanded_kernel<DS, RS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); attr = true; }
    hipLaunchKernelGGL((latent_expanded_kernel<DS, RS>), dim3(x.nunits, d.heads), dim3(256), lds, s, d, b, v, x);
    FH_CHECK_LAUNCH();
    return 0;
}
int latent_attention_expanded(const LatentDims& d, const LatentBuffers<bf16>& b, const BatchView& v, const LatentExpanded& x, hipStream_t s) {
    FH_REQUIRE(latent_expanded_supports(d), "latent attention: sizes the expanded form does not take");
    form_hit(FORM_LATENT_ATTN_EXPANDED);
    if (d.rp == 32) return d.dp == 32 ? launch_expanded<1, 1>(d, b, v, x, s) : d.dp == 64 ? launch_expanded<2, 1>(d, b, v, x, s) : launch_expanded<4, 1>(d, b, v, x, s);
    return d.dp == 32 ? launch_expanded<1, 2>(d, b, v, x, s) : d.dp == 64 ? launch_expanded<2, 2>(d, b, v, x, s) : launch_expanded<4, 2>(d, b, v, x, s);
}

template <typename E>
static int latent_plain(const LatentDims& d, const LatentBuffers<E>& b, const BatchView& v, hipStream_t s) {
    form_hit(FORM_LATENT_ATTN_PLAIN);
    const size_t lds = (size_t)(2 * d.kp + d.rp + 256 + 8) * 4;
    FH_REQUIRE(lds <= 64 * 1024, "latent attention: kv_rank %d + rotated %d do not fit LDS", d.kv_rank, d.rot_dim);
    hipLaunchKernelGGL(latent_attn_plain_kernel<E>, dim3(v.T, d.heads), dim3(256), lds, s, d, b, v);
    FH_CHECK_LAUNCH();
    return 0;
}
template <typename E>
static int latent_reduce(const LatentDims& d, const LatentBuffers<E>& b, const BatchView& v, int tiles, int rows, int ns, hipStream_t s) {
    const dim3 rg(tiles, cdiv(rows * (d.kp / 4), 256));
    if (ns == 2) hipLaunchKernelGGL((latent_attn_reduce_kernel<E, 2>), rg, dim3(256), 0, s, d, b, v, rows);
    else if (ns == 4) hipLaunchKernelGGL((latent_attn_reduce_kernel<E, 4>), rg, dim3(256), 0, s, d, b, v, rows);
    else if (ns == 8) hipLaunchKernelGGL((latent_attn_reduce_kernel<E, 8>), rg, dim3(256), 0, s, d, b, v, rows);
    else hipLaunchKernelGGL((latent_attn_reduce_kernel<E, 16>), rg, dim3(256), 0, s, d, b, v, rows);
    FH_CHECK_LAUNCH();
    return 0;
}
static int latent_mfma(const LatentDims& d, const LatentBuffers<bf16>& b, const BatchView& v, hipStream_t s) {
    // two 16-row tiles per workgroup where a token fills both and the batch is large: the keys are loaded and parked once for 32 heads
    // (below ≈ 128 tiles the launch is bound by latency, and one tile per workgroup has the shorter chain)
    const bool pair = knobs().latent_tiles > 0 ? knobs().latent_tiles == 2 : d.heads > 16 && (long)v.T * d.heads >= 128 * 16;
    const int mt = pair ? 2 : 1, rows = 16 * mt;
    const int tiles = v.single ? v.num_seqs * cdiv(d.heads, rows) : (int)(((long)v.T * d.heads) / rows) + v.num_seqs;      // upper bound of Σ ceil(rows of a sequence / rows)
    const int keys = (int)std::min<long>(v.max_keys, (long)d.window + 16);
    // split the keys while the launch has fewer workgroups than stay resident (2 per CU, 1 with two tiles) and a split keeps ≥ 128
    // keys (two steps); up to 256 keys the second launch costs more than it saves (a step of safolorn, one layer's cache of 120 keys, 32 rows: 206 µs whole, 210 in two)
    int ns = 1;
    while (ns < 16 && tiles * ns < 512 / mt && keys > 256 && keys >= 2 * ns * 128) ns *= 2;
    if (knobs().latent_splits > 0)
        for (ns = 1; ns < std::min(16, knobs().latent_splits); ns *= 2) {}
    while (ns > 1 && (size_t)tiles * ns * rows * (d.kp + LATENT_PARTIAL_PAD) * 4 > b.partial_bytes) ns /= 2;
    const dim3 grid(ns * tiles);         // (splits fastest: the row tiles of a sequence read a key range on the same XCD)
    form_hit(ns > 1 ? FORM_LATENT_ATTN_SPLIT : FORM_LATENT_ATTN);
    if (pair) form_hit(FORM_LATENT_ATTN_PAIR);
#define LATENT2(KS, RS)                                                                                           \
    do {                                                                                                          \
        if (mt == 1) hipLaunchKernelGGL((latent_attn_kernel<KS, RS, 1>), grid, dim3(256), 0, s, d, b, v, ns);      \
        else hipLaunchKernelGGL((latent_attn_kernel<KS, RS, 2>), grid, dim3(256), 0, s, d, b, v, ns);              \
    } while (0)
#define LATENT(KS)                              \
    do {                                        \
        if (d.rp == 32) LATENT2(KS, 1);         \
        else LATENT2(KS, 2);                    \
    } while (0)
    switch (d.kp) {
    case 32: LATENT(1); break;
    case 64: LATENT(2); break;
    case 128: LATENT(4); break;
    case 256: LATENT(8); break;
    case 384: LATENT(12); break;
    default: LATENT(16); break;
    }
#undef LATENT
#undef LATENT2
    FH_CHECK_LAUNCH();
    return ns > 1 ? latent_reduce(d, b, v, tiles, rows, ns, s) : 0;
}
static int latent_mfma(const LatentDims& d, const LatentBuffers<float>& b, const BatchView& v, hipStream_t s) {
    const int tiles = v.single ? v.num_seqs * cdiv(d.heads, 16) : (int)(((long)v.T * d.heads) / 16) + v.num_seqs;
    const int keys = (int)std::min<long>(v.max_keys, (long)d.window + 16);
    // Split the keys while there is less than a workgroup per CU and a split keeps ≥ 64 keys (a step, 4 µs of products, as much as the launch that joins them).  µs of a step of
    // nerenex, one such layer, with 1 | 2 | 4 | 8 splits: 1 × 120 keys 272 | 266 | 261 | 262, 1 × 200 285 | 270 | 260 | 261, 1 × 400 312 | 288 | 269 | 261,
    // 16 × 60 300 | 294 | 295 | 298, 16 × 200 321 | 305 | 295 | 298, 16 × 400 351 | 324 | 304 | 297.
    int ns = 1;
    while (ns < 16 && tiles * ns < 256 && keys >= 2 * ns * 64) ns *= 2;
    if (knobs().latent_splits > 0)
        for (ns = 1; ns < std::min(16, knobs().latent_splits); ns *= 2) {}
    while (ns > 1 && (size_t)tiles * ns * 16 * (d.kp + LATENT_PARTIAL_PAD) * 4 > b.partial_bytes) ns /= 2;
    form_hit(ns > 1 ? FORM_LATENT_ATTN_SPLIT : FORM_LATENT_ATTN);
#define LATENT(KS)                                                                                                                       \
    do {                                                                                                                                 \
        if (d.rp == 32) hipLaunchKernelGGL((latent_attn_f32_kernel<KS, 1>), dim3(tiles * ns), dim3(256), 0, s, d, b, v, ns);             \
        else hipLaunchKernelGGL((latent_attn_f32_kernel<KS, 2>), dim3(tiles * ns), dim3(256), 0, s, d, b, v, ns);                        \
    } while (0)
    switch (d.kp) {
    case 32: LATENT(1); break;
    case 64: LATENT(2); break;
    case 128: LATENT(4); break;
    case 256: LATENT(8); break;
    case 384: LATENT(12); break;
    default: LATENT(16); break;
    }
#undef LATENT
    FH_CHECK_LAUNCH();
    return ns > 1 ? latent_reduce(d, b, v, tiles, 16, ns, s) : 0;
}
template <> int latent_attention<float>(const LatentDims& d, const LatentBuffers<float>& b, const BatchView& v, hipStream_t s) {
    if (knobs().latent_plain || d.kp > 512 || d.rp > 64) return latent_plain(d, b, v, s);
    return latent_mfma(d, b, v, s);
}
template <> int latent_attention<bf16>(const LatentDims& d, const LatentBuffers<bf16>& b, const BatchView& v, hipStream_t s) {
    if (knobs().latent_plain || d.kp > 512 || d.rp > 64) return latent_plain(d, b, v, s);
    return latent_mfma(d, b, v, s);
}
template int latent_prepare<bf16>(const bf16*, const bf16*, long, const float*, const float*, float, const LatentDims&, const LatentBuffers<bf16>&,
                                  const BatchView&, bf16*, hipStream_t);
template int latent_prepare<float>(const float*, const float*, long, const float*, const float*, float, const LatentDims&,
                                   const LatentBuffers<float>&, const BatchView&, float*, hipStream_t);

}  // namespace fh
