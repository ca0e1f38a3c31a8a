// Residual stream of the layered models: fp32 throughout, with a copy in the projections' number format written by whoever changes it.
#include "common.h"
#include "knobs.h"
#include "layer_ops.h"
#include "route_device.h"

namespace fh {

// AT_ONCE: the waves' sums read together, for launches whose time is latency; of many rows the loop is no slower and leaves 16 registers (2048 × 2048 9.1, not 10.4 µs)
template <bool AT_ONCE = true>
__device__ __forceinline__ float block_sum(float q, float* red) {
    q = wave_reduce_sum(q);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = q;
    __syncthreads();
    if (!AT_ONCE) {
        float t = 0.f;
        for (int i = 0; i < (int)(blockDim.x >> 6); i++) t += red[i];
        return t;
    }
    float r[16], t = 0.f;                                              // (red holds 16, all read at once)
#pragma unroll
    for (int i = 0; i < 16; i++) r[i] = red[i];
#pragma unroll
    for (int i = 0; i < 16; i++) t += i < (int)(blockDim.x >> 6) ? r[i] : 0.f;
    return t;
}

// One workgroup per token.  VEC 1: a thread's 8 numbers stay in registers for the norm of the first block's input; 2: several such pieces, read back from x; 0: any length.
template <typename E, int VEC>
__global__ __launch_bounds__(256) void embed_kernel(Embedding<E> p, BatchView v, float* __restrict__ x, E* __restrict__ xb, int dim, int ldb) {
    __shared__ float red[16];
    const int t = blockIdx.x;
    float* xr = x + (long)t * dim;
    E *br = xb + (long)t * ldb, *raw = p.raw + (long)t * p.ld_raw;
    const uint32_t tok = v.tokens[t];
    const E *own = p.table + (long)tok * dim, *bigram = nullptr, *place = nullptr;
    if (p.bigram || p.positions) {
        const int seq = v.tok_seq[t], at = t - (int)v.cu[seq];
        if (p.bigram) {
            const int64_t prev = at == 0 ? (int64_t)v.prev[seq] : (int64_t)v.tokens[t - 1];
            bigram = p.bigram + dim * (prev < 0 ? (long)p.buckets : (long)(((uint64_t)prev * (uint64_t)p.mul_prev + (uint64_t)tok * (uint64_t)p.mul_cur) % (uint64_t)p.buckets));
        }
        if (p.positions) place = p.positions + (long)(v.pos[seq] + at) * dim;
    }
    float q = 0.f;
    if constexpr (VEC > 0) {
        typedef typename Frag<E>::v8 v8;
        floatx4 f[2], w[2] = {{1.f, 1.f, 1.f, 1.f}, {1.f, 1.f, 1.f, 1.f}};
        const int mine = threadIdx.x * 8;
        if (VEC == 1 && p.norm_w && mine < dim) {
            w[0] = *reinterpret_cast<const floatx4*>(p.norm_w + mine);
            w[1] = *reinterpret_cast<const floatx4*>(p.norm_w + mine + 4);
        }
        for (int i = mine; i < dim; i += 2048) {
            const v8 e = *reinterpret_cast<const v8*>(own + i);
            v8 g = e, l = e, o;
            if (bigram) g = *reinterpret_cast<const v8*>(bigram + i);
            if (place) l = *reinterpret_cast<const v8*>(place + i);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float y = (float)e[j] * p.factor + (bigram ? (float)g[j] : 0.f) + (place ? (float)l[j] : 0.f);
                f[j >> 2][j & 3] = y;
                q += y * y;
                o[j] = (E)y;
            }
            *reinterpret_cast<floatx4*>(xr + i) = f[0];
            *reinterpret_cast<floatx4*>(xr + i + 4) = f[1];
            if (p.raw) *reinterpret_cast<v8*>(raw + i) = o;
            if (!p.norm) *reinterpret_cast<v8*>(br + i) = o;
            if (VEC == 1) break;
        }
        if (!p.norm) return;
        const float inv = 1.0f / sqrtf(block_sum<VEC == 1>(q, red) / (float)dim + p.eps);
        for (int i = mine; i < dim; i += 2048) {
            if (VEC != 1) {                                       // (a thread's own numbers)
                f[0] = *reinterpret_cast<const floatx4*>(xr + i);
                f[1] = *reinterpret_cast<const floatx4*>(xr + i + 4);
                if (p.norm_w) {
                    w[0] = *reinterpret_cast<const floatx4*>(p.norm_w + i);
                    w[1] = *reinterpret_cast<const floatx4*>(p.norm_w + i + 4);
                }
            }
            v8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = (E)(f[j >> 2][j & 3] * inv * w[j >> 2][j & 3]);
            *reinterpret_cast<v8*>(br + i) = o;
            if (VEC == 1) break;
        }
        return;
    }
    for (int i = threadIdx.x; i < dim; i += 256) {
        float e = (float)own[i] * p.factor;
        if (bigram) e += (float)bigram[i];
        if (place) e += (float)place[i];
        xr[i] = e;
        q += e * e;
        if (p.raw) raw[i] = (E)e;
        if (!p.norm) br[i] = (E)e;
    }
    if (!p.norm) return;
    const float inv = 1.0f / sqrtf(block_sum<false>(q, red) / (float)dim + p.eps);
    for (int i = threadIdx.x; i < dim; i += 256) br[i] = (E)(p.norm_w ? xr[i] * inv * p.norm_w[i] : xr[i] * inv);
}

template <typename E>
int embed_tokens(const Embedding<E>& e, const BatchView& v, float* x, E* xb, int dim, int ldb, hipStream_t s) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(v.T), dim3(256), 0, s, e, v, x, xb, dim, ldb); };
    if (dim % 8) go(embed_kernel<E, 0>);
    else if (dim <= 2048) go(embed_kernel<E, 1>);
    else go(embed_kernel<E, 2>);
    FH_CHECK_LAUNCH();
    return 0;
}

// Σ over the slabs of a branch, in their order; TOGETHER: two, or up to four, are under way at once (one after the other each cost a round trip, 0.7 µs)
template <bool TOGETHER = true>
__device__ __forceinline__ floatx4 sum_slabs(const float* p, int slabs, long stride) {
    if (!TOGETHER || slabs == 1) {
        floatx4 v = *reinterpret_cast<const floatx4*>(p);
        for (int z = 1; z < slabs; z++) v += *reinterpret_cast<const floatx4*>(p + z * stride);
        return v;
    }
    if (slabs == 2) {
        const floatx4 a = *reinterpret_cast<const floatx4*>(p), b = *reinterpret_cast<const floatx4*>(p + stride);
        return a + b;
    }
    floatx4 t[4];
#pragma unroll
    for (int z = 0; z < 4; z++) t[z] = *reinterpret_cast<const floatx4*>(p + (z < slabs ? z : slabs - 1) * stride);
    floatx4 v = t[0];
#pragma unroll
    for (int z = 1; z < 4; z++)
        if (z < slabs) v += t[z];
    for (int z = 4; z < slabs; z++) v += *reinterpret_cast<const floatx4*>(p + z * stride);
    return v;
}

// x += Σ slabs of `sub` + Σ_j weights[row][j] · pairs[row·top + j]; elementwise, grid (rows, quads of columns / 256)
template <typename E, bool VEC>
__global__ __launch_bounds__(256) void branch_add_kernel(const float* __restrict__ sub, long ld_sub, int slabs, long slab_stride, const E* __restrict__ pairs,
                                                         long ld_pair, const float* __restrict__ weights, int top, float* __restrict__ x,
                                                         E* __restrict__ xb, int dim, int ldb) {
    const long row = blockIdx.x;
    const int i = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (i >= dim) return;
    const float* sr = sub + row * ld_sub + i;
    const E* pr = pairs + row * top * ld_pair + i;
    if (VEC) {
        typedef E e4 __attribute__((ext_vector_type(4)));
        const floatx4 xv = *reinterpret_cast<const floatx4*>(x + row * dim + i);
        floatx4 v = sum_slabs(sr, slabs, slab_stride);
#pragma unroll 4
        for (int j = 0; j < top; j++) {
            const e4 e = *reinterpret_cast<const e4*>(pr + j * ld_pair);
            const float w = weights[row * top + j];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] += w * (float)e[k];
        }
        v += xv;
        e4 o;
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = (E)v[k];
        *reinterpret_cast<floatx4*>(x + row * dim + i) = v;
        *reinterpret_cast<e4*>(xb + row * ldb + i) = o;
        return;
    }
    for (int k = 0; k < 4 && i + k < dim; k++) {
        float v = sr[k];
        for (int z = 1; z < slabs; z++) v += sr[z * slab_stride + k];
        for (int j = 0; j < top; j++) v += weights[row * top + j] * (float)pr[j * ld_pair + k];
        v += x[row * dim + i + k];
        x[row * dim + i + k] = v;
        xb[row * ldb + i + k] = (E)v;
    }
}
template <typename E>
int branch_add(const float* sub, long ld_sub, int slabs, long slab_stride, const E* pairs, long ld_pair, const float* weights, int top, float* x, E* xb,
               int rows, int dim, int ldb, hipStream_t s) {
    const bool vec = dim % 4 == 0 && ld_sub % 4 == 0 && ld_pair % 4 == 0 && ldb % 4 == 0 && slab_stride % 4 == 0;
    const dim3 grid(rows, cdiv(dim, 1024));
    if (vec) hipLaunchKernelGGL((branch_add_kernel<E, true>), grid, dim3(256), 0, s, sub, ld_sub, slabs, slab_stride, pairs, ld_pair, weights, top, x, xb, dim, ldb);
    else hipLaunchKernelGGL((branch_add_kernel<E, false>), grid, dim3(256), 0, s, sub, ld_sub, slabs, slab_stride, pairs, ld_pair, weights, top, x, xb, dim, ldb);
    FH_CHECK_LAUNCH();
    return 0;
}

// One workgroup per row; a thread holds VEC quads of the row in registers (0: any length, from memory), so the branch is read once.  NEXT: the copy is the row
// divided by its root mean square, times next_w where there is one: the input of a block that norms ahead of its sublayers, or of the head.
// One quad a thread (decode, and narrow rows): latency alone, so everything is requested at once, what the first sum does not need ahead of it.  Of
// several quads the row's own are requested first, and what is not needed yet does not take registers (all at once: rows of 6144 in two slabs
// 3.6 → 4.2 µs, 512 of them 7.7 → 9.1; the update below 1024 × 4096 8.5 → 15.5, 8192 × 2880 43 → 100).
template <typename E, int VEC, bool GATE, bool NEXT>
__global__ __launch_bounds__(1024) void post_norm_add_kernel(const float* __restrict__ sub, long ld_sub, int slabs, long slab_stride, const E* __restrict__ gate,
                                                             long ld_gate, const float* __restrict__ w, float mult, float eps,
                                                             const float* __restrict__ next_w, float* __restrict__ x, E* __restrict__ xb, int dim, int ldb) {
    __shared__ float red[32];
    const long row = blockIdx.x;
    const float* sr = sub + row * ld_sub;
    const E* gr = GATE ? gate + row * ld_gate : nullptr;
    float* xr = x + row * dim;
    E* br = xb + row * ldb;
    float q = 0.f, n = 0.f;
    if constexpr (VEC > 0) {
        typedef E e4 __attribute__((ext_vector_type(4)));
        floatx4 v[VEC ? VEC : 1], xv[VEC ? VEC : 1], wv[VEC ? VEC : 1], wn = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
        for (int c = 0; c < VEC; c++) {
            const int i = (c * blockDim.x + threadIdx.x) * 4;
            if (i < dim) {
                auto rest = [&] {
                    xv[c] = *reinterpret_cast<const floatx4*>(xr + i);
                    wv[c] = *reinterpret_cast<const floatx4*>(w + i);
                };
                if (VEC == 1) rest();
                if (VEC == 1 && NEXT && next_w) wn = *reinterpret_cast<const floatx4*>(next_w + i);
                e4 gv = {};
                if (GATE && VEC == 1) gv = *reinterpret_cast<const e4*>(gr + i);
                v[c] = sum_slabs<VEC == 1>(sr + i, slabs, slab_stride);
                if (GATE && VEC != 1) gv = *reinterpret_cast<const e4*>(gr + i);
                if (VEC != 1) rest();
#pragma unroll
                for (int j = 0; j < 4; j++) { if (GATE) v[c][j] *= (float)gv[j]; q += v[c][j] * v[c][j]; }
            }
        }
        const float inv = mult / sqrtf(block_sum<VEC == 1>(q, red) / (float)dim + eps);
#pragma unroll
        for (int c = 0; c < VEC; c++) {
            const int i = (c * blockDim.x + threadIdx.x) * 4;
            if (i < dim) {
#pragma unroll
                for (int j = 0; j < 4; j++) { xv[c][j] += v[c][j] * inv * wv[c][j]; n += xv[c][j] * xv[c][j]; }
                *reinterpret_cast<floatx4*>(xr + i) = xv[c];
            }
        }
        const float unit = NEXT ? 1.0f / sqrtf(block_sum<VEC == 1>(n, red + 16) / (float)dim + eps) : 1.0f;
#pragma unroll
        for (int c = 0; c < VEC; c++) {
            const int i = (c * blockDim.x + threadIdx.x) * 4;
            if (i < dim) {
                if (VEC != 1 && NEXT && next_w) wn = *reinterpret_cast<const floatx4*>(next_w + i);
                e4 o;
#pragma unroll
                for (int j = 0; j < 4; j++) o[j] = (E)(NEXT ? xv[c][j] * unit * wn[j] : xv[c][j]);
                *reinterpret_cast<e4*>(br + i) = o;
            }
        }
        return;
    }
    auto branch = [&](int i) {
        float t = sr[i];
        for (int z = 1; z < slabs; z++) t += sr[z * slab_stride + i];
        return GATE ? t * (float)gr[i] : t;
    };
    for (int i = threadIdx.x; i < dim; i += blockDim.x) { const float t = branch(i); q += t * t; }
    const float inv = mult / sqrtf(block_sum<VEC == 1>(q, red) / (float)dim + eps);
    for (int i = threadIdx.x; i < dim; i += blockDim.x) {
        const float t = xr[i] + branch(i) * inv * w[i];
        xr[i] = t;
        n += t * t;
        if (!NEXT) br[i] = (E)t;
    }
    if (NEXT) {
        const float unit = 1.0f / sqrtf(block_sum<VEC == 1>(n, red + 16) / (float)dim + eps);
        for (int i = threadIdx.x; i < dim; i += blockDim.x) br[i] = (E)(next_w ? xr[i] * unit * next_w[i] : xr[i] * unit);
    }
}

template <typename E>
int post_norm_add(const float* sub, long ld_sub, int slabs, long slab_stride, const E* gate, long ld_gate, const float* w, float mult, float eps, bool next_norm,
                  const float* next_w, float* x, E* xb, int rows, int dim, int ldb, hipStream_t s) {
    const int threads = rows <= 512 && dim >= 2048 ? 1024 : 256;
    const bool vec = dim % 4 == 0 && dim <= threads * 16 && ld_sub % 4 == 0 && ld_gate % 4 == 0 && ldb % 4 == 0 && slab_stride % 4 == 0;
    auto go = [&](auto v, auto g, auto n) {
        hipLaunchKernelGGL((post_norm_add_kernel<E, decltype(v)::value, decltype(g)::value, decltype(n)::value>), dim3(rows), dim3(threads), 0, s, sub, ld_sub, slabs,
                           slab_stride, gate, ld_gate, w, mult, eps, next_w, x, xb, dim, ldb);
    };
    auto with_next = [&](auto v, auto g) { next_norm ? go(v, g, std::true_type{}) : go(v, g, std::false_type{}); };
    auto with_gate = [&](auto v) { gate ? with_next(v, std::true_type{}) : with_next(v, std::false_type{}); };
    if (!vec) with_gate(std::integral_constant<int, 0>{});
    else if (dim <= threads * 4) with_gate(std::integral_constant<int, 1>{});
    else with_gate(std::integral_constant<int, 4>{});
    FH_CHECK_LAUNCH();
    return 0;
}

template <typename E>
__global__ __launch_bounds__(256) void rms_norm_rows_kernel(const float* __restrict__ x, const int32_t* __restrict__ row_idx,
                                                            const float* __restrict__ w, float eps, E* __restrict__ out, int dim, int ldo) {
    __shared__ float red[16];
    const float* xr = x + (row_idx ? (long)row_idx[blockIdx.x] : (long)blockIdx.x) * dim;
    float q = 0.f;
    // the row and its weights requested together, and read once
    auto held = [&](auto numbers) {
        constexpr int N = decltype(numbers)::value;
        float xv[N], wv[N];
#pragma unroll
        for (int c = 0; c < N; c++) {
            const int i = threadIdx.x + c * 256, at = i < dim ? i : 0;
            wv[c] = w ? w[at] : 1.f;
            xv[c] = xr[at];
        }
#pragma unroll
        for (int c = 0; c < N; c++) q += (int)threadIdx.x + c * 256 < dim ? xv[c] * xv[c] : 0.f;
        const float inv = 1.0f / sqrtf(block_sum(q, red) / (float)dim + eps);
#pragma unroll
        for (int c = 0; c < N; c++) {
            const int i = threadIdx.x + c * 256;
            if (i < dim) out[(long)blockIdx.x * ldo + i] = (E)(xv[c] * inv * wv[c]);
        }
    };
    if (dim <= 2 * 256) return held(std::integral_constant<int, 2>{});
    if (dim <= 8 * 256) return held(std::integral_constant<int, 8>{});
    for (int i = threadIdx.x; i < dim; i += 256) q += xr[i] * xr[i];
    const float inv = 1.0f / sqrtf(block_sum(q, red) / (float)dim + eps);
    for (int i = threadIdx.x; i < dim; i += 256) out[(long)blockIdx.x * ldo + i] = (E)(w ? xr[i] * inv * w[i] : xr[i] * inv);
}
template <typename E>
int rms_norm_rows(const float* x, const int32_t* row_idx, const float* w, float eps, E* out, int rows, int dim, int ldo, hipStream_t s) {
    hipLaunchKernelGGL(rms_norm_rows_kernel<E>, dim3(rows), dim3(256), 0, s, x, row_idx, w, eps, out, dim, ldo);
    FH_CHECK_LAUNCH();
    return 0;
}

// One workgroup per row; a thread holds VEC quads of the row in registers (0: any length, from memory).  POST: the sum itself is normed.
// `copy`: the row in the number format goes there, too.
template <typename E, int VEC, bool POST>
__device__ __forceinline__ void stream_update_row(const StreamUpdate<E>& u, float* red, E* copy) {
    const long row = blockIdx.x;
    const int dim = u.dim, nt = blockDim.x;
    const float *s1 = u.sub + row * u.ld_sub, *s2 = u.sub2 + row * u.ld_sub;
    float* xr = u.x + row * dim;
    const E* pr = u.pairs + row * u.top * u.ld_pair;
    E* out = u.out + row * u.ldo;
    const bool joined = !POST && u.sub2 != nullptr;
    float keep = u.replace ? 0.f : 1.f, factor = 1.f;
    if (POST) {
        keep *= u.keep;
        if (u.sub_scale) factor = u.sub_scale[row];
        if (u.pair_ids)
            for (int j = 0; j < u.top; j++)
                if (u.pair_ids[row * u.top + j] >= u.pair_limit) keep += u.weights[row * u.top + j];
    }
    auto listed = [&](int j) { return !POST || !u.pair_ids || u.pair_ids[row * u.top + j] < u.pair_limit; };
    if constexpr (VEC > 0) {
        typedef E e4 __attribute__((ext_vector_type(4)));
        floatx4 v[VEC ? VEC : 1], r[VEC ? VEC : 1], xv[VEC ? VEC : 1], w1[VEC ? VEC : 1], w2[VEC ? VEC : 1], wn[VEC ? VEC : 1];
        constexpr bool EARLY = VEC == 1;
        // weights, of one quad ahead of the sums that they are for (see above)
        auto branch_weights = [&](int c, int i) {
            if (POST) w1[c] = *reinterpret_cast<const floatx4*>(u.post_w + i);
            if (POST && u.gate) w2[c] = *reinterpret_cast<const floatx4*>(u.gate_w + i);
            if (joined) { w1[c] = *reinterpret_cast<const floatx4*>(u.w + i); w2[c] = *reinterpret_cast<const floatx4*>(u.w2 + i); }
        };
        auto next_weights = [&](int c, int i) {
            wn[c] = (floatx4){1.f, 1.f, 1.f, 1.f};
            if (u.out && u.next_w) wn[c] = *reinterpret_cast<const floatx4*>(u.next_w + i);
        };
        if (EARLY) {
            const int at = threadIdx.x * 4, i = at < dim ? at : 0;
            branch_weights(0, i);
            next_weights(0, i);
        }
        float q1 = 0.f, q2 = 0.f, n = 0.f;
#pragma unroll
        for (int c = 0; c < VEC; c++) {
            const int i = (c * nt + threadIdx.x) * 4;
            if (i < dim) {
                xv[c] = (floatx4){0.f, 0.f, 0.f, 0.f};
                if (EARLY && !u.replace) xv[c] = *reinterpret_cast<const floatx4*>(xr + i);
                if (EARLY && joined) r[c] = sum_slabs(s2 + i, u.slabs2, u.slab_stride2);
                v[c] = (floatx4){0.f, 0.f, 0.f, 0.f};
                if (u.sub) v[c] = sum_slabs<EARLY>(s1 + i, u.slabs, u.slab_stride);
                if (!EARLY && !u.replace) xv[c] = *reinterpret_cast<const floatx4*>(xr + i);
                if (POST)
#pragma unroll
                    for (int k = 0; k < 4; k++) v[c][k] *= factor;
                if (POST)
#pragma unroll
                    for (int k = 0; k < 4; k++) xv[c][k] *= keep;
                if (u.add) xv[c] += *reinterpret_cast<const floatx4*>(u.add + i);
                if (!POST && EARLY)
                    for (int j0 = 0; j0 < u.top; j0 += 8) {             // (eight at once)
                        e4 e[8];
                        float w[8];
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const int at = min(j0 + j, u.top - 1);
                            e[j] = *reinterpret_cast<const e4*>(pr + at * u.ld_pair + i);
                            w[j] = u.weights[row * u.top + at];
                        }
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            if (j0 + j < u.top)
#pragma unroll
                                for (int k = 0; k < 4; k++) v[c][k] += w[j] * (float)e[j][k];
                    }
                else
#pragma unroll 4
                for (int j = 0; j < u.top; j++) {
                    if (!listed(j)) continue;
                    const e4 e = *reinterpret_cast<const e4*>(pr + j * u.ld_pair + i);
                    const float w = u.weights[row * u.top + j];
#pragma unroll
                    for (int k = 0; k < 4; k++) v[c][k] += w * (float)e[k];
                }
                if (joined) {
                    if (!EARLY) r[c] = sum_slabs<false>(s2 + i, u.slabs2, u.slab_stride2);
#pragma unroll
                    for (int k = 0; k < 4; k++) { q1 += v[c][k] * v[c][k]; q2 += r[c][k] * r[c][k]; }
                }
            }
        }
        float i1 = 0.f, i2 = 0.f;
        if (joined) {
            i1 = 0.5f / sqrtf(block_sum<VEC == 1>(q1, red) / (float)dim + u.eps);
            i2 = 0.5f / sqrtf(block_sum<VEC == 1>(q2, red + 16) / (float)dim + u.eps);
        }
#pragma unroll
        for (int c = 0; c < VEC; c++) {
            const int i = (c * nt + threadIdx.x) * 4;
            if (i < dim) {
                if (joined) {
                    if (!EARLY) branch_weights(c, i);
#pragma unroll
                    for (int k = 0; k < 4; k++) v[c][k] = v[c][k] * i1 * w1[c][k] + r[c][k] * i2 * w2[c][k];
                }
                xv[c] += v[c];
#pragma unroll
                for (int k = 0; k < 4; k++) n += xv[c][k] * xv[c][k];
                if (!POST) *reinterpret_cast<floatx4*>(xr + i) = xv[c];
            }
        }
        if (POST) {
            const float inv = 1.0f / sqrtf(block_sum<VEC == 1>(n, red) / (float)dim + u.eps);
            float z = 0.f;
            n = 0.f;
#pragma unroll
            for (int c = 0; c < VEC; c++) {
                const int i = (c * nt + threadIdx.x) * 4;
                if (i < dim) {
                    if (!EARLY) branch_weights(c, i);
                    floatx4 g = {0.f, 0.f, 0.f, 0.f};
                    if (u.gate) g = w2[c];
#pragma unroll
                    for (int k = 0; k < 4; k++) { xv[c][k] *= inv * w1[c][k]; n += xv[c][k] * xv[c][k]; z += xv[c][k] * g[k]; }
                    *reinterpret_cast<floatx4*>(xr + i) = xv[c];
                }
            }
            if (u.gate) {
                z = block_sum<VEC == 1>(z, red + 16);
                if (threadIdx.x == 0) u.gate[row] = 1.0f / (1.0f + expf(-z));
            }
        }
        if (!u.out) return;
        const float unit = u.next_w ? 1.0f / sqrtf(block_sum<VEC == 1>(n, red + 32) / (float)dim + u.eps) : 1.0f;
#pragma unroll
        for (int c = 0; c < VEC; c++) {
            const int i = (c * nt + threadIdx.x) * 4;
            if (i < dim) {
                if (!EARLY) next_weights(c, i);
                e4 o;
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] = (E)(xv[c][k] * unit * wn[c][k]);
                *reinterpret_cast<e4*>(out + i) = o;
                if (copy) *reinterpret_cast<e4*>(copy + i) = o;
            }
        }
        return;
    }
    auto first = [&](int i) {
        float t = u.sub ? s1[i] : 0.f;
        for (int z = 1; z < u.slabs; z++) t += s1[z * u.slab_stride + i];
        t *= factor;
        for (int j = 0; j < u.top; j++)
            if (listed(j)) t += u.weights[row * u.top + j] * (float)pr[j * u.ld_pair + i];
        return t;
    };
    auto second = [&](int i) {
        float t = s2[i];
        for (int z = 1; z < u.slabs2; z++) t += s2[z * u.slab_stride2 + i];
        return t;
    };
    float i1 = 0.f, i2 = 0.f, n = 0.f;
    if (joined) {
        float q1 = 0.f, q2 = 0.f;
        for (int i = threadIdx.x; i < dim; i += nt) { const float a = first(i), b = second(i); q1 += a * a; q2 += b * b; }
        i1 = 0.5f / sqrtf(block_sum<VEC == 1>(q1, red) / (float)dim + u.eps);
        i2 = 0.5f / sqrtf(block_sum<VEC == 1>(q2, red + 16) / (float)dim + u.eps);
    }
    for (int i = threadIdx.x; i < dim; i += nt) {
        float t = joined ? first(i) * i1 * u.w[i] + second(i) * i2 * u.w2[i] : first(i);
        if (u.add) t += u.add[i];
        if (!u.replace) t += POST ? keep * xr[i] : xr[i];
        xr[i] = t;
        n += t * t;
    }
    if (POST) {
        const float inv = 1.0f / sqrtf(block_sum<VEC == 1>(n, red) / (float)dim + u.eps);
        float z = 0.f;
        n = 0.f;
        for (int i = threadIdx.x; i < dim; i += nt) {            // (a thread's own elements)
            const float t = xr[i] * inv * u.post_w[i];
            xr[i] = t;
            n += t * t;
            if (u.gate) z += t * u.gate_w[i];
        }
        if (u.gate) {
            z = block_sum<VEC == 1>(z, red + 16);
            if (threadIdx.x == 0) u.gate[row] = 1.0f / (1.0f + expf(-z));
        }
    }
    if (!u.out) return;
    const float unit = u.next_w ? 1.0f / sqrtf(block_sum<VEC == 1>(n, red + 32) / (float)dim + u.eps) : 1.0f;
    for (int i = threadIdx.x; i < dim; i += nt) out[i] = (E)(u.next_w ? xr[i] * unit * u.next_w[i] : xr[i]);
}
template <typename E, int VEC, bool POST>
__global__ __launch_bounds__(1024) void stream_update_kernel(StreamUpdate<E> u) {
    __shared__ float red[64];
    stream_update_row<E, VEC, POST>(u, red, nullptr);
}

// An update whose rows a router reads next, the router's logits, each row's choice of experts, and by the workgroup that comes last the sorted list of the pairs: one
// launch for three.  A workgroup has its row in LDS and the first of the router's weights, requested ahead of the row, in registers; a wave takes every nw-th step of K
// of all experts as the first operand of the matrix instruction (the row's numbers are alike in all columns), and the waves' sums meet in LDS.
// 32 bits: a wave's sums of 128 products, then sums of those, as in the few-row kernel (relative error of a logit at K = 1024 / 4096, emulated: 2.1 / 2.2e-7, parts summed whole
// 2.9 / 2.9e-7).
// The ids cross workgroups within the launch: written and read past the caches, behind a ticket that the last one puts back.
// Bound by latency: update, router and list of 32 rows of 2048 on 24 experts 4.8 + 5 + 10.5 µs in launches of their own, of which two of three are on the way to the first
// load of each; a step of four such layers 665 → 628 µs, of two layers of 2 rows on 30 experts 226 → 221.
template <typename E, bool POST, bool CORRECTED>
__global__ __launch_bounds__(1024) void stream_update_route_kernel(StreamUpdate<E> u, StreamRoute<E> r) {
    constexpr int EP = 16 / sizeof(E), SK = 4 * EP, AHEAD = 4, N = STREAM_ROUTE_MAX;
    typedef E piece __attribute__((ext_vector_type(EP)));
    __shared__ __attribute__((aligned(16))) E row_lds[4096];
    __shared__ __attribute__((aligned(16))) float part[16][N];
    __shared__ float red[64], logits[N];
    __shared__ int16_t hist[16][N];
    __shared__ int32_t offset[N];
    __shared__ int last;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int a = lane >> 4, b = lane & 15, steps = r.k / SK, tiles = r.n >> 4;
    auto weights = [&](int t, int s) { return *reinterpret_cast<const piece*>(r.w + ((long)t * steps + s) * (64 * EP) + lane * EP); };
    piece ahead[2][AHEAD];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < AHEAD; j++) ahead[t][j] = weights(t, min(wave + j * nw, steps - 1));
    for (int i = u.dim + threadIdx.x; i < r.k; i += blockDim.x) row_lds[i] = (E)0.f;
    stream_update_row<E, 1, POST>(u, red, row_lds);
    __syncthreads();
    floatx4 acc[N / 16];
#pragma unroll
    for (int t = 0; t < N / 16; t++) acc[t] = (floatx4){0.f, 0.f, 0.f, 0.f};
    auto numbers = [&](int s) { return *reinterpret_cast<const piece*>(row_lds + s * SK + a * EP); };
#pragma unroll
    for (int j = 0; j < AHEAD; j++) {
        const int s = wave + j * nw;
        if (s >= steps) continue;
        const piece x = numbers(s);
#pragma unroll
        for (int t = 0; t < N / 16; t++)
            if (t < 2) acc[t] = Frag<E>::mma(ahead[t < 2 ? t : 0][j], x, acc[t]);
            else if (t < tiles) acc[t] = Frag<E>::mma(weights(t, s), x, acc[t]);
    }
    constexpr int FOLD = sizeof(E) == 4 ? 128 / SK : 0;                    // steps of a sum
    floatx4 sums[FOLD ? N / 16 : 1] = {};
    static_assert(!FOLD || FOLD > AHEAD, "the first sum ends behind the steps that were requested ahead");
    int done = AHEAD;
    for (int s = wave + AHEAD * nw; s < steps; s += nw) {
        const piece x = numbers(s);
#pragma unroll
        for (int t = 0; t < N / 16; t++)
            if (t < tiles) acc[t] = Frag<E>::mma(weights(t, s), x, acc[t]);
        if constexpr (FOLD > 0)
            if (++done % FOLD == 0)
#pragma unroll
                for (int t = 0; t < N / 16; t++) {
                    sums[t] += acc[t];
                    acc[t] = (floatx4){0.f, 0.f, 0.f, 0.f};
                }
    }
    if constexpr (FOLD > 0)
#pragma unroll
        for (int t = 0; t < N / 16; t++) acc[t] += sums[t];
#pragma unroll
    for (int t = 0; t < N / 16; t++)
        if (b == 0 && t < tiles) *reinterpret_cast<floatx4*>(&part[wave][16 * t + 4 * a]) = acc[t];
    __syncthreads();
    const long row = blockIdx.x;
    if (wave == 0) {
        if (lane < r.experts) {
            float sum = 0.f;
            for (int w = 0; w < nw; w++) sum += part[w][lane];
            logits[lane] = sum * r.mul + (r.bias ? r.bias[lane] : 0.f);
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        int id;
        float w;
        if (CORRECTED) route_token_corrected<1>(logits, lane, r.experts, r.top, r.rule, id, w);
        else route_token<1>(logits, lane, r.experts, r.top, 1, id, w);
        if (lane < r.top) {
            __hip_atomic_store(r.ids + row * r.top + lane, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            r.weights[row * r.top + lane] = w;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane == 0) {
            last = __hip_atomic_fetch_add(r.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
            if (last) __hip_atomic_store(r.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    if (!last) return;
    const int pairs = u.rows * r.top, listed = r.experts - (CORRECTED ? r.rule.unlisted : 0);
    route_sort_pairs<N>([&] { return (int)threadIdx.x < pairs ? __hip_atomic_load(r.ids + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -1; }, pairs, listed,
                        r.block, r.sorted, r.block_ids, r.total, hist, offset);
}
template <typename E>
static int update_threads(const StreamUpdate<E>& u) { return u.rows <= 512 && u.dim >= 2048 ? 1024 : 256; }
template <typename E>
static int update_quads(const StreamUpdate<E>& u) {
    const int threads = update_threads(u);
    const bool vec = u.dim % 4 == 0 && u.dim <= threads * 16 && u.ld_sub % 4 == 0 && u.ld_pair % 4 == 0 && u.ldo % 4 == 0 && u.slab_stride % 4 == 0 && u.slab_stride2 % 4 == 0;
    return !vec ? 0 : u.dim <= threads * 4 ? 1 : u.dim <= threads * 8 ? 2 : 4;
}
template <typename E>
int stream_update(const StreamUpdate<E>& u, hipStream_t s) {
    FH_REQUIRE(!u.sub2 || (u.sub && u.w && u.w2 && !u.top), "stream update: a second branch needs both norms");
    FH_REQUIRE(u.sub || u.slabs == 1, "stream update: slabs of nothing");
    FH_REQUIRE(u.post_w ? !u.sub2 : u.keep == 1.f && !u.pair_ids && !u.sub_scale && !u.gate, "stream update: factors and the stream's own pairs belong to a normed sum of one branch");
    const int threads = update_threads(u), quads = update_quads(u);
#define UPDATE(V, P) hipLaunchKernelGGL((stream_update_kernel<E, V, P>), dim3(u.rows), dim3(threads), 0, s, u)
    if (u.post_w) { if (quads == 1) UPDATE(1, true); else if (quads == 2) UPDATE(2, true); else if (quads) UPDATE(4, true); else UPDATE(0, true); }
    else { if (quads == 1) UPDATE(1, false); else if (quads == 2) UPDATE(2, false); else if (quads) UPDATE(4, false); else UPDATE(0, false); }
#undef UPDATE
    FH_CHECK_LAUNCH();
    return 0;
}

// (a quad of the row a thread, a thread a pair)
template <typename E>
bool stream_update_route_supports(const StreamUpdate<E>& u, const StreamRoute<E>& r) {
    return update_quads(u) == 1 && u.out && u.dim <= r.k && r.k <= 4096 && r.k % 32 == 0 && r.n <= STREAM_ROUTE_MAX && r.n % 32 == 0 && r.experts <= r.n && u.rows * r.top <= update_threads(u);
}
template <typename E>
int stream_update_route(const StreamUpdate<E>& u, const StreamRoute<E>& r, bool corrected, hipStream_t s) {
    FH_REQUIRE(stream_update_route_supports(u, r) && u.rows > 0 && r.top > 0 && r.top <= r.experts && r.block > 0 && r.ticket, "stream update with a router: %d rows of %d, %d of %d experts",
               u.rows, u.dim, r.top, r.experts);
    FH_REQUIRE(!corrected || moe_route_corrected_supports(r.experts, r.top, r.rule), "stream update with a router: %d groups, %d kept", r.rule.groups, r.rule.keep);
    FH_REQUIRE(!u.sub2 || (u.sub && u.w && u.w2 && !u.top), "stream update: a second branch needs both norms");
    FH_REQUIRE(u.sub || u.slabs == 1, "stream update: slabs of nothing");
    FH_REQUIRE(u.post_w ? !u.sub2 : u.keep == 1.f && !u.pair_ids && !u.sub_scale && !u.gate, "stream update: factors and the stream's own pairs belong to a normed sum of one branch");
    form_hit(FORM_STREAM_ROUTE);
    form_hit(FORM_MOE_ROUTE_SORT);
#define UPDATE(P, C) hipLaunchKernelGGL((stream_update_route_kernel<E, P, C>), dim3(u.rows), dim3(update_threads(u)), 0, s, u, r)
    if (u.post_w) { if (corrected) UPDATE(true, true); else UPDATE(true, false); }
    else { if (corrected) UPDATE(false, true); else UPDATE(false, false); }
#undef UPDATE
    FH_CHECK_LAUNCH();
    return 0;
}

#define INSTANTIATE(E)                                                                                                                  \
    template int embed_tokens<E>(const Embedding<E>&, const BatchView&, float*, E*, int, int, hipStream_t);                              \
    template int branch_add<E>(const float*, long, int, long, const E*, long, const float*, int, float*, E*, int, int, int, hipStream_t); \
    template int post_norm_add<E>(const float*, long, int, long, const E*, long, const float*, float, float, bool, const float*, float*, \
                                  E*, int, int, int, hipStream_t);                                                                      \
    template int stream_update<E>(const StreamUpdate<E>&, hipStream_t);                                                                  \
    template bool stream_update_route_supports<E>(const StreamUpdate<E>&, const StreamRoute<E>&);                                        \
    template int stream_update_route<E>(const StreamUpdate<E>&, const StreamRoute<E>&, bool, hipStream_t);                               \
    template int rms_norm_rows<E>(const float*, const int32_t*, const float*, float, E*, int, int, int, hipStream_t);
INSTANTIATE(bf16)
INSTANTIATE(float)
#undef INSTANTIATE

}  // namespace fh
