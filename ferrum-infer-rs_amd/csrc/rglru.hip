// Real-gated linear recurrent unit behind a causal depthwise convolution.
//
//   u_t = Σ_j taps[j] · x_{t − taps + 1 + j} + b;   r, i = σ(block-diagonal projections of u);   log a = −8 · r · softplus(λ)
//   S_t = a · S_{t−1} + √(1 − a²) · i · u;   out_t = S_t · y_t
//
// The two gate projections of a channel are computed side by side on the matrix cores (tiles interleaved ra, ri), so one lane holds
// both gates of its (token, channel) and everything from the sigmoids to the state update stays in fp32 registers.  1 − a² is taken as
// 1 − e^(2 log a) by a series where it would cancel.  One token per sequence: that launch also updates the state and writes the output, for blocks of up to 128 channels behind the convolution too.  Portions: decay and drive go to
// memory and a chunked scan (64 tokens per workgroup; chunk totals, carry over chunks, final pass) produces the output.
// A sequence's first token starts from zero whatever its slot holds, so slots are reused without clearing.
#include "common.h"
#include "knobs.h"
#include "layer_ops.h"
#include "short_conv.h"

namespace fh {

template <typename E>
__host__ __device__ inline ShortConv<E> rglru_conv(const RglruDims& d, const RglruBuffers<E>& b) {
    return {b.x, b.ld, b.conv_w, b.conv_b, b.conv_state, b.u, d.wp, d.taps, false};
}

// σ and −expm1 to fp32 rounding with the hardware exponential, reciprocal and square root (a few units in the last place)
__device__ __forceinline__ float gate_sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
// 1 − e^t, t ≤ 0: series below 1/4, where the difference would cancel
__device__ __forceinline__ float one_minus_exp(float t) {
    const float series = -t * (1.0f + t * (0.5f + t * (1.0f / 6.0f + t * (1.0f / 24.0f + t * (1.0f / 120.0f + t * (1.0f / 720.0f + t * (1.0f / 5040.0f)))))));
    return t > -0.25f ? series : 1.0f - __expf(t);
}

// grid (tiles, row blocks, blocks of the block-diagonal projections); a wave owns one 16-channel tile (ra and ri)
template <typename E, int MT, bool STEP>
__global__ __launch_bounds__(256) void rglru_gates_kernel(RglruDims d, RglruBuffers<E> p, BatchView v) {
    constexpr int EP = 16 / sizeof(E), SK = 4 * EP;             // numbers of 16 bytes, K of a step
    typedef E piece_t __attribute__((ext_vector_type(EP)));
    const int lane = threadIdx.x & 63, a = lane >> 4, b = lane & 15, rb = blockIdx.y, g = blockIdx.z;
    const int tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (tile * 16 >= d.bp) return;
    const int ksteps = d.bp / SK;
    const E* xrow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int r = (rb * MT + mt) * 16 + b;
        xrow[mt] = p.u + (long)(r < v.T ? r : v.T - 1) * d.wp + g * d.bp + EP * a;
    }
    const E* wr = p.gate_w + ((long)(g * (d.bp >> 4) + tile) * 2) * ksteps * (64 * EP) + lane * EP;
    floatx4 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) { acc[mt][0] = (floatx4){0.f, 0.f, 0.f, 0.f}; acc[mt][1] = (floatx4){0.f, 0.f, 0.f, 0.f}; }
#pragma unroll 2
    for (int s = 0; s < ksteps; s++) {
        const piece_t w0 = *reinterpret_cast<const piece_t*>(wr + (long)s * (64 * EP)), w1 = *reinterpret_cast<const piece_t*>(wr + (long)(ksteps + s) * (64 * EP));
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const piece_t ax = *reinterpret_cast<const piece_t*>(xrow[mt] + s * SK);
            acc[mt][0] = Frag<E>::mma(ax, w0, acc[mt][0]);
            acc[mt][1] = Frag<E>::mma(ax, w1, acc[mt][1]);
        }
    }
    const int c = g * d.bp + tile * 16 + b;
    const float bra = p.ra_b[c], bri = p.ri_b[c], sp = p.lam[c];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int row = (rb * MT + mt) * 16 + 4 * a + q;
            if (row >= v.T) continue;
            const float r = gate_sigmoid(acc[mt][0][q] + bra), in = gate_sigmoid(acc[mt][1][q] + bri);
            const float log_a = -8.0f * r * sp, decay = __expf(log_a);
            const float drive = __builtin_amdgcn_sqrtf(one_minus_exp(2.0f * log_a)) * in * (float)p.u[(long)row * d.wp + c];
            if (STEP) {
                float* st = p.state + (long)v.slots[row] * d.wp + c;       // (token i belongs to sequence i)
                const float h = v.pos[row] == 0 ? drive : decay * *st + drive;
                *st = h;
                p.out[(long)row * d.wp + c] = (E)(h * (float)p.y[(long)row * p.ld + c]);
            } else {
                p.decay[(long)row * d.wp + c] = decay;
                p.drive[(long)row * d.wp + c] = drive;
            }
        }
}

// One token a sequence: convolution, gates, state and output of 16 rows × a block of up to 128 channels in a workgroup, which is the only one to touch these channels' stored
// inputs.  The gates' weights (64 KiB, in 32 bits 128) are requested ahead of the convolution, whose results its waves, a 16-channel tile each, read from LDS.
// Bound by latency: one row of 2048 channels in 16 blocks 3.7 + 4.0 µs in two launches → 4.4, four rows in 32 bits 4.6 + 8.0 → 7.1; a step of six layers, four of them such, 314 → 299 µs,
// of three in 32 bits with two 291 → 280; 32 rows of three layers 230 → 213 and 387 → 366.
constexpr int STEP_BLOCK = 128, STEP_TAPS = 4;
template <typename E>
__global__ __launch_bounds__(512) void rglru_step_kernel(RglruDims d, RglruBuffers<E> p, BatchView v) {
    constexpr int EP = 16 / sizeof(E), SK = 4 * EP, KS = STEP_BLOCK / SK, PITCH = STEP_BLOCK + EP;
    typedef E piece_t __attribute__((ext_vector_type(EP)));
    typedef typename Frag<E>::v8 v8;
    __shared__ __attribute__((aligned(16))) E u_lds[16 * PITCH];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, a = lane >> 4, b = lane & 15;
    const int g = blockIdx.x, row0 = blockIdx.y * 16, ksteps = d.bp / SK;       // (a wave for each 16 channels)
    const E* wr = p.gate_w + ((long)(g * (d.bp >> 4) + wave) * 2) * ksteps * (64 * EP) + lane * EP;
    piece_t w[2][KS];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int h = 0; h < 2; h++) w[h][s] = *reinterpret_cast<const piece_t*>(wr + (long)(h * ksteps + min(s, ksteps - 1)) * (64 * EP));
    const int c = g * d.bp + wave * 16 + b;
    const float bra = p.ra_b[c], bri = p.ri_b[c], sp = p.lam[c];
    float state[4], y[4];
    float* at[4];
    bool first[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int row = min(row0 + 4 * a + q, v.T - 1);                        // (token i belongs to sequence i)
        at[q] = p.state + (long)v.slots[row] * d.wp + c;
        first[q] = v.pos[row] == 0;
        state[q] = *at[q];
        y[q] = (float)p.y[(long)row * p.ld + c];
    }
    const ShortConv<E> conv = rglru_conv(d, p);
    const int per = d.bp >> 3;
    for (int i = threadIdx.x; i < 16 * per; i += blockDim.x) {
        const int r = i / per, cc = (i - r * per) * 8, ch = g * d.bp + cc, tok = row0 + r;
        if (tok >= v.T) break;
        const int slot = v.slots[tok];
        const bool fresh = v.pos[tok] == 0;
        v8 in[STEP_TAPS];                                                      // (of the token `back` ago; 0: this one)
#pragma unroll
        for (int back = 0; back < STEP_TAPS; back++) in[back] = conv_input(conv, tok, 0, min(back, conv.taps - 1), slot, fresh, ch);
        float acc[8];
#pragma unroll
        for (int k = 0; k < 8; k++) acc[k] = conv.b[ch + k];
#pragma unroll
        for (int back = STEP_TAPS - 1; back >= 0; back--)
            if (back < conv.taps)
#pragma unroll
                for (int k = 0; k < 8; k++) acc[k] += conv.w[(long)(conv.taps - 1 - back) * conv.wp + ch + k] * (float)in[back][k];
        v8 o;
#pragma unroll
        for (int k = 0; k < 8; k++) o[k] = (E)acc[k];
        *reinterpret_cast<v8*>(u_lds + r * PITCH + cc) = o;
#pragma unroll
        for (int back = 0; back < STEP_TAPS - 1; back++)                       // (entry j: the input taps − 2 − j tokens back)
            if (back < conv.taps - 1) *reinterpret_cast<v8*>(conv.state + ((long)slot * (conv.taps - 1) + conv.taps - 2 - back) * conv.wp + ch) = in[back];
    }
    __syncthreads();
    floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < KS; s++) {
        if (s >= ksteps) break;
        const piece_t ax = *reinterpret_cast<const piece_t*>(u_lds + b * PITCH + s * SK + EP * a);
#pragma unroll
        for (int h = 0; h < 2; h++) acc[h] = Frag<E>::mma(ax, w[h][s], acc[h]);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = 4 * a + q, row = row0 + r;
        if (row >= v.T) continue;
        const float gate = gate_sigmoid(acc[0][q] + bra), in = gate_sigmoid(acc[1][q] + bri);
        const float log_a = -8.0f * gate * sp, decay = __expf(log_a);
        const float drive = __builtin_amdgcn_sqrtf(one_minus_exp(2.0f * log_a)) * in * (float)u_lds[r * PITCH + wave * 16 + b];
        const float h = first[q] ? drive : decay * state[q] + drive;
        *at[q] = h;
        p.out[(long)row * d.wp + c] = (E)(h * y[q]);
    }
}

// totals of every chunk that another chunk of its sequence follows: Π decay and the state it would reach from zero
template <typename E>
__global__ __launch_bounds__(256) void rglru_chunk_totals_kernel(RglruDims d, RglruBuffers<E> p, BatchView v) {
    const int c = blockIdx.x * 256 + threadIdx.x, unit = blockIdx.y;
    const int seq = v.units[2 * unit], t0 = v.units[2 * unit + 1];
    if (c >= d.wp || t0 + RGLRU_CHUNK >= (int)v.cu[seq + 1]) return;
    float A = 1.f, h = 0.f;
#pragma unroll 8
    for (int t = 0; t < RGLRU_CHUNK; t++) {
        const float a = p.decay[(long)(t0 + t) * d.wp + c];
        h = a * h + p.drive[(long)(t0 + t) * d.wp + c];
        A *= a;
    }
    p.chunk_a[(long)unit * d.wp + c] = A;
    p.chunk_h[(long)unit * d.wp + c] = h;
}
// chunk_h[unit] ← state before the chunk (one thread per channel of a sequence walks its chunks)
template <typename E>
__global__ __launch_bounds__(64) void rglru_carry_kernel(RglruDims d, RglruBuffers<E> p, BatchView v) {
    const int c = blockIdx.x * 64 + threadIdx.x, unit0 = blockIdx.y;
    const int seq = v.units[2 * unit0];
    if (c >= d.wp || v.units[2 * unit0 + 1] != (int)v.cu[seq]) return;         // only a sequence's first chunk starts a walk
    const int n = cdiv_dev(v.cu[seq + 1] - v.cu[seq], RGLRU_CHUNK);
    float h = v.pos[seq] == 0 ? 0.f : p.state[(long)v.slots[seq] * d.wp + c];
    for (int i = 0; i < n; i += 8) {
        float A[8], H[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const long o = (long)(unit0 + min(i + j, n - 1)) * d.wp + c;
            A[j] = p.chunk_a[o];
            H[j] = p.chunk_h[o];
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (i + j < n) {
                p.chunk_h[(long)(unit0 + i + j) * d.wp + c] = h;
                h = A[j] * h + H[j];
            }
    }
}
// final pass: states of a chunk from its carry, output, and — last chunk of a sequence — the state and convolution tail it leaves
template <typename E>
__global__ __launch_bounds__(256) void rglru_apply_kernel(RglruDims d, RglruBuffers<E> p, BatchView v) {
    const int c = blockIdx.x * 256 + threadIdx.x, unit = blockIdx.y;
    if (c >= d.wp) return;
    const int seq = v.units[2 * unit], t0 = v.units[2 * unit + 1], tok0 = v.cu[seq], end = v.cu[seq + 1], slot = v.slots[seq];
    const int n = min(RGLRU_CHUNK, end - t0);
    const bool fresh = v.pos[seq] == 0, many = end - tok0 > RGLRU_CHUNK;
    float h = many ? p.chunk_h[(long)unit * d.wp + c] : (fresh ? 0.f : p.state[(long)slot * d.wp + c]);
#pragma unroll 8
    for (int t = 0; t < n; t++) {
        const long o = (long)(t0 + t) * d.wp + c;
        h = p.decay[o] * h + p.drive[o];
        p.out[o] = (E)(h * (float)p.y[(long)(t0 + t) * p.ld + c]);
    }
    if (t0 + n < end) return;
    p.state[(long)slot * d.wp + c] = h;
    if (!(c & 7)) conv_store_tail(rglru_conv(d, p), tok0, end - 1 - tok0, slot, fresh, c);
}

template <typename E>
int rglru_forward(const RglruDims& d, const RglruBuffers<E>& b, const BatchView& v, hipStream_t s) {
    const int cb = cdiv(d.wp, 256);
    // a wave for every 16 channels and the inputs in registers: wider blocks and longer convolutions take the two launches
    if (v.single && d.bp <= STEP_BLOCK && d.taps <= STEP_TAPS) {
        form_hit(FORM_RGLRU_STEP);
        hipLaunchKernelGGL(rglru_step_kernel<E>, dim3(d.blocks, cdiv(v.T, 16)), dim3(4 * d.bp), 0, s, d, b, v);
        FH_CHECK_LAUNCH();
        return 0;
    }
    if (int rc = short_conv(rglru_conv(d, b), v, s)) return rc;
    const int mt = v.T <= 16 ? 1 : (v.T <= 32 ? 2 : 4);
    // prompts: the waves of a workgroup share the rows they read; steps: one wave per workgroup, spread over the CUs
    const int nw = v.single ? 1 : 4;
    const dim3 grid(cdiv(d.bp / 16, nw), cdiv(v.T, 16 * mt), d.blocks);
    form_hit(v.single ? FORM_RGLRU_STEP : FORM_RGLRU_SCAN);
#define GATES(MT, ST) hipLaunchKernelGGL((rglru_gates_kernel<E, MT, ST>), grid, dim3(64 * nw), 0, s, d, b, v)
    if (v.single) { if (mt == 1) GATES(1, true); else if (mt == 2) GATES(2, true); else GATES(4, true); }
    else { if (mt == 1) GATES(1, false); else if (mt == 2) GATES(2, false); else GATES(4, false); }
#undef GATES
    FH_CHECK_LAUNCH();
    if (v.single) return 0;
    if (v.num_units > v.num_seqs) {          // some sequence has more than one chunk
        hipLaunchKernelGGL(rglru_chunk_totals_kernel<E>, dim3(cb, v.num_units), dim3(256), 0, s, d, b, v);
        FH_CHECK_LAUNCH();
        hipLaunchKernelGGL(rglru_carry_kernel<E>, dim3(cdiv(d.wp, 64), v.num_units), dim3(64), 0, s, d, b, v);
        FH_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(rglru_apply_kernel<E>, dim3(cb, v.num_units), dim3(256), 0, s, d, b, v);
    FH_CHECK_LAUNCH();
    return 0;
}
template int rglru_forward<bf16>(const RglruDims&, const RglruBuffers<bf16>&, const BatchView&, hipStream_t);
template int rglru_forward<float>(const RglruDims&, const RglruBuffers<float>&, const BatchView&, hipStream_t);

}  // namespace fh
