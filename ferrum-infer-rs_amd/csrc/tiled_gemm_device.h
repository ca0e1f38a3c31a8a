// What the epilogues of the projections' kernels share (tiled_gemm.hip, tiled_gemm_wide.hip).
#pragma once
#include "tiled_gemm.h"

namespace fh {

// N neighbouring columns of one section, whose kind of activation is a scalar: one chain of branches for all of them (one for each number made squared
// ReLUs cost a launch of 4096 × 6144 × 2048 21 µs of 115, now 3)
template <typename E, bool RARE, int N, typename V>
__device__ __forceinline__ void gemm_act(const GemmSection& sec, int act, V& v) {
#define EACH(...)                            \
    do {                                     \
        _Pragma("unroll") for (int e = 0; e < N; e++) { const float z = v[e]; v[e] = __VA_ARGS__; } \
        return;                              \
    } while (0)
    if (act == GEMM_ACT_NONE) return;
    if (act == GEMM_ACT_SIGMOID) EACH(ActMath<E>::sigmoid(z));
    if (act == GEMM_ACT_GELU_TANH) EACH(gelu_tanh_f32<E>(z));
    if (act == GEMM_ACT_XIELU) EACH(xielu_f32<E>(z, sec.p, sec.q));
    if (act == GEMM_ACT_RELU2) EACH(fmaxf(z, 0.f) * fmaxf(z, 0.f));
    if (act == GEMM_ACT_SILU) EACH(z * ActMath<E>::sigmoid(z));
    if (RARE && act == GEMM_ACT_SOFTPLUS) EACH(softplus_f32<E>(z));
    if (RARE && act == GEMM_ACT_LOG_SIGMOID) EACH(sec.p * log_sigmoid_f32<E>(z));
    if (RARE && act == GEMM_ACT_SOFTCAP) EACH(sec.p * ActMath<E>::tanh(z / sec.p));
#undef EACH
}
// output row of place r, −1: none
template <typename E>
__device__ __forceinline__ int gemm_out_row(const TiledGemm<E>& p, int r) {
    if (p.rows.id) r = p.rows.id[r];
    return r < p.m ? r : -1;
}
template <typename E, int N, typename V>
__device__ __forceinline__ void gemm_glu(const GemmSection& sec, int act, V& gate, const V& up) {
    if (act == GEMM_ACT_SILU_GLU) {
#pragma unroll
        for (int e = 0; e < N; e++) gate[e] = gate[e] * ActMath<E>::sigmoid(gate[e]) * up[e];
    } else if (act == GEMM_ACT_GELU_GLU) {
#pragma unroll
        for (int e = 0; e < N; e++) gate[e] = gelu_tanh_f32<E>(gate[e]) * up[e];
    } else {
#pragma unroll
        for (int e = 0; e < N; e++) gate[e] = clamped_glu_f32<E>(gate[e], up[e], sec.p, sec.q);
    }
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

// tiles of 256 × 256 (tiled_gemm_wide.hip): whether a launch can have the form (tiled_gemm.h: whether it takes it), and the launch
template <typename E> bool tiled_gemm_wide_supports(const TiledGemm<E>& g);
template <typename E> int tiled_gemm_wide(const TiledGemm<E>& g, hipStream_t s);

}  // namespace fh
