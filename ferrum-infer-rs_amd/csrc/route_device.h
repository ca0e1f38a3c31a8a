// Choice of a token's experts on one wave, and the sorted list of a decode batch's pairs in one workgroup (moe.hip, residual_stream.hip).
#pragma once
#include "common.h"
#include "kernels.h"

namespace fh {

// One expert a lane (64 at most), top_k of them by their place among all rather than one after the other: a maximum over the wave costs as much as
// six comparisons with a lane's value.  (A launch of 32 tokens, two a wave, on 24 experts in 8 groups of 3, top 8: 19 → 11 µs, of which
// 7.4 the choice; two tokens on 30, one group: 7.7 → 6.1; bound by the instructions of 16 waves on one CU, with few tokens by their latency.)
// place: how many of the first `n` lanes hold a larger v, the lower lane first on ties; −∞ and NaN are behind all and have no place (≥ 64)
__device__ __forceinline__ int route_place(float v, int lane, int n) {
    const bool in = v > -INFINITY;
    if (!in) v = -INFINITY;
    int place = 0;
    for (int l0 = 0; l0 < n; l0 += 8)                   // (lanes past the n-th hold −∞)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int l = l0 + j;
            const float x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l));
            place += x > v || (x == v && l < lane);
        }
    return in ? place : 64;
}
// Comparisons come in eights.  µs of a launch of 32 tokens, maxima | places: 32 experts, 8 of them 3.43 | 3.01, 6 3.19 | 3.08, 4 2.85 | 3.04; 48, 8 3.42 | 3.37,
// 6 3.18 | 3.42; 24, 4 2.86 | 2.86, 3 2.77 | 2.93; 64, 8 3.45 | 3.76.
__device__ __forceinline__ bool route_by_place(int per_lane, int num_experts, int top_k) { return per_lane == 1 && (num_experts + 7) / 8 * 8 <= 6 * top_k; }
// lane k < top_k: what the lane of place k has, `none` where no lane has it
template <typename T>
__device__ __forceinline__ T route_at_place(T x, int place, int lane, int top_k, T none) {
    static_assert(sizeof(T) == 4, "");
    const int got = __builtin_amdgcn_ds_permute((place < top_k ? place : 63) << 2, __builtin_bit_cast(int, x));
    const int places = __popcll(__ballot(place < top_k));
    return lane < places ? __builtin_bit_cast(T, got) : none;
}
// Router of one token on one wave (E ≤ 64·PER, lane l looks at experts l, l + 64, …): f32 softmax, k argmax-mask passes, ties → lowest
// index.  Lane k ends up with the k-th choice.
template <int PER, typename T>
__device__ __forceinline__ void route_token(const T* __restrict__ row, int lane, int num_experts, int top_k, int norm_topk_prob, int& id, float& weight) {
    float v[PER];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        int e = lane + i * 64;
        v[i] = e < num_experts ? (float)row[e] : -INFINITY;
        mx = fmaxf(mx, v[i]);
    }
    mx = wave_reduce_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        int e = lane + i * 64;
        v[i] = e < num_experts ? expf(v[i] - mx) : 0.f;
        sum += v[i];
    }
    sum = wave_reduce_sum(sum);
    const float inv_sum = 1.0f / sum;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        int e = lane + i * 64;
        v[i] = e < num_experts ? v[i] * inv_sum : -INFINITY;
    }
    float sel_sum = 0.f;
    weight = 0.f;
    id = 0;
    if (route_by_place(PER, num_experts, top_k)) {
        const int place = route_place(v[0], lane, num_experts);
        id = route_at_place(lane, place, lane, top_k, 0);
        weight = route_at_place(v[0], place, lane, top_k, -INFINITY);
        for (int k = 0; k < top_k; k++) sel_sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), k));
    } else
    for (int k = 0; k < top_k; k++) {
        float best = -INFINITY;
        int mine = 1 << 20;
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (v[i] > best) { best = v[i]; mine = lane + i * 64; }       // ascending e within a lane → first max
        const float top = wave_reduce_max(best);
        // lowest index among the lanes that hold the maximum (indices are exact in f32); all −inf: index 0 (router.rs keeps best_idx = 0)
        int best_idx = (int)-wave_reduce_max(best == top && best > -INFINITY ? -(float)mine : -(float)(1 << 20));
        if (best_idx == 1 << 20) best_idx = 0;
        sel_sum += top;
        if (lane == k) { weight = top; id = best_idx; }
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (lane + i * 64 == best_idx) v[i] = -INFINITY;
    }
    if (norm_topk_prob) weight = sel_sum > 0.f ? weight * (1.0f / sel_sum) : 1.0f / (float)top_k;
}

// expert of the largest v on the wave, lowest expert on ties; −1: every v is −∞.  The result is uniform.
template <int PER>
__device__ __forceinline__ int route_best(const float (&v)[PER], float& top) {
    float best = v[0];
#pragma unroll
    for (int i = 1; i < PER; i++) best = fmaxf(best, v[i]);
    top = wave_reduce_max(best);
    int e = -1;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const unsigned long long at = __ballot(v[i] == top && top > -INFINITY);
        if (e < 0 && at) e = i * 64 + __ffsll(at) - 1;
    }
    return e;
}
// x of the lane that differs in bit log2(off), once the lanes below that bit agree
__device__ __forceinline__ float route_partner(float x, int off) {
    return off == 1 ? dpp_move<0xB1>(x) : off == 2 ? dpp_move<0x4E>(x) : off == 4 ? dpp_move<0x141>(x) : off == 8 ? dpp_move<0x140>(x) : __shfl_xor(x, off, 64);
}
// v of experts outside the best rule.keep groups ← −∞; a group counts by the sum of its two largest v
template <int PER>
__device__ __forceinline__ void route_drop_groups(float (&v)[PER], const int (&grp)[PER], int lane, int per_group, const MoeCorrectedRule& rule) {
    if (per_group <= 64 && !(per_group & (per_group - 1))) {
        // groups are aligned runs of lanes: two largest by butterflies, then every group's place among them
        float score[PER];
        int place[PER];
#pragma unroll
        for (int i = 0; i < PER; i++) {
            float m1 = v[i], m2 = -INFINITY;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                if (off >= per_group) continue;
                const float o1 = route_partner(m1, off), o2 = route_partner(m2, off);
                m2 = fmaxf(fminf(m1, o1), fmaxf(m2, o2));
                m1 = fmaxf(m1, o1);
            }
            score[i] = per_group > 1 ? m1 + m2 : m1;
            place[i] = 0;
        }
        for (int g = 0; g < rule.groups; g++) {
            const int at = g * per_group;
            float x = 0.f;
#pragma unroll
            for (int i = 0; i < PER; i++)
                if (at >> 6 == i) x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(score[i]), at & 63));
#pragma unroll
            for (int i = 0; i < PER; i++) place[i] += x > score[i] || (x == score[i] && g < grp[i]);
        }
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (place[i] >= rule.keep) v[i] = -INFINITY;
        return;
    }
    if constexpr (PER == 1) {
        // every lane its own group's two largest, from the group's lanes, and its place among the others'
        const float x = v[0] > -INFINITY ? v[0] : -INFINITY;
        float m1 = -INFINITY, m2 = -INFINITY;
        for (int j = 0; j < per_group; j++) {
            const float o = __shfl(x, grp[0] * per_group + j, 64);
            m2 = fmaxf(m2, fminf(m1, o));
            m1 = fmaxf(m1, o);
        }
        float sum = per_group > 1 ? m1 + m2 : m1;
        if (!(sum > -INFINITY)) sum = -INFINITY;
        int place = 0, real = 0;
        for (int g = 0; g < rule.groups; g++) {
            const float o = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sum), g * per_group));
            place += o > sum || (o == sum && g < grp[0]);
            real += o > -INFINITY;
        }
        // (groups without a value are not chosen; in place of those missing, the first)
        if (!((sum > -INFINITY && place < rule.keep) || (real < rule.keep && grp[0] == 0))) v[0] = -INFINITY;
        return;
    }
    float mine = -INFINITY, top;                     // lane g: group g's
    for (int g = 0; g < rule.groups; g++) {
        float w[PER], second = 0.f;
#pragma unroll
        for (int i = 0; i < PER; i++) w[i] = grp[i] == g ? v[i] : -INFINITY;
        const int e = route_best<PER>(w, top);
        if (per_group > 1) {
            float other;
#pragma unroll
            for (int i = 0; i < PER; i++)
                if (lane + i * 64 == e) w[i] = -INFINITY;
            route_best<PER>(w, other);
            second = other;
        }
        if (lane == g) mine = top + second;
    }
    unsigned long long kept = 0;
    for (int k = 0; k < rule.keep; k++) {
        const float one[1] = {mine};
        const int g = route_best<1>(one, top);
        kept |= 1ull << (g < 0 ? 0 : g);
        if (lane == g) mine = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < PER; i++)
        if (!(kept >> (grp[i] & 63) & 1)) v[i] = -INFINITY;
}
// MoeCorrectedRule of one token on one wave, layout as route_token; ids of all experts, unlisted ones included
template <int PER>
__device__ __forceinline__ void route_token_corrected(const float* __restrict__ row, int lane, int num_experts, int top_k, const MoeCorrectedRule& rule, int& id, float& weight) {
    const int per_group = num_experts / rule.groups;
    float s[PER], v[PER], top;
    int grp[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int e = lane + i * 64;
        s[i] = e >= num_experts ? rule.softmax ? -INFINITY : 0.f : rule.softmax ? row[e] : 1.0f / (1.0f + expf(-row[e]));
        grp[i] = e / per_group;
    }
    if (rule.softmax) {
        float mx = s[0], total = 0.f;
#pragma unroll
        for (int i = 1; i < PER; i++) mx = fmaxf(mx, s[i]);
        mx = wave_reduce_max(mx);
#pragma unroll
        for (int i = 0; i < PER; i++) { s[i] = expf(s[i] - mx); total += s[i]; }
        const float inv = 1.0f / wave_reduce_sum(total);
#pragma unroll
        for (int i = 0; i < PER; i++) s[i] *= inv;
    }
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int e = lane + i * 64;
        v[i] = e < num_experts ? s[i] + rule.correction[e] : -INFINITY;
    }
    if (rule.keep < rule.groups) route_drop_groups<PER>(v, grp, lane, per_group, rule);
    float sum = 0.f;
    weight = 0.f;
    id = 0;
    if (route_by_place(PER, num_experts, top_k)) {
        const int place = route_place(v[0], lane, num_experts);
        id = route_at_place(lane, place, lane, top_k, 0);
        weight = route_at_place(s[0], place, lane, top_k, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[0]), 0)));
        for (int k = 0; k < top_k; k++) sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), k));
    } else
    for (int k = 0; k < top_k; k++) {
        const int e = max(route_best<PER>(v, top), 0);
        float score = 0.f;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            if (e >> 6 == i) score = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[i]), e & 63));
            if (lane + i * 64 == e) v[i] = -INFINITY;
        }
        sum += score;
        if (lane == k) { weight = score; id = e; }
    }
    weight = (rule.raw ? weight : weight / (sum + 1e-20f)) * rule.scale;
}

constexpr int ROUTE_SORT_PAIRS = 1024;
// Pairs sorted by expert, by all threads of a workgroup (as many as there are pairs at least): a thread owns a pair, whose expert `expert_of` names once the workgroup
// has come together (−1, or as many as are listed and more: none).  Its rank among the pairs of its expert is the count in earlier waves (histograms in LDS) plus the
// count in earlier lanes.  N: most experts.
template <int N, typename F>
__device__ __forceinline__ void route_sort_pairs(const F& expert_of, int n_pairs, int num_experts, int block_size, int32_t* __restrict__ sorted, int32_t* __restrict__ block_ids,
                                                 int32_t* __restrict__ total, int16_t (&hist)[16][N], int32_t (&offset)[N]) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, nw = (n_pairs + 63) >> 6;
    for (int i = lane; i < num_experts; i += 64) hist[wave][i] = 0;
    __syncthreads();
    int e = expert_of();
    if (e >= num_experts) e = -1;
    // the lanes with the same expert, bit by bit of its number
    unsigned long long alike = ~0ull;
    for (int bit = 0; (1 << bit) <= num_experts; bit++) {          // (as far as −1 differs from every number)
        const unsigned long long set = __ballot(e >> bit & 1);
        alike &= e >> bit & 1 ? set : ~set;
    }
    const int rank = __popcll(alike & ((1ull << lane) - 1)), same = __popcll(alike);
    if (e >= 0 && rank == 0) hist[wave][e] = (int16_t)same;
    __syncthreads();
    // counts of earlier waves per expert, and the padded start of every expert's rows
    int count = 0;
    if (tid < num_experts)
        for (int w = 0; w < nw; w++) { const int c = hist[w][tid]; hist[w][tid] = (int16_t)count; count += c; }
    if (tid < N) offset[tid] = tid < num_experts ? (count + block_size - 1) / block_size * block_size : 0;
    __syncthreads();
    if (wave == 0) {
        int run[N / 64], sum = 0;
#pragma unroll
        for (int i = 0; i < N / 64; i++) { run[i] = sum; sum += offset[lane * (N / 64) + i]; }
        int incl = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(incl, off, 64);
            if (lane >= off) incl += v;
        }
#pragma unroll
        for (int i = 0; i < N / 64; i++) offset[lane * (N / 64) + i] = incl - sum + run[i];
        if (lane == 63) total[0] = incl;
    }
    __syncthreads();
    if (e >= 0) sorted[offset[e] + hist[wave][e] + rank] = tid;
    if (tid < num_experts) {
        const int o = offset[tid], padded = (count + block_size - 1) / block_size * block_size;
        for (int i = count; i < padded; i++) sorted[o + i] = n_pairs;
        for (int i = 0; i < padded; i += block_size) block_ids[(o + i) / block_size] = tid;
    }
}

}  // namespace fh
