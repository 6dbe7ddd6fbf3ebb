// Grouped expert selection (GLM-4.5 router): sigmoid, + bias, group maximum, top groups, top-k experts, renormalised
// weights.  Reference: models/glm_v4_5/glm_select_experts.py:60-228 (kernel) and :274-313 (golden);
// python/tests/ut/interpreter/_ops/moe_gating_topk.py:223-287 (groups, -inf fill, scaling factor).
//
// The whole problem is a few MB (8192 x 160 logits): what bounds the kernels is vector instruction issue (many tokens) and
// the length of one wavefront's instruction chain (few), both mostly the sigmoid and the choice of the experts.  Groups are ranked
// by counting (rank of g = number of groups that come before g in the order "value descending, index ascending"), experts by
// merging sorted lists of (ordered score, ~id), or by top_k rounds of an arg-max on them where more than eight are selected.
// select_experts_rows_kernel puts four tokens in a wavefront (the router's shapes); select_experts_kernel, one token per
// wavefront, takes the shapes with more than 16 groups or 16 selected experts.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "kernels.h"
#include "timing.h"

namespace pto {
namespace {

constexpr int SE_MAX_NE = 256;
constexpr int SE_MAX_GROUPS = 64;
constexpr int SE_MAX_K = 32;

__device__ __forceinline__ float load_as_f32(const float* p, int64_t i) { return p[i]; }
__device__ __forceinline__ float load_as_f32(const uint16_t* p, int64_t i) { return __uint_as_float((uint32_t)p[i] << 16); }

// true when (v2, e2) comes before (v, e)
__device__ __forceinline__ int before(float v2, int e2, float v, int e) { return (v2 > v) || (v2 == v && e2 < e); }

// sigmoid(x) = 1 / (1 + exp(-x)) in double precision, rounded once to fp32: the correctly rounded value but for about one
// argument in 10^8, whose exact value lies within 1e-15 of the middle between two floats (as with any double-precision
// exp).  exp by Cody-Waite reduction to |r| <= ln2 / 2 and the Taylor polynomial of degree 12 (remainder below 2e-16), the
// reciprocal by two Newton steps: 33 instructions where the library's exp and division take about 110.  The argument is
// clamped where the fp32 result no longer changes (0 and 1 from |x| = 104 and 17 on).
__device__ __forceinline__ float sigmoid_f32(float x)
{
    const double t = -(double)fminf(fmaxf(x, -200.f), 200.f);
    const double k = __builtin_rint(t * 1.4426950408889634);
    double r = __builtin_fma(k, -0x1.62e42fefa0000p-1, t);     // ln 2 cut to 36 bits: k times it is exact
    r = __builtin_fma(k, -0x1.cf79abc9e3b398p-40, r);          // the rest of ln 2
    double p = 1.0 / 479001600.0;
    p = __builtin_fma(p, r, 1.0 / 39916800.0);
    p = __builtin_fma(p, r, 1.0 / 3628800.0);
    p = __builtin_fma(p, r, 1.0 / 362880.0);
    p = __builtin_fma(p, r, 1.0 / 40320.0);
    p = __builtin_fma(p, r, 1.0 / 5040.0);
    p = __builtin_fma(p, r, 1.0 / 720.0);
    p = __builtin_fma(p, r, 1.0 / 120.0);
    p = __builtin_fma(p, r, 1.0 / 24.0);
    p = __builtin_fma(p, r, 1.0 / 6.0);
    p = __builtin_fma(p, r, 0.5);
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, 1.0);
    const double d = 1.0 + __builtin_amdgcn_ldexp(p, (int)k);
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    return x == x ? (float)y : x; // (the clamp would lose a NaN)
}

// Wavefront-wide maximum of a u32, the same value in every lane, in the vector unit's own lane network (DPP row_shr
// steps inside the rows of 16 lanes, row_bcast15 / row_bcast31 across them).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t se_dpp_from(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}
__device__ __forceinline__ uint32_t se_wave_max(uint32_t v)
{
    v = max(v, se_dpp_from<0x111, 0xf>(v));
    v = max(v, se_dpp_from<0x112, 0xf>(v));
    v = max(v, se_dpp_from<0x114, 0xf>(v));
    v = max(v, se_dpp_from<0x118, 0xf>(v));
    v = max(v, se_dpp_from<0x142, 0xa>(v));
    v = max(v, se_dpp_from<0x143, 0xc>(v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ float ordered_to_f32(uint32_t k)
{
    return __builtin_bit_cast(float, (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// One wavefront per token, everything but the group maxima in registers: lane l holds experts l, l + 64, l + 128,
// l + 192.  Group maxima by LDS atomic maxima on order-preserving keys; group ranks by counting against the other groups'
// maxima read lane by lane (v_readlane); experts by top_k rounds of a wave-wide arg-max in two steps - the largest
// ordered score, then the smallest expert id among the lanes that hold it - both in the lane network (DPP), no trip
// through LDS.  The selected experts' sigmoid values are picked out of their owners' registers with v_readlane.
template <typename LT, typename BT>
__global__ __launch_bounds__(64) void select_experts_kernel(SelectExpertsArgs a)
{
    __shared__ uint32_t s_gkey[SE_MAX_GROUPS];

    const int lane = threadIdx.x;
    const int ne = a.ne, ng = a.n_group, gs = ne / ng;
    const LT* logits = static_cast<const LT*>(a.logits);
    const BT* bias = static_cast<const BT*>(a.bias);
    const float fill = a.fill_neg_inf ? -__builtin_inff() : 0.0f;
    // what does not depend on the token: this lane's experts' groups and bias
    int grp[4];
    float bs[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        grp[j] = e < ne ? e / gs : 0;
        bs[j] = e < ne ? load_as_f32(bias, e) : 0.f;
    }

    for (int64_t tok = blockIdx.x; tok < a.t; tok += gridDim.x) {
        float own_x[4], own_s[4];
        if (lane < ng) s_gkey[lane] = 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = lane + 64 * j;
            own_x[j] = 0.f;
            own_s[j] = 0.f;
            if (e < ne) {
                const float x = load_as_f32(logits, tok * ne + e);
                const float sg = sigmoid_f32(x);
                own_s[j] = sg;
                own_x[j] = sg + bs[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < ne) atomicMax(&s_gkey[grp[j]], f32_to_ordered(own_x[j]));
        __syncthreads();
        // lane g < ng: the maximum of group g, its rank among the groups (value descending, index ascending)
        const float m = ordered_to_f32(s_gkey[lane < ng ? lane : 0]);
        int rank = 0;
        for (int g2 = 0; g2 < ng; ++g2) {
            const float m2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), g2));
            rank += before(m2, g2, m, lane);
        }
        const uint64_t keep = __ballot(lane < ng && rank < a.topk_group);
        // ordered score and inverted id of this lane's experts (0 / 0 for the slots past the last expert and for the
        // experts already taken): the largest (score, ~id) is the largest score and, among equal scores, the smallest id
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = lane + 64 * j;
            if (!((keep >> grp[j]) & 1ull)) own_x[j] = fill;
            hi[j] = e < ne ? f32_to_ordered(own_x[j] + 0.0f) : 0u;
            lo[j] = e < ne ? (uint32_t)(~e) : 0u;
        }
        int my_id = 0;
        float my_w = 0.f, sum = 0.f;
        for (int r = 0; r < a.top_k; ++r) {
            const uint32_t hmax = se_wave_max(max(max(hi[0], hi[1]), max(hi[2], hi[3])));
            uint32_t cand = 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) cand = max(cand, hi[j] == hmax ? lo[j] : 0u);
            const uint32_t lmax = se_wave_max(cand);
            const int e = (int)~lmax;
            // the expert's sigmoid value sits in register e / 64 of lane e % 64
            const int ej = e >> 6;
            const float src = ej == 0 ? own_s[0] : ej == 1 ? own_s[1] : ej == 2 ? own_s[2] : own_s[3];
            const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, src), e & 63));
            sum += w;
            if (lane == r) {
                my_id = e;
                my_w = w;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) hi[j] = (hi[j] == hmax && lo[j] == lmax) ? 0u : hi[j];
        }
        if (lane < a.top_k) {
            a.topk_ids[tok * a.top_k + lane] = my_id;
            const float w = a.renormalize ? my_w / sum : my_w;
            a.topk_weights[tok * a.top_k + lane] = w * a.routed_scaling_factor;
        }
        __syncthreads(); // the group maxima are cleared for the next token only after every lane has read them
    }
}

// The same selection with four tokens per wavefront, one per row of 16 lanes: lane c of a row holds experts 32 i + 2 c and
// 32 i + 2 c + 1 (NS in all), so no lane idles at 160 experts, every cross-lane step serves four tokens at once and logits
// and bias come two to a load.  Reductions run inside the rows - a maximum by four rotations (row_ror 8, 4, 2, 1: every
// lane of the row ends up with it) - group ranks by rotating the row's group maxima past every lane.  For up to 16 groups
// and 16 selected experts (the router's shapes).
//
// (ordered score, ~id) of an expert are the mantissa of one double (order_word), so a comparison of both is one instruction.
// Up to eight selected experts (TOP8): every lane sorts its own and keeps eight, and four merges with the lanes 8, 4, 2 and 1
// places away leave the row's eight in order in all of its lanes - about 300 instructions where eight arg-max rounds over
// score and id took 800.  More: rounds of an arg-max.  The selected experts' sigmoid values are read back from LDS.
// A call with 160 experts, 8 of 4 of 8 groups: 8192 tokens 10.2 us with the library's exp and the rounds, 7.0 now; 8 tokens
// 7.6, 5.2 now (what is left is one wavefront's chain: loads, 33 dependent double-precision steps, the merges).
template <int N>
__device__ __forceinline__ uint32_t row_ror(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x120 + N, 0xf, 0xf, true);
}
template <int N>
__device__ __forceinline__ double row_ror_max(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint64_t o = ((uint64_t)row_ror<N>((uint32_t)(b >> 32)) << 32) | row_ror<N>((uint32_t)b);
    return __builtin_fmax(v, __builtin_bit_cast(double, o));
}
// (ordered value, smaller index first) as one double, exact: 2^52 + value * 256 + (255 - index)
__device__ __forceinline__ double order_word(uint32_t value, int index)
{
    return __builtin_bit_cast(double, 0x4330000000000000ull | ((uint64_t)value << 8) | (uint32_t)(255 - index));
}
__device__ __forceinline__ int order_word_index(double w) { return 255 - (int)(__builtin_bit_cast(uint64_t, w) & 255u); }
// rank of m among the row's words, by rotating the row past every lane: K = 1 .. LAST rotations (the words of a row that
// repeat with period 8 are all seen after 7)
template <int K, int LAST>
__device__ __forceinline__ void rank_step(int& rank, double m)
{
    if constexpr (K <= LAST) {
        const uint64_t b = __builtin_bit_cast(uint64_t, m);
        const uint64_t o = ((uint64_t)row_ror<K>((uint32_t)(b >> 32)) << 32) | row_ror<K>((uint32_t)b);
        rank += __builtin_bit_cast(double, o) > m ? 1 : 0;
        rank_step<K + 1, LAST>(rank, m);
    }
}

// a and b in descending order
__device__ __forceinline__ void order_pair(double& a, double& b)
{
    const double hi = __builtin_fmax(a, b), lo = __builtin_fmin(a, b);
    a = hi;
    b = lo;
}
// k[0 .. N) in descending order: Batcher's odd-even merge sort, N a power of two
template <int N>
__device__ __forceinline__ void sort_desc(double* k)
{
#pragma unroll
    for (int p = 1; p < N; p *= 2)
#pragma unroll
        for (int q = p; q >= 1; q /= 2)
#pragma unroll
            for (int j = q % p; j + q < N; j += 2 * q)
#pragma unroll
                for (int i = 0; i < q; ++i)
                    if (i + j + q < N && (i + j) / (2 * p) == (i + j + q) / (2 * p)) order_pair(k[i + j], k[i + j + q]);
}
// k[0 .. 8), a bitonic sequence, in descending order
__device__ __forceinline__ void merge8_desc(double* k)
{
#pragma unroll
    for (int q = 4; q >= 1; q /= 2)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if ((i & q) == 0) order_pair(k[i], k[i + q]);
}
// k: the eight largest words of the lane, descending -> those of the lane and the lane N places round the row
template <int N>
__device__ __forceinline__ void merge_lanes(double (&k)[8])
{
    double o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint64_t b = __builtin_bit_cast(uint64_t, k[i]);
        o[i] = __builtin_bit_cast(double, ((uint64_t)row_ror<N>((uint32_t)(b >> 32)) << 32) | row_ror<N>((uint32_t)b));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) k[i] = __builtin_fmax(k[i], o[7 - i]);
    merge8_desc(k);
}
// elements e and e + 1 (e even) of a row of n; `pairs`: n is even, so the pair is aligned and inside
__device__ __forceinline__ void load_pair(const float* p, int64_t row, int e, int n, bool pairs, float& a, float& b)
{
    if (pairs) {
        const float2 v = *reinterpret_cast<const float2*>(p + row * n + e);
        a = v.x;
        b = v.y;
    } else {
        a = p[row * n + e];
        b = p[row * n + min(e + 1, n - 1)];
    }
}
__device__ __forceinline__ void load_pair(const uint16_t* p, int64_t row, int e, int n, bool pairs, float& a, float& b)
{
    if (pairs) {
        const uint32_t v = *reinterpret_cast<const uint32_t*>(p + row * n + e);
        a = __uint_as_float(v << 16);
        b = __uint_as_float(v & 0xffff0000u);
    } else {
        a = load_as_f32(p, row * n + e);
        b = load_as_f32(p, row * n + min(e + 1, n - 1));
    }
}

template <typename LT, typename BT, int NS, bool TOP8>
__global__ __launch_bounds__(64) void select_experts_rows_kernel(SelectExpertsArgs a)
{
    __shared__ uint32_t s_gkey[4][16];
    __shared__ float s_sig[4][16 * NS];
    __shared__ __align__(16) float s_w[4][16];

    const int lane = threadIdx.x, row = lane >> 4, c = lane & 15;
    const int ne = a.ne, ng = a.n_group;
    const LT* logits = static_cast<const LT*>(a.logits);
    const BT* bias = static_cast<const BT*>(a.bias);
    const float fill = a.fill_neg_inf ? -__builtin_inff() : 0.0f;
    const bool pairs = (ne & 1) == 0;
    auto expert = [&](int j) { return 32 * (j >> 1) + 2 * c + (j & 1); };

    float bs[NS];
    bool have_bias = false;
    for (int64_t tok0 = (int64_t)blockIdx.x * 4; tok0 < a.t; tok0 += (int64_t)gridDim.x * 4) {
        const int64_t tok = tok0 + row;
        const bool live = tok < a.t;
        const int64_t tl = live ? tok : a.t - 1; // (rows past the last token work on the last one and store nothing)
        float x[NS];
        // (slots past the last expert load it again and are left out below)
#pragma unroll
        for (int j = 0; j < NS; j += 2) load_pair(logits, tl, min(expert(j), (ne - 1) & ~1), ne, pairs, x[j], x[j + 1]);
        if (!have_bias) {
#pragma unroll
            for (int j = 0; j < NS; j += 2) load_pair(bias, 0, min(expert(j), (ne - 1) & ~1), ne, pairs, bs[j], bs[j + 1]);
            have_bias = true;
        }
        float own_x[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const float sg = sigmoid_f32(x[j]);
            own_x[j] = sg + bs[j];
            s_sig[row][expert(j)] = sg;
        }
        uint64_t keep = ~0ull; // bit 16 row + g: group g is kept
        if (ng > 1) { // (uniform) one group is kept whole
            if (c < ng) s_gkey[row][c] = 0u;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NS; ++j)
                if (expert(j) < ne) atomicMax(&s_gkey[row][__umul24((uint32_t)expert(j), a.group_magic) >> 16], f32_to_ordered(own_x[j]));
            __syncthreads();
            // lane g < ng of a row: the maximum of the token's group g and its rank (value descending, index ascending);
            // up to eight groups are held twice by the row
            const int g = ng <= 8 ? c & 7 : c;
            const uint32_t gk = s_gkey[row][g < ng ? g : 0];
            const double m = g < ng ? order_word(f32_to_ordered(ordered_to_f32(gk) + 0.0f), g) : 0.0;
            int rank = 0;
            if (ng <= 8) rank_step<1, 7>(rank, m);
            else rank_step<1, 15>(rank, m);
            keep = __ballot(c < ng && rank < a.topk_group);
        }
        const uint32_t keep_row = (uint32_t)(keep >> (16 * row));
        double key[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int e = expert(j);
            const float v = (keep_row >> (__umul24((uint32_t)e, a.group_magic) >> 16)) & 1u ? own_x[j] : fill;
            const uint32_t hi = f32_to_ordered(v + 0.0f);
            key[j] = e < ne ? order_word(hi, e) : 0.0;
        }
        int my_id = 0;
        if constexpr (TOP8) {
            // the lane's eight largest, in order; then those of 2, 4, 8 and 16 lanes
            double top[8];
            sort_desc<8>(key);
            sort_desc<NS - 8>(key + 8);
#pragma unroll
            for (int i = 0; i < 8; ++i) top[i] = 7 - i < NS - 8 ? __builtin_fmax(key[i], key[15 - i]) : key[i];
            merge8_desc(top);
            merge_lanes<8>(top);
            merge_lanes<4>(top);
            merge_lanes<2>(top);
            merge_lanes<1>(top);
#pragma unroll
            for (int i = 0; i < 8; ++i) my_id = c == i ? order_word_index(top[i]) : my_id;
        } else {
            for (int r = 0; r < a.top_k; ++r) {
                double best = key[0];
#pragma unroll
                for (int j = 1; j < NS; ++j) best = __builtin_fmax(best, key[j]);
                best = row_ror_max<8>(best);
                best = row_ror_max<4>(best);
                best = row_ror_max<2>(best);
                best = row_ror_max<1>(best);
#pragma unroll
                for (int j = 0; j < NS; ++j) key[j] = key[j] == best ? 0.0 : key[j]; // (words are distinct)
                my_id = c == r ? order_word_index(best) : my_id;
            }
        }
        my_id = my_id < ne ? my_id : 0; // (fewer than eight experts in all: the lanes past the last have no word)
        __syncthreads();
        const float my_w = s_sig[row][my_id];
        s_w[row][c] = my_w;
        __syncthreads();
        float sum = 0.f;
        for (int r = 0; r < a.top_k; ++r) sum += s_w[row][r];
        if (live && c < a.top_k) {
            a.topk_ids[tok * a.top_k + c] = my_id;
            const float w = a.renormalize ? my_w / sum : my_w;
            a.topk_weights[tok * a.top_k + c] = w * a.routed_scaling_factor;
        }
        __syncthreads(); // LDS is written for the next tokens only after every lane has read it
    }
}

} // namespace

bool select_experts_supported(int ne, int n_group, int top_k)
{
    return ne > 0 && ne <= SE_MAX_NE && n_group > 0 && n_group <= SE_MAX_GROUPS && ne % n_group == 0 && top_k > 0 &&
           top_k <= SE_MAX_K && top_k <= ne;
}

template <typename LT, typename BT>
static void launch_typed(const SelectExpertsArgs& a, hipStream_t stream)
{
    if (a.n_group <= 16 && a.top_k <= 16) {
        const int64_t wgs = (a.t + 3) / 4;
        const int grid = (int)(wgs < 16384 ? wgs : 16384);
        const bool top8 = a.top_k <= 8;
        auto kern = a.ne <= 160 ? (top8 ? select_experts_rows_kernel<LT, BT, 10, true> : select_experts_rows_kernel<LT, BT, 10, false>)
                                : (top8 ? select_experts_rows_kernel<LT, BT, 16, true> : select_experts_rows_kernel<LT, BT, 16, false>);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(64), 0, stream, a);
    } else {
        const int grid = (int)(a.t < 16384 ? a.t : 16384);
        hipLaunchKernelGGL((select_experts_kernel<LT, BT>), dim3(grid), dim3(64), 0, stream, a);
    }
}

hipError_t select_experts_launch(const SelectExpertsArgs& args, hipStream_t stream)
{
    if (args.t == 0) return hipSuccess;
    SelectExpertsArgs a = args;
    // e / group size = e * ceil(2^16 / group size) >> 16 for e < 256: the product is off by less than e / 2^16 < 1 / group size
    const int gs = a.ne / a.n_group;
    a.group_magic = (uint32_t)((65536 + gs - 1) / gs);
    ScopedKernelTimer timer(KID_SELECT_EXPERTS, stream);
    if (a.logits_bf16) {
        if (a.bias_bf16) launch_typed<uint16_t, uint16_t>(a, stream);
        else launch_typed<uint16_t, float>(a, stream);
    } else {
        if (a.bias_bf16) launch_typed<float, uint16_t>(a, stream);
        else launch_typed<float, float>(a, stream);
    }
    return hipGetLastError();
}

} // namespace pto
