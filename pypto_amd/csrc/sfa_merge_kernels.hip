// Sparse flash attention: the merge of many KV splits' partial results - gfx950 kernels.  They have a code object of their own: beside
// the attention kernels they moved these to other addresses, which cost 32 tokens of 16 K contexts 56.1 -> 57.3 us a call, 26 packed ones 50.4 -> 50.9, with
// the same instructions.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace pto {
namespace {

// sfa_combine_kernel's merge (sfa_kernels.hip) for more than eight splits: a workgroup to each wavefront's part of that one - 16 heads x 64 columns, workgroup b + 2
// (cb / 2) of the block's four - whose four wavefronts take every fourth split, G of them in flight at a time, and whose four sums are then
// merged through LDS, a quarter of the columns to a wavefront.  Latency-bound: few tokens have many splits, and were 16 workgroups a
// token of the other kernel, each with a chain of groups of eight splits: 6.3 us at one token of 16, so 4.1 (with 32); decode calls of
// 2 tokens 33.8 -> 32.5 us, 4: 35.1 / 32.7, 8: 38.5 / 36.5, 16: 41.6 / 41.1, 20: 45.5 / 43.8.  For up to eight splits it is the slower one
// (26 tokens of 8 splits 47.9 -> 48.3, 40 of 6: 56.5 / 58.0).
// grid (tokens with several splits x head groups x 64), 256 lanes
template <int G, bool FP32>
__global__ __launch_bounds__(256) void sfa_combine_many_kernel(const void* __restrict__ partials, const float* __restrict__ part_ml, void* out, int nq,
                                                               int nsplit, int token0, int hgroups)
{
    using P = typename std::conditional<FP32, float, _Float16>::type;
    const P* part_o = static_cast<const P*>(partials);
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    constexpr int ROW = 64 * 2 + 16; // bytes per LDS row of the output block
    __shared__ __align__(16) f32x4 s_acc[4][4][64]; // [wavefront][h, j][lane]
    __shared__ float2 s_ml[4][64];
    __shared__ __align__(16) uint8_t tr[16 * ROW];
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int task = blockIdx.x >> 2, b = blockIdx.x & 1, cb = blockIdx.x & 2;
    const int hb = task & 1, wv = (task >> 1) & 7;
    const int th = task >> 4, hz = th % hgroups, tq = token0 + th / hgroups;
    const int64_t partial = (int64_t)(tq - token0) * nsplit;
    const int hh = wv & 1, dq = wv >> 1;
    const int head0 = hz * SFA_HEADS_PER_WG + 64 * hh + 32 * hb + 16 * b;
    if (head0 >= nq) return; // (uniform)
    float acc[2][8];
#pragma unroll
    for (int x = 0; x < 16; ++x) (&acc[0][0])[x] = 0.f;
    float M = -INFINITY, L = 0.f;
    const int64_t split_stride = (int64_t)hgroups * 8 * 8192;
    const P* frag0 = part_o + ((partial * hgroups + hz) * 8 + wv) * 8192 + hb * 4096 + cb * 1024 + b * 512;
    const float2* ml0 = reinterpret_cast<const float2*>(part_ml) + partial * nq + min(head0 + l16, nq - 1);
    for (int s0 = w; s0 < nsplit; s0 += 4 * G) { // (wave-uniform)
        typename std::conditional<FP32, f32x8, f16x8>::type v[G][2];
        float2 ml[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int s = min(s0 + 4 * j, nsplit - 1);
            const P* base = frag0 + s * split_stride;
            ml[j] = ml0[(int64_t)s * nq];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if constexpr (FP32) {
                    const f32x4 *lo = reinterpret_cast<const f32x4*>(base + h * 1024) + lane, *hi = lo + 64;
                    v[j][h] = __builtin_shufflevector(*lo, *hi, 0, 1, 2, 3, 4, 5, 6, 7);
                } else
                    v[j][h] = *reinterpret_cast<const f16x8*>(base + h * 1024 + lane * 8);
            }
            if (s0 + 4 * j >= nsplit) ml[j].y = 0.f;
        }
        __builtin_amdgcn_sched_barrier(0);
        float Mg = M;
#pragma unroll
        for (int j = 0; j < G; ++j) Mg = ml[j].y > 0.f ? fmaxf(Mg, ml[j].x) : Mg;
        if (Mg != -INFINITY) {
            if (s0 >= 4 * G) {
                const float back = exp2f(M - Mg);
                L *= back;
#pragma unroll
                for (int x = 0; x < 16; ++x) (&acc[0][0])[x] *= back;
            }
            M = Mg;
#pragma unroll
            for (int j = 0; j < G; ++j) {
                const float f = ml[j].y > 0.f ? exp2f(ml[j].x - M) * ml[j].y : 0.f;
                L += f;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[h][e] += (float)v[j][h][e] * f;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) s_acc[w][q][lane] = f32x4{acc[q >> 1][4 * (q & 1)], acc[q >> 1][4 * (q & 1) + 1], acc[q >> 1][4 * (q & 1) + 2], acc[q >> 1][4 * (q & 1) + 3]};
    s_ml[w][lane] = float2{M, L};
    __syncthreads();
    float2 ml[4];
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ml[i] = s_ml[i][lane];
        top = fmaxf(top, ml[i].x);
    }
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float f = ml[i].y > 0.f ? exp2f(ml[i].x - top) : 0.f; // (no split of it attended: M = -inf, L = 0)
        total += f * ml[i].y;
        sum += s_acc[i][w][lane] * f;
    }
    const float inv = total > 0.f ? 1.f / total : 0.f;
    // wavefront w: column run j = w % 2 of column block h = w / 2
    *reinterpret_cast<u32x2*>(tr + l16 * ROW + (32 * (w >> 1) + 16 * (w & 1) + 4 * g) * 2) =
        u32x2{pack_bf16x2(sum[0] * inv, sum[1] * inv), pack_bf16x2(sum[2] * inv, sum[3] * inv)};
    __syncthreads();
    const int r = threadIdx.x >> 3, c = threadIdx.x & 7;
    if (r < 16 && head0 + r < nq)
        *reinterpret_cast<u32x4*>(reinterpret_cast<uint8_t*>(out) + (((int64_t)tq * nq + head0 + r) * SFA_DN + 128 * dq + 32 * cb + 8 * c) * 2) =
            *reinterpret_cast<const u32x4*>(tr + r * ROW + c * 16);
}

} // namespace

hipError_t sfa_combine_many_launch(const SfaArgs& a, int n, int token0, hipStream_t stream)
{
    const int t = a.b * a.s1, hgroups = (a.nq + SFA_HEADS_PER_WG - 1) / SFA_HEADS_PER_WG;
    const dim3 grid((t - token0) * hgroups * 64);
    // (a last round's tokens have up to 16 splits; more are a single token's, or asked for)
    auto merge = token0 > 0 ? sfa_combine_many_kernel<4, true> : n <= 16 ? sfa_combine_many_kernel<4, false> : sfa_combine_many_kernel<8, false>;
    hipLaunchKernelGGL(merge, grid, dim3(256), 0, stream, static_cast<const void*>(a.part_o), a.part_ml, a.out, a.nq, n, token0, hgroups);
    return hipGetLastError();
}

} // namespace pto
