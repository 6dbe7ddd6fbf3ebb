// GLM-4.5 attention_pre_quant (the producer of the query / key / value rows of the paged GQA attention) - gfx950 kernels.
//
// Replaces the device side of attention_pre_quant (models/glm_v4_5/glm_attention_pre_quant.py:633-747; kernel
// quant_attention_pre_kernel :235-505), whose arithmetic is kept step by step:
//   s        = fp32(residual) + fp32(hidden_states);  residual_res = bf16(s)
//   x_norm   = bf16((s / sqrt(sum(s * s * (1 / h)) + eps)) * gamma + bias)                      (:361-386)
//   x_int8   = int8(saturate(rint(fp32(x_norm) * in_scale + in_offset)))                          (:389-396)
//   mm       = bf16(fp32(int32(x_int8 @ weight) + quant_bias) * deq_scale)                        (:398-403)
//   q | k | v = the first q_size, next kv_size, last kv_size outputs                              (:410-425)
//   q, k     = per head of 128: bf16((y / sqrt(sum(y * y / 128) + eps)) * norm_w + norm_b)       (:428-433, :188-218)
//              then on the head's first 2 * half dims (x1, x2): bf16(x1 cos - x2 sin), bf16(x2 cos + x1 sin)  (:446-490)
// Every product and sum above is a separately rounded fp32 operation (no contraction into fma).
//
// At decode sizes (8 - 64 tokens) the operator reads 9 MB of int8 weights once (hidden 5120 x 1792 outputs) and is bound by
// launch latency and that read; three launches:
//   apq_norm_kernel   one workgroup per token: the row is read once and stays in registers across the sum (up to 4 tokens of up to 6144 columns part of the next:
//                     apq_norm_gemm_kernel; up to 160 of hidden 2304 to 6144 a workgroup per 256 pieces of a row: apq_norm_pieces_kernel; where
//                     the sums take the place of an input always this one)
//   apq_gemm_kernel   one workgroup per (128 outputs, 256 to 1024 contraction rows, 32 tokens): the weight tile (output
//                     dimension contiguous in memory) is loaded in one go, parked in LDS and read back with 8-bit
//                     transposing reads as the A operand of the int8 MFMA; int32 partial sums to the workspace (exact,
//                     so the split over the contraction changes nothing)
//   apq_head_kernel   one wavefront per (head, token): sum of the partials, bias, dequantisation, head norm, rotary
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "common.h"
#include "gemm_tile.h"
#include "kernels.h"
#include "prolog_common.h"
#include "timing.h"

namespace pto {
namespace {

constexpr int AD = 128;      // head dim
constexpr int AK = 256;      // contraction rows per workgroup of apq_gemm_kernel
constexpr int AROW = 136;    // bytes per LDS row of the [256][128] int8 weight tile (padded, 8-byte aligned)
constexpr int ATOK = 32;     // tokens per workgroup of apq_gemm_kernel
constexpr int AMAX_H = 16384;

// sum over the 256 lanes of a workgroup in a fixed order; red is 4 floats of LDS (in the lanes' own network: six dependent
// permutes through LDS here and in apq_head_kernel were 0.4 us of the 12.1 of a call of 8 tokens x 14 heads)
__device__ __forceinline__ float block_sum_256(float v, float* red, int tid)
{
    v = wave_sum_descending(v);
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// ------------------------------------------------------------------------------------------------ residual + norm + quant
// grid (tokens), 256 lanes; lane l owns the 8-element pieces l, l + 256, ... of the row (NP of them at most)
template <int NP>
__global__ __launch_bounds__(256) void apq_norm_kernel(AttnPreArgs a)
{
#pragma clang fp contract(off)
    __shared__ float red[4];
    const int tok = blockIdx.x, tid = threadIdx.x;
    const int npieces = a.h / 8;
    const uint16_t* xrow = a.x + (int64_t)tok * a.h;
    const uint16_t* rrow = a.residual + (int64_t)tok * a.h;
    // every load of the kernel goes out before the first use (pieces past the row's end read its last piece again)
    u32x4 xr[NP], rr[NP], gr[NP], br[NP], sr[NP], fr[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int pc = min(tid + 256 * i, npieces - 1);
        xr[i] = reinterpret_cast<const u32x4*>(xrow)[pc];
        rr[i] = reinterpret_cast<const u32x4*>(rrow)[pc];
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int pc = min(tid + 256 * i, npieces - 1);
        gr[i] = reinterpret_cast<const u32x4*>(a.gamma)[pc];
        br[i] = reinterpret_cast<const u32x4*>(a.bias)[pc];
        sr[i] = reinterpret_cast<const u32x4*>(a.in_scale)[pc];
        fr[i] = reinterpret_cast<const u32x4*>(a.in_offset)[pc];
    }
    float s[NP][8];
    float part = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const bool live = tid + 256 * i < npieces;
        u32x4 ro;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float lo = bf16_bits_to_f32(rr[i][e] & 0xffffu) + bf16_bits_to_f32(xr[i][e] & 0xffffu);
            const float hi = bf16_bits_to_f32(rr[i][e] >> 16) + bf16_bits_to_f32(xr[i][e] >> 16);
            s[i][2 * e] = lo;
            s[i][2 * e + 1] = hi;
            ro[e] = pack_bf16x2(lo, hi);
            if (live) {
                part += (lo * lo) * a.mean_coff;
                part += (hi * hi) * a.mean_coff;
            }
        }
        if (live) reinterpret_cast<u32x4*>(a.residual_out + (int64_t)tok * a.h)[tid + 256 * i] = ro;
    }
    const float denom = sqrtf(block_sum_256(part, red, tid) + a.eps);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        if (tid + 256 * i >= npieces) continue;
        int8_t q[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int w = e >> 1, sh = (e & 1) * 16;
            const float g = bf16_bits_to_f32((gr[i][w] >> sh) & 0xffffu), b = bf16_bits_to_f32((br[i][w] >> sh) & 0xffffu);
            const float sc = bf16_bits_to_f32((sr[i][w] >> sh) & 0xffffu), of = bf16_bits_to_f32((fr[i][w] >> sh) & 0xffffu);
            const float xn = round_bf16((s[i][e] / denom) * g + b);
            const float v = __builtin_rintf(xn * sc + of);
            q[e] = (int8_t)(int)fminf(fmaxf(v, -128.f), 127.f);
        }
        *reinterpret_cast<u32x2*>(a.x_q + (int64_t)tok * a.h + 8 * (tid + 256 * i)) = __builtin_bit_cast(u32x2, q);
    }
}

// Eight columns of the sums (bf16, `sums`) and of the quantised row: what apq_norm_kernel does with a piece, of which these are the operands.
__device__ __forceinline__ u32x2 norm_piece(u32x4 x, u32x4 r, u32x4 gamma, u32x4 bias, u32x4 scale, u32x4 offset, float denom, u32x4& sums)
{
#pragma clang fp contract(off)
    int8_t q[8];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float s2[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int sh = e * 16;
            s2[e] = bf16_bits_to_f32((r[w] >> sh) & 0xffffu) + bf16_bits_to_f32((x[w] >> sh) & 0xffffu);
            const float ga = bf16_bits_to_f32((gamma[w] >> sh) & 0xffffu), b = bf16_bits_to_f32((bias[w] >> sh) & 0xffffu);
            const float sc = bf16_bits_to_f32((scale[w] >> sh) & 0xffffu), of = bf16_bits_to_f32((offset[w] >> sh) & 0xffffu);
            const float xn = round_bf16((s2[e] / denom) * ga + b);
            const float v = __builtin_rintf(xn * sc + of);
            q[2 * w + e] = (int8_t)(int)fminf(fmaxf(v, -128.f), 127.f);
        }
        sums[w] = pack_bf16x2(s2[0], s2[1]);
    }
    return __builtin_bit_cast(u32x2, q);
}

// The same with a workgroup to every 256 pieces of a token's row (norm_in_pieces): each adds up the whole row for itself, in the order
// above, and normalises its own piece a lane.  What bounds the kernel above at few tokens is one CU's vector issue: of a
// wavefront's 750 instructions 600 are the 20 to 24 columns that a lane normalises one piece behind the other.
// grid (tokens, pieces / 256 rounded up), 256 lanes
__global__ __launch_bounds__(256) void apq_norm_pieces_kernel(AttnPreArgs a)
{
#pragma clang fp contract(off)
    constexpr int NP = 3; // pieces of the row per lane, for the sum
    __shared__ float red[4];
    const int tok = blockIdx.x, tid = threadIdx.x, npieces = a.h / 8, own = tid + 256 * blockIdx.y, oc = min(own, npieces - 1);
    const u32x4* xrow = reinterpret_cast<const u32x4*>(a.x + (int64_t)tok * a.h);
    const u32x4* rrow = reinterpret_cast<const u32x4*>(a.residual + (int64_t)tok * a.h);
    u32x4 xr[NP], rr[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int pc = min(tid + 256 * i, npieces - 1);
        xr[i] = xrow[pc];
        rr[i] = rrow[pc];
    }
    const u32x4 ox = xrow[oc], orr = rrow[oc], g = reinterpret_cast<const u32x4*>(a.gamma)[oc], b = reinterpret_cast<const u32x4*>(a.bias)[oc];
    const u32x4 sc = reinterpret_cast<const u32x4*>(a.in_scale)[oc], of = reinterpret_cast<const u32x4*>(a.in_offset)[oc];
    __builtin_amdgcn_sched_barrier(0); // (every load is out)
    float part = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const bool live = tid + 256 * i < npieces;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float lo = bf16_bits_to_f32(rr[i][e] & 0xffffu) + bf16_bits_to_f32(xr[i][e] & 0xffffu);
            const float hi = bf16_bits_to_f32(rr[i][e] >> 16) + bf16_bits_to_f32(xr[i][e] >> 16);
            if (live) {
                part += (lo * lo) * a.mean_coff;
                part += (hi * hi) * a.mean_coff;
            }
        }
    }
    const float denom = sqrtf(block_sum_256(part, red, tid) + a.eps);
    if (own >= npieces) return;
    u32x4 sums;
    const u32x2 q = norm_piece(ox, orr, g, b, sc, of, denom, sums);
    const int64_t at = (int64_t)tok * npieces + own;
    reinterpret_cast<u32x4*>(a.residual_out)[at] = sums;
    reinterpret_cast<u32x2*>(a.x_q)[at] = q;
}

// ------------------------------------------------------------------------------------------------ int8 projection
// grid (n_out / 128, splits of the contraction, token tiles of 32), 256 lanes: wave w owns outputs [32 w, 32 w + 32) of
// the tile.  A workgroup takes PER consecutive stages of 256 contraction rows (one where the grid would otherwise not
// fill the chip, more where there are workgroups to spare: fewer partial sums to write and to add up); every load of all
// its stages goes out before the first is used.
template <int PER>
__global__ __launch_bounds__(256) void apq_gemm_kernel(AttnPreArgs a)
{
    __shared__ __align__(16) uint8_t wl[AK * AROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const int col0 = blockIdx.x * AD, split = blockIdx.y, tok0 = blockIdx.z * ATOK;
    const int stages = a.h / AK;
    // B operand (tokens): 16 contraction bytes per lane and MFMA, straight from the quantised rows
    i32x4 qf[PER][AK / 64][2];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int64_t kbase = (int64_t)min(split * PER + j, stages - 1) * AK; // past the end: the last stage again, dropped below
#pragma unroll
        for (int ks = 0; ks < AK / 64; ++ks)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
                qf[j][ks][tb] = *reinterpret_cast<const i32x4*>(a.x_q + (int64_t)min(tok0 + 16 * tb + l16, a.t - 1) * a.h +
                                                                kbase + ks * 64 + 16 * g);
    }
    // the weight tiles: 256 rows of 128 bytes per stage, 16 bytes per lane and load
    const int srow = tid >> 3, spc = tid & 7;
    u32x4 stg[PER][AK / 32];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int64_t kbase = (int64_t)min(split * PER + j, stages - 1) * AK;
#pragma unroll
        for (int i = 0; i < AK / 32; ++i)
            stg[j][i] = *reinterpret_cast<const u32x4*>(a.w + (kbase + srow + 32 * i) * a.n_out + col0 + 16 * spc);
    }
    i32x4 acc[2][2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) acc[db][tb] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (j > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < AK / 32; ++i) {
            u32x2* d = reinterpret_cast<u32x2*>(wl + (srow + 32 * i) * AROW + 16 * spc);
            d[0] = u32x2{stg[j][i][0], stg[j][i][1]};
            d[1] = u32x2{stg[j][i][2], stg[j][i][3]};
        }
        __syncthreads();
        if (split * PER + j >= stages) continue; // uniform over the workgroup
#pragma unroll
        for (int ks = 0; ks < AK / 64; ++ks) {
            // A operand: output 32 w + 16 db + l16, contraction bytes 16 g .. 16 g + 15 of the step.  An 8-bit transposing
            // read hands lane i of a 16-lane group byte i % 8 of the chunks addressed by lanes i / 8, i / 8 + 2, ...: with
            // lane i pointing at row i / 2, column half i % 2, lane i gets column i over rows 0 .. 7
            i32x4 wf[2];
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const uint8_t* p = wl + (ks * 64 + 16 * g + (l16 >> 1)) * AROW + 32 * wave + 16 * db + 8 * (l16 & 1);
                const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 8 * AROW);
                wf[db] = i32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
                    acc[db][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[db], qf[j][ks][tb], acc[db][tb], 0, 0, 0);
        }
    }
    // register e of acc[db][tb]: output 32 w + 16 db + 4 g + e, token 16 tb + l16
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        const int tok = tok0 + 16 * tb + l16;
        if (tok >= a.t) continue;
        int32_t* dst = a.part + ((int64_t)split * a.t + tok) * a.n_out + col0 + 32 * wave + 4 * g;
#pragma unroll
        for (int db = 0; db < 2; ++db) *reinterpret_cast<i32x4*>(dst + 16 * db) = acc[db][tb];
    }
}

// A few tokens' norm and projection in one kernel (norm_in_projection): every workgroup adds up the rows' squares for itself, beside the weights'
// way from memory, and quantises its own columns, so that a launch of one workgroup per token goes.  The operations and their order are
// apq_norm_kernel's, lane by lane; the first column tile's workgroups write the sums of hidden states and residual, and the quantised rows (no kernel reads
// them here, but the workspace's head holds them whatever the number of tokens, and the tests compare them).  T: most tokens,
// T / G of them to a group of 256 lanes.
// grid (n_out / 128, splits of the contraction), 256 G lanes.
template <int PER, int T, int G>
__global__ __launch_bounds__(256 * G) void apq_norm_gemm_kernel(AttnPreArgs a)
{
#pragma clang fp contract(off)
    constexpr int NP = 3, QROW = PER * AK + 16, PIECES = PER * AK / 8; // pieces of 8 elements: of a row per lane, of a token's columns here
    static_assert(G <= 2 && T % G == 0, "");
    constexpr int TG = T / G, LANES = 256 * G, OWN = (T * PIECES + LANES - 1) / LANES, DB = G == 1 ? 2 : 1;
    __shared__ __align__(16) uint8_t wl[AK * AROW];
    __shared__ __align__(16) uint8_t ql[T * QROW];
    __shared__ float red[T][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4, ltid = tid & 255, t0 = TG * (tid >> 8);
    const int col0 = blockIdx.x * AD, split = blockIdx.y;
    const int stages = a.h / AK, npieces = a.h / 8;
    u32x4 xr[TG][NP], rr[TG][NP];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int64_t at = (int64_t)min(t0 + t, a.t - 1) * npieces + min(ltid + 256 * i, npieces - 1);
            xr[t][i] = reinterpret_cast<const u32x4*>(a.x)[at];
            rr[t][i] = reinterpret_cast<const u32x4*>(a.residual)[at];
        }
    // this workgroup's columns: piece tid + LANES i, token by token
    u32x4 ox[OWN], orr[OWN], gr[OWN], br[OWN], sr[OWN], fr[OWN];
    int otok[OWN], opc[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        otok[i] = (tid + LANES * i) / PIECES;
        opc[i] = split * PIECES + (tid + LANES * i) % PIECES;
        const int pc = min(opc[i], npieces - 1);
        const int64_t at = (int64_t)min(otok[i], a.t - 1) * npieces + pc;
        ox[i] = reinterpret_cast<const u32x4*>(a.x)[at];
        orr[i] = reinterpret_cast<const u32x4*>(a.residual)[at];
        gr[i] = reinterpret_cast<const u32x4*>(a.gamma)[pc];
        br[i] = reinterpret_cast<const u32x4*>(a.bias)[pc];
        sr[i] = reinterpret_cast<const u32x4*>(a.in_scale)[pc];
        fr[i] = reinterpret_cast<const u32x4*>(a.in_offset)[pc];
    }
    const int srow = tid >> 3, spc = tid & 7;
    u32x4 stg[PER][AK / 32 / G];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int64_t kbase = (int64_t)min(split * PER + j, stages - 1) * AK;
#pragma unroll
        for (int i = 0; i < AK / 32 / G; ++i)
            stg[j][i] = *reinterpret_cast<const u32x4*>(a.w + (kbase + srow + 32 * G * i) * a.n_out + col0 + 16 * spc);
    }
    __builtin_amdgcn_sched_barrier(0); // (every load is out)
    float part[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        part[t] = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const bool live = ltid + 256 * i < npieces;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float lo = bf16_bits_to_f32(rr[t][i][e] & 0xffffu) + bf16_bits_to_f32(xr[t][i][e] & 0xffffu);
                const float hi = bf16_bits_to_f32(rr[t][i][e] >> 16) + bf16_bits_to_f32(xr[t][i][e] >> 16);
                if (live) {
                    part[t] += (lo * lo) * a.mean_coff;
                    part[t] += (hi * hi) * a.mean_coff;
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < TG; ++t) part[t] = wave_sum_descending(part[t]);
    if (lane == 0)
#pragma unroll
        for (int t = 0; t < TG; ++t) red[t0 + t][wave & 3] = part[t];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        if (otok[i] >= T) continue;
        const float denom = sqrtf(((red[otok[i]][0] + red[otok[i]][1]) + (red[otok[i]][2] + red[otok[i]][3])) + a.eps);
        u32x4 ro;
        const u32x2 q = norm_piece(ox[i], orr[i], gr[i], br[i], sr[i], fr[i], denom, ro);
        *reinterpret_cast<u32x2*>(ql + otok[i] * QROW + 8 * (opc[i] - split * PIECES)) = q;
        if (blockIdx.x == 0 && otok[i] < a.t && opc[i] < npieces) {
            const int64_t at = (int64_t)otok[i] * npieces + opc[i];
            reinterpret_cast<u32x4*>(a.residual_out)[at] = ro;
            reinterpret_cast<u32x2*>(a.x_q)[at] = q;
        }
    }
    i32x4 acc[DB]; // wave w: outputs [16 DB w, +16 DB)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (j > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < AK / 32 / G; ++i) {
            u32x2* d = reinterpret_cast<u32x2*>(wl + (srow + 32 * G * i) * AROW + 16 * spc);
            d[0] = u32x2{stg[j][i][0], stg[j][i][1]};
            d[1] = u32x2{stg[j][i][2], stg[j][i][3]};
        }
        __syncthreads(); // (and ql)
        if (split * PER + j >= stages) continue; // uniform over the workgroup
#pragma unroll
        for (int ks = 0; ks < AK / 64; ++ks) {
            const i32x4 qf = *reinterpret_cast<const i32x4*>(ql + min(l16, T - 1) * QROW + j * AK + 64 * ks + 16 * g);
#pragma unroll
            for (int db = 0; db < DB; ++db) { // (the byte-transposing read: see apq_gemm_kernel)
                const uint8_t* p = wl + (ks * 64 + 16 * g + (l16 >> 1)) * AROW + 16 * (DB * wave + db) + 8 * (l16 & 1);
                const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 8 * AROW);
                acc[db] = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{lo[0], lo[1], hi[0], hi[1]}, qf, acc[db], 0, 0, 0);
            }
        }
    }
    if (l16 >= a.t) return;
    int32_t* dst = a.part + ((int64_t)split * a.t + l16) * a.n_out + col0 + 16 * DB * wave + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db) *reinterpret_cast<i32x4*>(dst + 16 * db) = acc[db];
}

// The projection of a rank's few heads at small prefill sizes (attention_pre_kernel): a workgroup owns 128 tokens x 128 outputs
// over one split of the contraction, so that 14 heads fill the chip where tiles of 256 outputs leave most of it idle (14 heads:
// 144 tokens 21.4 us a call against 23.1, 28 heads, 64 tokens: 19.8 / 21.7).  It walks the split in stages of 128 rows, both
// operands staged through LDS with the next stage's global loads in flight while the current stage is multiplied.  Wave (wr, wc) owns tokens [64 wr, +64) x outputs [64 wc, +64):
// every operand fragment read from LDS feeds four MFMAs, and the weights are read once per 128 tokens instead of once
// per 32.  Same int32 partial sums as apq_gemm_kernel (exact, so neither the tiling nor the split shows).
// grid (n_out / 128, splits, token tiles of 128), 256 lanes.
constexpr int BTOK = 128, BK = 128;
constexpr int BQROW = BK + 16; // bytes per LDS row of the [token][k] int8 tile (padded against bank conflicts)
__global__ __launch_bounds__(256, 3) void apq_gemm_mid_kernel(AttnPreArgs a, int per)
{
    __shared__ __align__(16) uint8_t wl[BK * AROW];
    __shared__ __align__(16) uint8_t ql[BTOK * BQROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4, wr = wave >> 1, wc = wave & 1;
    const int col0 = blockIdx.x * AD, split = blockIdx.y, tok0 = blockIdx.z * BTOK;
    const int st0 = split * per, stages = min(a.h / BK, st0 + per) - st0; // this split's stages of 128 rows
    // 128 rows x 128 bytes of either operand per stage = 4 pieces of 16 bytes per lane (rows tid / 8 + 32 i, piece tid % 8)
    const int srow = tid >> 3, spc = tid & 7;
    const int8_t* wp = a.w + ((int64_t)st0 * BK + srow) * a.n_out + col0 + 16 * spc;
    const int8_t* qp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) qp[i] = a.x_q + (int64_t)min(tok0 + srow + 32 * i, a.t - 1) * a.h + (int64_t)st0 * BK + 16 * spc;
    u32x4 wst[4], qst[4];
    auto load = [&](int st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) qst[i] = *reinterpret_cast<const u32x4*>(qp[i] + st * BK);
#pragma unroll
        for (int i = 0; i < 4; ++i) wst[i] = *reinterpret_cast<const u32x4*>(wp + ((int64_t)st * BK + 32 * i) * a.n_out);
    };
    i32x4 acc[4][4]; // [db][tb]
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) acc[db][tb] = i32x4{0, 0, 0, 0};
    load(0);
    for (int st = 0; st < stages; ++st) {
        __syncthreads(); // everyone is done with the previous stage's tiles
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            u32x2* d = reinterpret_cast<u32x2*>(wl + (srow + 32 * i) * AROW + 16 * spc);
            d[0] = u32x2{wst[i][0], wst[i][1]};
            d[1] = u32x2{wst[i][2], wst[i][3]};
            *reinterpret_cast<u32x4*>(ql + (srow + 32 * i) * BQROW + 16 * spc) = qst[i];
        }
        __syncthreads();
        load(min(st + 1, stages - 1)); // (unconditional: past the end the last stage is fetched again and dropped)
#pragma unroll
        for (int ks = 0; ks < BK / 64; ++ks) {
            i32x4 qf[4], wf[4];
#pragma unroll
            for (int tb = 0; tb < 4; ++tb)
                qf[tb] = *reinterpret_cast<const i32x4*>(ql + (64 * wr + 16 * tb + l16) * BQROW + ks * 64 + 16 * g);
            // (the byte-transposing read: see apq_gemm_kernel)
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const uint8_t* p = wl + (ks * 64 + 16 * g + (l16 >> 1)) * AROW + 64 * wc + 16 * db + 8 * (l16 & 1);
                const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 8 * AROW);
                wf[db] = i32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int tb = 0; tb < 4; ++tb)
                    acc[db][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[db], qf[tb], acc[db][tb], 0, 0, 0);
        }
    }
    // register e of acc[db][tb]: output 64 wc + 16 db + 4 g + e, token 64 wr + 16 tb + l16
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
        const int tok = tok0 + 64 * wr + 16 * tb + l16;
        if (tok >= a.t) continue;
        int32_t* dst = a.part + ((int64_t)split * a.t + tok) * a.n_out + col0 + 64 * wc + 4 * g;
#pragma unroll
        for (int db = 0; db < 4; ++db) *reinterpret_cast<i32x4*>(dst + 16 * db) = acc[db][tb];
    }
}

// a over lanes l and l + 32 in the lower half, b in the upper; of rows of 16 lanes: a over rows 0 and 1, b, a over rows 2 and 3, b
__device__ __forceinline__ float add_halves32(float a, float b)
{
    const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)sw[0]) + __builtin_bit_cast(float, (unsigned)sw[1]);
}
__device__ __forceinline__ float add_rows16(float a, float b)
{
    const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)sw[0]) + __builtin_bit_cast(float, (unsigned)sw[1]);
}

// The projection at prefill sizes and larger decode batches (attention_pre_kernel): a workgroup owns 32 TB tokens x 256 outputs -
// two heads - over one split of the contraction (gemm_tile.h; an odd last head is taken twice and dropped).  An XCD takes
// neighbouring heads.  Where one split covers the whole contraction the head's epilogue runs on the tile: the sums never go to
// memory (777 tokens x 112 heads: 45 MB written and read again, and a kernel of 87 K small workgroups).  Same operations in the
// same order as apq_head_kernel, so the same bits: its sum over the 128 squares is a butterfly over dims 32, 16, .. 1 apart, which
// here are register, lane and register exchanges.
//
// All tiles reach the epilogue together, so nothing covers it; it is bound by its vector instructions, 14336 to 32768 elements to a
// SIMD.  At 224 tokens it took 38 K ticks beside the product's 99 K, of which a division per element and sums exchanged through
// LDS 21 K, rotary pairs from an LDS tile with their cos and sin two loads at a time 15 K; now 20 K:
//  - a quotient is two fused multiply-adds on the product with the reciprocal, which for a bf16 dividend gives the rounded
//    quotient for every pair of mantissas (all 2^30 compared).  It needs that no step under- or overflows: positive scales of
//    2^-60 to 2^60 (a value is 0 or a scale times 1 to 2^32) and divisors of 2^-20 to 2^100, or the wave divides.  (A divisor is
//    the root of an fp32, below 2^64 where it is finite: the least quotient but 0 is above 2^-124, no subnormal);
//  - pairs of rotary dims 16 or 32 apart are registers of one lane, whose cos and sin are loaded before the sums.  The half of a
//    head that has none belongs to every second wave: the two waves of a SIMD get one of each (gt_wave_across);
//  - each wave turns 16 tokens x 64 dims at a time into rows through LDS of its own and stores them while it goes on.
// (777 tokens x 112 heads 82.4 -> 75.0 us a call, 1024 tokens 95.9 -> 88.9.  Tiles of 256 tokens keep 4 registers in scratch memory
// from there on; the product's loop has none.)
// Other rotary widths have pairs in two waves or in broken pieces: the tile goes through LDS.
// grid (heads / 2 rounded up, splits, token tiles), 512 lanes.
template <int TB, bool WHOLE>
__global__ __launch_bounds__(GT_LANES, 2) void apq_gemm_big_kernel(AttnPreArgs a, int per)
{
#pragma clang fp contract(off)
    using T = GtTile<TB>;
    constexpr int OROW = AD * 2 + 16; // bytes per LDS row of a head's bf16 output tile (padded against bank conflicts)
    constexpr int EPI = 2 * T::TOK * OROW + 4 * T::TOK * 4; // two heads' output tiles, sums of squares of [wc][tokens]
    __shared__ __align__(16) uint8_t lds[WHOLE && EPI > T::LDS ? EPI : T::LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = gt_wave_across();
    const int l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    const int tile = gridDim.x % 8 == 0 ? (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8) : (int)blockIdx.x;
    const int heads = a.q_heads + 2 * a.kv_heads, head0 = 2 * tile, head = head0 + (wc >> 1); // of the tile, of this wave
    const int split = blockIdx.y, tok0 = blockIdx.z * T::TOK;
    const int st0 = split * per, stages = min(a.h / GT_KI8, st0 + per) - st0; // this split's stages
    i32x4 acc[4][TB]; // [db][tb]
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[db][tb] = i32x4{0, 0, 0, 0};
    const int8_t* w = a.w + (int64_t)st0 * GT_KI8 * a.n_out;
    gt_product_i8<TB>(acc, w + head0 * AD, w + min(head0 + 1, heads - 1) * AD, a.n_out, a.x_q + (int64_t)st0 * GT_KI8, a.h, tok0, a.t,
                      stages, lds, wave);
    const bool live = head < heads;
    const int hw = 64 * (wc & 1), col0 = min(head, heads - 1) * AD; // this wave's half of its head; the head's columns
    // register e of acc[db][tb]: dim hw + 16 db + 4 g + e of the head, token 16 TB wr + 16 tb + l16
    if constexpr (!WHOLE) {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const int tok = tok0 + 16 * TB * wr + 16 * tb + l16;
            if (tok >= a.t || !live) continue;
            int32_t* dst = a.part + ((int64_t)split * a.t + tok) * a.n_out + col0 + hw + 4 * g;
#pragma unroll
            for (int db = 0; db < 4; ++db) *reinterpret_cast<i32x4*>(dst + 16 * db) = acc[db][tb];
        }
        return;
    }
    float* sums = reinterpret_cast<float*>(lds + 2 * T::TOK * OROW); // [wc][tokens]
    const bool is_q = head < a.q_heads, is_v = head >= a.q_heads + a.kv_heads; // uniform over the wave
    const uint16_t* gp = is_q ? a.q_gamma : a.k_gamma;
    const uint16_t* bp = is_q ? a.q_bias : a.k_bias;
    uint32_t y[4][TB][2]; // [db][tb][e / 2], bf16
    float least = HUGE_VALF, most = 0.f; // of the scales
#pragma unroll
    for (int db = 0; db < 4; ++db) {
        const int dim = hw + 16 * db + 4 * g;
        const f32x4 deq = *reinterpret_cast<const f32x4*>(a.deq + col0 + dim);
        const i32x4 qb = *reinterpret_cast<const i32x4*>(a.qbias + col0 + dim);
        least = fminf(fminf(least, deq[0]), fminf(deq[1], fminf(deq[2], deq[3])));
        most = fmaxf(fmaxf(most, deq[0]), fmaxf(deq[1], fmaxf(deq[2], deq[3])));
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int e = 0; e < 4; e += 2)
                y[db][tb][e / 2] = pack_bf16x2((float)(acc[db][tb][e] + qb[e]) * deq[e], (float)(acc[db][tb][e + 1] + qb[e + 1]) * deq[e + 1]);
    }
    __builtin_amdgcn_sched_barrier(0); // (the loads below once the sums' registers are free)
    const bool here = hw == 0 && !is_v && (a.half == 16 || a.half == 32); // rotary pairs of this wave, in one lane each
    u32x2 cosr[TB][2], sinr[TB][2], gr[4], br[4];
    if (!is_v) {
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            gr[db] = *reinterpret_cast<const u32x2*>(gp + hw + 16 * db + 4 * g);
            br[db] = *reinterpret_cast<const u32x2*>(bp + hw + 16 * db + 4 * g);
        }
        if (here) {
            const uint16_t* cp = a.cos + (int64_t)tok0 * a.half;
            const uint16_t* sp = a.sin + (int64_t)tok0 * a.half;
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int i = 0; i < 2; ++i) { // (16 dims: the same ones twice)
                    const uint32_t at = min(16 * TB * wr + 16 * tb + l16, a.t - 1 - tok0) * a.half + (16 * i & (a.half - 1)) + 4 * g;
                    cosr[tb][i] = *reinterpret_cast<const u32x2*>(cp + at);
                    sinr[tb][i] = *reinterpret_cast<const u32x2*>(sp + at);
                }
        }
        // sums of squares: over dims 32, 16 (registers), 8, 4 (16-lane rows), 2, 1 (registers) apart.  An exchange adds up two
        // values at once, one to either half of the lanes, then to every other row: the four values of e, then four token blocks
        float s[(TB + 3) / 4 * 4];
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            float m[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float sq[4];
#pragma unroll
                for (int db = 0; db < 4; ++db) {
                    const float v = half_of(y[db][tb][e >> 1], e & 1);
                    sq[db] = (v * v) * (1.0f / AD);
                }
                m[e] = (sq[0] + sq[2]) + (sq[1] + sq[3]);
            }
            s[tb] = add_rows16(add_halves32(m[0], m[2]), add_halves32(m[1], m[3])); // in row e the sum for e
        }
#pragma unroll
        for (int tb = TB; tb < (int)(sizeof(s) / sizeof(float)); ++tb) s[tb] = s[TB - 1];
#pragma unroll
        for (int tb = 0; tb < TB; tb += 4) {
            const float sum = add_rows16(add_halves32(s[tb], s[tb + 1]), add_halves32(s[tb + 2], s[tb + 3]));
            const int mine = min(tb + ((g & 1) << 1 | g >> 1), TB - 1); // rows 0, 1, 2, 3: blocks 0, 2, 1, 3
            sums[wc * T::TOK + 16 * TB * wr + 16 * mine + l16] = sum;
        }
    }
    __syncthreads();
    if (!is_v) {
        float denom[TB];
        bool plain = least >= 0x1p-60f && most <= 0x1p60f;
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const int tl = 16 * TB * wr + 16 * tb + l16;
            denom[tb] = sqrtf((sums[(wc & 2) * T::TOK + tl] + sums[(wc | 1) * T::TOK + tl]) + a.eps);
            plain = plain && denom[tb] >= 0x1p-20f && denom[tb] <= 0x1p100f;
        }
        auto norm = [&](auto quotient) {
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
#pragma unroll
                for (int db = 0; db < 4; ++db) // (taken apart anew, not kept in fp32 since the sums)
                    asm("" : "+v"(y[db][tb][0]), "+v"(y[db][tb][1]));
                const float r = 1.0f / denom[tb];
#pragma unroll
                for (int db = 0; db < 4; ++db)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        float x[2];
#pragma unroll
                        for (int e = 0; e < 2; ++e)
                            x[e] = quotient(half_of(y[db][tb][i], e), denom[tb], r) * half_of(gr[db][i], e) + half_of(br[db][i], e);
                        y[db][tb][i] = pack_bf16x2(x[0], x[1]);
                    }
            }
        };
        if (__all(plain))
            norm([](float x, float d, float r) {
                const float q = x * r;
                return __builtin_fmaf(__builtin_fmaf(-q, d, x), r, q);
            });
        else
            norm([](float x, float d, float) { return x / d; });
    }
    if (a.half == 16 || a.half == 32) {
        auto rotate = [&](auto first, auto second, int tb, int j) { // blocks of 16 dims that hold a pair's dims
            uint32_t(&lo)[2] = y[decltype(first)::value][tb];
            uint32_t(&hi)[2] = y[decltype(second)::value][tb];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float r[2][2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float x1 = half_of(lo[i], e), x2 = half_of(hi[i], e), c = half_of(cosr[tb][j][i], e), sn = half_of(sinr[tb][j][i], e);
                    r[0][e] = x1 * c - x2 * sn;
                    r[1][e] = x2 * c + x1 * sn;
                }
                lo[i] = pack_bf16x2(r[0][0], r[0][1]);
                hi[i] = pack_bf16x2(r[1][0], r[1][1]);
            }
        };
        using std::integral_constant;
        constexpr integral_constant<int, 0> b0{};
        constexpr integral_constant<int, 1> b1{};
        constexpr integral_constant<int, 2> b2{};
        constexpr integral_constant<int, 3> b3{};
        if (here) {
            if (a.half == 32) {
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) rotate(b0, b2, tb, 0), rotate(b1, b3, tb, 1);
            } else {
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) rotate(b0, b1, tb, 0);
            }
        }
        // 16 tokens x 64 dims at a time to where the wave alone reads them back as pieces of 16 bytes
        constexpr int WROW = 128 + 16;
        uint8_t* own = lds + wave * (2 * 16 * WROW);
        static_assert(8 * 2 * 16 * WROW <= 2 * T::TOK * OROW, "the sums lie behind");
        uint16_t* dst = is_v ? a.v + (int64_t)(head - a.q_heads - a.kv_heads) * AD
                             : is_q ? a.q + (int64_t)head * AD
                                    : a.k + (int64_t)(head - a.q_heads) * AD;
        const int64_t pitch = (int64_t)(is_q ? a.q_heads : a.kv_heads) * AD;
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            uint8_t* at = own + (tb & 1) * (16 * WROW);
#pragma unroll
            for (int db = 0; db < 4; ++db)
                *reinterpret_cast<u32x2*>(at + l16 * WROW + 32 * db + 8 * g) = u32x2{y[db][tb][0], y[db][tb][1]};
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = 8 * i + (lane >> 3), tok = tok0 + 16 * TB * wr + 16 * tb + row;
                const u32x4 o = *reinterpret_cast<const u32x4*>(at + row * WROW + 16 * (lane & 7));
                if (tok < a.t && live) *reinterpret_cast<u32x4*>(dst + (int64_t)tok * pitch + hw + 8 * (lane & 7)) = o;
            }
            __builtin_amdgcn_wave_barrier();
        }
        return;
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int db = 0; db < 4; ++db)
            *reinterpret_cast<u32x2*>(lds + ((wc >> 1) * T::TOK + 16 * TB * wr + 16 * tb + l16) * OROW + (hw + 16 * db + 4 * g) * 2) =
                u32x2{y[db][tb][0], y[db][tb][1]};
    __syncthreads();
    // tokens x 16 pieces of 8 dims, a head to four waves; a piece's rotary partners are half dims further on or back
    const int ohead = head0 + (tid >> 8), otid = tid & 255;
    if (ohead >= heads) return;
    const bool oq = ohead < a.q_heads, ov = ohead >= a.q_heads + a.kv_heads;
    const int d0 = 8 * (otid & 15), half = a.half;
    uint16_t* dst = ov   ? a.v + (int64_t)(ohead - a.q_heads - a.kv_heads) * AD
                    : oq ? a.q + (int64_t)ohead * AD
                         : a.k + (int64_t)(ohead - a.q_heads) * AD;
    const int64_t pitch = (int64_t)(oq ? a.q_heads : a.kv_heads) * AD;
#pragma unroll 2
    for (int i = 0; i < T::TOK / 16; ++i) {
        const int tl = (otid >> 4) + 16 * i, tok = tok0 + tl;
        if (tok >= a.t) break;
        const uint16_t* row = reinterpret_cast<const uint16_t*>(lds + ((tid >> 8) * T::TOK + tl) * OROW);
        u32x4 o = *reinterpret_cast<const u32x4*>(row + d0);
        if (!ov && d0 < 2 * half) {
            const uint16_t* cp = a.cos + (int64_t)tok * half;
            const uint16_t* sp = a.sin + (int64_t)tok * half;
            if (half % 8 == 0) { // whole pieces on either side
                const bool first = d0 < half;
                const int ci = first ? d0 : d0 - half;
                const u32x4 x = *reinterpret_cast<const u32x4*>(row + (first ? d0 + half : d0 - half));
                const u32x4 cv = *reinterpret_cast<const u32x4*>(cp + ci), sv = *reinterpret_cast<const u32x4*>(sp + ci);
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    float r[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int sh = 16 * e;
                        const float yn = bf16_bits_to_f32((o[w] >> sh) & 0xffffu), xp = bf16_bits_to_f32((x[w] >> sh) & 0xffffu);
                        const float cs = bf16_bits_to_f32((cv[w] >> sh) & 0xffffu), sn = bf16_bits_to_f32((sv[w] >> sh) & 0xffffu);
                        const float p0 = yn * cs, p1 = xp * sn;
                        r[e] = first ? p0 - p1 : p0 + p1;
                    }
                    o[w] = pack_bf16x2(r[0], r[1]);
                }
            } else {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    float r[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int dim = d0 + 2 * w + e;
                        r[e] = bf16_to_f32(row[dim]);
                        if (dim < half)
                            r[e] = r[e] * bf16_to_f32(cp[dim]) - bf16_to_f32(row[dim + half]) * bf16_to_f32(sp[dim]);
                        else if (dim < 2 * half)
                            r[e] = r[e] * bf16_to_f32(cp[dim - half]) + bf16_to_f32(row[dim - half]) * bf16_to_f32(sp[dim - half]);
                    }
                    o[w] = pack_bf16x2(r[0], r[1]);
                }
            }
        }
        *reinterpret_cast<u32x4*>(dst + (int64_t)tok * pitch + d0) = o;
    }
}

// ------------------------------------------------------------------------------------------------ heads
// grid (q_heads + 2 kv_heads, tokens / 4 rounded up), 256 lanes: a wave owns a head of a token, a lane its dims l and 64 + l.
// Latency-bound: one or two trips for the partial sums (S: splits whose loads are out together; in eights, and what is left over one by one, 20 splits
// were six trips: a call of 8 tokens x 28 heads 14.2 us, 13.7 this way, GLM layer of 8 sequences 30.7 / 29.8; 24 and 32 splits by 20 are loads for 40: in
// eights / by 20 / by 16, 14 heads, 32 tokens, 24 splits 14.8 / 14.6 / 14.3, 32: 17.6 / 17.8 / 17.6, 28 heads, 8 tokens, 24: 13.6 / 12.2 / 12.0, 32: 15.1 / 15.2 /
// 15.0, 32 tokens, 16: 13.6 / 13.3 / 13.1), the rest in registers (the sum over the dims adds in the order of 64-lane halves, 32, 16, .. 1 apart, then the halves).
template <int S>
__global__ __launch_bounds__(256) void apq_head_kernel(AttnPreArgs a)
{
#pragma clang fp contract(off)
    const int head = blockIdx.x, tok = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (tok >= a.t) return;
    const bool is_q = head < a.q_heads, is_v = head >= a.q_heads + a.kv_heads;
    // what the epilogue reads goes out first
    const uint16_t* gp = is_q ? a.q_gamma : a.k_gamma;
    const uint16_t* bp = is_q ? a.q_bias : a.k_bias;
    const int rot = 2 * a.half;
    float deq[2], gam[2], bia[2], cs[2], sn[2];
    int32_t qb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int dim = 64 * j + lane;
        deq[j] = a.deq[head * AD + dim];
        qb[j] = a.qbias[head * AD + dim];
        gam[j] = bf16_to_f32(gp[dim]);
        bia[j] = bf16_to_f32(bp[dim]);
        const int ci = dim < a.half ? dim : (dim < rot ? dim - a.half : 0);
        cs[j] = bf16_to_f32(a.cos[(int64_t)tok * a.half + ci]);
        sn[j] = bf16_to_f32(a.sin[(int64_t)tok * a.half + ci]);
    }
    int32_t sum[2] = {0, 0};
    const int32_t* pp = a.part + (int64_t)tok * a.n_out + head * AD + lane;
    const int64_t pstride = (int64_t)a.t * a.n_out;
    // S splits' loads in flight together (a split past the end is the last one again and adds nothing)
    for (int s0 = 0; s0 < a.ksplits; s0 += S) {
        int32_t v[S][2];
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const int32_t* p = pp + min(s0 + i, a.ksplits - 1) * pstride;
            v[i][0] = p[0];
            v[i][1] = p[64];
        }
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) sum[j] += s0 + i < a.ksplits ? v[i][j] : 0;
    }
    float y[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) y[j] = round_bf16((float)(sum[j] + qb[j]) * deq[j]);
    if (is_v) {
        uint16_t* dst = a.v + ((int64_t)tok * a.kv_heads + head - a.q_heads - a.kv_heads) * AD + lane;
        dst[0] = f32_to_bf16(y[0]);
        dst[64] = f32_to_bf16(y[1]);
        return;
    }
    const float m[2] = {wave_sum_descending((y[0] * y[0]) * (1.0f / AD)), wave_sum_descending((y[1] * y[1]) * (1.0f / AD))};
    const float denom = sqrtf((m[0] + m[1]) + a.eps);
    float yn[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) yn[j] = round_bf16((y[j] / denom) * gam[j] + bia[j]);
    uint16_t* dst = is_q ? a.q + ((int64_t)tok * a.q_heads + head) * AD : a.k + ((int64_t)tok * a.kv_heads + head - a.q_heads) * AD;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int dim = 64 * j + lane;
        const int from = dim < a.half ? dim + a.half : dim - a.half; // the rotary partner, if the dim has one
        const float x0 = __shfl(yn[0], from & 63, 64), x1 = __shfl(yn[1], from & 63, 64), x = from & 64 ? x1 : x0;
        float o = yn[j];
        if (dim < a.half)
            o = yn[j] * cs[j] - x * sn[j];
        else if (dim < rot)
            o = yn[j] * cs[j] + x * sn[j];
        dst[dim] = f32_to_bf16(o);
    }
}

} // namespace

bool attention_pre_supported(int64_t h, int64_t d, int64_t half)
{
    return d == AD && h > 0 && h % AK == 0 && h <= AMAX_H && half >= 1 && 2 * half <= AD;
}

static uint64_t align256(uint64_t v) { return (v + 255) & ~(uint64_t)255; }

// stages of 256 contraction rows per workgroup of apq_gemm_kernel: as many (1, 2 or 4) as still leave enough workgroups
// (14 heads, 33 tokens, 560 workgroups of one stage: 17.0 us a call, 280 of two 15.6; 28 heads, 32 tokens: 18.9 / 18.1)
static int stages_per_split(int64_t t, int64_t h, int64_t n_out)
{
    const int64_t wgs = (n_out / AD) * (h / AK) * ((t + ATOK - 1) / ATOK);
    return wgs >= 8 * 448 ? 4 : wgs >= 480 ? 2 : 1;
}

// stages of 128 rows per workgroup of apq_gemm_mid_kernel - all of them while that still leaves 256 workgroups, otherwise as
// many as do
static int mid_stages_per_split(int64_t t, int64_t h, int64_t n_out)
{
    const int64_t tiles = (n_out / AD) * ((t + BTOK - 1) / BTOK), stages = h / BK;
    const int64_t splits = std::min<int64_t>(stages, std::max<int64_t>(1, (256 + tiles - 1) / tiles));
    return (int)((stages + splits - 1) / splits);
}

// Prefill sizes: token blocks of the tile and stages of 128 rows per workgroup of apq_gemm_big_kernel, by the time they should
// take in ns (gt_time_ns); partial sums are written, read again at 8 TB/s (the caches hold them) and cost the head kernel.
struct BigPlan { int tb, per; };
static BigPlan big_plan(int64_t t, int64_t h, int64_t n_out)
{
    const int64_t cols = (n_out / AD + 1) / 2, stages = h / GT_KI8;
    BigPlan best = {8, (int)stages};
    int64_t best_ns = INT64_MAX;
    for (const int64_t want : {1, 2, 3, 4, 5, 6, 8, 10}) {
        const int64_t per = (stages + want - 1) / want, splits = (stages + per - 1) / per;
        const int64_t sums = splits > 1 ? 4000 + t * n_out * 8 * splits / 8000 : 0;
        for (int tb = 4; tb <= 8; ++tb) {
            const int64_t ns = gt_time_ns(cols * splits * ((t + 32 * tb - 1) / (32 * tb)), per, tb) + sums;
            if (ns < best_ns) best = {tb, (int)per}, best_ns = ns;
        }
    }
    return best;
}

// The projection's kernel.  The streamed one up to 32 tokens, but only up to 8 where the weights are large (112 heads: 12 tokens
// 24.8 us a call against 22.2 by tiles of 256 outputs, 24: 29.6 / 24.3, 100: 77 / 32; 28 heads and 12 tokens are the same, 14
// heads 13.1 / 14.3), and up to 128 tokens with up to 16 heads (14 heads, 128 x 128 tiles in the middle, 256 outputs last: 33 tokens
// 15.6 / 16.6 / 17.0, 97: 19.9 / 20.6 / 21.3, 128: 22.4 / 22.4 / 23.6, 129: 22.5 / 21.0 / 23.2).  128 x 128 tiles with up to 16 heads
// up to 192 tokens, with up to 32 up to 160, and again where a third token tile has just begun (14 heads: 160 tokens 22.6
// against 23.9, 192: 23.7 / 24.0, 224: 24.8 / 24.5, 257: 25.8 / 26.8, 320: 28.0 / 26.8; 28 heads: 97 tokens 22.7 / 23.8, 160:
// 25.2 / 26.5, 161: 25.3 / 24.7, 288: 31.9 / 32.6; 56 heads, 64 tokens: 24.8 / 22.6).
enum class ApqKernel { stream, mid, tiles };
static ApqKernel attention_pre_kernel(int64_t t, int64_t n_out)
{
    if (t <= 8 || (t <= 32 && n_out < 8192) || (t <= 128 && n_out <= 16 * AD)) return ApqKernel::stream;
    const int64_t two_tiles = n_out <= 16 * AD ? 192 : 160;
    return n_out <= 32 * AD && (t <= two_tiles || (t > 256 && t <= 288)) ? ApqKernel::mid : ApqKernel::tiles;
}

int attention_pre_ksplits(int64_t t, int64_t h, int64_t n_out)
{
    const ApqKernel kernel = attention_pre_kernel(t, n_out);
    const int per = kernel == ApqKernel::tiles ? big_plan(t, h, n_out).per
                                               : kernel == ApqKernel::mid ? mid_stages_per_split(t, h, n_out) : stages_per_split(t, h, n_out);
    const int rows = kernel == ApqKernel::tiles ? GT_KI8 : kernel == ApqKernel::mid ? BK : AK;
    return (int)((h / rows + per - 1) / per);
}

// one split at prefill sizes: the projection's workgroups finish their heads themselves, no sums go through memory
static bool attention_pre_whole(int64_t t, int64_t n_out, int ksplits)
{
    return attention_pre_kernel(t, n_out) == ApqKernel::tiles && ksplits == 1;
}

uint64_t attention_pre_workspace_bytes(int64_t t, int64_t h, int64_t n_out)
{
    if (attention_pre_whole(t, n_out, attention_pre_ksplits(t, h, n_out))) return align256((uint64_t)t * h);
    return align256((uint64_t)t * h) + (uint64_t)attention_pre_ksplits(t, h, n_out) * t * n_out * sizeof(int32_t);
}

void attention_pre_bind_workspace(AttnPreArgs& a, void* ws)
{
    a.x_q = static_cast<int8_t*>(ws);
    a.part = reinterpret_cast<int32_t*>(static_cast<uint8_t*>(ws) + align256((uint64_t)a.t * a.h));
}

// f(integral constants: stages per split, most tokens, groups of lanes) for norm_in_projection's kernel
template <class F>
static void norm_gemm_dispatch(int per, int t, F&& f)
{
    auto tokens = [&](auto p) {
        if (t == 1)
            f(p, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
        else if (t == 2)
            f(p, std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
        else
            f(p, std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
    };
    if (per == 4)
        tokens(std::integral_constant<int, 4>{});
    else if (per == 2)
        tokens(std::integral_constant<int, 2>{});
    else
        tokens(std::integral_constant<int, 1>{});
}

// The sums of hidden states and residual may take the place of either: then one workgroup has to read and write a row.
static bool rows_apart(const AttnPreArgs& a)
{
    const uint64_t bytes = (uint64_t)a.t * a.h * 2, to = (uint64_t)a.residual_out, x = (uint64_t)a.x, r = (uint64_t)a.residual;
    return (to + bytes <= x || x + bytes <= to) && (to + bytes <= r || r + bytes <= to);
}
// Up to 4 tokens the norm joins the projection: every workgroup reads all rows, 20 KB a token (us a call, a kernel of its own / joined, three sets of
// operands: 14 heads, 1 token 10.8 / 8.4, 2: 11.0 / 9.0, 4: 11.7 / 10.8, 8: 12.1 / 14.7; 28 heads 12.9 / 9.7, 13.2 / 10.4, 13.6 / 11.9, 14.1 / 16.6; 112
// heads 20.9 / 17.4, 21.4 / 18.4, 22.0 / 21.1, 23.1 / 35.6; two tokens by one group of lanes 9.1, 10.7, 19.0, four by four groups 12.0, 12.8, 26.0).
static bool norm_in_projection(const AttnPreArgs& a)
{
    return a.t <= 4 && a.h <= 3 * 2048 && rows_apart(a) && attention_pre_kernel(a.t, a.n_out) == ApqKernel::stream;
}

// A workgroup to a token leaves CUs idle at few tokens: pieces on workgroups of their own up to 160 (us a call, three sets of operands, hidden 5120, a workgroup to
// a token / to 256 pieces: 14 heads, 16 tokens 14.1 / 13.6, 32: 16.1 / 15.3, 64: 18.7 / 17.9, 160: 21.6 / 21.2, 200: 23.0 / 23.0, 256: 23.6 / 23.6, 777: 37.4 / 38.9;
// 28 heads, 8: 15.2 / 14.3, 32: 18.1 / 17.4, 128: 23.8 / 22.9; 112 heads, 8: 23.2 / 22.4, 64: 26.5 / 25.3, 160: 37.5 / 36.6, 256: 45.9 / 45.8, 1024: 82.1 / 83.9).
static bool norm_in_pieces(const AttnPreArgs& a)
{
    return a.t <= 160 && a.h > 2048 && a.h <= 3 * 2048 && rows_apart(a);
}

hipError_t attention_pre_launch(const AttnPreArgs& a, hipStream_t stream)
{
    if (a.t == 0) return hipSuccess;
    const bool whole = attention_pre_whole(a.t, a.n_out, a.ksplits), together = norm_in_projection(a);
    hipError_t e;
    if (!together)
    {
        ScopedKernelTimer tm(KID_APQ_NORM, stream);
        if (norm_in_pieces(a))
            hipLaunchKernelGGL(apq_norm_pieces_kernel, dim3(a.t, (a.h / 8 + 255) / 256), dim3(256), 0, stream, a);
        else if (a.h <= 3 * 2048)
            hipLaunchKernelGGL(apq_norm_kernel<3>, dim3(a.t), dim3(256), 0, stream, a);
        else
            hipLaunchKernelGGL(apq_norm_kernel<AMAX_H / 2048>, dim3(a.t), dim3(256), 0, stream, a);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    {
        ScopedKernelTimer tm(KID_APQ_GEMM, stream);
        const dim3 grid(a.n_out / AD, a.ksplits, (a.t + ATOK - 1) / ATOK);
        const int per = stages_per_split(a.t, a.h, a.n_out);
        if (a.ksplits != attention_pre_ksplits(a.t, a.h, a.n_out)) return hipErrorInvalidValue;
        const ApqKernel kernel = attention_pre_kernel(a.t, a.n_out);
        if (kernel == ApqKernel::tiles) {
            const BigPlan big = big_plan(a.t, a.h, a.n_out);
            gt_dispatch(big.tb, [&](auto tb) {
                constexpr int TB = decltype(tb)::value;
                hipLaunchKernelGGL((whole ? apq_gemm_big_kernel<TB, true> : apq_gemm_big_kernel<TB, false>),
                                   dim3((a.n_out / AD + 1) / 2, a.ksplits, (a.t + 32 * TB - 1) / (32 * TB)), dim3(GT_LANES), 0, stream, a,
                                   big.per);
            });
        } else if (together) {
            norm_gemm_dispatch(per, a.t, [&](auto p, auto t, auto g) {
                constexpr int PER = decltype(p)::value, T = decltype(t)::value, G = decltype(g)::value;
                hipLaunchKernelGGL((apq_norm_gemm_kernel<PER, T, G>), grid, dim3(256 * G), 0, stream, a);
            });
        } else if (kernel == ApqKernel::mid)
            hipLaunchKernelGGL(apq_gemm_mid_kernel, dim3(a.n_out / AD, a.ksplits, (a.t + BTOK - 1) / BTOK), dim3(256), 0, stream, a,
                               mid_stages_per_split(a.t, a.h, a.n_out));
        else if (per == 4)
            hipLaunchKernelGGL(apq_gemm_kernel<4>, grid, dim3(256), 0, stream, a);
        else if (per == 2)
            hipLaunchKernelGGL(apq_gemm_kernel<2>, grid, dim3(256), 0, stream, a);
        else
            hipLaunchKernelGGL(apq_gemm_kernel<1>, grid, dim3(256), 0, stream, a);
    }
    if ((e = hipGetLastError()) != hipSuccess || whole) return e;
    {
        ScopedKernelTimer tm(KID_APQ_HEAD, stream);
        const dim3 grid(a.q_heads + 2 * a.kv_heads, (a.t + 3) / 4);
        if (a.ksplits <= 4)
            hipLaunchKernelGGL(apq_head_kernel<4>, grid, dim3(256), 0, stream, a);
        else if (a.ksplits <= 10)
            hipLaunchKernelGGL(apq_head_kernel<10>, grid, dim3(256), 0, stream, a);
        else if (a.ksplits <= 16 || a.ksplits > 20)
            hipLaunchKernelGGL(apq_head_kernel<16>, grid, dim3(256), 0, stream, a);
        else
            hipLaunchKernelGGL(apq_head_kernel<20>, grid, dim3(256), 0, stream, a);
    }
    return hipGetLastError();
}

} // namespace pto
