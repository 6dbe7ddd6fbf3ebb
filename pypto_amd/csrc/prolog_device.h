// Lightning-indexer prolog: device bodies of the query and the key kernels, shared by the operator's own kernels
// (prolog_kernels.hip) and by the fused MLA + indexer prolog (mla_prolog_kernels.hip).
#pragma once
#include "gemm_tile.h"
#include "kernels.h"
#include "prolog_common.h"

namespace pto {
namespace {


constexpr int PD = 128;      // index head dim
constexpr int PROPE = 64;    // rotary dims
constexpr int PTOK = 32;     // tokens per workgroup tile
constexpr int XW_K = 256;    // contraction rows per workgroup of the x @ [w_k | w_proj] product
constexpr int XROW = PD * 2 + 8; // bytes per LDS row of the 32 x 128 bf16 tile (padded: 32 rows two banks apart)
constexpr int QK = 128;      // contraction rows per stage of prolog_q_kernel
constexpr int QROW = 136;    // bytes per LDS row of a [k][128] int8 weight stage (padded, 8-byte aligned)
constexpr int QGROUPS = 4;   // wave groups of prolog_q_kernel, each with its own stages
constexpr int QMAX_R = 2048; // largest q_lora_rank
constexpr int QMAXS = QMAX_R / QK / QGROUPS;   // stages per group at the largest q_lora_rank
constexpr int QQP = PTOK * (QMAX_R / 16) / 1024; // 16-byte pieces of the q_norm tile per lane at the largest q_lora_rank

constexpr int QAUX = 2 * PTOK * PROPE * 2 + PD * 4 + PTOK * 4; // cos and sin rows of the token tile, w_qb_scale, q_norm_scale

__host__ __device__ constexpr int prolog_q_lds_bytes(int r) { return QGROUPS * QK * QROW + PTOK * (r + 16) + QAUX; }
static_assert(QGROUPS * QK * QROW >= PD * PD * 2 + PTOK * XROW + 4 * PTOK * 4, "the epilogue fits in the stage buffers");

// Rotary embedding of the first 64 dims of the 32 x 128 bf16 tile in LDS, fp32 arithmetic with every product and sum
// rounded (the golden's x * cos + rotate_half(x) * sin), back to bf16.  256 lanes: 4 (token, pair) items each.  csl is the
// tile's [2][32][64] cos and sin rows in LDS.
__device__ __forceinline__ void rope_tile(uint8_t* xt, const uint16_t* csl, int tid)
{
#pragma clang fp contract(off)
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int item = tid + 256 * it;
        const int tok = item >> 5, i = item & 31;
        uint16_t* row = reinterpret_cast<uint16_t*>(xt + tok * XROW);
        const uint16_t* cosp = csl + tok * PROPE;
        const uint16_t* sinp = csl + (PTOK + tok) * PROPE;
        const float x1 = bf16_to_f32(row[i]), x2 = bf16_to_f32(row[i + 32]);
        const float c1 = bf16_to_f32(cosp[i]), c2 = bf16_to_f32(cosp[i + 32]);
        const float s1 = bf16_to_f32(sinp[i]), s2 = bf16_to_f32(sinp[i + 32]);
        const float o1 = x1 * c1 + (-x2) * s1;
        const float o2 = x2 * c2 + x1 * s2;
        row[i] = f32_to_bf16(o1);
        row[i + 32] = f32_to_bf16(o2);
    }
}

// What follows the index query's product for one head and 32 TB tokens, 256 lanes (ht), on the bf16 tile xt [32 TB][XROW] - the one
// place for the operations behind every form of the product: Hadamard and quantisation here, the rotary embedding in front of them in
// prolog_q_finish (from memory) or rope_tile (from LDS).  had: hadamard_q, smax: per-wave maxima.  Every lane of the workgroup
// passes its barriers; heads past the last one are dropped.
template <int TB>
__device__ __forceinline__ void prolog_q_quantise(const PrologArgs& a, int head, int tok0, int ht, const uint8_t* had, const uint8_t* xt,
                                                  float (*smax)[32 * TB])
{
#pragma clang fp contract(off)
    const int lane = ht & 63, hwave = ht >> 6, l32 = lane & 31, hl = lane >> 5;
    // Y^T[n, token] = H^T[n, k] . X^T[k, token]: wave w of a head owns n in [32 w, 32 w + 32) for the blocks of 32 tokens.  A (H^T) by
    // transposing reads of the row-major H: lane jj of 16-lane group G points at row k0 + 4 hl + jj / 4 (+ 8), columns 32 w + 16 (G & 1)
    // + 4 (jj & 3); they hand lane half hl the contraction rows {4 hl .. 4 hl + 3} and {8 + 4 hl .. 8 + 4 hl + 3} of a 16-row step, so
    // the B operand takes the same rows of X: two 8-byte pieces
    f32x16 y[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int e = 0; e < 16; ++e) y[tb][e] = 0.f;
    {
        const int jj = lane & 15, mh = (lane >> 4) & 1;
        const uint8_t* hp = had + (4 * hl + (jj >> 2)) * (PD * 2) + (32 * hwave + 16 * mh + 4 * (jj & 3)) * 2;
        const uint8_t* xp = xt + l32 * XROW + hl * 8;
        bf16x8 av[2], bv[2][TB]; // a step's operands are read while the step before is multiplied
        auto read = [&](int ks) {
            const s16x4 lo = lds_read_tr(hp + ks * 16 * (PD * 2));
            const s16x4 hi = lds_read_tr(hp + (ks * 16 + 8) * (PD * 2));
            av[ks & 1] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                const u32x2 b0 = *reinterpret_cast<const u32x2*>(xp + 32 * tb * XROW + ks * 32);
                const u32x2 b1 = *reinterpret_cast<const u32x2*>(xp + 32 * tb * XROW + ks * 32 + 16);
                bv[ks & 1][tb] = __builtin_bit_cast(bf16x8, u32x4{b0[0], b0[1], b1[0], b1[1]});
            }
        };
        read(0);
#pragma unroll
        for (int ks = 0; ks < PD / 16; ++ks) {
            if (ks + 1 < PD / 16) read(ks + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) y[tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[ks & 1], bv[ks & 1][tb], y[tb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // register e of y[tb]: n = 32 w + 8 (e/4) + 4 hl + e%4, token 32 tb + l32.  Round to bf16, per-token absmax over the 128 n
    float mx[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        mx[tb] = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            y[tb][e] = bf16_to_f32(f32_to_bf16(y[tb][e]));
            mx[tb] = fmaxf(mx[tb], fabsf(y[tb][e]));
        }
        mx[tb] = fmaxf(mx[tb], __shfl_xor(mx[tb], 32));
        if (hl == 0) smax[hwave][32 * tb + l32] = mx[tb];
    }
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const int tl = 32 * tb + l32;
        const float m = fmaxf(fmaxf(smax[0][tl], smax[1][tl]), fmaxf(smax[2][tl], smax[3][tl]));
        const float sq = quant_scale(m);
        const int gt = tok0 + tl;
        // pieces of 4 dims, 8 apart; with the other lane half's: 16 dims in a row to a lane, one store
        uint32_t pk[4];
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            uint32_t r[4]; // at most 127: behind 1.5 * 2^23 the low byte is the value rounded to even (0 of a NaN, and of an infinity by a scale
                           // that a maximum below 2^-121 makes infinite: the golden's bytes)
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = __builtin_bit_cast(uint32_t, y[tb][4 * e4 + e] * sq + 12582912.f);
            pk[e4] = __builtin_amdgcn_perm(r[1], r[0], 0x0c0c0400u) | __builtin_amdgcn_perm(r[3], r[2], 0x04000c0cu);
        }
        const auto even = __builtin_amdgcn_permlane32_swap(pk[0], pk[2], false, false);
        const auto odd = __builtin_amdgcn_permlane32_swap(pk[1], pk[3], false, false);
        if (gt < a.t && head < a.n) {
            *reinterpret_cast<u32x4*>(a.q_int8 + ((int64_t)gt * a.n + head) * PD + 32 * hwave + 16 * hl) =
                u32x4{(unsigned)even[0], (unsigned)even[1], (unsigned)odd[0], (unsigned)odd[1]};
            if (hwave == 0 && hl == 0) a.q_scale[(int64_t)gt * a.n + head] = __builtin_bit_cast(uint16_t, (_Float16)(1.0f / sq));
        }
    }
}
template <int TB>
__device__ __forceinline__ void prolog_q_finish(const PrologArgs& a, int head, int tok0, int ht, const uint8_t* had, uint8_t* xt,
                                                float (*smax)[32 * TB])
{
#pragma clang fp contract(off)
    // rotary on the first 64 dims: 32 pairs a token (the arithmetic of rope_tile)
#pragma unroll 4
    for (int it = 0; it < TB * 32 * 32 / 256; ++it) {
        const int item = ht + 256 * it;
        const int tok = item >> 5, i = item & 31;
        uint16_t* row = reinterpret_cast<uint16_t*>(xt + tok * XROW);
        const int64_t gtc = (int64_t)min(tok0 + tok, a.t - 1) * PROPE;
        const uint16_t* cosp = a.cos + gtc;
        const uint16_t* sinp = a.sin + gtc;
        const float x1 = bf16_to_f32(row[i]), x2 = bf16_to_f32(row[i + 32]);
        const float c1 = bf16_to_f32(cosp[i]), c2 = bf16_to_f32(cosp[i + 32]);
        const float s1 = bf16_to_f32(sinp[i]), s2 = bf16_to_f32(sinp[i + 32]);
        const float o1 = x1 * c1 + (-x2) * s1;
        const float o2 = x2 * c2 + x1 * s2;
        row[i] = f32_to_bf16(o1);
        row[i + 32] = f32_to_bf16(o2);
    }
    __syncthreads();
    prolog_q_quantise<TB>(a, head, tok0, ht, had, xt, smax);
}

// ------------------------------------------------------------------------------------------------ query path
// One workgroup of 1024 lanes = 4 groups of 4 wavefronts per (head, token tile of 32); plds is its dynamic LDS
// (prolog_q_lds_bytes).
__device__ __forceinline__ void prolog_q_body(const PrologArgs& a, int head, int tok0, uint8_t* plds)
{
    // LDS: [4 groups][QK x QROW] weight stages | [32][r + 16] q_norm tile | cos, sin rows and scales for the epilogue.
    // Once the GEMM is done the first region is
    // reused for hadamard_q [128][128] bf16, the head's bf16 tile [32][XROW] and the per-wave maxima.
    uint8_t* had = plds;
    uint8_t* xt = plds + PD * PD * 2;
    float(*smax)[PTOK] = reinterpret_cast<float(*)[PTOK]>(plds + PD * PD * 2 + PTOK * XROW);

    const int tid = threadIdx.x & 255, grp = threadIdx.x >> 8, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4, l32 = lane & 31, hl = lane >> 5;
    const int r = a.r, qrowb = r + 16;
    const int64_t nd = (int64_t)a.n * PD;
    uint8_t* wl = plds + grp * (QK * QROW);
    uint8_t* ql = plds + QGROUPS * (QK * QROW);
    uint8_t* aux = ql + PTOK * qrowb; // [2][32][64] bf16 cos, sin | [128] w_qb_scale | [32] q_norm_scale
    const uint16_t* csl = reinterpret_cast<const uint16_t*>(aux);
    const float* wsl = reinterpret_cast<const float*>(aux + 2 * PTOK * PROPE * 2);
    const float* qsl = wsl + PD;

    // loads in the order they are needed: hadamard_q (parked in registers until the GEMM is over), the q_norm tile,
    // then every weight stage of this group - all in flight together
    u32x4 hst[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) hst[i] = reinterpret_cast<const u32x4*>(a.had_q)[threadIdx.x + 1024 * i];
    const int qpieces = PTOK * (r / 16);
    u32x4 qst[QQP];
#pragma unroll
    for (int i = 0; i < QQP; ++i) {
        const int pc = min((int)threadIdx.x + 1024 * i, qpieces - 1);
        const int row = pc / (r / 16), c = pc % (r / 16);
        qst[i] = *reinterpret_cast<const u32x4*>(a.q_norm + (int64_t)min(tok0 + row, a.t - 1) * r + 16 * c);
    }
    // what the epilogue reads (rotary rows, scales): fetched now, so that it waits for nothing later
    // (every lane loads - a load under a condition would be waited for on the spot; lanes past 544 fetch piece 0 again)
    const int ai = threadIdx.x < 544 ? (int)threadIdx.x : 0;
    const uint8_t* ap = ai < 512 ? reinterpret_cast<const uint8_t*>((ai >> 8 ? a.sin : a.cos) +
                                                                     (int64_t)min(tok0 + ((ai & 255) >> 3), a.t - 1) * PROPE + 8 * (ai & 7))
                                 : reinterpret_cast<const uint8_t*>(a.w_qb_scale + (int64_t)head * PD + 4 * (ai - 512));
    const u32x4 ast = *reinterpret_cast<const u32x4*>(ap);
    const float qst1 = a.q_norm_scale[min(tok0 + (int)(threadIdx.x & 31), a.t - 1)];
    const int stages = r / QK;
    const int srow = tid >> 3, spc = tid & 7;
    const int8_t* sp = a.w_qb + (int64_t)srow * nd + head * PD + 16 * spc;
    u32x4 stg[QMAXS][4];
#pragma unroll
    for (int j = 0; j < QMAXS; ++j) {
        const int s = min(grp + QGROUPS * j, stages - 1); // past the end: the last stage again, dropped below
#pragma unroll
        for (int i = 0; i < 4; ++i) stg[j][i] = *reinterpret_cast<const u32x4*>(sp + ((int64_t)s * QK + 32 * i) * nd);
    }
#pragma unroll
    for (int i = 0; i < QQP; ++i) {
        const int pc = (int)threadIdx.x + 1024 * i;
        if (pc < qpieces) *reinterpret_cast<u32x4*>(ql + (pc / (r / 16)) * qrowb + 16 * (pc % (r / 16))) = qst[i];
    }
    if (threadIdx.x < 544) reinterpret_cast<u32x4*>(aux)[threadIdx.x] = ast;
    if (threadIdx.x < 32) reinterpret_cast<float*>(aux)[4 * 544 + threadIdx.x] = qst1;
    // C^T[dim, token] = W^T[dim, :] . q_norm[token, :]: wave w owns dims [32 w, 32 w + 32) x 32 tokens
    i32x4 acc[2][2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) acc[db][tb] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < QMAXS; ++j) {
        const int s = grp + QGROUPS * j;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            u32x2* d = reinterpret_cast<u32x2*>(wl + (srow + 32 * i) * QROW + 16 * spc);
            d[0] = u32x2{stg[j][i][0], stg[j][i][1]};
            d[1] = u32x2{stg[j][i][2], stg[j][i][3]};
        }
        __syncthreads();
        if (s < stages) {
#pragma unroll
            for (int ks = 0; ks < QK / 64; ++ks) {
                i32x4 qf[2], wf[2];
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
                    qf[tb] = *reinterpret_cast<const i32x4*>(ql + (16 * tb + l16) * qrowb + s * QK + ks * 64 + 16 * g);
                // A operand: dim 32 w + 16 db + l16, contraction bytes 16 g .. 16 g + 15 of the step.  An 8-bit
                // transposing read hands lane i of a 16-lane group byte i % 8 of the chunks addressed by lanes
                // i / 8, i / 8 + 2, ..., i / 8 + 14: with lane i pointing at row i / 2, column half i % 2, lane i gets
                // column i over rows 0 .. 7 - eight of its sixteen contraction bytes per read
#pragma unroll
                for (int db = 0; db < 2; ++db) {
                    const uint8_t* p = wl + (ks * 64 + 16 * g + (l16 >> 1)) * QROW + 32 * wave + 16 * db + 8 * (l16 & 1);
                    const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 8 * QROW);
                    wf[db] = i32x4{lo[0], lo[1], hi[0], hi[1]};
                }
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb)
                        acc[db][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[db], qf[tb], acc[db][tb], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // add the groups' int32 sums (exact): groups 1.. leave theirs in their own stage buffer, group 0 collects
    if (grp > 0) {
        i32x4* red = reinterpret_cast<i32x4*>(wl);
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) red[(2 * db + tb) * 256 + tid] = acc[db][tb];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int og = 1; og < QGROUPS; ++og) {
            const i32x4* red = reinterpret_cast<const i32x4*>(plds + og * (QK * QROW));
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) acc[db][tb] += red[(2 * db + tb) * 256 + tid];
        }
    }
    __syncthreads();
    // the stage buffers are free now: hadamard_q moves in
#pragma unroll
    for (int i = 0; i < 2; ++i) reinterpret_cast<u32x4*>(had)[threadIdx.x + 1024 * i] = hst[i];
    __syncthreads();
    if (grp > 0) return; // the barriers below are among the first group's waves (a finished wave does not count)
    // register e of acc[db][tb]: dim 32 w + 16 db + 4 g + e, token 16 tb + l16
    {
#pragma clang fp contract(off)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const int tok = 16 * tb + l16;
            const float qs = qsl[tok];
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const int dim = 32 * wave + 16 * db + 4 * g;
                const f32x4 ws = *reinterpret_cast<const f32x4*>(wsl + dim);
                uint16_t* dst = reinterpret_cast<uint16_t*>(xt + tok * XROW) + dim;
#pragma unroll
                for (int e = 0; e < 4; ++e) dst[e] = f32_to_bf16(((float)acc[db][tb][e] * qs) * ws[e]);
            }
        }
    }
    __syncthreads();
    rope_tile(xt, csl, tid);
    __syncthreads();
    prolog_q_quantise<1>(a, head, tok0, tid, had, xt, smax);
}

// ------------------------------------------------------------------------------------------------ query path, prefill sizes
// The same product for 128 tokens and more: a workgroup of 256 lanes owns (head, 128 tokens) and walks the contraction
// in stages of 128 rows, both operands staged through LDS with the loads of the next DEPTH stages in flight.  Wave
// (wr, wc) owns tokens [64 wr, +64) x dims [64 wc, +64): every operand fragment read from LDS feeds four MFMAs, and the
// head's weight slice is fetched once per 128 tokens instead of once per 32.  Then, in LDS, for all 128 tokens: scale
// and round to bf16, rotary, hadamard (wave w: outputs [32 w, +32) of all tokens, every hadamard fragment feeding four
// MFMAs), quantisation.  The int32 sums are exact and the rest is the same operations in the same order, so the
// results are the bits of prolog_q_body's.
constexpr int QB_TOK = 128;
constexpr int QB_QROW = QK + 16; // bytes per LDS row of the [token][k] int8 tile (padded against bank conflicts)
constexpr int QB_STAGE_BYTES = QK * QROW + QB_TOK * QB_QROW;
constexpr int QB_EPI_BYTES = PD * PD * 2 + QB_TOK * XROW + 4 * QB_TOK * 4; // hadamard_q | bf16 tile | per-wave maxima
constexpr int QB_LDS_BYTES = QB_EPI_BYTES > QB_STAGE_BYTES ? QB_EPI_BYTES : QB_STAGE_BYTES;
constexpr int QB_DEPTH = 3; // stages of loads in flight (the epilogue's 68 KB of LDS leave two workgroups to a CU whatever the
                            // register count, so the depth costs no occupancy)

template <int DEPTH>
__device__ __forceinline__ void prolog_q_big_body(const PrologArgs& a, int head, int tok0, uint8_t* lds)
{
#pragma clang fp contract(off)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4, l32 = lane & 31, hl = lane >> 5, wr = wave >> 1, wc = wave & 1;
    const int r = a.r;
    const int64_t nd = (int64_t)a.n * PD;
    uint8_t* wl = lds;
    uint8_t* ql = lds + QK * QROW;
    const int stages = r / QK;
    // 128 rows x 128 bytes of either operand per stage = 4 pieces of 16 bytes per lane (rows tid / 8 + 32 i, piece tid % 8)
    const int srow = tid >> 3, spc = tid & 7;
    const int8_t* wp = a.w_qb + (int64_t)srow * nd + head * PD + 16 * spc;
    const int8_t* qp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) qp[i] = a.q_norm + (int64_t)min(tok0 + srow + 32 * i, a.t - 1) * r + 16 * spc;
    u32x4 wst[DEPTH][4], qst[DEPTH][4];
    auto load = [&](int st, int u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) qst[u][i] = *reinterpret_cast<const u32x4*>(qp[i] + st * QK);
#pragma unroll
        for (int i = 0; i < 4; ++i) wst[u][i] = *reinterpret_cast<const u32x4*>(wp + ((int64_t)st * QK + 32 * i) * nd);
    };
    // the epilogue's scales, requested first
    float qs_pre[4];
    f32x4 ws_pre[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) qs_pre[tb] = a.q_norm_scale[min(tok0 + 64 * wr + 16 * tb + l16, a.t - 1)];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) ws_pre[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + (int64_t)head * PD + 64 * wc + 16 * nb + 4 * g);
    i32x4 acc[4][4]; // [nb][tb]
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) load(min(u, stages - 1), u);
    for (int st0 = 0; st0 < stages; st0 += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if (st0 + u < stages) { // (uniform over the workgroup)
                __syncthreads();    // everyone is done with the previous stage's tiles
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    u32x2* d = reinterpret_cast<u32x2*>(wl + (srow + 32 * i) * QROW + 16 * spc);
                    d[0] = u32x2{wst[u][i][0], wst[u][i][1]};
                    d[1] = u32x2{wst[u][i][2], wst[u][i][3]};
                    *reinterpret_cast<u32x4*>(ql + (srow + 32 * i) * QB_QROW + 16 * spc) = qst[u][i];
                }
                __syncthreads();
                load(min(st0 + u + DEPTH, stages - 1), u); // (unconditional: past the end the last stage is fetched again and dropped)
#pragma unroll
                for (int ks = 0; ks < QK / 64; ++ks) {
                    i32x4 qf[4], wf[4];
#pragma unroll
                    for (int tb = 0; tb < 4; ++tb)
                        qf[tb] = *reinterpret_cast<const i32x4*>(ql + (64 * wr + 16 * tb + l16) * QB_QROW + ks * 64 + 16 * g);
                    // (the byte-transposing read: see prolog_q_body)
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb) {
                        const uint8_t* p = wl + (ks * 64 + 16 * g + (l16 >> 1)) * QROW + 64 * wc + 16 * nb + 8 * (l16 & 1);
                        const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 8 * QROW);
                        wf[nb] = i32x4{lo[0], lo[1], hi[0], hi[1]};
                    }
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
                        for (int tb = 0; tb < 4; ++tb)
                            acc[nb][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[nb], qf[tb], acc[nb][tb], 0, 0, 0);
                }
            }
        }
    }
    __syncthreads(); // the operand tiles are free: hadamard_q and the bf16 tile take their place
    uint8_t* had = lds;
    uint8_t* xt = lds + PD * PD * 2;
    float(*smax)[QB_TOK] = reinterpret_cast<float(*)[QB_TOK]>(lds + PD * PD * 2 + QB_TOK * XROW);
#pragma unroll
    for (int i = 0; i < PD * PD * 2 / 16 / 256; ++i) reinterpret_cast<u32x4*>(had)[tid + 256 * i] = reinterpret_cast<const u32x4*>(a.had_q)[tid + 256 * i];
    // register e of acc[nb][tb]: dim 64 wc + 16 nb + 4 g + e, token 64 wr + 16 tb + l16
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
        const int tl = 64 * wr + 16 * tb + l16;
        const float qs = qs_pre[tb];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const int dim = 64 * wc + 16 * nb + 4 * g;
            const f32x4 ws = ws_pre[nb];
            uint16_t vb[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) vb[e] = f32_to_bf16(((float)acc[nb][tb][e] * qs) * ws[e]);
            *reinterpret_cast<u32x2*>(xt + tl * XROW + dim * 2) = u32x2{(uint32_t)vb[0] | ((uint32_t)vb[1] << 16), (uint32_t)vb[2] | ((uint32_t)vb[3] << 16)};
        }
    }
    __syncthreads();
    prolog_q_finish<QB_TOK / 32>(a, head, tok0, tid, had, xt, smax);
}

// 4 x 4 pieces of 8 bytes, [row of 16 lanes][register]: out[j] of row g = x[g] of row j
__device__ __forceinline__ void transpose_rows(uint32_t (&out)[4][2], const u32x4 (&x)[2])
{
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto a = __builtin_amdgcn_permlane32_swap(x[0][i], x[1][i], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(x[0][2 + i], x[1][2 + i], false, false);
        const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a[0], (unsigned)b[0], false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)a[1], (unsigned)b[1], false, false);
        out[0][i] = lo[0], out[1][i] = lo[1], out[2][i] = hi[0], out[3][i] = hi[1];
    }
}

// Above 128 tokens: 32 TB tokens x two heads per workgroup (gemm_tile.h), four waves to a head behind the product; the
// operations are prolog_q_big_body's, so are the bits (51 us at 1501 tokens there).  512 lanes; an odd last head is taken twice
// and dropped.
// Nothing covers what follows the product, which at 192 tokens x 1536 rows took 33 K ticks beside the product's 30 K: rotary pairs
// out of LDS, cos and sin loaded in single elements; pairs of LDS rows in the same banks in front of the Hadamard product; four
// stores of 4 bytes a lane.  Now 22 K: pairs are rotated where they are, in registers of a lane, by one wave of each SIMD
// (gt_wave_across), cos and sin loaded 16 bytes at a time (loads of 8 cost the memory pipe twice as much, 13 K ticks in all, not 8);
// rows two banks apart; one store of 16 bytes.  Call of 1501 tokens 239.6 -> 232.9 us, 300: 80.7 -> 76.5.
// 256 tokens' tiles of both heads do not fit LDS: there the two halves of the tokens, which are two rows of waves, go through one
// after the other (three rounds of workgroups for 1501 tokens instead of four of 192: a call 215.7 -> 207.0 us).
constexpr int prolog_q_wide_parts(int tb) { return tb > 7 ? 2 : 1; }
constexpr int prolog_q_wide_lds(int tb) // the product's stages, or hadamard_q | [2] bf16 tiles | [2] per-wave maxima
{
    const int tok = 32 * tb / prolog_q_wide_parts(tb), ring = gt_lds_bytes(tb);
    const int epi = PD * PD * 2 + 2 * tok * XROW + 2 * 4 * tok * 4;
    return epi > ring ? epi : ring;
}
template <int TB>
__device__ __forceinline__ void prolog_q_wide_body(const PrologArgs& a, int head0, int tok0, uint8_t* lds)
{
#pragma clang fp contract(off)
    constexpr int PARTS = prolog_q_wide_parts(TB), TILE = 32 * TB / PARTS;
    static_assert(PARTS == 1 || TILE == 16 * TB, "a part is a row of waves");
    static_assert(prolog_q_wide_lds(TB) <= 160 * 1024 && prolog_q_wide_lds(TB) >= GtTile<TB>::LDS, "LDS");
    const int tid = threadIdx.x, lane = tid & 63, wave = gt_wave_across();
    const int l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    const int64_t nd = (int64_t)a.n * PD;
    i32x4 acc[4][TB]; // [nb][tb]
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
    gt_product_i8<TB>(acc, a.w_qb + head0 * PD, a.w_qb + min(head0 + 1, a.n - 1) * PD, nd, a.q_norm, a.r, tok0, a.t, a.r / GT_KI8, lds,
                      wave);
    u32x4 hadr[PD * PD * 2 / 16 / 512];
#pragma unroll
    for (int i = 0; i < PD * PD * 2 / 16 / 512; ++i) hadr[i] = reinterpret_cast<const u32x4*>(a.had_q)[tid + 512 * i];
    // register e of acc[nb][tb]: dim 64 (wc & 1) + 16 nb + 4 g + e of head wc / 2, token 16 TB wr + 16 tb + l16
    const int hw = 64 * (wc & 1);
    uint32_t y[4][TB][2]; // bf16
    {
        f32x4 ws[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
            ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + (int64_t)min(head0 + (wc >> 1), a.n - 1) * PD + hw + 16 * nb + 4 * g);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const float qs = a.q_norm_scale[min(tok0 + 16 * TB * wr + 16 * tb + l16, a.t - 1)];
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs) * ws[nb][e];
                y[nb][tb][0] = pack_bf16x2(v[0], v[1]);
                y[nb][tb][1] = pack_bf16x2(v[2], v[3]);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0); // (the loads below once the sums' registers are free)
    if (hw == 0) { // rotary pairs are 32 dims apart: registers of a lane
        const uint16_t* cp = a.cos + (int64_t)tok0 * PROPE;
        const uint16_t* sp = a.sin + (int64_t)tok0 * PROPE;
        // a lane loads dims 16 g .. 16 g + 15 of its token, four pieces of 4, and gets its pieces 16 nb + 4 g by exchange of rows
        u32x4 cr[TB][2], sr[TB][2];
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t at = min(16 * TB * wr + 16 * tb + l16, a.t - 1 - tok0) * PROPE + 16 * g + 8 * i;
                cr[tb][i] = *reinterpret_cast<const u32x4*>(cp + at);
                sr[tb][i] = *reinterpret_cast<const u32x4*>(sp + at);
            }
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            uint32_t c[4][2], sn[4][2];
            transpose_rows(c, cr[tb]);
            transpose_rows(sn, sr[tb]);
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float o[2][2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) { // (the arithmetic of rope_tile)
                        const float x1 = half_of(y[nb][tb][i], e), x2 = half_of(y[nb + 2][tb][i], e);
                        o[0][e] = x1 * half_of(c[nb][i], e) + (-x2) * half_of(sn[nb][i], e);
                        o[1][e] = x2 * half_of(c[nb + 2][i], e) + x1 * half_of(sn[nb + 2][i], e);
                    }
                    y[nb][tb][i] = pack_bf16x2(o[0][0], o[0][1]);
                    y[nb + 2][tb][i] = pack_bf16x2(o[1][0], o[1][1]);
                }
        }
    }
    const int hs = tid >> 8, ht = tid & 255, head = head0 + hs; // behind the tile four waves to a head
    uint8_t* xt = lds + PD * PD * 2 + hs * TILE * XROW;
    float(*smax)[TILE] = reinterpret_cast<float(*)[TILE]>(lds + PD * PD * 2 + 2 * TILE * XROW + hs * 4 * TILE * 4);
#pragma unroll
    for (int i = 0; i < PD * PD * 2 / 16 / 512; ++i) reinterpret_cast<u32x4*>(lds)[tid + 512 * i] = hadr[i];
#pragma unroll
    for (int part = 0; part < PARTS; ++part) {
        if (part > 0) __syncthreads(); // the tile and the maxima before are read
        if (PARTS == 1 || wr == part) {
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb)
                    *reinterpret_cast<u32x2*>(lds + PD * PD * 2 + ((wc >> 1) * TILE + 16 * TB * wr - part * TILE + 16 * tb + l16) * XROW +
                                              (hw + 16 * nb + 4 * g) * 2) = u32x2{y[nb][tb][0], y[nb][tb][1]};
        }
        __syncthreads();
        prolog_q_quantise<TB / PARTS>(a, head, tok0 + part * TILE, ht, lds, xt, smax);
    }
}

// Up to 32 tokens: one head per workgroup of 256 lanes behind the streamed product; the bits of prolog_q_body.
// lds: the stages, afterwards the bf16 tile and the per-wave maxima | hadamard_q, copied along with the first stages
constexpr int PROLOG_STREAM_LDS = GtStream::LDS + PD * PD * 2;
static_assert(PTOK * XROW + 4 * PTOK * 4 <= GtStream::LDS && PTOK == GtStream::TOK, "tile and maxima take the stages' place");
__device__ __forceinline__ void prolog_q_stream_body(const PrologArgs& a, int head, uint8_t* lds)
{
#pragma clang fp contract(off)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    uint8_t* had = lds + GtStream::LDS;
    float qs[2];
    f32x4 ws[2];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) qs[tb] = a.q_norm_scale[min(16 * tb + l16, a.t - 1)];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + (int64_t)head * PD + 32 * wave + 16 * nb + 4 * g);
#pragma unroll
    for (int i = 0; i < PD * PD * 2 / 4096; ++i) gt_copy(a.had_q, (uint32_t)(4096 * i + 16 * tid), had + 4096 * i + 1024 * wave);
    i32x4 acc[2][2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
    gt_stream_i8(acc, a.w_qb + head * PD, (int64_t)a.n * PD, a.q_norm, a.r, a.t, a.r / GT_KI8, lds);
    uint8_t* xt = lds;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs[tb]) * ws[nb][e];
            *reinterpret_cast<u32x2*>(xt + (16 * tb + l16) * XROW + (32 * wave + 16 * nb + 4 * g) * 2) =
                u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
    __syncthreads();
    prolog_q_finish<1>(a, head, 0, tid, had, xt, reinterpret_cast<float(*)[PTOK]>(lds + PTOK * XROW));
}

// 33 to 160 tokens: one head per workgroup of 512 lanes behind the streamed product of all tokens; two groups of four waves to the
// halves of the tokens behind it.  Rotary pairs are registers of a lane; hadamard_q, cos and sin come ahead of the stages.  lds: the stages, afterwards hadamard_q | bf16 tile | [2] per-wave maxima
template <int TT>
__device__ __forceinline__ void prolog_q_batch_body(const PrologArgs& a, int head, uint8_t* lds)
{
#pragma clang fp contract(off)
    using T = GtBatch<TT>;
    constexpr int HB = (TT + 1) / 2, HTOK = 32 * HB; // token blocks of a group
    static_assert(PD * PD * 2 + 2 * HTOK * XROW + 2 * 4 * HTOK * 4 <= T::LDS, "the epilogue takes the stages' place");
    const int tid = threadIdx.x, lane = tid & 63, wave = gt_wave(), l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    float qs[TT];
    f32x4 ws[2];
#pragma unroll
    for (int tb = 0; tb < TT; ++tb) qs[tb] = a.q_norm_scale[min(16 * TT * wr + 16 * tb + l16, a.t - 1)];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + (int64_t)head * PD + 16 * gt_batch_block(wc, nb) + 4 * g);
    u32x4 hadr[PD * PD * 2 / 16 / 512];
#pragma unroll
    for (int i = 0; i < PD * PD * 2 / 16 / 512; ++i) hadr[i] = reinterpret_cast<const u32x4*>(a.had_q)[tid + 512 * i];
    // cos and sin of the rotary dims 16 wc + 4 g .. + 3 and the ones 32 on (waves 0 and 1 of a row)
    u32x2 cs[TT][2], sn[TT][2];
#pragma unroll
    for (int tb = 0; tb < TT; ++tb)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int at = min(16 * TT * wr + 16 * tb + l16, a.t - 1) * PROPE + 32 * i + 16 * (wc & 1) + 4 * g;
            cs[tb][i] = *reinterpret_cast<const u32x2*>(a.cos + at);
            sn[tb][i] = *reinterpret_cast<const u32x2*>(a.sin + at);
        }
    i32x4 acc[2][TT];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int tb = 0; tb < TT; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
    gt_batch_i8<TT>(acc, a.w_qb + head * PD, (int64_t)a.n * PD, a.q_norm, a.r, a.t, a.r / GT_KI8, lds);
    uint8_t* xt = lds + PD * PD * 2;
#pragma unroll
    for (int tb = 0; tb < TT; ++tb) {
        uint32_t y[2][2];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs[tb]) * ws[nb][e];
            y[nb][0] = pack_bf16x2(v[0], v[1]);
            y[nb][1] = pack_bf16x2(v[2], v[3]);
        }
        if (wc < 2) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float o[2][2];
#pragma unroll
                for (int e = 0; e < 2; ++e) { // (the arithmetic of rope_tile)
                    const float x1 = half_of(y[0][i], e), x2 = half_of(y[1][i], e);
                    o[0][e] = x1 * half_of(cs[tb][0][i], e) + (-x2) * half_of(sn[tb][0][i], e);
                    o[1][e] = x2 * half_of(cs[tb][1][i], e) + x1 * half_of(sn[tb][1][i], e);
                }
                y[0][i] = pack_bf16x2(o[0][0], o[0][1]);
                y[1][i] = pack_bf16x2(o[1][0], o[1][1]);
            }
        }
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
            *reinterpret_cast<u32x2*>(xt + (16 * TT * wr + 16 * tb + l16) * XROW + (16 * gt_batch_block(wc, nb) + 4 * g) * 2) = u32x2{y[nb][0], y[nb][1]};
    }
#pragma unroll
    for (int i = 0; i < PD * PD * 2 / 16 / 512; ++i) reinterpret_cast<u32x4*>(lds)[tid + 512 * i] = hadr[i];
    __syncthreads();
    const int hs = tid >> 8; // (of an odd number of blocks the second group has one less: rows past the tile, dropped)
    float(*smax)[HTOK] = reinterpret_cast<float(*)[HTOK]>(xt + 2 * HTOK * XROW + hs * 4 * HTOK * 4);
    prolog_q_quantise<HB>(a, head, HTOK * hs, tid & 255, lds, xt + HTOK * hs * XROW, smax);
}
constexpr int PROLOG_BIG_T = 128;   // token count from which the query product runs per 128 tokens

// ------------------------------------------------------------------------------------------------ key path, weights
__device__ __forceinline__ float block_sum128(float v, float* red)
{
    v = wave_sum_butterfly(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1];
}
__device__ __forceinline__ float block_max128(float v, float* red)
{
    v = wave_max_f32(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(red[0], red[1]);
}

// One workgroup of 128 lanes per token: lane = output dim
template <int S = 16>
__device__ __forceinline__ void prolog_k_body(const PrologArgs& a, int tok)
{
#pragma clang fp contract(off)
    __shared__ float red[2];
    __shared__ __align__(16) float kb[PD], yb[PD];
    const int tid = threadIdx.x;
    // everything that does not depend on the sums is loaded first (its latency hides behind them), and no load sits
    // under a condition (the compiler would wait for it on the spot)
    const int64_t row = a.k_cache_index[tok];
    const float gam = bf16_to_f32(a.ln_gamma[tid]), bet = bf16_to_f32(a.ln_beta[tid]);
    const int ri = tid & (PROPE - 1);
    const float rc = bf16_to_f32(a.cos[(int64_t)tok * PROPE + ri]), rs = bf16_to_f32(a.sin[(int64_t)tok * PROPE + ri]);
    float kv = 0.f, wv = 0.f;
    const int wcol = PD + min(tid, a.n - 1);
    // S splits' loads in flight together (a split past the end re-reads the last one and adds zero); the order of the
    // additions is the order of the splits
    float v0[S], v1[S];
    auto load = [&](int s0) {
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const float* p = a.xw_part + ((int64_t)min(s0 + j, a.ksplits - 1) * a.t + tok) * a.xw_stride + a.xw_col0;
            v0[j] = p[tid];
            v1[j] = p[wcol];
        }
    };
    auto add = [&](int s0) {
#pragma unroll
        for (int j = 0; j < S; ++j) {
            kv += s0 + j < a.ksplits ? v0[j] : 0.f;
            wv += s0 + j < a.ksplits ? v1[j] : 0.f;
        }
    };
    load(0);
    __builtin_amdgcn_sched_barrier(0);
    // the Hadamard matrix behind the sums in the memory pipe: the wave's half of the rows, two columns to a lane (a wave per half of
    // the columns asked for twice as many loads, 256 of 2 bytes a lane, in front of the sums)
    const int hw = __builtin_amdgcn_readfirstlane(tid >> 6), hc = 2 * (tid & 63);
    uint32_t hk[PD / 2];
#pragma unroll
    for (int k = 0; k < PD / 2; ++k) hk[k] = *reinterpret_cast<const uint32_t*>(a.had_k + (PD / 2 * hw + k) * PD + hc);
    __builtin_amdgcn_sched_barrier(0);
    add(0);
    for (int s0 = S; s0 < a.ksplits; s0 += S) load(s0), add(s0);
    // LayerNorm in fp32 (biased variance), -> bf16
    const float mean = block_sum128(kv, red) / (float)PD;
    const float dlt = kv - mean;
    const float var = block_sum128(dlt * dlt, red) / (float)PD;
    float xn = dlt / sqrtf(var + a.eps);
    xn = xn * gam + bet;
    kb[tid] = bf16_to_f32(f32_to_bf16(xn));
    __syncthreads();
    // rotary on the first 64 dims
    float kr = kb[tid];
    if (tid < PROPE) {
        const float other = tid < 32 ? -kb[tid + 32] : kb[tid - 32];
        kr = bf16_to_f32(f32_to_bf16(kb[tid] * rc + other * rs));
    }
    __syncthreads();
    kb[tid] = kr;
    __syncthreads();
    // hadamard: y[n] = sum_k kr[k] H[k][n], fp32, k in order (the second wave goes on from the first's sums), -> bf16
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
        if (hw == part) {
            float2 h = part ? *reinterpret_cast<const float2*>(yb + hc) : float2{0.f, 0.f};
#pragma unroll
            for (int k = 0; k < PD / 2; ++k) {
                asm("" : "+v"(hk[k])); // (taken apart here, not in front of the loop for 64 registers more)
                const float x = kb[PD / 2 * hw + k];
                h.x = __builtin_fmaf(x, half_of(hk[k], 0), h.x);
                h.y = __builtin_fmaf(x, half_of(hk[k], 1), h.y);
            }
            *reinterpret_cast<float2*>(yb + hc) = h;
        }
        __syncthreads();
    }
    const float y = bf16_to_f32(f32_to_bf16(yb[tid]));
    const float mx = block_max128(fabsf(y), red);
    const float sq = quant_scale(mx);
    if (row >= 0 && row < a.cache_rows) {
        a.k_cache[row * PD + tid] = (int8_t)(int)__builtin_rintf(y * sq);
        if (tid == 0) a.k_scale_cache[row] = __builtin_bit_cast(uint16_t, (_Float16)(1.0f / sq));
    }
    if (tid < a.n) {
        const float w = bf16_to_f32(f32_to_bf16(wv));
        a.weights[(int64_t)tok * a.n + tid] = __builtin_bit_cast(uint16_t, (_Float16)((w * a.wscale_n) * a.wscale_d));
    }
}

} // namespace
} // namespace pto
