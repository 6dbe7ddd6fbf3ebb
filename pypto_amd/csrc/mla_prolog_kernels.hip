// MLA prolog, int8 form (the producer of the query and of the paged int8 cache that sparse flash attention reads) -
// gfx950 kernels.
//
// Replaces the device side of mla_prolog_quant_d / mla_prolog_quant_p
// (models/deepseek_v32_exp/mla_prolog_quant_impl.py:364-727, entry points :745-951); arithmetic follows the operator
// (RmsNorm with its epsilon, :127-163) and otherwise the golden mla_prolog_quant_v32_compute
// (models/deepseek_v32_exp/deepseekv32_mla_prolog_quant.py:131-283):
//   q_a   = bf16(x @ w_dq);  q_rms = bf16(gamma_cq * (q_a / sqrt(mean(q_a^2) + eps)))
//   q_norm, q_norm_scale = int8 rint(q_rms * 127 / max|q_rms|), fp32 max|q_rms| / 127         (per token)
//   q_b   = bf16(int32(q_norm @ w_uq_qr) * q_norm_scale * w_qb_scale)                          [t, n, 192]
//   q_nope[t, head] = bf16(q_b[t, head, :128] @ w_uk[head])                                    [t, n, 512]
//   q_rope = rotary(q_b[t, head, 128:])  (interleaved pairs (2i, 2i+1) -> positions (i, 32+i))  [t, n, 64]
//   kv    = bf16(x @ w_dkv_kr) [t, 576];  k_rms = bf16 RmsNorm(kv[:, :512], gamma_ckv)
//   cache row cache_index[t]: four groups of 128 of k_rms quantised like q_norm (int8 + 4 fp32 scales), rotary(kv[:, 512:])
//
// At decode sizes the operator streams 85 MB of weights once (w_dq 22, w_uq_qr 38, w_uk 17, w_dkv_kr 8) and is bound
// by that read.  All four weight matrices are stored with the output dimension contiguous, the opposite of what the
// MFMA operands want (contraction contiguous per lane), so every weight tile goes through LDS and is read back
// transposed: bf16 tiles with ds_read_b64_tr_b16, the int8 tile with ds_read_b64_tr_b8.
//   mla_xa_kernel    x @ [w_dq | w_dkv_kr], 1024 contraction rows x 64 outputs per workgroup, fp32 partials
//   mla_norm_kernel  two workgroups per token: fixed-order sum of the partials, an RmsNorm each, the quantisations, the
//                    key's rotary embedding, the three cache writes, q_norm / q_norm_scale
//   mla_qb_kernel    int8 MFMA GEMM q_norm @ w_uq_qr, 128 outputs x 32 tokens per workgroup, weights streamed to LDS
//                    (gemm_tile.h); dequantisation and the query's rotary embedding on the tile
//   mla_wuk_kernel   per (head, 128 outputs): q_b[:, head, :128] @ w_uk[head]; for many tokens or heads per head (mla_wuk_wide_kernel)
// The last two are one kernel wherever that is faster (head_units): a head's dims and its absorbed product in one workgroup.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdint.h>

#include "common.h"
#include "gemm_tile.h"
#include "kernels.h"
#include "prolog_common.h"
#include "prolog_device.h"
#include "timing.h"

namespace pto {
namespace {

constexpr int MTOK = 32;          // tokens per workgroup tile
constexpr int MNOPE = 128, MROPE = 64, MQH = MNOPE + MROPE, MC = 512, MKV = MC + MROPE;
constexpr int MAX_R = 2048;       // largest q_lora_rank (LDS of mla_norm_kernel)
constexpr int XA_K = 256;         // the hidden size is a multiple
constexpr int XA_SPLIT = 1024;    // contraction rows per workgroup of mla_xa_kernel (one fp32 partial sum each)
constexpr int TROW = 128 * 2 + 32; // bytes per LDS row of a [k][128] bf16 weight tile (padded against bank conflicts)
constexpr int BIG_T = 33;         // token count from which the query kernels that hold more than 32 tokens take over: the others read the
                                  // weights once per 32 tokens (fused prolog, 32 tokens 30.5 us and 40: 31.2; with the weights read
                                  // twice 63.6)
constexpr int BATCH16_T = 128;    // token count to which the bf16 form's query product streams its weights beside all tokens
constexpr int BIG_T2 = 256;       // token count above which the x product's tiles are 256 outputs wide, in splits of its own

// Output tile `tile` (64 columns) of x @ [w_dq | w_dkv_kr | w_k | w_proj]: its weight columns and their row stride.
__device__ __forceinline__ const uint16_t* xa_source(const MlaPrologArgs& a, int tile, int& ld)
{
    const int qtiles = a.r / 64;
    if (tile < qtiles) {
        ld = a.r;
        return a.w_dq + tile * 64;
    }
    if (tile < qtiles + MKV / 64) {
        ld = MKV;
        return a.w_dkv_kr + (tile - qtiles) * 64;
    }
    if (tile < qtiles + MKV / 64 + PD / 64) { // fused with the indexer prolog: its x @ [w_k | w_proj] rides along
        ld = PD;
        return a.w_k + (tile - qtiles - MKV / 64) * 64;
    }
    ld = a.n_idx;
    return a.w_proj + (tile - qtiles - MKV / 64 - PD / 64) * 64;
}

// ------------------------------------------------------------------------------------------------ x @ [w_dq | w_dkv_kr]
// Up to 256 tokens a workgroup owns all tokens x 64 columns over one 1024-row split of the contraction and streams it in stages of
// 64 rows straight to LDS (gemm_tile.h), so that the weights are read once.  x is the A operand here, so a result register holds one
// token's value for 32 consecutive columns across the lanes and the partial sums leave as 128-byte runs.  The sums are chains of 128
// rows added up in order, whatever the number of tokens (a decode step's selection can hang on the last bit of a score, so batches of
// different sizes see the same numbers).
// What bounds it: the weights' stream (34 MB, 6.5 us), and from some 100 tokens on what 252 workgroups draw of x from the L2 (2 KB a
// token and split each, 10 TB/s).
// To 32 tokens 1024 lanes with the whole split in registers, the token rows in operand layout (a different row with every lane: a
// cycle of the texture addresser each, 8192 to a workgroup): a call of the bf16 form of 24 tokens 34.6 us, 32.6 this way, the fused
// operator of 8 and 32 tokens 30.5 -> 29.3 and 32.4 -> 30.7.  Above, tiles of 128 tokens through registers took 13.3 us at 40 tokens
// and 20.9 at 160 (two tiles); so 10.4 and 16.0.
// Three stages ahead: with seven 33.4 at 24 tokens, with eleven 34.3 (fused, 96 tokens: 40.3 with seven, 39.0 with three; two ahead are as good).
// grid (splits, output tiles of 64), 512 lanes: up to four blocks of 32 tokens wave w owns block w / 2 x 32 columns, above block w x 64.
constexpr int XB_KS = 64; // contraction rows per stage
template <int TT>
__global__ __launch_bounds__(512, 2) void mla_xa_kernel(MlaPrologArgs a)
{
    constexpr int XBYTES = TT * 32 * 128, STAGE = XBYTES + XB_KS * 128, FIT = 160 * 1024 / STAGE, RING = FIT < 4 ? FIT : 4;
    constexpr int NB = TT <= 4 ? 1 : 2, XC = (TT + 1) / 2;
    static_assert(XA_K % (2 * XB_KS) == 0, "whole chains of 128 rows in every split");
    __shared__ __align__(16) uint8_t lds[RING * STAGE];
    const int lane = threadIdx.x & 63, wave = gt_wave();
    const int l32 = lane & 31, hl = lane >> 5, jj = lane & 15, mh = (lane >> 4) & 1;
    int ld;
    const uint16_t* src = xa_source(a, blockIdx.y, ld);
    const int split = blockIdx.x, kbeg = split * XA_SPLIT, stages = (min(a.h, kbeg + XA_SPLIT) - kbeg) / XB_KS;
    const uint16_t* x = a.x + kbeg;
    src += (int64_t)kbeg * ld;
    // copies of a wave (layout and exchange of the pieces: gemm_tile.h): token rows 64 i + 8 w + lane / 8 (the last rows again where
    // eight waves have more hands than rows), weight rows 8 w + lane / 8.  Eight token rows are a base of their own: all of them can be
    // more than 4 GB
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    const uint16_t* xp[XC];
    uint32_t xo[XC];
    int xd[XC];
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        const int c = min(8 * i + wave, 4 * TT - 1), xrow = 8 * c + (lane >> 3), xrow0 = min(8 * c, a.t - 1);
        xd[i] = 1024 * c;
        xp[i] = x + (int64_t)xrow0 * a.h;
        xo[i] = (uint32_t)(min(xrow, a.t - 1) - xrow0) * a.h * 2 + 16 * (pos ^ ((xrow >> 1) & 7));
    }
    const uint32_t wo = (uint32_t)(row * ld * 2 + 16 * (pos ^ ((row << 1) & 4)));
    const int tb = TT <= 4 ? wave >> 1 : wave, nb0 = TT <= 4 ? wave & 1 : 0;
    const bool busy = tb < TT; // (the barriers are everybody's)
    const uint8_t* xr = lds + (32 * (busy ? tb : 0) + l32) * 128;
    const int xf = (l32 >> 1) & 7;
    const uint8_t* wrow = lds + XBYTES + (8 * hl + (jj >> 2)) * 128 + 8 * (jj & 1);
    const int wpos = 16 * ((4 * nb0 + 2 * mh + ((jj >> 1) & 1)) ^ ((jj >> 1) & 4));
    f32x16 acc[NB], sum[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[nb][e] = sum[nb][e] = 0.f;
    gt_stages<RING, STAGE, XC + 1>(
        stages,
        [&](int st, int b) {
            gt_copy(src + (int64_t)st * XB_KS * ld, wo, lds + b + XBYTES + 1024 * wave);
#pragma unroll
            for (int i = 0; i < XC; ++i) gt_copy(xp[i] + st * XB_KS, xo[i], lds + b + xd[i]);
        },
        [&](int st, int b) {
            if (!busy) return;
            bf16x8 xv[XB_KS / 16], wv[XB_KS / 16][NB];
#pragma unroll
            for (int ks = 0; ks < XB_KS / 16; ++ks) {
                xv[ks] = *reinterpret_cast<const bf16x8*>(xr + b + 16 * ((2 * ks + hl) ^ xf));
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const uint8_t* p = wrow + b + 2048 * ks + (wpos ^ (64 * nb));
                    const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 512);
                    wv[ks][nb] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
            }
#pragma unroll
            for (int ks = 0; ks < XB_KS / 16; ++ks)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv[ks], wv[ks][nb], acc[nb], 0, 0, 0);
            if (st & 1) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[nb][e] += acc[nb][e], acc[nb][e] = 0.f;
            }
        });
    if (!busy) return;
    // register e of sum[nb]: token 32 tb + 8 (e / 4) + 4 hl + e % 4, column 32 (nb0 + nb) + lane % 32
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int tok = 32 * tb + 8 * (e >> 2) + 4 * hl + (e & 3);
        if (tok >= a.t) continue;
        float* out = a.xa_part + ((int64_t)split * a.t + tok) * a.ncols + blockIdx.y * 64 + 32 * nb0 + l32;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) out[32 * nb] = sum[nb][e];
    }
}

// Above 256 tokens the workgroup owns 128 tokens x 256 outputs (gemm_tile.h) over one split of the contraction, whole stages of
// 64 rows, so that the workgroups fill the CUs once: few splits, so few partial sums.  Seven splits of 1024 rows
// with 256 x 64 tiles wrote 97 MB of partial sums at 1501 tokens, which the norm kernel read again.  An XCD takes neighbouring
// workgroups in the order token tile, output tile, split.  grid (workgroups rounded up to a multiple of 8), 512 lanes.
__global__ __launch_bounds__(GT_LANES, 2) void mla_xa_wide_kernel(MlaPrologArgs a, int ttiles, int ntiles, int rows)
{
    using T = GtTile<4>;
    __shared__ __align__(16) uint8_t lds[T::LDS];
    const int id = (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8);
    const int tok0 = id % ttiles * T::TOK, nt = id / ttiles % ntiles, split = id / ttiles / ntiles;
    if (split >= a.ksplits) return; // uniform over the workgroup
    const int kbeg = split * rows, stages = (min(a.h, kbeg + rows) - kbeg) / GT_KBF;
    const uint16_t* src[4];
    int ld[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { // (blocks past the last one: that one again, dropped below)
        src[i] = xa_source(a, min(4 * nt + i, a.ncols / 64 - 1), ld[i]);
        src[i] += (int64_t)kbeg * ld[i];
    }
    f32x16 acc[2][2];
    gt_product_bf16<XA_SPLIT, XA_SPLIT>(acc, src, ld, a.x + kbeg, a.h, tok0, a.t, stages, lds);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, hl = lane >> 5, wr = wave >> 2, wc = wave & 3;
    const int col0 = (4 * nt + wc) * 64;
    if (col0 >= a.ncols) return;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int gt = tok0 + 64 * wr + 32 * tb + 8 * (e >> 2) + 4 * hl + (e & 3);
            if (gt >= a.t) continue;
            float* out = a.xa_part + ((int64_t)split * a.t + gt) * a.ncols + col0 + l32;
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) out[32 * nb] = acc[tb][nb][e];
        }
}
// its contraction rows per split: as many splits as there are CUs for, and no more than the workspace holds, as even as whole
// stages allow (in pieces of 256 rows, where three or five splits of 7168 end on an emptier one: fused prolog of 600 tokens 108.6 us a
// call, so 107.1, 1024: 155.2 / 154.2; bf16 form of 600 118.4 / 116.4).  The same with and without the indexer's columns (counted in), so that the fused operator's sums are the others'.
static int xa_wide_rows(int64_t t, int64_t h, int64_t r)
{
    const int64_t tiles = ((t + 127) / 128) * ((r + MKV + PD + 64 + 255) / 256), most = (h + XA_SPLIT - 1) / XA_SPLIT;
    const int64_t splits = std::max<int64_t>(1, std::min<int64_t>(most, 256 / tiles));
    return (int)((h / GT_KBF + splits - 1) / splits) * GT_KBF;
}

// Four blocks of 64 outputs of q_b, TOK tokens each, from LDS rows of QBS_ROW bytes (padded against bank conflicts) to memory in
// 16-byte pieces: a block is half of a head's 128 first dims, or its rotary dims, rotated on the way.  PER lanes to a block (two waves: two
// blocks in 256 lanes); step: from one of them to the next.
constexpr int QBS_ROW = 64 * 2 + 16;
template <int TOK, int PER = 128>
__device__ __forceinline__ void qb_store_blocks(const MlaPrologArgs& a, const uint8_t* lds, int block0, int tok0, int step = 1)
{
#pragma clang fp contract(off)
    const int tid = threadIdx.x, blocks = a.n * MQH / 64;
    const int bl = tid / PER, block = block0 + step * bl, head = block / 3;
    if (block >= blocks) return;
    const uint8_t* tile = lds + bl * TOK * QBS_ROW;
    if (block % 3 < 2) { // 8 pieces of 8 dims
        uint16_t* dst = a.qb_nope + head * MNOPE + block % 3 * 64 + 8 * (tid & 7);
#pragma unroll
        for (int i = 0; i < TOK * 8 / PER; ++i) {
            const int tl = (tid % PER >> 3) + PER / 8 * i;
            if (tok0 + tl < a.t)
                *reinterpret_cast<u32x4*>(dst + (int64_t)(tok0 + tl) * a.n * MNOPE) =
                    *reinterpret_cast<const u32x4*>(tile + tl * QBS_ROW + 16 * (tid & 7));
        }
    } else { // 4 times 8 pairs, rotated into the two halves
        const int i0 = 8 * (tid & 3);
#pragma unroll
        for (int i = 0; i < (TOK * 4 + PER - 1) / PER; ++i) {
            const int tl = (tid % PER >> 2) + PER / 4 * i, gt = tok0 + tl;
            if (tl >= TOK || gt >= a.t) continue;
            const u32x4* x = reinterpret_cast<const u32x4*>(tile + tl * QBS_ROW + 4 * i0);
            const uint16_t* cp = a.cos + (int64_t)gt * MROPE + i0;
            const uint16_t* sp = a.sin + (int64_t)gt * MROPE + i0;
            const u32x4 xa = x[0], xb = x[1];
            const u32x4 c1 = *reinterpret_cast<const u32x4*>(cp), c2 = *reinterpret_cast<const u32x4*>(cp + 32);
            const u32x4 s1 = *reinterpret_cast<const u32x4*>(sp), s2 = *reinterpret_cast<const u32x4*>(sp + 32);
            u32x4 o1, o2;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float r1[2], r2[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t pair = w < 2 ? xa[2 * w + e] : xb[2 * w + e - 4];
                    const int sh = 16 * e;
                    const float xe = bf16_bits_to_f32(pair & 0xffffu), xo = bf16_bits_to_f32(pair >> 16);
                    r1[e] = xe * bf16_bits_to_f32((c1[w] >> sh) & 0xffffu) + (-xo) * bf16_bits_to_f32((s1[w] >> sh) & 0xffffu);
                    r2[e] = xo * bf16_bits_to_f32((c2[w] >> sh) & 0xffffu) + xe * bf16_bits_to_f32((s2[w] >> sh) & 0xffffu);
                }
                o1[w] = pack_bf16x2(r1[0], r1[1]);
                o2[w] = pack_bf16x2(r2[0], r2[1]);
            }
            uint16_t* out = a.q_rope + ((int64_t)gt * a.n + head) * MROPE + i0;
            *reinterpret_cast<u32x4*>(out) = o1;
            *reinterpret_cast<u32x4*>(out + 32) = o2;
        }
    }
}

// bf16 form of the operator, up to 32 tokens: q_b = q_norm (bf16 [t, r]) @ w_uq_qr (bf16 [r, n * 192]), a stream of 75 MB of
// weights.  A workgroup owns 128 outputs (192 of them at model sizes) and keeps three stages of 64 rows x 256 bytes in flight
// straight to LDS (call of 24 tokens 30.8 us, with six 31.3; out of HBM 35.9 and 36.3).  Splits of 1024 rows loaded in one go through registers, their fp32 partial sums through memory and a kernel
// behind them took 24.4 + 4.8 us at 24 tokens.  The sums: chains of 128 rows added up in order, then splits of 1024 rows.
// 256 lanes: wave w owns outputs [32 w, +32); the two blocks of 64 begin at w0 and w1.  run(copy, multiply) goes through the stages.
// Register e of sum: output 32 w + 8 (e / 4) + 4 hl + e % 4, token lane % 32.
struct Qb16Stream { // a stage: token rows | [2] weight rows of 128 bytes
    static constexpr int XB = MTOK * 128, STAGE = XB + 2 * 64 * 128, RING = 4, LDS = RING * STAGE;
};
template <class Run>
__device__ __forceinline__ void qb16_stream(f32x16& sum, const MlaPrologArgs& a, const uint16_t* w0, const uint16_t* w1, uint8_t* lds, Run&& run)
{
#pragma clang fp contract(off)
    constexpr int XB = Qb16Stream::XB;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, hl = lane >> 5, jj = lane & 15, mh = (lane >> 4) & 1;
    const int nq = a.n * MQH;
    const uint16_t* x = reinterpret_cast<const uint16_t*>(a.q_norm);
    // copies of a wave (layout and exchange of the pieces: gemm_tile.h): token rows 8 w + lane / 8, weight rows 32 i + that
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    const uint32_t xo = (uint32_t)(min(row, a.t - 1) * a.r * 2 + 16 * (pos ^ ((row >> 1) & 7)));
    uint32_t wo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) wo[i] = (uint32_t)((row + 32 * i) * nq * 2 + 16 * (pos ^ ((row << 1) & 4)));
    const uint8_t* xr = lds + l32 * 128;
    const int xf = (l32 >> 1) & 7;
    const uint8_t* wrow = lds + XB + (wave >> 1) * 8192 + (8 * hl + (jj >> 2)) * 128 + 8 * (jj & 1);
    const int wpos = 16 * ((4 * (wave & 1) + 2 * mh + ((jj >> 1) & 1)) ^ ((jj >> 1) & 4));
    f32x16 acc, part;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = part[e] = sum[e] = 0.f;
    const int stages = a.r / 64;
    run(
        [&](int st, int b) {
            uint8_t* d = lds + b + 1024 * wave;
            gt_copy(x + st * 64, xo, d);
#pragma unroll
            for (int i = 0; i < 4; ++i) gt_copy((i < 2 ? w0 : w1) + (int64_t)st * 64 * nq, wo[i & 1], d + XB + 4096 * i);
        },
        [&](int st, int b) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const uint8_t* p = wrow + b + 2048 * ks + wpos;
                const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 512);
                const bf16x8 wv = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                const bf16x8 xv = *reinterpret_cast<const bf16x8*>(xr + b + 16 * ((2 * ks + hl) ^ xf));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, xv, acc, 0, 0, 0);
            }
            const bool last = st + 1 == stages;
            if (st % 2 == 1 || last) {
#pragma unroll
                for (int e = 0; e < 16; ++e) part[e] += acc[e], acc[e] = 0.f;
            }
            if ((st + 1) % (XA_SPLIT / 64) == 0 || last) {
#pragma unroll
                for (int e = 0; e < 16; ++e) sum[e] += part[e], part[e] = 0.f;
            }
        });
}
// the sums as bf16 rows [2 blocks][32 tokens] of QBS_ROW bytes
__device__ __forceinline__ void qb16_tile(const f32x16& sum, uint8_t* tile)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, hl = lane >> 5;
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4)
        *reinterpret_cast<u32x2*>(tile + ((wave >> 1) * MTOK + l32) * QBS_ROW + (32 * (wave & 1) + 8 * e4 + 4 * hl) * 2) =
            u32x2{pack_bf16x2(sum[4 * e4], sum[4 * e4 + 1]), pack_bf16x2(sum[4 * e4 + 2], sum[4 * e4 + 3])};
}
// grid (n * 192 / 128), 256 lanes
__global__ __launch_bounds__(256) void mla_qb16_kernel(MlaPrologArgs a)
{
    using S = Qb16Stream;
    static_assert(2 * MTOK * QBS_ROW <= S::LDS, "the output tile takes the stages' place");
    __shared__ __align__(16) uint8_t lds[S::LDS];
    const uint16_t* w = static_cast<const uint16_t*>(a.w_uq_qr) + 128 * blockIdx.x;
    f32x16 sum;
    qb16_stream(sum, a, w, w + 64, lds, [&](auto&& copy, auto&& multiply) { gt_stages<S::RING, S::STAGE, 5>(a.r / 64, copy, multiply); });
    qb16_tile(sum, lds);
    __syncthreads();
    qb_store_blocks<MTOK>(a, lds, 2 * blockIdx.x, 0);
}

// The bf16 form at more tokens: 128 tokens x 256 outputs per workgroup over the whole contraction (gemm_tile.h), the epilogue
// on the tile: 91 us at 1024 tokens, where a kernel that read the weights once per 32 tokens took 811.  The sums are
// mla_qb16_kernel's bit for bit (in chains of 256 rows, added up in order, they took 5 us less there and 2 at 33 tokens, and were 10 %
// further off).  grid (n * 192 / 256 rounded up, token tiles of 128), 512 lanes.
__global__ __launch_bounds__(GT_LANES, 2) void mla_qb16_wide_kernel(MlaPrologArgs a)
{
#pragma clang fp contract(off)
    using T = GtTile<4>;
    static_assert(4 * T::TOK * QBS_ROW <= T::LDS, "the output tile takes the operand tiles' place");
    __shared__ __align__(16) uint8_t lds[T::LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hl = lane >> 5, wr = wave >> 2, wc = wave & 3;
    const int blocks = a.n * MQH / 64, block0 = 4 * blockIdx.x, tok0 = blockIdx.y * T::TOK;
    const uint16_t* src[4];
    int ld[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { // (blocks past the last one: that one again, dropped below)
        src[i] = static_cast<const uint16_t*>(a.w_uq_qr) + min(block0 + i, blocks - 1) * 64;
        ld[i] = a.n * MQH;
    }
    f32x16 acc[2][2];
    gt_product_bf16<128, XA_SPLIT>(acc, src, ld, reinterpret_cast<const uint16_t*>(a.q_norm), a.r, tok0, a.t, a.r / GT_KBF, lds);
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int tl = 64 * wr + 32 * tb + 8 * (e >> 2) + 4 * hl + (e & 3);
            uint16_t* row = reinterpret_cast<uint16_t*>(lds + (wc * T::TOK + tl) * QBS_ROW) + l32;
            row[0] = f32_to_bf16(acc[tb][0][e]);
            row[32] = f32_to_bf16(acc[tb][1][e]);
        }
    __syncthreads();
    qb_store_blocks<T::TOK>(a, lds, block0, tok0);
}

// ------------------------------------------------------------------------------------------------ norms, quantisation, cache
__device__ __forceinline__ float wave_sum(float v) { return wave_sum_butterfly(v); }
__device__ __forceinline__ float wave_max(float v) { return wave_max_f32(v); }

// Columns col0 + 4 tid + 1024 j .. + 3, j < NP, of a token's row: partial sums in a fixed order, rounded to bf16, into x and buf (n
// columns, a multiple of 4; S: splits whose partial sums are in flight together).  Four columns a load: a load costs the memory
// pipe its 64 lanes whatever their width, and single columns were 64 loads a lane of the query's chain at seven splits (with the
// indexer's key path, prolog_k_body: call of 1 token 34.6 -> 33.0 us, MLA alone 38.5 -> 36.4, 1501 tokens 232 -> 225).  Every
// load is unconditional (columns past the end re-read the last ones and are dropped): a load under a condition makes the compiler
// wait for it on the spot, one memory round trip per load.
template <int S, int NP>
__device__ __forceinline__ void mla_sums(const MlaPrologArgs& a, int tok, int col0, int n, float (&x)[NP][4], float* buf)
{
    const int tid = threadIdx.x;
    int cj[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        cj[j] = col0 + min(1024 * j + 4 * tid, n - 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[j][e] = 0.f;
    }
    // (a split past the end re-reads the last one and adds zero)
    for (int s0 = 0; s0 < a.ksplits; s0 += S) {
        f32x4 v[S][NP];
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const float* p = a.xa_part + ((int64_t)min(s0 + i, a.ksplits - 1) * a.t + tok) * a.ncols;
#pragma unroll
            for (int j = 0; j < NP; ++j) v[i][j] = *reinterpret_cast<const f32x4*>(p + cj[j]);
        }
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][e] += s0 + i < a.ksplits ? v[i][j][e] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < NP; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[j][e] = round_bf16(x[j][e]);
        if (1024 * j + 4 * tid < n) *reinterpret_cast<f32x4*>(buf + 1024 * j + 4 * tid) = f32x4{x[j][0], x[j][1], x[j][2], x[j][3]};
    }
}

// The two norms of a token are independent chains of loads, reductions and barriers: a workgroup of 256 lanes for either (one
// workgroup for both, one chain behind the other: 1.6 us more a call, at 1 token as at 600).
// Query: RmsNorm over r, then per-token quantisation.
template <int S>
__device__ __forceinline__ void mla_norm_query_body(const MlaPrologArgs& a, int tok)
{
#pragma clang fp contract(off)
    __shared__ __align__(16) float buf[MAX_R];
    __shared__ float red[8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = a.r;
    // (what does not depend on the sums is loaded first, so that its latency hides behind them)
    constexpr int NP = MAX_R / 1024;
    u32x2 gq[NP];
    float x[NP][4];
#pragma unroll
    for (int j = 0; j < NP; ++j) gq[j] = *reinterpret_cast<const u32x2*>(a.gamma_cq + min(1024 * j + 4 * tid, r - 4));
    mla_sums<S, NP>(a, tok, 0, r, x, buf);
    __syncthreads();
    const float coff = 1.0f / (float)r;
    float ss = 0.f;
    for (int c = tid; c < r; c += 256) ss += (buf[c] * buf[c]) * coff;
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    const float y = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) + a.eps_cq);
    float mx = 0.f; // (columns past the end are the last ones again)
#pragma unroll
    for (int j = 0; j < NP; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[j][e] = round_bf16(half_of(gq[j][e >> 1], e & 1) * (x[j][e] * y));
            mx = fmaxf(mx, fabsf(x[j][e]));
        }
    mx = wave_max(mx);
    if (lane == 0) red[4 + wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
    if (a.quant) {
        const float sq = quant_scale(mx);
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int c = 1024 * j + 4 * tid;
            uint32_t pk = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) pk |= ((uint32_t)(int)__builtin_rintf(x[j][e] * sq) & 0xffu) << (8 * e);
            if (c < r) *reinterpret_cast<uint32_t*>(a.q_norm + (int64_t)tok * r + c) = pk;
        }
        if (tid == 0) a.q_norm_scale[tok] = 1.0f / sq;
    } else { // bf16 form: q_norm is the normalised row itself
        uint16_t* qo = reinterpret_cast<uint16_t*>(a.q_norm) + (int64_t)tok * r;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int c = 1024 * j + 4 * tid;
            if (c < r) *reinterpret_cast<u32x2*>(qo + c) = u32x2{pack_bf16x2(x[j][0], x[j][1]), pack_bf16x2(x[j][2], x[j][3])};
        }
    }
}

// Key: RmsNorm over 512 (lane: elements tid and tid + 256), groups of 128 quantised on their own, rotary, the cache rows.
template <int S>
__device__ __forceinline__ void mla_norm_key_body(const MlaPrologArgs& a, int tok)
{
#pragma clang fp contract(off)
    __shared__ __align__(16) float buf[MKV];
    __shared__ float red[8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = a.cache_index[tok];
    const bool row_ok = row >= 0 && row < a.cache_rows;
    const uint16_t gk0 = a.gamma_ckv[tid], gk1 = a.gamma_ckv[256 + tid];
    const int ri = tid & 31;
    const float rc0 = bf16_to_f32(a.cos[(int64_t)tok * MROPE + ri]), rc1 = bf16_to_f32(a.cos[(int64_t)tok * MROPE + ri + 32]);
    const float rs0 = bf16_to_f32(a.sin[(int64_t)tok * MROPE + ri]), rs1 = bf16_to_f32(a.sin[(int64_t)tok * MROPE + ri + 32]);
    float x[1][4];
    mla_sums<S, 1>(a, tok, a.r, MKV, x, buf);
    __syncthreads();
    {
        const float x0 = buf[tid], x1 = buf[256 + tid];
        float ss = wave_sum((x0 * x0) * (1.0f / MC) + (x1 * x1) * (1.0f / MC));
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        const float y = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) + a.eps_ckv);
        const float v0 = round_bf16(bf16_to_f32(gk0) * (x0 * y));
        const float v1 = round_bf16(bf16_to_f32(gk1) * (x1 * y));
        // waves 0, 1 hold group 0 (v0) and group 2 (v1); waves 2, 3 groups 1 and 3
        const float m0 = wave_max(fabsf(v0)), m1 = wave_max(fabsf(v1));
        __syncthreads();
        if (lane == 0) {
            red[wave] = m0;
            red[4 + wave] = m1;
        }
        __syncthreads();
        const int pair = wave & 2;
        const float sq0 = quant_scale(fmaxf(red[pair], red[pair + 1]));
        const float sq1 = quant_scale(fmaxf(red[4 + pair], red[4 + pair + 1]));
        if (row_ok && a.quant) {
            a.kv_cache[row * MC + tid] = (int8_t)(int)__builtin_rintf(v0 * sq0);
            a.kv_cache[row * MC + 256 + tid] = (int8_t)(int)__builtin_rintf(v1 * sq1);
            if ((tid & 127) == 0) {
                a.k_scale_cache[row * 4 + (tid >> 7)] = 1.0f / sq0;
                a.k_scale_cache[row * 4 + 2 + (tid >> 7)] = 1.0f / sq1;
            }
        } else if (row_ok) { // bf16 form: the cache row is the normalised key itself, no scales
            uint16_t* kvo = reinterpret_cast<uint16_t*>(a.kv_cache) + row * MC;
            kvo[tid] = f32_to_bf16(v0);
            kvo[256 + tid] = f32_to_bf16(v1);
        }
    }
    // key rotary: pair i = elements (2i, 2i+1) -> positions (i, 32 + i)
    if (tid < MROPE / 2 && row_ok) {
        const float xe = buf[MC + 2 * tid], xo = buf[MC + 2 * tid + 1];
        const float o1 = xe * rc0 + (-xo) * rs0;
        const float o2 = xo * rc1 + xe * rs1;
        a.kr_cache[row * MROPE + tid] = f32_to_bf16(o1);
        a.kr_cache[row * MROPE + 32 + tid] = f32_to_bf16(o2);
    }
}

// The fused operator's norms above 256 tokens where the x product has at most eight splits: a wavefront to each of a
// token's three chains, the sums of the workgroups above bit for bit - what they spread over four wavefronts (lane l of wave w: columns
// l + 64 w + 256 i) are four sums of a lane here, and no barrier is passed.  The fused operator has the int8 form only.
// What bounds it: the partial sums' way from memory (28 MB at 1501 tokens).  A workgroup to a chain went through barriers with
// eight chains in flight to a CU, and every token's fetched hadamard_k's 32 KB out of the L2 in 128 loads: the kernel at 1501 tokens 15.1 us, so 11.6,
// a call 210.7 -> 208.1, 900: 140.4 / 138.1; with five to seven splits, 218 registers, three sets of operands in turn, 257: 63.7 / 63.2, 410: 78.6 / 77.2,
// 600: 100.8 / 99.2; to 256 tokens slower (200: 57.9 / 58.0, 96: 41.2 / 42.0).  The MLA prolog's two chains alone are no faster (1024 tokens 8.3 / 8.4, a
// call of 300 60.3 / 61.5).
// request(i, split) asks for what a chain reads of a split, all S of them in flight together (a split past the end is the last one
// again, dropped), add(i, first, real) adds it up in order.
template <int S, class Request, class Add>
__device__ __forceinline__ void each_split(int ksplits, Request&& request, Add&& add)
{
#pragma unroll
    for (int i = 0; i < S; ++i) request(i, min(i, ksplits - 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < S; ++i) add(i, i == 0, i < ksplits);
}

template <int S, int NP>
__device__ __forceinline__ void mla_norm_query_wave(const MlaPrologArgs& a, int tok, float* buf)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, r = a.r;
    f32x4 x[NP], v[S][NP];
    each_split<S>(
        a.ksplits,
        [&](int i, int split) {
            const float* p = a.xa_part + ((int64_t)split * a.t + tok) * a.ncols;
#pragma unroll
            for (int j = 0; j < NP; ++j) v[i][j] = *reinterpret_cast<const f32x4*>(p + min(256 * j + 4 * lane, r - 4));
        },
        [&](int i, bool first, bool real) {
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][e] = first ? v[i][j][e] : x[j][e] + (real ? v[i][j][e] : 0.f);
        });
    u32x2 gq[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) gq[j] = *reinterpret_cast<const u32x2*>(a.gamma_cq + min(256 * j + 4 * lane, r - 4));
#pragma unroll
    for (int j = 0; j < NP; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[j][e] = round_bf16(x[j][e]);
        *reinterpret_cast<f32x4*>(buf + 256 * j + 4 * lane) = 256 * j + 4 * lane < r ? x[j] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __builtin_amdgcn_wave_barrier();
    const float coff = 1.0f / (float)r;
    float ss[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        ss[w] = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const float b = buf[256 * i + 64 * w + lane]; // (zero past the end)
            ss[w] += (b * b) * coff;
        }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) ss[w] = wave_sum(ss[w]);
    const float y = 1.0f / sqrtf(((ss[0] + ss[1]) + (ss[2] + ss[3])) + a.eps_cq);
    float mx = 0.f; // (columns past the end are the last ones again)
#pragma unroll
    for (int j = 0; j < NP; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[j][e] = round_bf16(half_of(gq[j][e >> 1], e & 1) * (x[j][e] * y));
            mx = fmaxf(mx, fabsf(x[j][e]));
        }
    const float sq = quant_scale(wave_max(mx));
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        const int c = 256 * j + 4 * lane;
        uint32_t pk = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) pk |= ((uint32_t)(int)__builtin_rintf(x[j][e] * sq) & 0xffu) << (8 * e);
        if (c < r) *reinterpret_cast<uint32_t*>(a.q_norm + (int64_t)tok * r + c) = pk;
    }
    if (lane == 0) a.q_norm_scale[tok] = 1.0f / sq;
}

// lane l: columns l + 64 m of the 512 normalised ones, and (l < 32) the rotary pair 2 l, 2 l + 1
template <int S>
__device__ __forceinline__ void mla_norm_key_wave(const MlaPrologArgs& a, int tok)
{
#pragma clang fp contract(off)
    constexpr int M = MC / 64;
    const int lane = threadIdx.x & 63, ri = lane & 31;
    const int64_t row = a.cache_index[tok];
    uint16_t gk[M];
#pragma unroll
    for (int m = 0; m < M; ++m) gk[m] = a.gamma_ckv[64 * m + lane];
    const float rc0 = bf16_to_f32(a.cos[(int64_t)tok * MROPE + ri]), rc1 = bf16_to_f32(a.cos[(int64_t)tok * MROPE + ri + 32]);
    const float rs0 = bf16_to_f32(a.sin[(int64_t)tok * MROPE + ri]), rs1 = bf16_to_f32(a.sin[(int64_t)tok * MROPE + ri + 32]);
    float x[M], pv[S][M];
    float2 pair, pp[S];
    each_split<S>(
        a.ksplits,
        [&](int i, int split) {
            const float* p = a.xa_part + ((int64_t)split * a.t + tok) * a.ncols + a.r;
#pragma unroll
            for (int m = 0; m < M; ++m) pv[i][m] = p[64 * m + lane];
            pp[i] = *reinterpret_cast<const float2*>(p + MC + 2 * ri);
        },
        [&](int i, bool first, bool real) {
#pragma unroll
            for (int m = 0; m < M; ++m) x[m] = first ? pv[i][m] : x[m] + (real ? pv[i][m] : 0.f);
            pair.x = first ? pp[i].x : pair.x + (real ? pp[i].x : 0.f);
            pair.y = first ? pp[i].y : pair.y + (real ? pp[i].y : 0.f);
        });
    const bool row_ok = row >= 0 && row < a.cache_rows;
    float ss[4], v[M];
#pragma unroll
    for (int m = 0; m < M; ++m) x[m] = round_bf16(x[m]);
#pragma unroll
    for (int w = 0; w < 4; ++w) ss[w] = wave_sum((x[w] * x[w]) * (1.0f / MC) + (x[w + 4] * x[w + 4]) * (1.0f / MC));
    const float y = 1.0f / sqrtf(((ss[0] + ss[1]) + (ss[2] + ss[3])) + a.eps_ckv);
#pragma unroll
    for (int m = 0; m < M; ++m) v[m] = round_bf16(bf16_to_f32(gk[m]) * (x[m] * y));
#pragma unroll
    for (int g = 0; g < M / 2; ++g) { // groups of 128
        const float sq = quant_scale(wave_max(fmaxf(fabsf(v[2 * g]), fabsf(v[2 * g + 1]))));
        if (row_ok) {
            a.kv_cache[row * MC + 128 * g + lane] = (int8_t)(int)__builtin_rintf(v[2 * g] * sq);
            a.kv_cache[row * MC + 128 * g + 64 + lane] = (int8_t)(int)__builtin_rintf(v[2 * g + 1] * sq);
            if (lane == 0) a.k_scale_cache[row * 4 + g] = 1.0f / sq;
        }
    }
    if (lane < MROPE / 2 && row_ok) {
        const float xe = round_bf16(pair.x), xo = round_bf16(pair.y);
        a.kr_cache[row * MROPE + lane] = f32_to_bf16(xe * rc0 + (-xo) * rs0);
        a.kr_cache[row * MROPE + 32 + lane] = f32_to_bf16(xo * rc1 + xe * rs1);
    }
}

// The indexer's key path and weights (prolog_k_body's arithmetic); had: hadamard_k in LDS
template <int S>
__device__ __forceinline__ void prolog_k_wave(const PrologArgs& a, int tok, const uint32_t* had)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int64_t row = a.k_cache_index[tok];
    float gam[2], bet[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        gam[m] = bf16_to_f32(a.ln_gamma[64 * m + lane]);
        bet[m] = bf16_to_f32(a.ln_beta[64 * m + lane]);
    }
    const float rc = bf16_to_f32(a.cos[(int64_t)tok * PROPE + lane]), rs = bf16_to_f32(a.sin[(int64_t)tok * PROPE + lane]);
    float kv[2], wv[2], v0[S][2], v1[S][2];
    each_split<S>(
        a.ksplits,
        [&](int i, int split) {
            const float* p = a.xw_part + ((int64_t)split * a.t + tok) * a.xw_stride + a.xw_col0;
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                v0[i][m] = p[64 * m + lane];
                v1[i][m] = p[PD + min(64 * m + lane, a.n - 1)];
            }
        },
        [&](int i, bool first, bool real) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                kv[m] = first ? v0[i][m] : kv[m] + (real ? v0[i][m] : 0.f);
                wv[m] = first ? v1[i][m] : wv[m] + (real ? v1[i][m] : 0.f);
            }
        });
    const float mean = (wave_sum(kv[0]) + wave_sum(kv[1])) / (float)PD;
    float dlt[2], kb[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) dlt[m] = kv[m] - mean;
    const float var = (wave_sum(dlt[0] * dlt[0]) + wave_sum(dlt[1] * dlt[1])) / (float)PD;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        float xn = dlt[m] / sqrtf(var + a.eps);
        xn = xn * gam[m] + bet[m];
        kb[m] = round_bf16(xn);
    }
    // rotary on the first 64 dims: the partner is 32 lanes away
    const float far = __shfl_xor(kb[0], 32);
    kb[0] = round_bf16(kb[0] * rc + (lane < 32 ? -far : far) * rs);
    // hadamard: columns 2 l, 2 l + 1, k in order
    float2 h = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < PD; ++k) {
        const float x = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, kb[k >> 6]), k & 63));
        const uint32_t hk = had[64 * k + lane];
        h.x = __builtin_fmaf(x, half_of(hk, 0), h.x);
        h.y = __builtin_fmaf(x, half_of(hk, 1), h.y);
    }
    const float y0 = round_bf16(h.x), y1 = round_bf16(h.y);
    const float sq = quant_scale(wave_max(fmaxf(fabsf(y0), fabsf(y1))));
    if (row >= 0 && row < a.cache_rows) {
        const uint32_t q0 = (uint32_t)(int)__builtin_rintf(y0 * sq) & 0xffu, q1 = (uint32_t)(int)__builtin_rintf(y1 * sq) & 0xffu;
        *reinterpret_cast<uint16_t*>(a.k_cache + row * PD + 2 * lane) = (uint16_t)(q0 | (q1 << 8));
        if (lane == 0) a.k_scale_cache[row] = __builtin_bit_cast(uint16_t, (_Float16)(1.0f / sq));
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
        if (64 * m + lane < a.n) {
            const float w = bf16_to_f32(f32_to_bf16(wv[m]));
            a.weights[(int64_t)tok * a.n + 64 * m + lane] = __builtin_bit_cast(uint16_t, (_Float16)((w * a.wscale_n) * a.wscale_d));
        }
}

// grid (3 ceil(t / 4): the indexer's keys, queries, keys; four tokens to a workgroup), 256 lanes
template <int S, int NP>
__global__ __launch_bounds__(256) void fused_norm_wide_kernel(MlaPrologArgs m, PrologArgs p)
{
    constexpr int QB = 4 * NP * 256 * 4, HB = PD * PD * 2;
    __shared__ __align__(16) uint8_t lds[HB > QB ? HB : QB];
    const int groups = (m.t + 3) / 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = blockIdx.x / groups, tok = 4 * (blockIdx.x % groups) + wave;
    if (part == 0) {
        u32x4 h[HB / 4096];
#pragma unroll
        for (int i = 0; i < HB / 4096; ++i) h[i] = reinterpret_cast<const u32x4*>(p.had_k)[threadIdx.x + 256 * i];
#pragma unroll
        for (int i = 0; i < HB / 4096; ++i) reinterpret_cast<u32x4*>(lds)[threadIdx.x + 256 * i] = h[i];
        __syncthreads();
    }
    if (tok >= m.t) return;
    if (part == 0)
        prolog_k_wave<S>(p, tok, reinterpret_cast<const uint32_t*>(lds));
    else if (part == 1)
        mla_norm_query_wave<S, NP>(m, tok, reinterpret_cast<float*>(lds) + wave * NP * 256);
    else
        mla_norm_key_wave<S>(m, tok);
}

// The head of a weight slice, read and dropped: the first `rows` rows of 16 `pieces` bytes (rows a multiple of what 256 lanes
// cover in one go, up to 24 times that), so that the workgroup of the next launch that streams the slice finds them in
// its XCD's L2.  The second half of a row's pieces lies `gap` bytes further on.
__device__ __forceinline__ void touch_rows(const uint8_t* base, int64_t stride, int rows, int pieces, int gap)
{
    const int per = 256 / pieces, row = threadIdx.x / pieces, n = rows / per, piece = threadIdx.x % pieces;
    const uint8_t* p = base + row * stride + piece * 16 + (2 * piece >= pieces ? gap : 0);
    u32x4 v[24];
#pragma unroll
    for (int i = 0; i < 24; ++i)
        if (i < n) v[i] = *reinterpret_cast<const u32x4*>(p + i * per * stride);
#pragma unroll
    for (int i = 0; i < 24; ++i)
        if (i < n) asm volatile("" ::"v"(v[i]));
}

// ------------------------------------------------------------------------------------------------ q_norm @ w_uq_qr
// Up to 32 tokens: 128 outputs per workgroup of 256 lanes behind the streamed product (gemm_tile.h); dequantisation and the
// query's rotary embedding on the tile.  The int32 sums are exact.  The outputs are two times 64, `gap` columns apart.
struct QbScales {
    float qs[2];
    f32x4 ws[2];
    __device__ __forceinline__ void load(const MlaPrologArgs& a, int col0, int gap)
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) qs[tb] = a.q_norm_scale[min(16 * tb + l16, a.t - 1)];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
            ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + col0 + (wave >> 1) * gap + 32 * wave + 16 * nb + 4 * g);
    }
    // bf16 rows [2 blocks][32 tokens] of QBS_ROW bytes
    __device__ __forceinline__ void tile(const i32x4 (&acc)[2][2], uint8_t* to) const
    {
#pragma clang fp contract(off)
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs[tb]) * ws[nb][e];
                *reinterpret_cast<u32x2*>(to + ((wave >> 1) * MTOK + 16 * tb + l16) * QBS_ROW + (32 * (wave & 1) + 16 * nb + 4 * g) * 2) =
                    u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            }
    }
};
__device__ __forceinline__ void mla_qb_body(const MlaPrologArgs& a, int tile, uint8_t* lds)
{
    QbScales scales;
    scales.load(a, 128 * tile, 0);
    i32x4 acc[2][2] = {};
    gt_stream_i8(acc, static_cast<const int8_t*>(a.w_uq_qr) + 128 * tile, (int64_t)a.n * MQH, a.q_norm, a.r, a.t, a.r / GT_KI8, lds);
    scales.tile(acc, lds);
    __syncthreads();
    qb_store_blocks<MTOK>(a, lds, 2 * tile, 0);
}

// Up to 32 tokens and one workgroup to a CU (head_units): a head's 128 first dims of q_b in one workgroup, which goes on to
// the absorbed product with the head's w_uk, whose 128 KB follow the other weights through the same stages; the rotary dims of two heads
// in another.  The three workgroups of two heads, which share cache lines of the int8 weights, go to one XCD, in the last of the rounds of eight pairs too,
// whose other workgroups have nothing to do (int8 form, us a call of 8 tokens with the last pairs' workgroups side by side / so: 100 heads 23.4 / 21.0, 120:
// 25.3 / 21.8, 170: 28.2 / 26.5; fused, 126 heads 30.3 / 25.0).  The bf16 form's share none: 170 heads 29.5 side by side, 35.5 so, with 33 workgroups
// to some XCDs' 32 CUs.
// A kernel of its own for the absorbed product, 512 workgroups behind a launch and a round trip of q_b through memory, took 4.2 to 5 us.
constexpr int WUK_CHUNKS = MC / 64; // stages of w_uk: 128 rows x 64 columns
struct HeadUnit {
    int head, col0, gap; // (the first) head, first output, from the first 64 outputs to the others
    bool nope;
};
__device__ __forceinline__ HeadUnit head_unit(const MlaPrologArgs& a, int id)
{
    const bool rounds = a.quant || a.n % 16 == 0; // of the XCDs, a pair to each
    const int pair = rounds ? id / 24 * 8 + id % 8 : id / 3, k = rounds ? id / 8 % 3 : id % 3;
    if (2 * pair >= a.n) return HeadUnit{-1, 0, 0, false}; // none
    return k < 2 ? HeadUnit{2 * pair + k, (2 * pair + k) * MQH, 0, true} : HeadUnit{2 * pair, 2 * pair * MQH + MNOPE, MQH - 64, false};
}
__host__ __device__ inline int head_grid(const MlaPrologArgs& a) { return a.quant ? 24 * ((a.n + 15) / 16) : a.n * MQH / 128; }
struct Absorbed { // wave w: columns 32 (w % 2) of the chunks 2 i + w / 2
    static constexpr int TILE = 2 * MTOK * QBS_ROW, OROW = MC * 2 + 16; // bytes of q_b's tile, of an LDS row of the outputs
    f32x16 acc[WUK_CHUNKS / 2];

    // five copies of a wave, as many as a stage of the other weights (the first is not used)
    static __device__ __forceinline__ void copy(const MlaPrologArgs& a, int head, int c, uint8_t* slot)
    {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int row = 8 * wave + (lane >> 3), pos = lane & 7;
        const uint16_t* w = a.w_uk + (int64_t)head * MNOPE * MC + 64 * c;
        const uint32_t at = (uint32_t)(row * MC * 2 + 16 * (pos ^ ((row << 1) & 4)));
        uint8_t* d = slot + 1024 * wave;
        gt_copy(w, at, d);
#pragma unroll
        for (int i = 0; i < 4; ++i) gt_copy(w + 32 * i * MC, at, d + MTOK * 128 + 4096 * i);
    }
    // (the operands and the order of mla_wuk_kernel)
    template <int C>
    __device__ __forceinline__ void multiply(const uint8_t* tile, const uint8_t* slot)
    {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if ((wave >> 1) != (C & 1)) return;
        const int l32 = lane & 31, hl = lane >> 5, jj = lane & 15, mh = (lane >> 4) & 1;
        const uint8_t* wrow = slot + MTOK * 128 + (8 * hl + (jj >> 2)) * 128 + 8 * (jj & 1) +
                              16 * ((4 * (wave & 1) + 2 * mh + ((jj >> 1) & 1)) ^ ((jj >> 1) & 4));
        f32x16& o = acc[C / 2];
#pragma unroll
        for (int e = 0; e < 16; ++e) o[e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < MNOPE / 16; ++ks) {
            const s16x4 lo = lds_read_tr(wrow + 2048 * ks), hi = lds_read_tr(wrow + 2048 * ks + 512);
            const bf16x8 wv = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            const bf16x8 xv = *reinterpret_cast<const bf16x8*>(tile + ((ks >> 2) * MTOK + l32) * QBS_ROW + 32 * (ks & 3) + 16 * hl);
            o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, xv, o, 0, 0, 0);
        }
    }
    // through LDS, a token's 512 outputs to a wavefront's store
    __device__ __forceinline__ void store(const MlaPrologArgs& a, int head, uint8_t* lds) const
    {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, hl = lane >> 5;
#pragma unroll
        for (int i = 0; i < WUK_CHUNKS / 2; ++i)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4)
                *reinterpret_cast<u32x2*>(lds + l32 * OROW + (64 * (2 * i + (wave >> 1)) + 32 * (wave & 1) + 8 * e4 + 4 * hl) * 2) =
                    u32x2{pack_bf16x2(acc[i][4 * e4], acc[i][4 * e4 + 1]), pack_bf16x2(acc[i][4 * e4 + 2], acc[i][4 * e4 + 3])};
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MTOK / 4; ++i) {
            const int tok = 4 * i + wave;
            if (tok < a.t) // (wave-uniform)
                *reinterpret_cast<u32x4*>(a.q_nope + ((int64_t)tok * a.n + head) * MC + 8 * lane) = *reinterpret_cast<const u32x4*>(lds + tok * OROW + 16 * lane);
        }
    }
};
constexpr int HEAD_LDS = GtStream::LDS + Absorbed::TILE; // the stages, later the outputs | q_b's tile
static_assert(Qb16Stream::STAGE == GtStream::STAGE && Qb16Stream::RING == GtStream::RING && Qb16Stream::XB == GtStream::QBYTES &&
                  GtStream::QBYTES == MTOK * 128 && MTOK * Absorbed::OROW <= GtStream::LDS, "one layout");
// lds: HEAD_LDS bytes
template <bool QUANT>
__device__ __forceinline__ void mla_head_body(const MlaPrologArgs& a, int id, uint8_t* lds)
{
    using S = GtStream;
    const HeadUnit u = head_unit(a, id);
    if (u.head < 0) return; // (uniform)
    uint8_t* tile = lds + S::LDS;
    QbScales scales;
    i32x4 acc[2][2] = {};
    f32x16 sum;
    if constexpr (QUANT) scales.load(a, u.col0, u.gap);
    const int stages = a.r / (QUANT ? GT_KI8 : 64);
    auto product = [&](auto&& run) {
        if constexpr (QUANT)
            gt_stream_i8(acc, static_cast<const int8_t*>(a.w_uq_qr) + u.col0, u.gap, (int64_t)a.n * MQH, a.q_norm, a.r, a.t, lds, run);
        else
            qb16_stream(sum, a, static_cast<const uint16_t*>(a.w_uq_qr) + u.col0, static_cast<const uint16_t*>(a.w_uq_qr) + u.col0 + 64 + u.gap, lds, run);
    };
    auto to_tile = [&]() {
        if constexpr (QUANT)
            scales.tile(acc, tile);
        else
            qb16_tile(sum, tile);
    };
    if (u.nope) { // uniform over the workgroup
        Absorbed o;
        product([&](auto&& copy, auto&& multiply) {
            gt_stages_more<S::RING, S::STAGE, 5, WUK_CHUNKS>(
                stages, copy, multiply, [&](int c, int b) { Absorbed::copy(a, u.head, c, lds + b); }, to_tile,
                [&](auto ic, int b) { o.template multiply<decltype(ic)::value>(tile, lds + b); });
        });
        o.store(a, u.head, lds);
    } else {
        product([&](auto&& copy, auto&& multiply) { gt_stages<S::RING, S::STAGE, 5>(stages, copy, multiply); });
        to_tile();
        __syncthreads();
        qb_store_blocks<MTOK>(a, tile, 3 * u.head + 2, 0, 3);
    }
}
// grid (head_grid), 256 lanes
template <bool QUANT>
__global__ __launch_bounds__(256) void mla_head_kernel(MlaPrologArgs a)
{
    __shared__ __align__(16) uint8_t lds[HEAD_LDS];
    mla_head_body<QUANT>(a, blockIdx.x, lds);
}

// Decode batches: while the norms' few workgroups go through their chains, the rest of the chip has nothing to do, and the
// next launch starts with a stream of weights.  The workgroups from `first` on (a multiple of eight: workgroups go to the XCDs
// round-robin) read the head of the slice that the workgroup of the same number past `first` streams next, `bytes` of it.
//
// How much: what an XCD's slices come to has to stay in its 4 MB L2 beside all else, and has to be there when the norms are done.
// 96 KB of each slice, however many there are, took longer than none from about 250 slices on.  Weights out of HBM (six sets
// in turn), us a call with none / 96 KB / 2 MB to an XCD: int8, 8 tokens, 128 heads 33.8 / 33.5 / 33.2, 192: 45.8 / 47.1 / 45.9,
// 256: 48.0 / 51.5 / 47.9; bf16, 32 tokens, 144 heads 46.2 / 47.0 / 46.5, 256: 65.2 / 67.9 / 64.8; fused, 8 tokens, 144 heads
// 47.9 / 48.6 / 47.0, 256: 52.4 / 55.9 / 52.3.  The fused operator's norms take longer; to 256 slices they cover 3 MB (128 heads,
// 1 token 36.4, 35.5 with 3 MB, 36.0 with 2; 64 heads 33.8 / 32.3).
constexpr int TOUCH_BYTES = 96 * 1024; // of a slice, at most: touch_rows' registers
inline int touch_bytes(int slices, bool fused)
{
    const int xcd = fused && slices <= 256 ? 3 << 20 : 2 << 20;
    return std::min(TOUCH_BYTES, xcd / ((slices + 7) / 8));
}

__device__ __forceinline__ void mla_touch(const MlaPrologArgs& a, int tile, int bytes, bool heads)
{
    const int value = a.quant ? 1 : 2, pieces = 8 * value; // 128 outputs
    const int64_t stride = (int64_t)a.n * MQH * value;
    const int rows = min(a.r, bytes / (16 * pieces)) & ~31;
    const HeadUnit u = heads ? head_unit(a, tile) : HeadUnit{0, 128 * tile, 0, true};
    if (u.head < 0) return;
    touch_rows(static_cast<const uint8_t*>(a.w_uq_qr) + (int64_t)u.col0 * value, stride, rows, pieces, u.gap * value);
}

// grid (2 x tokens: query, key | TOUCH: touching workgroups from `first` on), 256 lanes.  Without them (above 32 tokens) 40 registers
// instead of 98, all of a token's chain that a SIMD can hold.
template <int S, bool TOUCH>
__global__ __launch_bounds__(256) void mla_norm_kernel(MlaPrologArgs a, int first, int touch, bool heads)
{
    const int id = blockIdx.x;
    if (id < a.t)
        mla_norm_query_body<S>(a, id);
    else if (id < 2 * a.t)
        mla_norm_key_body<S>(a, id - a.t);
    else if constexpr (TOUCH) {
        if (id >= first) mla_touch(a, id - first, touch, heads);
    }
}

// grid (n * 192 / 128), 256 lanes
__global__ __launch_bounds__(256) void mla_qb_kernel(MlaPrologArgs a)
{
    __shared__ __align__(16) uint8_t lds[GtStream::LDS];
    mla_qb_body(a, blockIdx.x, lds);
}

// For more tokens than mla_qb_batch_kernel takes (qb_batch), of few heads: 32 TB tokens x 256 outputs per workgroup (gemm_tile.h), the same exact
// sums and the same operations behind them.  128 x 128 tiles through registers are bound by the operands' way into LDS: MLA prolog
// of 200 tokens 66.2 us a call against 57.2.
constexpr int mla_qb_wide_lds(int tb) // the product's stages, or four blocks of the output tile
{
    const int tok = 32 * tb, ring = gt_lds_bytes(tb);
    return 4 * tok * QBS_ROW > ring ? 4 * tok * QBS_ROW : ring;
}
template <int TB>
__device__ __forceinline__ void mla_qb_wide_body(const MlaPrologArgs& a, int tile, int tok0, uint8_t* lds)
{
#pragma clang fp contract(off)
    using T = GtTile<TB>;
    static_assert(mla_qb_wide_lds(TB) >= T::LDS, "LDS");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    const int nq = a.n * MQH, col0 = 256 * tile; // (nq is a multiple of 128)
    i32x4 acc[4][TB]; // [nb][tb]
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
    const int8_t* w = static_cast<const int8_t*>(a.w_uq_qr);
    gt_product_i8<TB>(acc, w + col0, w + min(col0 + 128, nq - 128), nq, a.q_norm, a.r, tok0, a.t, a.r / GT_KI8, lds,
                      gt_wave());
    // register e of acc[nb][tb]: output 64 wc + 16 nb + 4 g + e, token 16 TB wr + 16 tb + l16
    f32x4 ws[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + min(col0 + 64 * wc, nq - 64) + 16 * nb + 4 * g);
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const int tl = 16 * TB * wr + 16 * tb + l16;
        const float qs = a.q_norm_scale[min(tok0 + tl, a.t - 1)];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs) * ws[nb][e];
            *reinterpret_cast<u32x2*>(lds + (wc * T::TOK + tl) * QBS_ROW + 32 * nb + 8 * g) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
    }
    __syncthreads();
    qb_store_blocks<T::TOK>(a, lds, 4 * tile, tok0);
}
// grid (n * 192 / 256 rounded up, token tiles), 512 lanes
template <int TB>
__global__ __launch_bounds__(GT_LANES, 2) void mla_qb_wide_kernel(MlaPrologArgs a)
{
    __shared__ __align__(16) uint8_t lds[mla_qb_wide_lds(TB)];
    mla_qb_wide_body<TB>(a, blockIdx.x, blockIdx.y * 32 * TB, lds);
}

// q_b[:, head, :128] @ w_uk[head] behind a tile of q_b, by the workgroup of 512 lanes that has it in LDS: wave w owns outputs [64 w, +64),
// whose weights lie in its registers (64 a lane) and come straight from memory: a lane loads 4 neighbouring outputs of 8 contraction rows at a
// time and turns them by byte permutes into what the matrix instructions want.  Which 4 of the 64 is chosen so that a lane's
// results for a token are runs of 8 neighbouring outputs; exchanged between tokens 8 apart, a store is 8 whole lines of 128 bytes.
//
// As a kernel of its own (mla_wuk_wide_kernel) the product waits for memory: at 1501 tokens 49 MB of q_b out and in again and 197 MB
// of outputs, 45 us in which the matrix pipes stand still, behind a query product of 91 that writes little.  Here the outputs of some workgroups
// leave while others multiply, and q_b's first dims stay in LDS.  Call of 1501 tokens, us: two kernels 203.4; one, with halves of lines to
// a store, 198.5; whole lines 198.9; and streaming stores (they do not push the operands out of the L2) 183.1, halves of lines 183.0 (int8 form
// alone 161.8 and 170.4); long workgroups sent out first and short ones kept for the end 174.4 (wide_unit).
struct AbsorbedWide {
    static constexpr int ROW = MNOPE * 2 + 16; // bytes of a tile's LDS row, padded: 16 rows in 16 different places
    u32x2 raw[MNOPE / 4];
    bf16x8 w[4][MNOPE / 32];

    __device__ __forceinline__ void load(const MlaPrologArgs& a, int head)
    {
        const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
        const uint16_t* src = a.w_uk + ((int64_t)head * MNOPE + 8 * g) * MC + 64 * gt_wave() + 4 * (2 * (l16 >> 2) + (l16 & 1) + 4 * (l16 & 2));
#pragma unroll
        for (int ks = 0; ks < MNOPE / 32; ++ks)
#pragma unroll
            for (int k = 0; k < 8; ++k) raw[8 * ks + k] = *reinterpret_cast<const u32x2*>(src + (32 * ks + k) * MC);
    }
    // The weights of HEADS heads from `head` on into the XCD's L2, a line to a lane, four bytes of which land in 256 bytes of LDS at `drop`.
    // Nothing waits for them but the first stage of the product that follows, whose copies are younger.  The first token tile of a head does it
    // for all (they are one XCD's).  Three sets of operands in turn, us a call without / with: fused, 200 tokens 61.2 / 57.0, 512: 89.9 / 86.5, 1501:
    // 193.3 / 189.3; int8 form 300: 64.2 / 59.4; bf16 form 256: 73.0 / 65.0, 1024: 177.6 / 174.0; one set, bf16 form 256: 57.4 / 59.5.
    template <int HEADS>
    static __device__ __forceinline__ void touch(const MlaPrologArgs& a, int head, uint8_t* drop)
    {
        const uint16_t* src = a.w_uk + (int64_t)head * MNOPE * MC;
#pragma unroll
        for (int i = 0; i < HEADS * MNOPE * MC / 64 / 512; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                         :
                         : "s"((gt_lds*)drop), "v"((uint32_t)(128 * (threadIdx.x + 512 * i))), "s"(src)
                         : "memory");
    }
    __device__ __forceinline__ void turn()
    {
#pragma unroll
        for (int ks = 0; ks < MNOPE / 32; ++ks)
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                u32x4 v;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    v[k] = __builtin_amdgcn_perm(raw[8 * ks + 2 * k + 1][cb >> 1], raw[8 * ks + 2 * k][cb >> 1], cb & 1 ? 0x07060302u : 0x05040100u);
                w[cb][ks] = __builtin_bit_cast(bf16x8, v);
            }
    }
    // 16 BLOCKS tokens from tok0 on, their rows at `tile`
    template <int BLOCKS, bool STREAM>
    __device__ __forceinline__ void multiply(const MlaPrologArgs& a, int head, int tok0, const uint8_t* tile) const
    {
        const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
        uint16_t* dst = a.q_nope + ((int64_t)(tok0 + (l16 & 7)) * a.n + head) * MC + 64 * gt_wave() + 8 * g + 4 * (l16 & 8);
#pragma unroll
        for (int tb = 0; tb < BLOCKS; ++tb) {
            f32x4 acc[4];
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < MNOPE / 32; ++ks) {
                const bf16x8 x = *reinterpret_cast<const bf16x8*>(tile + (16 * tb + l16) * ROW + 64 * ks + 16 * g);
#pragma unroll
                for (int cb = 0; cb < 4; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[cb][ks], x, acc[cb], 0, 0, 0);
            }
            // register e of acc[cb]: output 8 g + 32 (e / 2) + 4 (e % 2) + cb of token l16
            const bool up = l16 >= 8;
            u32x4 o[2];
#pragma unroll
            for (int h = 0; h < 2; ++h)
                o[h] = u32x4{pack_bf16x2(acc[0][2 * h], acc[1][2 * h]), pack_bf16x2(acc[2][2 * h], acc[3][2 * h]),
                             pack_bf16x2(acc[0][2 * h + 1], acc[1][2 * h + 1]), pack_bf16x2(acc[2][2 * h + 1], acc[3][2 * h + 1])};
            u32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(up ? o[0][i] : o[1][i]), 0x128, 0xf, 0xf, true);
                lo[i] = up ? v : o[0][i];
                hi[i] = up ? o[1][i] : v;
            }
            auto store = [&](u32x4 v, int tok) {
                if (tok0 + tok + (l16 & 7) >= a.t) return;
                u32x4* to = reinterpret_cast<u32x4*>(dst + (int64_t)tok * a.n * MC);
                if constexpr (STREAM)
                    __builtin_nontemporal_store(v, to);
                else
                    *to = v;
            };
            store(lo, 16 * tb);
            store(hi, 16 * tb + 8);
        }
    }
};

constexpr int mla_heads_wide_lds(int tb) // the product's stages, or two heads' tile
{
    const int epi = 2 * 32 * tb * AbsorbedWide::ROW, ring = gt_lds_bytes(tb);
    return epi > ring ? epi : ring;
}
// mla_qb_wide_body's product and arithmetic by other units: two heads' first dims and the absorbed products behind them, or (rope) four heads'
// rotary dims.  What bounds it at 1501 tokens: without the outputs' stores a call takes 172 us, without the absorbed products 159.
template <int TB>
__device__ __forceinline__ void mla_heads_wide_body(const MlaPrologArgs& a, int unit, bool rope, int tok0, uint8_t* lds)
{
#pragma clang fp contract(off)
    using T = GtTile<TB>;
    static_assert(mla_heads_wide_lds(TB) >= mla_qb_wide_lds(TB), "LDS");
    const int tid = threadIdx.x, lane = tid & 63, wave = gt_wave(), l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    i32x4 acc[4][TB]; // [nb][tb]
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
    const int nq = a.n * MQH;
    // first columns of the two halves, and of this wave's 64 (a last unit with two heads takes them twice; the second time is dropped)
    const int c0 = rope ? 4 * unit * MQH + MNOPE : 2 * unit * MQH, c1 = rope ? min(4 * unit + 2, a.n - 2) * MQH + MNOPE : c0 + MQH;
    const int gap = rope ? MQH - 64 : 0, cw = (wc >> 1 ? c1 : c0) + (wc & 1) * (64 + gap);
    const int8_t* w = static_cast<const int8_t*>(a.w_uq_qr);
    if (!rope && tok0 == 0) AbsorbedWide::touch<2>(a, 2 * unit, lds + (T::RING - 1) * T::QBYTES);
    gt_product_i8<TB>(acc, w + c0, w + c1, nq, a.q_norm, a.r, tok0, a.t, a.r / GT_KI8, lds, wave, gap);
    AbsorbedWide ab;
    if (!rope) ab.load(a, 2 * unit);
    // register e of acc[nb][tb]: output 64 wc + 16 nb + 4 g + e, token 16 TB wr + 16 tb + l16
    f32x4 ws[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + cw + 16 * nb + 4 * g);
    const int row = rope ? QBS_ROW : AbsorbedWide::ROW;
    uint8_t* to = lds + (rope ? wc * T::TOK * QBS_ROW : (wc >> 1) * T::TOK * AbsorbedWide::ROW + (wc & 1) * 128) + (16 * TB * wr + l16) * row + 8 * g;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const float qs = a.q_norm_scale[min(tok0 + 16 * TB * wr + 16 * tb + l16, a.t - 1)];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs) * ws[nb][e];
            *reinterpret_cast<u32x2*>(to + 16 * tb * row + 32 * nb) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
    }
    __syncthreads();
    if (rope) {
        qb_store_blocks<T::TOK>(a, lds, 3 * 4 * unit + 2, tok0, 3);
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        ab.turn();
        if (h == 0) ab.load(a, 2 * unit + 1);
        ab.multiply<2 * TB, true>(a, 2 * unit + h, tok0, lds + h * T::TOK * AbsorbedWide::ROW);
    }
}
// Workgroup id's unit where n1 long units go out among n2 short ones: all of them first (share 256; grid n1 + n2, so that every XCD gets as many
// workgroups), or eight of a kind at a time (an XCD each), `share` / 256 of the groups long ones while they last (grid wide_grid).  kind -1: none.  Up to
// two rounds of workgroups long ones first (fused, 612 tokens: evenly mixed 97.1 us, two thirds 95.8, all first 91.4; int8 form 512 tokens 79.4 / 79.4 /
// 71.8 in tiles of 128); in more, some short ones among them, so that not all CUs store at the same time.  How many matters little: of 256, with 170 / 210
// / 256, three sets of operands in turn, fused, 900 tokens 128.4 / 128.9 / 128.7, 1200: 168.8 / 167.2 / 169.5, 1501: 188.3 / 186.0 / 186.3; int8 form 1501: 174.5 /
// 169.2 / 169.2; bf16 form 700: 138.5 / 131.6 / 132.1, 900: 164.3 / 162.8 / 154.7, 1200: 212.4 / 204.5 / 201.6 (runs of one differ by 1 %).
struct WideUnit {
    int kind, at;
};
__device__ __forceinline__ WideUnit wide_unit(int id, int n1, int n2, int share)
{
    if (share == 256) return id < n1 ? WideUnit{0, id} : WideUnit{1, id - n1};
    const int g1 = (n1 + 7) / 8, g2 = (n2 + 7) / 8, j = id / 8;
    auto firsts = [&](int k) { return max(k - g2, min(g1, (k * share + 255) / 256)); };
    const int before = firsts(j);
    const bool first = firsts(j + 1) > before;
    const int at = 8 * (first ? before : j - before) + id % 8;
    return {at >= (first ? n1 : n2) ? -1 : first ? 0 : 1, at};
}
inline int wide_share(int n1, int n2) { return n1 + n2 <= 512 ? 256 : 210; }
inline unsigned wide_grid(int n1, int n2) { return wide_share(n1, n2) == 256 ? n1 + n2 : 8 * ((n1 + 7) / 8 + (n2 + 7) / 8); }

// Number `at` of units x rows of tiles: whole rounds of the XCDs keep a unit, and its weights, on one of them in all rows; the tiles of the units left over
// go to all.  (In row order 65 or 85 units are on other XCDs in every row, and rounded up to eights the workgroups of one round are more than some
// XCDs have CUs: 170 heads, int8 form 256 tokens 68.8 us a call, 57.5 this way, bf16 form 512 tokens 133 / 114; 130 heads, int8 form 700: 118.8 / 100.9,
// fused 257: 81.2 / 69.3.)
struct WidePlace {
    int unit, row;
};
__device__ __forceinline__ WidePlace wide_place(int at, int units, int rows)
{
    const int most = units & ~7, left = units - most, b = at - most * rows;
    if (b < 0) return {at % most, at / most};
    return {most + b % left, b / left};
}

// The bf16 form by the same units: 33 to 128 tokens beside a head's first dims or two heads' rotary dims, the weights streamed (gt_batch_bf16);
// sums and operations are mla_qb16_kernel's.  In tiles of 128 x 256 the 75 MB of weights were 96 workgroups' work on 256 CUs, 23 us, and the absorbed
// product 7 to 9 behind them.  A call of 33, 64 and 128 tokens 38.4 -> 29.6 us, 40.1 -> 31.2, 46.0 -> 39.4 (three sets of operands 45.3 -> 36.1, 48.5 ->
// 39.8, 57.9 -> 48.5); 16 heads, 64 tokens 36.8 -> 27.6.  A head's w_uk goes to registers ahead of the stages (behind them, from the L2, 1.4 us more).
// grid (n * 192 / 128), 512 lanes
template <int TT>
__global__ __launch_bounds__(GT_LANES, 2) void mla_heads16_batch_kernel(MlaPrologArgs a)
{
    using T = GtBatch16<TT>;
    static_assert(2 * T::TOK * QBS_ROW <= T::LDS && T::TOK * AbsorbedWide::ROW <= T::LDS, "the output tile takes the stages' place");
    __shared__ __align__(16) uint8_t lds[T::LDS];
    const int lane = threadIdx.x & 63, wave = gt_wave(), l32 = lane & 31, hl = lane >> 5, wr = wave >> 2, wc = wave & 3;
    const bool nope = (int)blockIdx.x < a.n;
    const int pair = blockIdx.x - a.n, col0 = nope ? blockIdx.x * MQH : 2 * pair * MQH + MNOPE;
    AbsorbedWide ab;
    if (nope) ab.load(a, blockIdx.x);
    f32x16 sum[T::NB];
    const uint16_t* w = static_cast<const uint16_t*>(a.w_uq_qr) + col0;
    gt_batch_bf16<TT, 128, XA_SPLIT>(sum, w, w + (nope ? 64 : MQH), a.n * MQH, reinterpret_cast<const uint16_t*>(a.q_norm), a.r, a.t, a.r / GT_KBF, lds);
    const int row = nope ? AbsorbedWide::ROW : QBS_ROW;
    uint8_t* to = lds + l32 * row + (wc >> 1) * (nope ? 128 : T::TOK * QBS_ROW) + 64 * (wc & 1) + 8 * hl;
#pragma unroll
    for (int i = 0; i < T::NB; ++i)
        if (wr + 2 * i < TT) // (wave-uniform)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4)
                *reinterpret_cast<u32x2*>(to + 32 * (wr + 2 * i) * row + 16 * e4) =
                    u32x2{pack_bf16x2(sum[i][4 * e4], sum[i][4 * e4 + 1]), pack_bf16x2(sum[i][4 * e4 + 2], sum[i][4 * e4 + 3])};
    __syncthreads();
    if (nope) {
        ab.turn();
        ab.multiply<2 * TT, false>(a, blockIdx.x, 0, lds);
    } else
        qb_store_blocks<T::TOK, 256>(a, lds, 6 * pair + 2, 0, 3);
}

// More tokens: tiles of 128 tokens x two heads' first dims or four heads' rotary dims (mla_qb16_wide_kernel's product).  Three sets of operands in
// turn: 200 tokens 64.5 -> 61.8 us, 289: 92.0 -> 81.3, 384: 98.7 -> 84.5, 512: 107.9 -> 103.4, 1024: 175.2 -> 174.0 (one set 176.7 -> 168.5).
// grid (wide_grid), 512 lanes
__global__ __launch_bounds__(GT_LANES, 2) void mla_heads16_wide_kernel(MlaPrologArgs a, int share)
{
    using T = GtTile<4>;
    static_assert(4 * T::TOK * QBS_ROW <= T::LDS && 2 * T::TOK * AbsorbedWide::ROW <= T::LDS, "the output tile takes the operand tiles' place");
    __shared__ __align__(16) uint8_t lds[T::LDS];
    const int lane = threadIdx.x & 63, wave = gt_wave(), l32 = lane & 31, hl = lane >> 5, wr = wave >> 2, wc = wave & 3;
    const int nab = a.n / 2, nro = (a.n + 3) / 4, rows = (a.t + T::TOK - 1) / T::TOK;
    const WideUnit u = wide_unit(blockIdx.x, nab * rows, nro * rows, share);
    if (u.kind < 0) return;
    const bool rope = u.kind == 1;
    const WidePlace place = wide_place(u.at, rope ? nro : nab, rows);
    const int unit = place.unit, tok0 = place.row * T::TOK;
    const uint16_t* src[4];
    int ld[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { // (heads past the last one: that one again, dropped below)
        src[i] = static_cast<const uint16_t*>(a.w_uq_qr) + (rope ? min(4 * unit + i, a.n - 1) * MQH + MNOPE : (2 * unit + (i >> 1)) * MQH + 64 * (i & 1));
        ld[i] = a.n * MQH;
    }
    f32x16 sum[2][2];
    if (!rope && tok0 == 0) AbsorbedWide::touch<2>(a, 2 * unit, lds + (T::RING - 1) * T::QBYTES);
    gt_product_bf16<128, XA_SPLIT>(sum, src, ld, reinterpret_cast<const uint16_t*>(a.q_norm), a.r, tok0, a.t, a.r / GT_KBF, lds);
    AbsorbedWide ab;
    __builtin_amdgcn_sched_barrier(0); // (once the sums' registers are free)
    if (!rope) ab.load(a, 2 * unit);
    const int row = rope ? QBS_ROW : AbsorbedWide::ROW;
    uint8_t* to = lds + (rope ? wc * T::TOK * QBS_ROW : (wc >> 1) * T::TOK * AbsorbedWide::ROW + (wc & 1) * 128) + 2 * l32;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
                *reinterpret_cast<uint16_t*>(to + (64 * wr + 32 * tb + 8 * (e >> 2) + 4 * hl + (e & 3)) * row + 64 * nb) = f32_to_bf16(sum[tb][nb][e]);
    __syncthreads();
    if (rope) {
        qb_store_blocks<T::TOK>(a, lds, 12 * unit + 2, tok0, 3);
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        ab.turn();
        if (h == 0) ab.load(a, 2 * unit + 1);
        ab.multiply<T::TOK / 16, true>(a, 2 * unit + h, tok0, lds + h * T::TOK * AbsorbedWide::ROW);
    }
}

// 33 to QB_BATCH_T tokens: 128 outputs per workgroup of 512 lanes, all tokens, the weights streamed (gt_batch_i8); the same exact sums
// and the same operations behind them.  ABSORB (head_units): a head's first dims and the absorbed product behind them, or the rotary dims of two heads.  Its 192 workgroups at model sizes keep twice as many CUs at the weights as tiles of 256
// outputs.  Call of 40 tokens 33.8 -> 30.6 us, 96: 37.9 -> 35.0, 160: 50.6 -> 46.4.
template <int TT, bool ABSORB>
__device__ __forceinline__ void mla_qb_batch_body(const MlaPrologArgs& a, int tile, uint8_t* lds)
{
#pragma clang fp contract(off)
    using T = GtBatch<TT>;
    static_assert(2 * T::TOK * QBS_ROW <= T::LDS && T::TOK * AbsorbedWide::ROW <= T::LDS, "the output tile takes the stages' place");
    const int lane = threadIdx.x & 63, wave = gt_wave(), l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    const bool nope = ABSORB && tile < a.n; // a head's first dims, then two heads' rotary dims
    const int pair = tile - a.n, gap = ABSORB && !nope ? MQH - 64 : 0;
    const int col0 = !ABSORB ? 128 * tile : nope ? tile * MQH : 2 * pair * MQH + MNOPE;
    float qs[TT];
    f32x4 ws[2];
#pragma unroll
    for (int tb = 0; tb < TT; ++tb) qs[tb] = a.q_norm_scale[min(16 * TT * wr + 16 * tb + l16, a.t - 1)];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) ws[nb] = *reinterpret_cast<const f32x4*>(a.w_qb_scale + col0 + (wc >> 1) * gap + 16 * gt_batch_block(wc, nb) + 4 * g);
    AbsorbedWide ab;
    if (nope) ab.load(a, tile);
    i32x4 acc[2][TT];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int tb = 0; tb < TT; ++tb) acc[nb][tb] = i32x4{0, 0, 0, 0};
    gt_batch_i8<TT>(acc, static_cast<const int8_t*>(a.w_uq_qr) + col0, (int64_t)a.n * MQH, a.q_norm, a.r, a.t, a.r / GT_KI8, lds, gap);
    const int row = nope ? AbsorbedWide::ROW : QBS_ROW;
    uint8_t* to = lds + (16 * TT * wr + l16) * row + 8 * g;
#pragma unroll
    for (int tb = 0; tb < TT; ++tb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = ((float)acc[nb][tb][e] * qs[tb]) * ws[nb][e];
            const int cb = gt_batch_block(wc, nb);
            *reinterpret_cast<u32x2*>(to + 16 * tb * row + 32 * (cb & 3) + (cb >> 2) * (nope ? 128 : T::TOK * QBS_ROW)) =
                u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
    __syncthreads();
    if (nope) {
        ab.turn();
        ab.multiply<2 * TT, false>(a, tile, 0, lds);
    } else
        qb_store_blocks<T::TOK, 256>(a, lds, ABSORB ? 6 * pair + 2 : 2 * tile, 0, ABSORB ? 3 : 1);
}
// grid (n * 192 / 128), 512 lanes
template <int TT, bool ABSORB>
__global__ __launch_bounds__(GT_LANES, 2) void mla_qb_batch_kernel(MlaPrologArgs a)
{
    __shared__ __align__(16) uint8_t lds[GtBatch<TT>::LDS];
    mla_qb_batch_body<TT, ABSORB>(a, blockIdx.x, lds);
}

// ------------------------------------------------------------------------------------------------ fused with the indexer prolog
// The fused operator runs the two prologs' per-token kernels side by side in one launch, and likewise the two int8
// GEMMs on q_norm (192 + 64 workgroups at model sizes: one per compute unit); the indexer's x @ [w_k | w_proj] rides along
// in mla_xa_kernel as three more output tiles.
// grid (3 x tokens: the MLA norms, the indexer's key path and weights (128 lanes) | TOUCH: touching workgroups from `first` on),
// 256 lanes
template <int S, bool TOUCH>
__global__ __launch_bounds__(256) void fused_norm_kernel(MlaPrologArgs m, PrologArgs p, int first, int touch, bool heads)
{
    const int id = blockIdx.x;
    if (id < m.t)
        mla_norm_query_body<S>(m, id);
    else if (id < 2 * m.t)
        mla_norm_key_body<S>(m, id - m.t);
    else if (id < 3 * m.t) {
        if (threadIdx.x >= 128) return; // the barriers inside are among the two remaining waves
        prolog_k_body<S>(p, id - 2 * m.t);
    } else if (TOUCH && id >= first) {
        const int tile = id - first, nqb = heads ? head_grid(m) : m.n * MQH / 128;
        if (tile < nqb)
            mla_touch(m, tile, touch, heads);
        else
            touch_rows(reinterpret_cast<const uint8_t*>(p.w_qb) + (int64_t)(tile - nqb) * PD, (int64_t)p.n * PD, min(p.r, touch / PD) & ~31, 8, 0);
    }
}

// Up to 32 tokens, grid (n * 192 / 128 + index heads), 256 lanes.  With a workgroup of 1024 lanes per tile that loaded all its
// weights into registers at once and took them through LDS: 15.7 us at one token, 3.2 TB/s.
__global__ __launch_bounds__(256) void fused_qb_kernel(MlaPrologArgs m, PrologArgs p)
{
    __shared__ __align__(16) uint8_t lds[PROLOG_STREAM_LDS];
    const int nqb = m.n * MQH / 128;
    if ((int)blockIdx.x < nqb)
        mla_qb_body(m, blockIdx.x, lds);
    else
        prolog_q_stream_body(p, blockIdx.x - nqb, lds);
}

// The same with a head's absorbed product behind it (mla_head_body).
__global__ __launch_bounds__(256) void fused_head_kernel(MlaPrologArgs m, PrologArgs p)
{
    __shared__ __align__(16) uint8_t lds[PROLOG_STREAM_LDS > HEAD_LDS ? PROLOG_STREAM_LDS : HEAD_LDS];
    const int nqb = head_grid(m);
    if ((int)blockIdx.x < nqb)
        mla_head_body<true>(m, blockIdx.x, lds);
    else
        prolog_q_stream_body(p, blockIdx.x - nqb, lds);
}

// The same pair at 33 to QB_BATCH_T tokens.  The kernel at model sizes: 40 tokens 13.8 us, 96: 16.0, 128: 18.4, 160: 22.1; tiles of
// 128 x 128 through registers, three stages of loads in flight and two barriers a stage, took 20.7 up to 128 tokens, tiles of 256
// outputs 24.4 at 160.  grid (index heads + n * 192 / 128), 512 lanes
template <int TT, bool ABSORB>
__global__ __launch_bounds__(GT_LANES, 2) void fused_qb_batch_kernel(MlaPrologArgs m, PrologArgs p)
{
    __shared__ __align__(16) uint8_t lds[GtBatch<TT>::LDS];
    if ((int)blockIdx.x < p.n) // (the index heads have the longer epilogue)
        prolog_q_batch_body<TT>(p, blockIdx.x, lds);
    else
        mla_qb_batch_body<TT, ABSORB>(m, blockIdx.x - p.n, lds);
}

// For more tokens than that (qb_batch), of few heads, the two products in one launch of gemm_tile.h's tiles: the index heads' part alone is half a round of workgroups
// up to 512 tokens (call of 257 tokens 83.0 us as two launches, 72.2 as one, 512: 104.4 / 96.3, 1024: 163.6 / 160.7, 1344: 211.5 /
// 194.6, 4096: 604.7 / 591.0).  Tiles of 128 to 256 tokens, by modelled time (with 224 at most: 512 tokens 94.5 us a call, 1024: 159.8,
// 1501: 215.7; so 91.9, 153.6, 207.0).
// The index heads' tiles take the longer, 26 us at 192 tokens against 19, and come first, those of all tokens: as columns of each
// token tile they began again in the last round of workgroups (104 us for the kernel at 1501 tokens,
// 92 so; the call 240.8 -> 236.8, no difference where the rounds come out even).
// grid ((index heads / 2 rounded up + n * 192 / 256 rounded up) x token tiles), 512 lanes
template <int TB>
__global__ __launch_bounds__(GT_LANES, 2) void fused_qb_wide_kernel(MlaPrologArgs m, PrologArgs p)
{
    constexpr int A = mla_qb_wide_lds(TB), B = prolog_q_wide_lds(TB);
    __shared__ __align__(16) uint8_t lds[A > B ? A : B];
    const int nqt = (p.n + 1) / 2, nqb = (m.n * MQH + 255) / 256, rows = (m.t + 32 * TB - 1) / (32 * TB);
    int id = blockIdx.x;
    if (id < nqt * rows)
        prolog_q_wide_body<TB>(p, 2 * (id % nqt), id / nqt * 32 * TB, lds);
    else {
        id -= nqt * rows;
        mla_qb_wide_body<TB>(m, id % nqb, id / nqb * 32 * TB, lds);
    }
}

// The same with the absorbed products behind the heads' first dims, and alone.  grid (wide_grid), 512 lanes
template <int TB>
__global__ __launch_bounds__(GT_LANES, 2) void fused_heads_wide_kernel(MlaPrologArgs m, PrologArgs p, int share)
{
    constexpr int A = mla_heads_wide_lds(TB), B = prolog_q_wide_lds(TB);
    __shared__ __align__(16) uint8_t lds[A > B ? A : B];
    const int nqt = (p.n + 1) / 2, nab = m.n / 2, nro = (m.n + 3) / 4, rows = (m.t + 32 * TB - 1) / (32 * TB);
    const WideUnit u = wide_unit(blockIdx.x, nab * rows, (nqt + nro) * rows, share);
    if (u.kind < 0) return;
    const bool rope = u.kind == 1 && u.at >= nqt * rows;
    const WidePlace place = wide_place(rope ? u.at - nqt * rows : u.at, u.kind == 0 ? nab : rope ? nro : nqt, rows);
    if (u.kind == 0)
        mla_heads_wide_body<TB>(m, place.unit, false, place.row * 32 * TB, lds);
    else if (!rope)
        prolog_q_wide_body<TB>(p, 2 * place.unit, place.row * 32 * TB, lds);
    else
        mla_heads_wide_body<TB>(m, place.unit, true, place.row * 32 * TB, lds);
}
template <int TB>
__global__ __launch_bounds__(GT_LANES, 2) void mla_heads_wide_kernel(MlaPrologArgs a, int share)
{
    __shared__ __align__(16) uint8_t lds[mla_heads_wide_lds(TB)];
    const int nab = a.n / 2, nro = (a.n + 3) / 4, rows = (a.t + 32 * TB - 1) / (32 * TB);
    const WideUnit u = wide_unit(blockIdx.x, nab * rows, nro * rows, share);
    if (u.kind < 0) return;
    const WidePlace place = wide_place(u.at, u.kind == 0 ? nab : nro, rows);
    mla_heads_wide_body<TB>(a, place.unit, u.kind == 1, place.row * 32 * TB, lds);
}

// ------------------------------------------------------------------------------------------------ q_b[:, head, :128] @ w_uk[head]
// Tiles of 32 TB tokens (TB 1 or 2) x 128 outputs, one to a workgroup: grid (heads, 512 / 128, token tiles), 256 lanes; wave w owns
// outputs [32 w, 32 w + 32) of the tile.
template <int TB>
__global__ __launch_bounds__(256) void mla_wuk_kernel(MlaPrologArgs a)
{
    constexpr int WTOK = MTOK * TB;    // tokens
    constexpr int OROW = 128 * 2 + 16; // bytes per LDS row of the WTOK x 128 bf16 output tile (padded)
    __shared__ __align__(16) uint8_t wl[MNOPE * TROW];
    __shared__ __align__(16) uint8_t bt[WTOK * OROW]; // the operand rows
    __shared__ __align__(16) uint8_t ot[WTOK * OROW]; // the outputs
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hl = lane >> 5;
    const int head = blockIdx.x, ct = blockIdx.y, tok0 = blockIdx.z * WTOK;
    const uint16_t* src = a.w_uk + (int64_t)head * MNOPE * MC + ct * 128;
    // the operand rows: WTOK tokens x 256 bytes, fetched once by the workgroup in 16-byte pieces (16 lanes per row) and
    // handed to the waves through LDS - a wave loading its own operand would fetch a different row with every lane pair,
    // which costs the texture addresser a cycle per row and instruction, four times over for the four waves
    const int prow = tid >> 4, pcol = tid & 15;
    u32x4 q[2 * TB];
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i)
        q[i] = *reinterpret_cast<const u32x4*>(a.qb_nope + ((int64_t)min(tok0 + prow + 16 * i, a.t - 1) * a.n + head) * MNOPE + 8 * pcol);
#pragma unroll
    for (int i = tid; i < MNOPE * 16; i += 256) {
        const int k = i >> 4, c = i & 15;
        *reinterpret_cast<u32x4*>(wl + k * TROW + c * 16) = *reinterpret_cast<const u32x4*>(src + (int64_t)k * MC + c * 8);
    }
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i) *reinterpret_cast<u32x4*>(bt + (prow + 16 * i) * OROW + 16 * pcol) = q[i];
    __syncthreads();
    const int jj = lane & 15, mh = (lane >> 4) & 1;
    const uint8_t* hp = wl + (8 * hl + (jj >> 2)) * TROW + (32 * wave + 16 * mh + 4 * (jj & 3)) * 2;
    f32x16 acc[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[tb][e] = 0.f;
    // The weight fragment by transposing reads.  Lane jj of a 16-lane group points at row 8 hl + jj / 4 (+ 4 for the second read) of the
    // step, columns 16 mh + 4 (jj & 3); a read hands lane i the column 16 mh + i over the four rows its group's lanes i / 4, i / 4 + 4,
    // .. point at, so lane half hl ends up with the contraction rows 8 hl .. 8 hl + 7 - and B takes the same rows with one 16-byte read.
#pragma unroll
    for (int ks = 0; ks < MNOPE / 16; ++ks) {
        const s16x4 lo = lds_read_tr(hp + ks * 16 * TROW);
        const s16x4 hi = lds_read_tr(hp + (ks * 16 + 4) * TROW);
        const bf16x8 av = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const bf16x8 bx = *reinterpret_cast<const bf16x8*>(bt + (32 * tb + l32) * OROW + (ks * 16 + 8 * hl) * 2);
            acc[tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bx, acc[tb], 0, 0, 0);
        }
    }
    // through LDS, so that a token's 128 outputs leave as one 256-byte run (16 lanes x 16 bytes)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const u32x2 pk = {(uint32_t)f32_to_bf16(acc[tb][4 * e4]) | ((uint32_t)f32_to_bf16(acc[tb][4 * e4 + 1]) << 16),
                              (uint32_t)f32_to_bf16(acc[tb][4 * e4 + 2]) | ((uint32_t)f32_to_bf16(acc[tb][4 * e4 + 3]) << 16)};
            *reinterpret_cast<u32x2*>(ot + (32 * tb + l32) * OROW + (32 * wave + 8 * e4 + 4 * hl) * 2) = pk;
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i) {
        const int tok = prow + 16 * i;
        if (tok0 + tok < a.t)
            *reinterpret_cast<u32x4*>(a.q_nope + ((int64_t)(tok0 + tok) * a.n + head) * MC + ct * 128 + 8 * pcol) =
                *reinterpret_cast<const u32x4*>(ot + tok * OROW + 16 * pcol);
    }
}

// The same product for more tiles than WUK_TILES where it is a kernel of its own (the bf16 form; few heads).  Bound by the outputs' way to memory (1501 tokens x 128
// heads: 197 MB out, 49 in, 47 us at the rate of a large copy).  By tiles of 64 tokens x 128 outputs, two workgroups to a CU with
// the weights in LDS, every tile's rows were read four times over and a tile passed two barriers: 65 us.  So a workgroup of 512
// lanes owns a head's whole 512 outputs and walks the token tiles of 64, z of them side by side (z: one workgroup to a CU); wave w
// owns outputs [64 w, +64), whose weights stay in its registers (64 a lane) and whose outputs leave through LDS of its own; a
// tile's rows are in one of two buffers, and one barrier ends it.  Call of 1501 tokens 236.7 -> 224.5 us, 300: 81.7 -> 77.2, 128:
// 56.4 -> 54.7; at 64 tokens, a single tile for half as many waves, 48.9 -> 49.4, so not there.
// Where the tiles of 128 outputs all fit side by side, two workgroups to a CU, they are the faster ones: a workgroup here starts
// with four times their weights.  The kernel, wide and by tiles: 16 heads x 128 tokens 5.6 us and 4.1, 512: 6.4 / 5.8, 1024: 8.1 /
// 9.3; 64 heads x 128 tokens 6.8 / 6.2, 192: 7.4 / 8.4; 128 heads x 65 tokens 7.7 / 10.2 (256 heads 15.1 / 16.8).
// grid (heads, z), 512 lanes.
constexpr int WUK_TILES = 2 * 256;
constexpr int WW_TOK = 64;
__global__ __launch_bounds__(512, 2) void mla_wuk_wide_kernel(MlaPrologArgs a)
{
    constexpr int BROW = MNOPE * 2 + 16; // bytes per LDS row of a tile's operand rows (padded)
    constexpr int OROW = 64 * 2 + 16;    // of a wave's 64 outputs, or of its slice of the weights
    constexpr int OWN = 2 * 32 * OROW;   // two blocks of 32 tokens of a wave's outputs
    constexpr int BT = WW_TOK * BROW, WL = MNOPE * OROW;
    __shared__ __align__(16) uint8_t lds[8 * WL]; // the weights on their way to the registers; then [2] operand rows, outputs
    static_assert(2 * BT + 8 * OWN <= 8 * WL, "LDS");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hl = lane >> 5, head = blockIdx.x;
    const int ttiles = (a.t + WW_TOK - 1) / WW_TOK;
    const int prow = tid >> 4, pcol = tid & 15; // the operand rows' pieces of 16 bytes, 32 rows a load
    auto fetch = [&](u32x4 (&q)[2], int tt) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            q[i] = *reinterpret_cast<const u32x4*>(a.qb_nope + ((int64_t)min(tt * WW_TOK + prow + 32 * i, a.t - 1) * a.n + head) * MNOPE + 8 * pcol);
    };
    auto park = [&](const u32x4 (&q)[2], uint8_t* bt) {
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(bt + (prow + 32 * i) * BROW + 16 * pcol) = q[i];
    };
    u32x4 q[2];
    fetch(q, blockIdx.y);
    bf16x8 w[2][MNOPE / 16];
    {
        const uint16_t* src = a.w_uk + (int64_t)head * MNOPE * MC + 64 * wave;
        uint8_t* wl = lds + wave * WL;
        const int r = lane >> 3, c = lane & 7;
        u32x4 x[MNOPE / 8];
#pragma unroll
        for (int i = 0; i < MNOPE / 8; ++i) x[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)(8 * i + r) * MC + 8 * c);
#pragma unroll
        for (int i = 0; i < MNOPE / 8; ++i) *reinterpret_cast<u32x4*>(wl + (8 * i + r) * OROW + 16 * c) = x[i];
        __builtin_amdgcn_wave_barrier();
        // (the weight fragment by transposing reads: see mla_wuk_kernel)
        const int jj = lane & 15, mh = (lane >> 4) & 1;
        const uint8_t* hp = wl + (8 * hl + (jj >> 2)) * OROW + (16 * mh + 4 * (jj & 3)) * 2;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int ks = 0; ks < MNOPE / 16; ++ks) {
                const s16x4 lo = lds_read_tr(hp + 64 * nb + ks * 16 * OROW), hi = lds_read_tr(hp + 64 * nb + (ks * 16 + 4) * OROW);
                w[nb][ks] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
    }
    __syncthreads(); // every wave has its weights
    park(q, lds);
    __syncthreads();
    uint8_t* own = lds + 2 * BT + wave * OWN;
    uint16_t* dst = a.q_nope + (int64_t)head * MC + 64 * wave + 8 * (lane & 7);
    for (int tt = blockIdx.y, cur = 0; tt < ttiles; tt += gridDim.y, cur ^= 1) {
        const bool more = tt + (int)gridDim.y < ttiles; // (uniform over the workgroup)
        if (more) fetch(q, tt + gridDim.y);
        const uint8_t* bt = lds + cur * BT + l32 * BROW + 16 * hl;
        f32x16 acc[2][2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[tb][nb][e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < MNOPE / 16; ++ks)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                const bf16x8 bx = *reinterpret_cast<const bf16x8*>(bt + 32 * tb * BROW + 32 * ks);
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) acc[tb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[nb][ks], bx, acc[tb][nb], 0, 0, 0);
            }
        if (more) park(q, lds + (cur ^ 1) * BT); // (read last before the barrier behind the tile before)
        // through LDS of the wave's own, so that a token's 64 outputs leave as one run of 128 bytes
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4)
                    *reinterpret_cast<u32x2*>(own + (32 * tb + l32) * OROW + (32 * nb + 8 * e4 + 4 * hl) * 2) =
                        u32x2{pack_bf16x2(acc[tb][nb][4 * e4], acc[tb][nb][4 * e4 + 1]), pack_bf16x2(acc[tb][nb][4 * e4 + 2], acc[tb][nb][4 * e4 + 3])};
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 32 * tb + 8 * i + (lane >> 3), tok = tt * WW_TOK + row;
                const u32x4 o = *reinterpret_cast<const u32x4*>(own + row * OROW + 16 * (lane & 7));
                if (tok < a.t) *reinterpret_cast<u32x4*>(dst + (int64_t)tok * a.n * MC) = o;
            }
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads(); // the next tile's rows are parked, this one's read
    }
}

} // namespace

bool mla_prolog_supported(int64_t h, int64_t r, int64_t n, int64_t d_nope, int64_t d_rope, int64_t c)
{
    return d_nope == MNOPE && d_rope == MROPE && c == MC && n > 0 && (n * MQH) % 128 == 0 && r > 0 && r % 128 == 0 &&
           r <= MAX_R && h > 0 && h % XA_K == 0;
}

static uint64_t up256(uint64_t x) { return (x + 255) & ~(uint64_t)255; }

static uint64_t xa_part_bytes(int64_t t, int64_t h, int64_t ncols)
{
    return up256((uint64_t)((h + XA_SPLIT - 1) / XA_SPLIT) * t * ncols * sizeof(float));
}

uint64_t mla_prolog_workspace_bytes(int64_t t, int64_t h, int64_t r, int64_t n, int64_t n_idx)
{
    return xa_part_bytes(t, h, r + MKV + (n_idx ? PD + n_idx : 0)) + up256((uint64_t)t * n * MNOPE * 2);
}

void mla_prolog_bind_workspace(MlaPrologArgs& a, void* ws)
{
    uint8_t* p = static_cast<uint8_t*>(ws);
    if (a.t > BIG_T2) {
        const int rows = xa_wide_rows(a.t, a.h, a.r);
        a.ksplits = (a.h + rows - 1) / rows;
    }
    a.xa_part = reinterpret_cast<float*>(p);
    p += xa_part_bytes(a.t, a.h, a.ncols);
    a.qb_nope = reinterpret_cast<uint16_t*>(p);
}

bool fused_prolog_supported(int64_t n_idx) { return n_idx % 64 == 0; }

void fused_prolog_bind(MlaPrologArgs& m, PrologArgs& p, void* ws)
{
    m.w_k = p.w_k;
    m.w_proj = p.w_proj;
    m.n_idx = p.n;
    m.ncols = m.r + MKV + PD + p.n;
    mla_prolog_bind_workspace(m, ws);
    p.xw_part = m.xa_part;
    p.xw_stride = m.ncols;
    p.xw_col0 = m.r + MKV;
    p.ksplits = m.ksplits;
}

// f(integral constant: blocks of 32 tokens) for up to 256 tokens
template <class F>
static void token_blocks(int t, F&& f)
{
    switch ((t + 31) / 32) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    default: f(std::integral_constant<int, 2>{}); break;
    }
}

// The int8 products by workgroups of 128 outputs and all tokens: one round of workgroups to the CUs, one to a CU.  Alone to 160
// tokens where they are one round (us a call, tiles of 256 outputs and these: 40 tokens, 16 heads 31.7 / 26.7, 160 heads 36.4 / 34.5,
// 192: 37.8 / 41.7; 150 tokens, 16 heads 39.9 / 38.0, 160: 55.2 / 52.2, 192: 61.4 / 71.4; 128 heads, 192 tokens 50.9 / 50.7, 224:
// 52.2 / 53.5).  Beside the index heads' up to 128 tokens (against 128 x 128 tiles, 96 tokens: 16 heads 39.6 / 35.5, 256 heads, two
// rounds: 69.1 / 65.4), to 160 where 256 outputs leave the chip half empty and these fill it: by slices of 128 outputs, index heads among
// them, at 129, 145 and 160 tokens 88: 41.4 / 41.4, 41.1 / 41.8, 41.5 / 42.5; 160: 45.4 / 45.2, 44.4 / 45.0, 44.8 / 45.7; 172: 45.5 / 44.9,
// 45.5 / 45.3, 46.1 / 46.1; 184: 46.4 / 45.3, 46.4 / 45.6, 46.8 / 46.6; 196: 49.7 / 47.0, 50.0 / 47.3, 50.9 / 48.5; 256: 52.6 / 50.2, 51.7 / 49.5,
// 52.4 / 50.2 (352, two rounds, at 150: 70.3 / 74.4; 256 slices, 192 tokens: 61.9 / 61.7).
constexpr int QB_BATCH_T = 160;
static bool qb_batch(const MlaPrologArgs& a, const PrologArgs* p)
{
    const int slices = a.n * MQH / 128 + (p ? p->n : 0);
    if (a.t > QB_BATCH_T) return false;
    return p ? a.t <= 128 || (slices > 172 && slices <= 256) : slices <= 256;
}

// Where the absorbed product goes behind the heads' query product.  All figures us a call, two kernels / one; "warm": the same weights call after call, else three
// sets of them in turn, as a stack of layers has it.  Where the two disagree the sets in turn decide.
//
// Up to 32 tokens while that is a workgroup to a CU (warm: fused, 1 token 27.1 / 24.7, 8: 28.5 / 26.0, 32: 30.1 / 27.5, of 16 heads 23.1 / 21.6; bf16
// form, 24 tokens 29.8 / 27.6, out of HBM 36.0 / 33.9, of 16 heads 23.3 / 22.4; int8 form, 8 tokens 23.8 / 22.3, out of HBM 28.4 / 28.2).  The int8 form of
// few heads has short streams behind each other: of 16 19.8 / 20.0, 32: 20.0 / 20.5, 64: 20.7 / 20.7.
//
// From 33 to QB_BATCH_T tokens (bf16 form BATCH16_T), one workgroup to a CU still, the first weights of the absorbed product are fetched ahead of the stream of the
// others (fused, 33 tokens 36.0 / 33.7, 64: 39.3 / 36.6, 96: 46.4 / 41.8; warm, 48: 31.6 / 31.4, 96: 38.6 / 36.4, 128: 42.7 / 39.1, 160: 50.4 / 44.0, of
// 16 heads 64: 27.9 / 26.0).  The int8 form from 65 tokens and 96 heads on, where the warm call gains nothing: 48 tokens 29.8 / 29.7, warm 26.8 / 28.0;
// 65: 34.2 / 32.4, warm 30.9 / 31.3; 96: 38.0 / 35.5, warm 32.7 / 33.0; 128: 41.5 / 39.3, warm 35.8 / 35.3; 160: 48.0 / 44.8, warm 43.5 / 41.4; of 64 heads 96: 27.9
// / 28.4.  In two rounds (256 heads) 128 tokens take 67.2 / 67.6 fused, 58.5 / 59.8 alone, bf16 form of 192 heads 64.4 / 67.1.
//
// Above, tiles of two heads, by heads x tokens (warm: fused, 200 tokens 55.7 / 51.4, 300: 64.4 / 56.9, 512: 83.6 / 73.3, 800: 121.0 / 111.2, 1024: 142.3 /
// 126.2, 1501: 203.3 / 174.4; int8 form 512: 71.0 / 67.0, 640: 81.3 / 80.5, 1024: 126.7 / 118.1, 1501: 179.1 / 159.9).  Few heads are few long workgroups (warm:
// fused, 16 heads 512: 54.1 / 54.5, 700: 64.7 / 63.4; 32 heads 250: 46.4 / 47.2, 400: 54.3 / 52.8; int8 form 64 heads 330: 47.1 / 47.6, 400: 50.7 / 49.8; 32 heads
// 512: 49.4 / 51.2, 1024: 68.0 / 66.1; bf16 form 128 heads 129: 58.2 / 58.5, 64 heads 200: 49.5 / 52.7, 512: 61.6 / 60.2, 16 heads 1024: 71.9 / 74.1).  Near the line
// the warm call loses what the other gains: int8 form 200 tokens 53.9 / 50.5, warm 49.0 / 48.9; 384: 69.2 / 63.3, warm 62.6 / 63.5; bf16 form 200: 64.2 / 61.9, warm 58.8
// / 61.0; 256: 68.4 / 64.9, warm 62.1 / 62.8; 160 heads, int8 form 188: 58.1 / 53.5, warm 51.5 / 53.6; 256 heads, bf16 form 1024: 309.8 / 318.7, warm 311.4 / 305.0.
// To 256 tokens the int8 form only of up to 160 heads, whose long and short workgroups are one round (170 heads, 188 tokens 57.2 / 57.5, warm 51.9 / 56.9, 200:
// 61.1 / 58.7, warm 54.8 / 57.0; 192 heads, 128: 53.9 / 53.8, warm 43.8 / 47.0, 256: 71.2 / 71.8, warm 65.2 / 66.6, 257: 82.5 / 71.2; 256 heads, 128: 57.9 / 58.7,
// warm 48.1 / 52.7, 256: 76.5 / 76.9), and the bf16 form of 161 to 170 heads, a full round of the two kernels' tiles, later (170 heads, 144 tokens 66.2 / 68.0, warm 61.8 /
// 64.5, 180: 69.5 / 69.8, warm 62.8 / 66.4, 200: 74.0 / 71.0, warm 67.7 / 67.2; 160 heads, 160: 66.5 / 65.8, warm 61.6 / 63.1; 192 heads, 129: 86.0 / 76.3).
static bool head_units(const MlaPrologArgs& a, const PrologArgs* p)
{
    const int slices = a.n * MQH / 128 + (p ? p->n : 0);
    const int64_t size = (int64_t)a.n * a.t;
    if (a.t < BIG_T) return slices <= 256 && (p || !a.quant || a.n > 64);
    if (!a.quant) {
        if (a.t <= BATCH16_T) return slices <= 256;
        return size >= (a.t <= 256 && a.n > 160 && a.n <= 170 ? 32000 : 24000);
    }
    if (qb_batch(a, p)) return slices <= 256 && (p || (a.n >= 96 && a.t > 64));
    if (p) return size >= 10000;
    return size >= 24000 && (a.n <= 160 || a.t > 256);
}

// Token blocks (4 to 8) of the tiles with the absorbed product behind: the end of the last of n1 long and n2 short workgroups on 256
// CUs, long ones first, with times (in no unit) that rank the tiles as measured (best of 4 .. 8 taken for 257, 300, 410, 512, 612, 800, 958 and 1501 tokens
// fused, within 1 us of it alone).
static double heads_end(int64_t n1, int64_t n2, double t1, double t2)
{
    const double begin = n1 / 256 * t1;
    const int64_t rest = n1 % 256;
    double end = begin + (rest ? t1 : 0);
    for (int64_t k = 0;; ++k) // k, k + 1, .. rounds of short ones beside the last long ones
        for (const double e : {begin + k * t2, begin + t1 + k * t2}) {
            const int64_t behind = rest ? std::max<int64_t>(0, (int64_t)((e - begin - t1) / t2 + 1e-9)) : 0;
            if ((256 - rest) * (int64_t)((e - begin) / t2 + 1e-9) + rest * behind >= n2) return std::max(end, e);
        }
}
static int heads_token_blocks(const MlaPrologArgs& a, const PrologArgs* p)
{
    int best = 4;
    double best_end = 1e30;
    for (int tb = 4; tb <= 8; ++tb) {
        const int64_t rows = (a.t + 32 * tb - 1) / (32 * tb);
        const double depth = a.r / 1536.0 * tb;
        const double end = p ? heads_end(a.n / 2 * rows, ((a.n + 3) / 4 + (p->n + 1) / 2) * rows, 8.0 + 1.2 * depth, 3.3 + 1.3 * depth)
                             : heads_end(a.n / 2 * rows, (a.n + 3) / 4 * rows, 9.9 + 1.17 * depth, 5.3 + 1.16 * depth);
        if (end < best_end) best = tb, best_end = end;
    }
    return best;
}

// p == nullptr: the MLA prolog on its own; otherwise the fused operator (m and p bound by fused_prolog_bind)
static hipError_t launch_prologs(const MlaPrologArgs& a, const PrologArgs* p, hipStream_t stream)
{
    if (a.t == 0) return hipSuccess;
    const int ttiles = (a.t + MTOK - 1) / MTOK;
    hipError_t e;
    const bool big = a.t >= BIG_T; // the kernels that own an output tile
    const bool heads = head_units(a, p);
    {
        ScopedKernelTimer tm(KID_MLA_XA, stream);
        if (a.t <= BIG_T2) {
            token_blocks(a.t, [&](auto tt) {
                constexpr int TT = decltype(tt)::value;
                hipLaunchKernelGGL(mla_xa_kernel<TT>, dim3(a.ksplits, a.ncols / 64), dim3(512), 0, stream, a);
            });
        } else {
            const int xtiles = (a.t + 127) / 128, ntiles = (a.ncols + 255) / 256, rows = xa_wide_rows(a.t, a.h, a.r);
            if (a.ksplits != (a.h + rows - 1) / rows) return hipErrorInvalidValue;
            hipLaunchKernelGGL(mla_xa_wide_kernel, dim3((xtiles * ntiles * a.ksplits + 7) / 8 * 8), dim3(GT_LANES), 0, stream, a, xtiles,
                               ntiles, rows);
        }
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    {
        ScopedKernelTimer tm(KID_MLA_NORM, stream);
        // all partial sums of an output in flight at once for the usual seven splits and fewer, none of them twice for one or two
        const int in_flight = a.ksplits <= 2 ? 2 : a.ksplits <= 4 ? 4 : 8;
        const int norms = (p ? 3 : 2) * a.t, first = (norms + 7) / 8 * 8;
        const int slices = a.n * MQH / 128 + (p ? p->n : 0), bytes = touch_bytes(slices, p != nullptr);
        const bool ahead = !big && bytes >= 32 * 256; // (32 rows; the kernels above BIG_T tokens do not wait for their weights)
        const unsigned grid = ahead ? first + (heads ? head_grid(a) + (p ? p->n : 0) : slices) : norms;
        auto launch = [&](auto splits, auto touch) {
            constexpr int S = decltype(splits)::value;
            constexpr bool TOUCH = decltype(touch)::value;
            if (p)
                hipLaunchKernelGGL((fused_norm_kernel<S, TOUCH>), dim3(grid), dim3(256), 0, stream, a, *p, first, bytes, heads);
            else
                hipLaunchKernelGGL((mla_norm_kernel<S, TOUCH>), dim3(grid), dim3(256), 0, stream, a, first, bytes, heads);
        };
        auto launch_with = [&](auto touch) {
            if (in_flight == 2)
                launch(std::integral_constant<int, 2>{}, touch);
            else if (in_flight == 4)
                launch(std::integral_constant<int, 4>{}, touch);
            else
                launch(std::integral_constant<int, 8>{}, touch);
        };
        if (p && a.t > BIG_T2 && a.ksplits <= 8) {
            auto wide = [&](auto splits, auto pieces) {
                hipLaunchKernelGGL((fused_norm_wide_kernel<decltype(splits)::value, decltype(pieces)::value>), dim3(3 * ((a.t + 3) / 4)), dim3(256), 0,
                                   stream, a, *p);
            };
            auto wide_with = [&](auto splits) {
                if (a.r <= 1536)
                    wide(splits, std::integral_constant<int, 6>{});
                else
                    wide(splits, std::integral_constant<int, MAX_R / 256>{});
            };
            if (in_flight == 2)
                wide_with(std::integral_constant<int, 2>{});
            else if (in_flight == 4)
                wide_with(std::integral_constant<int, 4>{});
            else
                wide_with(std::integral_constant<int, 8>{});
        } else if (ahead)
            launch_with(std::true_type{});
        else
            launch_with(std::false_type{});
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    {
        ScopedKernelTimer tm(KID_MLA_QB, stream);
        if (heads && !big) {
            if (p)
                hipLaunchKernelGGL(fused_head_kernel, dim3(head_grid(a) + p->n), dim3(256), 0, stream, a, *p);
            else
                hipLaunchKernelGGL((a.quant ? mla_head_kernel<true> : mla_head_kernel<false>), dim3(head_grid(a)), dim3(256), 0, stream, a);
        } else if (!a.quant && heads && a.t <= BATCH16_T) {
            token_blocks(a.t, [&](auto tt) {
                hipLaunchKernelGGL(mla_heads16_batch_kernel<std::clamp(decltype(tt)::value, 2, 4)>, dim3(a.n * MQH / 128), dim3(GT_LANES), 0, stream, a);
            });
        } else if (!a.quant && heads) {
            const int rows = (a.t + 127) / 128, first = a.n / 2 * rows, second = (a.n + 3) / 4 * rows;
            hipLaunchKernelGGL(mla_heads16_wide_kernel, dim3(wide_grid(first, second)), dim3(GT_LANES), 0, stream, a, wide_share(first, second));
        } else if (!a.quant && big) {
            hipLaunchKernelGGL(mla_qb16_wide_kernel, dim3((a.n * MQH + 255) / 256, (a.t + 127) / 128), dim3(GT_LANES), 0, stream, a);
        } else if (!a.quant) {
            hipLaunchKernelGGL(mla_qb16_kernel, dim3(a.n * MQH / 128), dim3(256), 0, stream, a);
        } else if (big) {
            if (qb_batch(a, p)) {
                token_blocks(a.t, [&](auto tt) {
                    constexpr int TT = std::clamp(decltype(tt)::value, 2, QB_BATCH_T / 32);
                    auto launch = [&](auto absorb) {
                        constexpr bool ABSORB = decltype(absorb)::value;
                        if (p)
                            hipLaunchKernelGGL((fused_qb_batch_kernel<TT, ABSORB>), dim3(a.n * MQH / 128 + p->n), dim3(GT_LANES), 0, stream, a, *p);
                        else
                            hipLaunchKernelGGL((mla_qb_batch_kernel<TT, ABSORB>), dim3(a.n * MQH / 128), dim3(GT_LANES), 0, stream, a);
                    };
                    if (heads)
                        launch(std::true_type{});
                    else
                        launch(std::false_type{});
                });
            } else if (heads) {
                const int qcols = p ? (p->n + 1) / 2 : 0;
                gt_dispatch(heads_token_blocks(a, p), [&](auto tb) {
                    constexpr int TB = decltype(tb)::value;
                    const int rows = (a.t + 32 * TB - 1) / (32 * TB), first = a.n / 2 * rows, second = ((a.n + 3) / 4 + qcols) * rows;
                    const int share = wide_share(first, second);
                    const dim3 grid(wide_grid(first, second));
                    if (p)
                        hipLaunchKernelGGL(fused_heads_wide_kernel<TB>, grid, dim3(GT_LANES), 0, stream, a, *p, share);
                    else
                        hipLaunchKernelGGL(mla_heads_wide_kernel<TB>, grid, dim3(GT_LANES), 0, stream, a, share);
                });
            } else {
                const int cols = (a.n * MQH + 255) / 256, qcols = p ? (p->n + 1) / 2 : 0, stages = a.r / GT_KI8;
                if (p)
                    gt_dispatch(gt_token_blocks(a.t, cols + qcols, stages, 8), [&](auto tb) {
                        constexpr int TB = decltype(tb)::value;
                        hipLaunchKernelGGL(fused_qb_wide_kernel<TB>, dim3((qcols + cols) * ((a.t + 32 * TB - 1) / (32 * TB))), dim3(GT_LANES), 0, stream,
                                           a, *p);
                    });
                else
                    gt_dispatch(gt_token_blocks(a.t, cols, stages, 8), [&](auto tb) {
                        constexpr int TB = decltype(tb)::value;
                        hipLaunchKernelGGL(mla_qb_wide_kernel<TB>, dim3(cols, (a.t + 32 * TB - 1) / (32 * TB)), dim3(GT_LANES), 0, stream, a);
                    });
            }
        } else if (p) {
            hipLaunchKernelGGL(fused_qb_kernel, dim3(a.n * MQH / 128 + p->n), dim3(256), 0, stream, a, *p);
        } else {
            hipLaunchKernelGGL(mla_qb_kernel, dim3(a.n * MQH / 128), dim3(256), 0, stream, a);
        }
    }
    if ((e = hipGetLastError()) != hipSuccess || heads) return e;
    {
        ScopedKernelTimer tm(KID_MLA_WUK, stream);
        const int wtiles = (a.t + WW_TOK - 1) / WW_TOK;
        if (!big)
            hipLaunchKernelGGL(mla_wuk_kernel<1>, dim3(a.n, MC / 128), dim3(256), 0, stream, a);
        else if (wtiles == 1 || (int64_t)a.n * (MC / 128) * wtiles <= WUK_TILES)
            hipLaunchKernelGGL(mla_wuk_kernel<2>, dim3(a.n, MC / 128, wtiles), dim3(256), 0, stream, a);
        else
            hipLaunchKernelGGL(mla_wuk_wide_kernel, dim3(a.n, std::min(wtiles, std::max(1, 256 / a.n))), dim3(512), 0, stream, a);
    }
    return hipGetLastError();
}

hipError_t mla_prolog_launch(const MlaPrologArgs& a, hipStream_t stream) { return launch_prologs(a, nullptr, stream); }

hipError_t fused_prolog_launch(const MlaPrologArgs& m, const PrologArgs& p, hipStream_t stream)
{
    return launch_prologs(m, &p, stream);
}

} // namespace pto
