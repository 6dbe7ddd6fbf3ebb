// Main loop of the products at prefill sizes: a workgroup of 512 lanes owns 32 TB tokens (128 to 256) x 256 outputs.
//
// What bounds these products at prefill sizes is first what the CUs draw from the L2: with the matrix instructions taken out, the
// copies of 128 x 128 tiles alone (1.03 GB for 777 tokens x 5120 x 14336) take 77 us, 13 TB/s, wherever the tiles lie.  So the
// tile is as large as LDS and registers hold (537 MB there).  Then a CU's own pipes: of a stage of 224 x 256 x 128 the matrix
// instructions take 1792 ticks, the LDS reads and the copies' writes some 1250, the copies' instructions 960, and the loop is as
// good as these overlap.  40 such stages take 122.6 K ticks with the copies issued first and the fragments read in front of
// their products, 111 K with the copies between the matrix instructions, 107 K with the products half a stage behind the reads
// besides (a call of 777 tokens x 112 heads 90.8 us, 88.7, 86.4; 1024 tokens 101.0, 98.3, 95.9).  With the reads between the matrix
// instructions too, instead of in one go behind the barrier, a stage by itself takes 2295 ticks, not 2440 (256 tokens 2490 / 2717, 128:
// 1488 / 1551).  A whole call keeps little of it (777 tokens 73.6 -> 72.6 us, 1024: 87.4 -> 86.1, 300: 53.4 -> 54.2, and 50.3 -> 48.7 with warm weights): the
// chip's power decides, matrix instructions 78 % of the time hold the clock at 1.85 GHz (four waves with half again the tile each read a
// quarter less of LDS, and the compiler moves their sums between register files: 57 -> 74 us at 256 tokens).  The waves' priorities make no
// difference: the second wave of a SIMD is done when it would be anyway, the first waits for it at the barrier.  And
//  - a stage's operands are copied to LDS by the memory pipe itself (global_load_lds_dwordx4: no registers, no LDS store
//    instructions), into the buffer that is not being read, so that a stage has one barrier;
//  - rows of 128 bytes are kept unpadded (a copy writes 64 lanes x 16 bytes in a row) and spread over the banks by
//    exchanging their 16-byte pieces, piece c of row r at position c ^ f(r): the copy takes the exchange on its global
//    side, where the 8 lanes of a row cover the same 128 bytes in another order.
// Wave (wr, wc) owns tokens [16 TB wr, +16 TB) x outputs [64 wc, +64).  Contraction lengths are multiples of a stage; rows past
// the last token re-read it and are dropped by the epilogue.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "prolog_common.h"

namespace pto {
namespace {

constexpr int GT_LANES = 512;
constexpr int GT_KI8 = 128;                  // contraction rows per stage
constexpr int gt_lds_bytes(int tb) // of an int8 tile's stages
{
    const int q = 32 * tb * 128, w = 2 * 128 * 128;
    return (3 * (q + w) <= 160 * 1024 ? 3 : 2) * q + 3 * w;
}
template <int TB>
struct GtTile {
    static constexpr int TOK = 32 * TB;             // tokens of the tile
    static constexpr int QBYTES = TOK * 128;        // a stage's token rows, 128 bytes each, and [2] weight rows: either
                                                    // operand in a ring of its own
    static constexpr int WBYTES = 2 * 128 * 128, STAGE = QBYTES + WBYTES;
    // stages in LDS, one workgroup to a CU: two in flight, of the token rows above 160 tokens one (what LDS holds)
    static constexpr int WRING = 3, RING = 3 * STAGE <= 160 * 1024 ? 3 : 2;
    static constexpr int WOFF = RING * QBYTES, LDS = gt_lds_bytes(TB); // int8: the token rows' buffers, the weights'
    static_assert(LDS == WOFF + WRING * WBYTES && LDS <= 160 * 1024, "");
};

typedef __attribute__((address_space(3))) uint8_t gt_lds;

// 64 lanes x 16 bytes from base + each lane's offset to 1 KB of LDS at d, in lane order; base and d are wave-uniform.  Written
// out because the compiler, which cannot tell the buffers apart, waits for every copy in flight before the next LDS read; the
// copies are waited for in gt_landed alone.  (One wait state between writing M0 and the copy that uses it; M0 is no register
// that the compiler keeps values in, and nothing else in these kernels reads it.)
__device__ __forceinline__ void gt_copy(const void* base, uint32_t offset, uint8_t* d)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"((gt_lds*)d), "v"(offset), "s"(base)
                 : "memory");
}

// All but the last N of this wave's copies have landed and all of its LDS reads are done, and with the barrier everybody's.  The
// wait for the reads is written out: gt_product_i8's and gt_product_bf16's last reads of a stage are used behind this barrier
// only, and what is copied right behind it goes into the buffer that they read.  Left to __syncthreads, the compiler drops that
// wait where the reads come over the loop's back edge (12 to 14 of them were outstanding at the barrier).  They were issued a
// half stage of matrix instructions before: no time.
template <int N>
__device__ __forceinline__ void gt_landed()
{
    static_assert(N < 64, "the counter's six bits");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | (N >> 4 << 14)); // vmcnt(N) lgkmcnt(0)
    __syncthreads();
}

// copy(stage, byte offset of the buffer) and multiply(byte offset) over the stages, RING - 1 of them ahead; COPIES: what copy
// issues per wave.  Past the end the last stage is copied again (the landings stay countable) and dropped.  On return nothing
// is in flight and LDS is the caller's again.
template <int RING, int STAGE, int COPIES, class Copy, class Multiply>
__device__ __forceinline__ void gt_stages(int stages, Copy&& copy, Multiply&& multiply)
{
#pragma unroll
    for (int s = 0; s < RING - 1; ++s) copy(min(s, stages - 1), s * STAGE);
    int in = (RING - 1) * STAGE, out = 0;
    for (int st = 0; st < stages; ++st) {
        gt_landed<(RING - 2) * COPIES>(); // stage st is there, and everyone is done with the buffer of the stage before
        copy(min(st + RING - 1, stages - 1), in);
        multiply(st, out);
        in = in == (RING - 1) * STAGE ? 0 : in + STAGE;
        out = out == (RING - 1) * STAGE ? 0 : out + STAGE;
    }
    gt_landed<0>();
}

// f(integral_constant 0) .. f(integral_constant N - 1), written out
template <class F, int... I>
__device__ __forceinline__ void gt_unroll_seq(std::integer_sequence<int, I...>, F&& f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void gt_unroll(F&& f)
{
    gt_unroll_seq(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// The same with MORE stages of something else behind them, whose copies (as many) follow without a gap: copy_more(stage, byte offset),
// between() in front of the first of them (what it leaves in LDS is there for multiply_more), multiply_more(integral constant stage,
// byte offset).
template <int RING, int STAGE, int COPIES, int MORE, class Copy, class Multiply, class CopyMore, class Between, class MultiplyMore>
__device__ __forceinline__ void gt_stages_more(int stages, Copy&& copy, Multiply&& multiply, CopyMore&& copy_more, Between&& between,
                                               MultiplyMore&& multiply_more)
{
    static_assert(MORE >= RING - 1, "no copies past the end");
    auto any = [&](int st, int b) { // (uniform)
        if (st < stages)
            copy(st, b);
        else
            copy_more(st - stages, b);
    };
#pragma unroll
    for (int s = 0; s < RING - 1; ++s) any(s, s * STAGE);
    int in = (RING - 1) * STAGE, out = 0;
    auto turn = [&]() {
        in = in == (RING - 1) * STAGE ? 0 : in + STAGE;
        out = out == (RING - 1) * STAGE ? 0 : out + STAGE;
    };
    for (int st = 0; st < stages; ++st) {
        gt_landed<(RING - 2) * COPIES>();
        any(st + RING - 1, in);
        multiply(st, out);
        turn();
    }
    between();
    gt_unroll<MORE>([&](auto ic) {
        constexpr int c = ic, ahead = c + RING - 2 < MORE - 1 ? RING - 2 : MORE - 1 - c;
        gt_landed<ahead * COPIES>();
        if constexpr (c + RING - 1 < MORE) copy_more(c + RING - 1, in);
        multiply_more(ic, out);
        turn();
    });
    gt_landed<0>();
}

// The tiles' loop: the operands in rings of their own, the weights one stage further ahead where they have one more buffer, and
// the copies between the matrix instructions.  A copy keeps the CU's texture addresser busy for 16 ticks: issued in one go at
// the head of a stage, the 60 of a 224 x 256 tile held the last wave up for 960 ticks, after which all matrix instructions
// were still to come.  copy_q(i, stage, byte offset of the buffer), i < QC, and copy_w(..), i < WC: one copy of a wave;
// multiply(byte offsets of both, issue): calls issue(i) for all QC + WC in order, somewhere.
template <int QRING, int QSTAGE, int QC, int WRING, int WSTAGE, int WC, class CopyQ, class CopyW, class Multiply>
__device__ __forceinline__ void gt_tile_stages(int stages, CopyQ&& copy_q, CopyW&& copy_w, Multiply&& multiply)
{
    static_assert(QRING == WRING || QRING + 1 == WRING, "the order of the copies that the wait counts on");
    // behind a stage's token rows: the weights of their round, where those are of a later stage, and the rounds since
    constexpr int BEHIND = (QRING - 2) * (QC + WC) + (QRING < WRING ? WC : 0);
#pragma unroll
    for (int s = 0; s < WRING - 1; ++s) { // (the token rows of the first stage with the weights of the last one ahead)
        if (s >= WRING - QRING)
#pragma unroll
            for (int i = 0; i < QC; ++i) copy_q(i, min(s - (WRING - QRING), stages - 1), (s - (WRING - QRING)) * QSTAGE);
#pragma unroll
        for (int i = 0; i < WC; ++i) copy_w(i, min(s, stages - 1), s * WSTAGE);
    }
    int qin = (QRING - 1) * QSTAGE, qout = 0, win = (WRING - 1) * WSTAGE, wout = 0;
    for (int st = 0; st < stages; ++st) {
        gt_landed<BEHIND>(); // stage st is there, and everyone is done with the buffers of the stage before
        const int qst = min(st + QRING - 1, stages - 1), wst = min(st + WRING - 1, stages - 1);
        multiply(st, qout, wout, [&](int i) {
            if (i < QC)
                copy_q(i, qst, qin);
            else
                copy_w(i - QC, wst, win);
        });
        qin = qin == (QRING - 1) * QSTAGE ? 0 : qin + QSTAGE;
        qout = qout == (QRING - 1) * QSTAGE ? 0 : qout + QSTAGE;
        win = win == (WRING - 1) * WSTAGE ? 0 : win + WSTAGE;
        wout = wout == (WRING - 1) * WSTAGE ? 0 : wout + WSTAGE;
    }
    gt_landed<0>();
}

// Waves by their number; and with the column blocks of the second token half exchanged in pairs, so that the two waves of a SIMD
// (numbers four apart) have an even and an odd one, for epilogues that give these different work.
__device__ __forceinline__ int gt_wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
__device__ __forceinline__ int gt_wave_across()
{
    const int wave = gt_wave();
    return wave ^ (wave >> 2);
}

// acc[nb][tb] += w[k, col0 + ..]^T . q[token, k], int8, by wave 4 wr + wc.  w0, w1: first contraction row of the two halves' columns, ldw bytes a
// row, the second 64 of either half `gap` columns further on; q: [t, ldq], column of the first contraction row.  Register e of acc[nb][tb]: output 64 wc + 16 nb + 4 g + e, token
// 16 TB wr + 16 tb + l16.
template <int TB>
__device__ __forceinline__ void gt_product_i8(i32x4 (&acc)[4][TB], const int8_t* w0, const int8_t* w1, int64_t ldw, const int8_t* q,
                                              int64_t ldq, int tok0, int t, int stages, uint8_t* lds, int wave, int gap = 0)
{
    using T = GtTile<TB>;
    const int lane = threadIdx.x & 63;
    const int l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    // copy i of a wave: rows 64 i + 8 wave + lane / 8 of either operand
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    constexpr int QC = (TB + 1) / 2; // (the last rows again where eight waves have more hands than rows)
    const int8_t* qb = q + (int64_t)tok0 * ldq;
    uint32_t qo[QC], wo[2];
    int qd[QC];
#pragma unroll
    for (int i = 0; i < QC; ++i) {
        const int c = min(8 * i + wave, 4 * TB - 1), qrow = 8 * c + (lane >> 3);
        qd[i] = 1024 * c;
        qo[i] = (uint32_t)(min(qrow, t - 1 - tok0) * (int)ldq + 16 * (pos ^ ((qrow >> 1) & 7)));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int piece = pos ^ (((row >> 1) & 3) | ((row >> 2) & 4));
        wo[i] = (uint32_t)((row + 64 * i) * (int)ldw + 16 * piece + (piece >= 4 ? gap : 0));
    }
    auto copy_q = [&](int i, int st, int b) { gt_copy(qb + st * GT_KI8, qo[i], lds + b + qd[i]); };
    auto copy_w = [&](int i, int st, int b) {
        gt_copy((i < 2 ? w0 : w1) + (int64_t)st * GT_KI8 * ldw, wo[i & 1], lds + T::WOFF + b + 8192 * i + 1024 * wave);
    };
    // token fragments: row 16 TB wr + 16 tb + l16, piece 4 ks + g.  Weight fragments by the byte-transposing read, which hands
    // lane i of a 16-lane group byte i % 8 of the chunks addressed by lanes i / 8, i / 8 + 2, ...: lane i points at row i / 2
    // (+ 8 for the second read), half i % 2 of the 16-column piece 4 (wc & 1) + nb, and gets column i over rows 0 .. 7
    const uint8_t* qr = lds + (16 * TB * wr + l16) * 128;
    const int qpos = 16 * (g ^ ((l16 >> 1) & 7));
    const uint8_t* wrow = lds + T::WOFF + (wc >> 1) * 16384 + (16 * g + (l16 >> 1)) * 128 + 8 * (l16 & 1);
    int wpos[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) wpos[nb] = 16 * ((4 * (wc & 1) + nb) ^ (((l16 >> 2) & 3) | ((g & 1) << 2)));
    // Half a stage behind: what follows a barrier is the second half of the stage before, whose fragments are in registers,
    // while the first half's are read.  (With the reads of a stage in front of its own products the matrix pipes waited
    // some 600 ticks of 2760 for all eight waves' fragments to come out of LDS.)
    i32x4 qf[2][TB], wf[2][4];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) qf[1][tb] = i32x4{0, 0, 0, 0}; // ("the stage before" the first: products of zero)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) wf[1][nb] = i32x4{0, 0, 0, 0};
    auto mfma = [&](int ks, auto&& between) {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
                acc[nb][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[ks][nb], qf[ks][tb], acc[nb][tb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            between(tb);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    gt_tile_stages<T::RING, T::QBYTES, QC, T::WRING, T::WBYTES, 4>(stages, copy_q, copy_w, [&](int, int b, int bw, auto&& issue) {
        auto read = [&](int ks, int i) { // token block i's fragment, and with the first four the weights'
            if (i < 4) {
                const uint8_t* p = wrow + bw + 8192 * ks + wpos[i];
                const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 1024);
                wf[ks][i] = i32x4{lo[0], lo[1], hi[0], hi[1]};
            }
            qf[ks][i] = *reinterpret_cast<const i32x4*>(qr + b + 2048 * i + (qpos ^ (64 * ks)));
        };
        mfma(1, [&](int tb) {
            read(0, tb);
            if (tb < QC + 4) issue(tb);
        });
        mfma(0, [&](int tb) {
            read(1, tb);
            if (TB + tb < QC + 4) issue(TB + tb);
        });
    });
    mfma(1, [](int) {});
}

// Up to 32 tokens x 128 outputs, 256 lanes: a stream of weights, three stages of 128 rows in flight straight to LDS (with five, or
// two, the fused prolog of 8 tokens takes 0.4 us longer: 28.4 us, weights out of HBM 32.8).  Wave w owns outputs [32 w, +32).
// Register e of acc[nb][tb]: output 32 w + 16 nb + 4 g + e, token 16 tb + l16.
struct GtStream { // (a stage's token rows first)
    static constexpr int TOK = 32, QBYTES = TOK * 128, STAGE = QBYTES + 128 * 128, RING = 4, LDS = RING * STAGE;
};
// The outputs are two times 64 that lie `gap` columns apart (0: 128 in a row).  run(copy, multiply) goes through the stages.
template <class Run>
__device__ __forceinline__ void gt_stream_i8(i32x4 (&acc)[2][2], const int8_t* w, int gap, int64_t ldw, const int8_t* q, int64_t ldq, int t,
                                             uint8_t* lds, Run&& run)
{
    using T = GtStream;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    // copies of a wave: token rows 8 w + lane / 8; weight rows 32 i + that
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    const uint32_t qo = (uint32_t)(min(row, t - 1) * (int)ldq + 16 * (pos ^ ((row >> 1) & 7)));
    uint32_t wo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int piece = pos ^ (((row >> 1) & 3) | ((row >> 2) & 4));
        wo[i] = (uint32_t)((row + 32 * i) * (int)ldw + 16 * piece + (piece >= 4 ? gap : 0));
    }
    const uint8_t* qr = lds + l16 * 128;
    const int qpos = 16 * (g ^ ((l16 >> 1) & 7));
    const uint8_t* wrow = lds + T::QBYTES + (16 * g + (l16 >> 1)) * 128 + 8 * (l16 & 1);
    const int wf0 = ((l16 >> 2) & 3) | ((g & 1) << 2); // (transposing reads: see gt_product_i8)
    run(
        [&](int st, int b) {
            uint8_t* d = lds + b + 1024 * wave;
            gt_copy(q + st * GT_KI8, qo, d);
#pragma unroll
            for (int i = 0; i < 4; ++i) gt_copy(w + (int64_t)st * GT_KI8 * ldw, wo[i], d + T::QBYTES + 4096 * i);
        },
        [&](int, int b) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                i32x4 qf[2], wf[2];
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) qf[tb] = *reinterpret_cast<const i32x4*>(qr + b + 2048 * tb + (qpos ^ (64 * ks)));
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) {
                    const uint8_t* p = wrow + b + 8192 * ks + 16 * ((2 * wave + nb) ^ wf0);
                    const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 1024);
                    wf[nb] = i32x4{lo[0], lo[1], hi[0], hi[1]};
                }
#pragma unroll
                for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb)
                        acc[nb][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[nb], qf[tb], acc[nb][tb], 0, 0, 0);
            }
        });
}
__device__ __forceinline__ void gt_stream_i8(i32x4 (&acc)[2][2], const int8_t* w, int64_t ldw, const int8_t* q, int64_t ldq, int t,
                                             int stages, uint8_t* lds)
{
    using T = GtStream;
    gt_stream_i8(acc, w, 0, ldw, q, ldq, t, lds, [&](auto&& copy, auto&& multiply) { gt_stages<T::RING, T::STAGE, 5>(stages, copy, multiply); });
}

// 33 to 160 tokens x 128 outputs, 512 lanes: a stream of weights still, all tokens beside them, two stages in flight (fused prolog of 40
// tokens, weights out of HBM, 38.1 us; with three 38.6, with five 39.2).  Wave (wr, wc) owns tokens [16 TT wr, +16 TT) x two blocks of
// 16 outputs 32 apart, gt_batch_block(wc, nb): what a rotary embedding pairs is in one lane.  Register e of acc[nb][tb]: output
// 16 gt_batch_block + 4 g + e, token 16 TT wr + 16 tb + l16.  The second 64 outputs lie `gap` columns further on.
template <int TT>
struct GtBatch {
    static constexpr int TOK = 32 * TT, QBYTES = TOK * 128, STAGE = QBYTES + 128 * 128, FIT = 160 * 1024 / STAGE, RING = FIT < 3 ? FIT : 3, LDS = RING * STAGE;
};
__device__ __forceinline__ int gt_batch_block(int wc, int nb) { return (wc & 1) + 2 * nb + 4 * (wc >> 1); }
template <int TT>
__device__ __forceinline__ void gt_batch_i8(i32x4 (&acc)[2][TT], const int8_t* w, int64_t ldw, const int8_t* q, int64_t ldq, int t, int stages,
                                            uint8_t* lds, int gap = 0)
{
    using T = GtBatch<TT>;
    const int lane = threadIdx.x & 63, wave = gt_wave();
    const int l16 = lane & 15, g = lane >> 4, wr = wave >> 2, wc = wave & 3;
    // copies of a wave: token rows 64 i + 8 w + lane / 8 (the last rows again where eight waves have more hands than rows), weight rows
    // alike, eight of them from a base of their own (128 can be more than 4 GB)
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    w += (int64_t)(8 * wave) * ldw;
    constexpr int QC = (TT + 1) / 2;
    uint32_t qo[QC], wo;
    int qd[QC];
#pragma unroll
    for (int i = 0; i < QC; ++i) {
        const int c = min(8 * i + wave, 4 * TT - 1), qrow = 8 * c + (lane >> 3);
        qd[i] = 1024 * c;
        qo[i] = (uint32_t)(min(qrow, t - 1) * (int)ldq + 16 * (pos ^ ((qrow >> 1) & 7)));
    }
    const int piece = pos ^ (((row >> 1) & 3) | ((row >> 2) & 4)); // (the same 64 rows on)
    wo = (uint32_t)(lane >> 3) * (uint32_t)ldw + 16 * piece + (piece >= 4 ? gap : 0);
    const uint8_t* qr = lds + (16 * TT * wr + l16) * 128;
    const int qpos = 16 * (g ^ ((l16 >> 1) & 7));
    const uint8_t* wrow = lds + T::QBYTES + (16 * g + (l16 >> 1)) * 128 + 8 * (l16 & 1);
    int wpos[2]; // (transposing reads: see gt_product_i8)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) wpos[nb] = 16 * (gt_batch_block(wc, nb) ^ (((l16 >> 2) & 3) | ((g & 1) << 2)));
    gt_stages<T::RING, T::STAGE, QC + 2>(
        stages,
        [&](int st, int b) {
#pragma unroll
            for (int i = 0; i < 2; ++i) gt_copy(w + (int64_t)(st * GT_KI8 + 64 * i) * ldw, wo, lds + b + T::QBYTES + 8192 * i + 1024 * wave);
#pragma unroll
            for (int i = 0; i < QC; ++i) gt_copy(q + st * GT_KI8, qo[i], lds + b + qd[i]);
        },
        [&](int, int b) {
            i32x4 qf[2][TT], wf[2][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) {
                    const uint8_t* p = wrow + b + 8192 * ks + wpos[nb];
                    const v2i lo = lds_read_tr8(p), hi = lds_read_tr8(p + 1024);
                    wf[ks][nb] = i32x4{lo[0], lo[1], hi[0], hi[1]};
                }
#pragma unroll
                for (int tb = 0; tb < TT; ++tb) qf[ks][tb] = *reinterpret_cast<const i32x4*>(qr + b + 2048 * tb + (qpos ^ (64 * ks)));
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int tb = 0; tb < TT; ++tb)
#pragma unroll
                    for (int nb = 0; nb < 2; ++nb)
                        acc[nb][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[ks][nb], qf[ks][tb], acc[nb][tb], 0, 0, 0);
        });
}

// The same loop in bf16 for 128 tokens x 256 outputs, the outputs in four blocks of 64 columns at src[i], ld[i] values a row;
// x: [t, ldx], column of the first contraction row.  Wave (wr, wc) owns tokens [64 wr, +64) x block wc.  Register e of
// sum[tb][nb]: token 64 wr + 32 tb + 8 (e / 4) + 4 hl + e % 4, column 32 nb + lane % 32 of the block.  Sums are chains of at most
// CHAIN contraction rows, added up in order within GROUP rows, and those sums in order.
constexpr int GT_KBF = 64; // contraction rows per stage
template <int CHAIN, int GROUP>
__device__ __forceinline__ void gt_product_bf16(f32x16 (&sum)[2][2], const uint16_t* const (&src)[4], const int (&ld)[4], const uint16_t* x,
                                                int64_t ldx, int tok0, int t, int stages, uint8_t* lds)
{
    using T = GtTile<4>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, hl = lane >> 5, jj = lane & 15, mh = (lane >> 4) & 1, wr = wave >> 2, wc = wave & 3;
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    const uint16_t* xb = x + (int64_t)tok0 * ldx;
    uint32_t xo[2], wo[4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        xo[i] = (uint32_t)(min(row + 64 * i, t - 1 - tok0) * (int)ldx * 2 + 16 * (pos ^ ((row >> 1) & 7)));
#pragma unroll
    for (int i = 0; i < 4; ++i) wo[i] = (uint32_t)(row * ld[i] * 2 + 16 * (pos ^ ((row << 1) & 4)));
    auto copy_x = [&](int i, int st, int b) { gt_copy(xb + st * GT_KBF, xo[i], lds + b + 1024 * wave + 8192 * i); };
    auto copy_w = [&](int i, int st, int b) { gt_copy(src[i] + (int64_t)st * GT_KBF * ld[i], wo[i], lds + T::WOFF + b + 1024 * wave + 8192 * i); };
    // token fragments: row 64 wr + 32 tb + l32, piece 2 ks + hl.  Weight fragments by 16-bit transposing reads: lane jj of a
    // 16-lane group points at row 8 hl + jj / 4 (+ 4 for the second read) of the step, columns 16 mh + 4 (jj & 3), and gets
    // column 16 mh + jj over those rows
    const uint8_t* xr = lds + (64 * wr + l32) * 128;
    const int xf = (l32 >> 1) & 7;
    const uint8_t* wrow = lds + T::WOFF + wc * 8192 + (8 * hl + (jj >> 2)) * 128 + 8 * (jj & 1);
    const int wpos = 16 * ((2 * mh + ((jj >> 1) & 1)) ^ ((jj >> 1) & 4));
    static_assert(GROUP % CHAIN == 0 && CHAIN % GT_KBF == 0, "whole chains");
    constexpr bool TWO = GROUP > CHAIN; // (else a chain goes straight to the sums)
    f32x16 acc[2][2], part[TWO ? 2 : 1][TWO ? 2 : 1];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[tb][nb][e] = sum[tb][nb][e] = 0.f;
                if constexpr (TWO) part[tb][nb][e] = 0.f;
            }
    auto add = [&](auto& to, auto& from) { // from is empty again
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    to[tb][nb][e] += from[tb][nb][e];
                    from[tb][nb][e] = 0.f;
                }
    };
    // (a step behind, as in gt_product_i8: after a barrier the last step of the stage before, and with it the end of a chain)
    constexpr int STEPS = GT_KBF / 16;
    bf16x8 xv[2][2], wv[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[1][i][e] = wv[1][i][e] = (__bf16)0.f;
    auto mfma = [&](int set, auto&& between) {
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
                acc[tb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv[set][tb], wv[set][nb], acc[tb][nb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            between(tb);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto finish = [&](int done, bool last) { // `done` stages are summed up
        if constexpr (TWO) {
            if (done % (CHAIN / GT_KBF) == 0 || last) add(part, acc);
            if (done % (GROUP / GT_KBF) == 0 || last) add(sum, part);
        } else {
            if (done % (CHAIN / GT_KBF) == 0 || last) add(sum, acc);
        }
    };
    static_assert(STEPS % 2 == 0, "the last step's fragments are in set 1");
    gt_tile_stages<T::RING, T::QBYTES, 2, T::WRING, T::WBYTES, 4>(stages, copy_x, copy_w, [&](int st, int b, int bw, auto&& issue) {
        auto read = [&](int ks) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                const uint8_t* p = wrow + bw + 2048 * ks + (wpos ^ (64 * nb));
                const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 512);
                wv[ks & 1][nb] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) xv[ks & 1][tb] = *reinterpret_cast<const bf16x8*>(xr + b + 4096 * tb + 16 * ((2 * ks + hl) ^ xf));
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks) {
            read(ks);
            mfma(1 - (ks & 1), [&](int tb) {
                if (2 * ks + tb < 6) issue(2 * ks + tb);
            });
            if (ks == 0 && st > 0) finish(st, false);
        }
    });
    mfma(1, [](int) {});
    finish(stages, true);
}

// gt_batch_i8's stream in bf16, 33 to 128 tokens: w0, w1 are the two blocks of 64 outputs, ldw values a row.  Wave (wr, wc) owns outputs [32 wc, +32) of
// the token blocks wr, wr + 2.  Register e of sum[i]: output 32 wc + 8 (e / 4) + 4 hl + e % 4, token 32 (wr + 2 i) + lane % 32.  The sums are
// gt_product_bf16's, to the bit.
template <int TT>
struct GtBatch16 {
    static constexpr int TOK = 32 * TT, XBYTES = TOK * 128, STAGE = XBYTES + 2 * 64 * 128, FIT = 160 * 1024 / STAGE, RING = FIT < 4 ? FIT : 4, LDS = RING * STAGE;
    static constexpr int NB = (TT + 1) / 2; // token blocks of a wave
};
template <int TT, int CHAIN, int GROUP>
__device__ __forceinline__ void gt_batch_bf16(f32x16 (&sum)[GtBatch16<TT>::NB], const uint16_t* w0, const uint16_t* w1, int64_t ldw, const uint16_t* x,
                                              int64_t ldx, int t, int stages, uint8_t* lds)
{
#pragma clang fp contract(off)
    using T = GtBatch16<TT>;
    constexpr int NB = T::NB, XC = (TT + 1) / 2;
    const int lane = threadIdx.x & 63, wave = gt_wave();
    const int l32 = lane & 31, hl = lane >> 5, jj = lane & 15, mh = (lane >> 4) & 1, wr = wave >> 2, wc = wave & 3;
    // copies of a wave: token rows 64 i + 8 w + lane / 8 (the last rows again where eight waves have more hands than rows), weight rows 8 w + lane / 8
    // of either block
    const int row = 8 * wave + (lane >> 3), pos = lane & 7;
    uint32_t xo[XC];
    int xd[XC];
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        const int c = min(8 * i + wave, 4 * TT - 1), xrow = 8 * c + (lane >> 3);
        xd[i] = 1024 * c;
        xo[i] = (uint32_t)(min(xrow, t - 1) * (int)ldx * 2 + 16 * (pos ^ ((xrow >> 1) & 7)));
    }
    const uint32_t wo = (uint32_t)row * (uint32_t)ldw * 2 + 16 * (pos ^ ((row << 1) & 4));
    const uint8_t* xr = lds + (32 * wr + l32) * 128;
    const int xf = (l32 >> 1) & 7;
    const uint8_t* wrow = lds + T::XBYTES + (wc >> 1) * 8192 + (8 * hl + (jj >> 2)) * 128 + 8 * (jj & 1);
    const int wpos = 16 * ((4 * (wc & 1) + 2 * mh + ((jj >> 1) & 1)) ^ ((jj >> 1) & 4));
    f32x16 acc[NB], part[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = part[i][e] = sum[i][e] = 0.f;
    gt_stages<T::RING, T::STAGE, XC + 2>(
        stages,
        [&](int st, int b) {
            gt_copy(w0 + (int64_t)st * GT_KBF * ldw, wo, lds + b + T::XBYTES + 1024 * wave);
            gt_copy(w1 + (int64_t)st * GT_KBF * ldw, wo, lds + b + T::XBYTES + 8192 + 1024 * wave);
#pragma unroll
            for (int i = 0; i < XC; ++i) gt_copy(x + st * GT_KBF, xo[i], lds + b + xd[i]);
        },
        [&](int st, int b) {
            bf16x8 xv[GT_KBF / 16][NB], wv[GT_KBF / 16];
#pragma unroll
            for (int ks = 0; ks < GT_KBF / 16; ++ks) {
                const uint8_t* p = wrow + b + 2048 * ks + wpos;
                const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 512);
                wv[ks] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                for (int i = 0; i < NB; ++i) // (an odd last block: both rows of waves have it, one drops it)
                    xv[ks][i] = *reinterpret_cast<const bf16x8*>(xr + b + min(2 * i, TT - 1 - wr) * 4096 + 16 * ((2 * ks + hl) ^ xf));
            }
#pragma unroll
            for (int ks = 0; ks < GT_KBF / 16; ++ks)
#pragma unroll
                for (int i = 0; i < NB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[ks], xv[ks][i], acc[i], 0, 0, 0);
            const int done = st + 1;
            const bool last = done == stages;
            if (done % (CHAIN / GT_KBF) == 0 || last) {
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int e = 0; e < 16; ++e) part[i][e] += acc[i][e], acc[i][e] = 0.f;
            }
            if (done % (GROUP / GT_KBF) == 0 || last) {
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[i][e] += part[i][e], part[i][e] = 0.f;
            }
        });
}

// Token blocks TB (4 .. most) of an int8 product's tile, by the time it should take in ns: the grid runs in rounds of one
// workgroup to each of the 256 CUs; a stage costs its matrix instructions, as the token blocks, and the weights' copies, like
// about two of them; a round has its ends; the copies together have 26 TB/s.
inline int64_t gt_time_ns(int64_t wgs, int64_t stages, int tb)
{
    return (wgs + 255) / 256 * (stages * (tb + 2) * 160 + 12000) + wgs * stages * (tb + 8) * 4096 / 26000;
}
inline int gt_token_blocks(int64_t t, int64_t cols, int64_t stages, int most)
{
    int best = 4;
    int64_t best_ns = INT64_MAX;
    for (int tb = 4; tb <= most; ++tb) {
        const int64_t ns = gt_time_ns(cols * ((t + 32 * tb - 1) / (32 * tb)), stages, tb);
        if (ns < best_ns) best = tb, best_ns = ns;
    }
    return best;
}

// f(integral constant TB) for the run-time value tb
template <class F>
inline void gt_dispatch(int tb, F&& f)
{
    switch (tb) {
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: f(std::integral_constant<int, 8>{}); break;
    }
}

} // namespace
} // namespace pto
