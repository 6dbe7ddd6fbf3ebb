// Sparse flash attention over a paged, int8, MLA-compressed KV cache - gfx950 kernels.
//
// Replaces the device side of sparse_flash_attention_quant_compute / sparse_attention_antiquant_compute
// (models/deepseek_v32_exp/sparse_flash_attention_quant_impl.py:45-286,
//  models/deepseek_v32_exp/sparse_attention_antiquant_impl.py:44-266,422-720); the arithmetic follows the
// online-softmax golden (models/deepseek_v32_exp/deepseekv32_sparse_attention_antiquant.py:359-457):
//   K row = [ bf16(fp32(int8) * scale[col/128]) | rope bf16 ],  V = first 512 columns of K
//   S = q K^T in fp32 from bf16 operands, * softmax_scale
//   P~ = exp(S - m) rounded to bf16 un-normalised, l summed in fp32 from the unrounded values
//   O = (sum P~ V) / l, one rounding to bf16
//
// Work decomposition.  One workgroup of eight wavefronts owns one (query token, KV split, group of 128 heads) and
// walks its share of the token's top-k list in tiles of 32 selected cache rows; every gathered row is dequantised
// once for all 128 heads.  The dequantised tile sits row-major in LDS (16-byte chunks XOR-swizzled with the row), three
// tiles deep, and serves as K (row reads) and as V (transposing reads, ds_read_b64_tr_b16).  A SIMD holds a pair of
// wavefronts, which owns 32 heads; the two do different work, so that one has vector and memory work to do while the other
// issues MFMAs (v_mfma_f32_16x16x32_bf16):
//   * the score wave holds Q (B operand, 30 of its 36 fragments in registers, six parked in LDS), computes S^T = K Q^T over
//     the whole contraction, runs the online softmax (two heads per lane) and accumulates O^T = V^T P~ for the first 128
//     value columns, with P~ straight out of its registers: S^T comes out in the B-operand order of the values product;
//   * the value wave produces the tiles - eight of the 32 rows each: gather into registers, dequantisation, store to LDS -
//     with the matrix instructions of the other 384 value columns between the pieces; P~ and the rescale factors come to it
//     through LDS.
// Between two barriers, one per tile: the scores and the softmax of tile i, the values of tile i - 1, the production of
// tile i + 1 and the gather of tile i + 2.  Nothing is exchanged within a tile.
//
// What bounds it: where every CU has long lists (1000 query tokens, 2048 rows each), the chip's power.  Its clock falls to 1.65 GHz
// there, from 2.35, and the time follows the energy of a tile more than its ticks: v_mfma_f32_16x16x32_bf16 adds up twice the
// products per accumulator it reads and writes of v_mfma_f32_32x32x16_bf16, and takes 3900 ticks a tile here where that one took
// 3580, but 546 us for the 1000 tokens instead of 572.  (Matrix instructions alone, out of registers, on random numbers: 1.82
// PFLOP/s and 1.63; on zeros, at full clock, 2.3 either way.  Only the values in the one and the scores in the other: 572.)  Short
// of that the issue of the two waves of a SIMD: a tile's values, scores and softmax take the score wave 0.8, 1.9 and 1.0 K ticks, the
// production and the values the value wave 3.5 K; the matrix pipes are busy 2.3 K, LDS 2.0 K.  Not faster: the values between the
// pieces of the softmax, or between the scores; more fragments ahead; the int8 shares' stores free of bank conflicts (LDS 1.8 K);
// equal priorities (4700).
//
// KV splits write their output normalised by their own sum as fp16 or fp32, in the accumulators' fragment order, plus (m, l);
// sfa_combine_kernel merges them and turns the result into rows.
#include <algorithm>
#include <utility>

#include "common.h"
#include "kernels.h"
#include "timing.h"

namespace pto {
namespace {

constexpr int T = 32;                  // selected rows per tile
constexpr int DN = SFA_DN;             // nope / value width
constexpr int DR = 64;                 // rope width
constexpr int KSTEPS = (DN + DR) / 32; // 18 MFMA k-steps for S
constexpr int KROW = (DN + DR) * 2;    // 1152 bytes per tile row = 72 chunks of 16 bytes
constexpr int STAGE = T * KROW;        // 36864
constexpr int MAX_SPLIT_TOKENS = 2048; // largest share of a top-k list one workgroup may own
constexpr int HEADS_PER_WG = SFA_HEADS_PER_WG;
constexpr int WAVES = 8, PAIRS = 4;    // a pair of waves, one of each role, to 32 heads
constexpr int NDB = DN / 16;           // 32 blocks of 16 value columns ...
constexpr int NDB_S = 8;               // ... of which the score wave of a pair takes the first eight
// of the score wave's 36 fragments of Q (k-step, block of 16 heads), every sixth is parked in LDS (16 bytes per lane each): what its
// 256 registers do not hold beside its part of O and the scores
constexpr int QFRAGS = 2 * KSTEPS, PARK_EVERY = 6, NPARK = QFRAGS / PARK_EVERY, NREG = QFRAGS - NPARK;
// LDS layout: three tile stages | parked Q | P~ [2][pair], 2 KB each | rescale factors [2][pair][32], flags [2][pair] |
// per-split arrays sized by SfaArgs::split_cap (validity words, rows).  At the start the query lies in front, on its way to operand
// layout, and behind it this sequence's page table (when it fits), while the share is looked up.
constexpr int QPARK_OFF = 3 * STAGE;
constexpr int PBUF_OFF = QPARK_OFF + PAIRS * NPARK * 1024;
constexpr int ALPHA_OFF = PBUF_OFF + 2 * PAIRS * 2048;
constexpr int FLAG_OFF = ALPHA_OFF + 2 * PAIRS * 32 * 4;
constexpr int SPLIT_OFF = FLAG_OFF + 2 * PAIRS * 4;
constexpr int LDS_LIMIT = 160 * 1024;
constexpr int OUT_ROW = DN * 2;  // epilogue staging: 128 heads x 512 values of 16 bits, reusing the front of LDS
constexpr int LSUM_OFF = ALPHA_OFF; // the epilogue's row sums [pair][32], where the rescale factors were
// start-up: each pair's query in LDS of its own, [32 heads] x 1024 bytes of nope columns, then x 128 of rope columns; behind them
// the page table
constexpr int QPAIR = 32 * (DN + DR) * 2, BT_OFF = PAIRS * QPAIR;
constexpr int BT_MAX = 1280;     // entries of a page table that is looked up in LDS (a wider one is read from memory, out of the L2: 24
                                 // tokens of 50 to 56 K contexts, 1750 entries each in LDS or 3500 in memory, 36.0 us a call either way)
static_assert(HEADS_PER_WG * OUT_ROW <= LSUM_OFF && BT_OFF + BT_MAX * 4 <= SPLIT_OFF && BT_OFF % 16 == 0, "what uses the front of LDS ends below the per-split arrays");
__host__ __device__ constexpr int tmask_bytes(int cap) { return (cap / T + 2) * 4; }
__host__ __device__ constexpr int split_bytes(int cap) { return tmask_bytes(cap) + cap * 4; }
static_assert(QPARK_OFF % 16 == 0 && SPLIT_OFF % 16 == 0, "16-byte LDS accesses");
static_assert(SPLIT_OFF + split_bytes(MAX_SPLIT_TOKENS) <= LDS_LIMIT, "a whole top-k list must fit one workgroup");


typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i receives element i%4 of the 8-byte chunks
// addressed by lanes i/4, 4 + i/4, 8 + i/4 and 12 + i/4 of the group.
__device__ __forceinline__ s16x4 lds_read_tr(uint8_t* p) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p); }

// Chunk swizzle of tile row t.  A row is 32 banks more than a multiple of the 64, so rows of one parity share their
// banks.  A b128 read serves 16 lanes at a time, 16 rows in the scores' K fragments: the eight rows of a parity need eight
// different values.  A transposing read serves 32 lanes, 32 bytes of eight rows: the four rows of a parity need different
// values of bits 1 and 2.
__host__ __device__ constexpr int swz(int t) { return ((t & 2) << 1) | (((t >> 1) ^ (t >> 2)) & 2) | ((t >> 3) & 1); }

// f(integral_constant 0), f(integral_constant 1) .. f(integral_constant N - 1), written out
template <class F, int... I>
__device__ __forceinline__ void unroll_seq(std::integer_sequence<int, I...>, F&& f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unroll(F&& f)
{
    unroll_seq(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// v, in a form that the compiler does not keep what follows from it in registers across the tiles: it would spill other
// such values, and a spilled value read back waits for every gather in flight
__device__ __forceinline__ int fresh(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// A value wave's share of one gathered tile, in registers: rows 8 pair .. 8 pair + 7 of the tile and 16 bytes of the rope
// columns of row lane / 8 of them.  int8: 16 columns (of the row's 512) of rows 4 (lane / 32) .. + 3 and the dequantisation
// scale of (row lane % 8, column group lane / 8 % 4) - 16 bytes a lane, because a load occupies the memory pipe by its
// lanes, not by its bytes.  bf16: 8 columns of all eight rows.
template <bool QUANT>
struct RawTile;
template <>
struct RawTile<true> {
    static constexpr int LOADS = 4;
    u32x4 nope[LOADS];
    u32x4 rope;
    float sc;
};
template <>
struct RawTile<false> {
    static constexpr int LOADS = 8;
    u32x4 nope[LOADS];
    u32x4 rope;
};

// rows[] holds valid cache rows only (absent entries point at row 0); the tile's validity word says which rows are
// absent, and their data is zeroed when it is consumed, so that no load depends on it.  All loads are unconditional.
// r points at the share's eight rows in LDS; what a load needs is read from there a few steps ahead of it (a register instead of ten).
// An address is one 64-bit multiply-add in the vector unit: the row comes out of LDS in every lane, and in scalar
// registers it would take a read of the lane, two multiplies and two additions per row, all issued by the same wave.
template <bool QUANT, int K>
__device__ __forceinline__ uint32_t nope_row(const int* r, int lane)
{
    return (uint32_t)(QUANT ? r[4 * (fresh(lane) >> 5) + K] : r[K]);
}
__device__ __forceinline__ uint32_t rope_row(const int* r, int lane) { return (uint32_t)r[fresh(lane) >> 3]; }
__device__ __forceinline__ uint32_t scale_row(const int* r, int lane) { return (uint32_t)r[fresh(lane) & 7]; }
template <bool QUANT, int K>
__device__ __forceinline__ void gather_nope(RawTile<QUANT>& r, uint32_t row, const SfaArgs& a, int lane)
{
    const int l = QUANT ? lane & 31 : fresh(lane);
    r.nope[K] = *reinterpret_cast<const u32x4*>(a.kn + l * 16 + (uint64_t)row * a.kn_stride);
}
template <bool QUANT>
__device__ __forceinline__ void gather_rope(RawTile<QUANT>& r, uint32_t row, const SfaArgs& a, int lane)
{
    lane = fresh(lane);
    r.rope = *reinterpret_cast<const u32x4*>(a.kr + (lane & 7) * 16 + (uint64_t)row * a.kr_stride);
}
template <bool QUANT>
__device__ __forceinline__ void gather_scale(RawTile<QUANT>& r, uint32_t row, const SfaArgs& a, int lane)
{
    lane = fresh(lane);
    if constexpr (QUANT) r.sc = *reinterpret_cast<const float*>(a.ks + ((lane >> 3) & 3) * 4 + (uint64_t)row * a.ks_stride);
}
template <bool QUANT>
__device__ __forceinline__ void gather_tile(RawTile<QUANT>& t, const SfaArgs& a, const int* r, int lane)
{
    gather_scale<QUANT>(t, scale_row(r, lane), a, lane);
    unroll<RawTile<QUANT>::LOADS>([&](auto k) { gather_nope<QUANT, k>(t, nope_row<QUANT, k>(r, lane), a, lane); });
    gather_rope<QUANT>(t, rope_row(r, lane), a, lane);
}

// Dequantisation of the share.  Two int8 of a row at a time: their bytes, sign bits flipped, are x + 128 and as the low
// bytes of two fp16 read (x + 128) 2^-24 (fp16 denormals, exact); one fma per element with the scale times 2^24 and -128
// times the scale, both exact (scales up to 2^103), rounds once, like the product x * s that the golden rounds.  (A
// conversion per element instead of one byte permute for two costs a quarter more instructions.)  In 35 pieces: a piece is the permute of one
// pair, the fmas of the pair before and the packing of the one before that, because a wave issues a vector instruction
// that depends on the one ahead of it at half the rate of an independent one.  A share with a scale from 2^104 on, where 2^24
// times the scale overflows and the product with an int8 need not, is stored once more by plain_share.
constexpr int PIECES = 35;
template <bool QUANT>
struct Production {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    float v;          // the loaded scale, of (row lane % 8, column group lane / 8 % 4)
    float sc;         // the scale of the row to come
    float s, c;       // of the row in hand: times 2^24 and times -128
    int from;         // where the scales of this lane's rows and columns are: 4 times the lane
    f16x2 h;
    float f0, f1;
    uint32_t pk[4];
    uint32_t at;      // LDS address of this lane's first chunk, stage included
    bool large;       // uniform: some scale of the share is 2^104 or more

    __device__ __forceinline__ void begin(const RawTile<QUANT>& r, uint32_t present, uint32_t stage, int pair, int lane)
    {
        lane = fresh(lane);
        if constexpr (QUANT) {
            v = r.sc;
            if (present != 0xffffffffu) { // (an absent row is stored as zeros)
                if (!((present >> (8 * pair + (lane & 7))) & 1u)) v = 0.f;
            }
            large = __any(fabsf(v) >= 0x1p104f);
            from = 4 * (4 * (lane >> 5) + (lane & 24));
            fetch_scale<0>();
            // rows t = 8 pair + 4 (lane / 32) + k, chunks 2 (lane % 32) and the next: swz(t) is swz(t - k) ^ 4 (k / 2)
            const int t = 8 * pair + 4 * (lane >> 5);
            at = stage + t * KROW + (((2 * (lane & 31)) ^ swz(t)) << 4);
        } else {
            at = stage + 8 * pair * KROW + ((lane ^ swz(8 * pair)) << 4); // rows 8 pair + k, chunk lane
        }
    }
    template <int K>
    __device__ __forceinline__ void fetch_scale()
    {
        sc = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from + 4 * K, __builtin_bit_cast(int, v)));
    }
    template <int P>
    __device__ __forceinline__ void piece(const RawTile<QUANT>& r, uint32_t present, uint8_t* lds, uint32_t stage, int pair, int lane)
    {
        if constexpr (QUANT) {
            if constexpr (P >= 2 && P < 34) {
                constexpr int K = (P - 2) / 8, H = (P - 2) / 4 % 2, Q = (P - 2) % 4;
                pk[Q] = pack_bf16x2(f0, f1);
                if constexpr (Q == 3) *reinterpret_cast<u32x4*>(lds + (at ^ (16 * H + 64 * (K / 2))) + K * KROW) = u32x4{pk[0], pk[1], pk[2], pk[3]};
            }
            if constexpr (P >= 1 && P < 33) {
                f0 = __builtin_fmaf((float)h[0], s, c);
                f1 = __builtin_fmaf((float)h[1], s, c);
            }
            if constexpr (P < 32) {
                constexpr int K = P / 8, J = P % 8;
                if constexpr (J == 0) {
                    s = sc * 16777216.f;
                    c = sc * -128.f;
                }
                if constexpr (J == 1 && K < 3) fetch_scale<K + 1>();
                h = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0u, r.nope[K][J / 2] ^ 0x80808080u, J % 2 ? 0x0c030c02u : 0x0c010c00u));
            }
        } else if constexpr (P < 32 && P % 4 == 3) {
            constexpr int K = P / 4; // (a multiple of eight rows changes swz only in the bits that `at` has)
            u32x4 v = r.nope[K];
            if (!((present >> (8 * pair + K)) & 1u)) v = u32x4{0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4*>(lds + (at ^ (swz(K) << 4)) + K * KROW) = v;
        }
        if constexpr (P == 34) { // (an absent row's scores are masked: its rope columns may be anything)
            lane = fresh(lane);
            const int t = 8 * pair + (lane >> 3);
            *reinterpret_cast<u32x4*>(lds + stage + t * KROW + DN * 2 + (((lane & 7) ^ swz(t)) << 4)) = r.rope;
        }
    }
};

// The int8 columns of a wave's share by the plain product, from memory: r points at the share's eight rows.
__device__ __forceinline__ void plain_share(const SfaArgs& a, const int* r, uint32_t present, uint8_t* stage, int pair, int lane)
{
    lane = fresh(lane);
#pragma unroll 1
    for (int e = 0; e < 8; ++e) {
        const int t = 8 * pair + e;
        const uint32_t row = (uint32_t)r[e];
        const u32x2 x = *reinterpret_cast<const u32x2*>(a.kn + lane * 8 + (uint64_t)row * a.kn_stride);
        const float sc = *reinterpret_cast<const float*>(a.ks + (lane >> 4) * 4 + (uint64_t)row * a.ks_stride);
        const float s = (present >> t) & 1u ? sc : 0.f;
        uint32_t pk[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int w = (int)(x[k >> 1] >> (k & 1 ? 16 : 0));
            pk[k] = pack_bf16x2((float)(int8_t)w * s, (float)(int8_t)(w >> 8) * s);
        }
        *reinterpret_cast<u32x4*>(stage + t * KROW + ((lane ^ swz(t)) << 4)) = u32x4{pk[0], pk[1], pk[2], pk[3]};
    }
}

// A workgroup's share of a token's top-k list: tiles [tile0, tile0 + ntiles) of the first `cur` entries.
struct SplitRange {
    int cur, tile0, ntiles;
};
__device__ __forceinline__ SplitRange split_range(int cur, int nsplit, int sp)
{
    const int ntiles_all = (cur + T - 1) / T;
    const int per = (ntiles_all + nsplit - 1) / nsplit;
    const int tile0 = sp * per;
    return {cur, tile0, max(min(ntiles_all, tile0 + per) - tile0, 0)};
}

// Resolves the workgroup's share: logical indices -> physical cache rows (absent entries: row 0 and a cleared bit in
// the tile's validity word), in LDS.  NT lanes.  The sequence's length, its page table and the share's top-k entries
// are requested together: the entries are fetched for the share a full list would give (the usual case) and only
// fetched again if the length, once known, moves the share.  The other waves pass its two barriers beside it.  Returns the share.
__device__ __forceinline__ SplitRange share_of(const SfaArgs& a, int act, int si, int nsplit, int sp)
{
    return split_range(min(max(act - a.s1 + 1 + si, 0), a.topk), nsplit, sp);
}
template <int NT>
__device__ __forceinline__ SplitRange resolve_split(const SfaArgs& a, int bi, int si, int tq, int nsplit, int sp, uint32_t* tmask,
                                                    int* rows, int* bt_lds, int tid, int lane)
{
    constexpr int PER_LANE = MAX_SPLIT_TOKENS / NT;
    const int32_t* list = a.topk_idx + (int64_t)tq * a.topk_stride;
    const SplitRange guess = split_range(a.topk, nsplit, sp);
    int my_idx[PER_LANE];
    auto fetch = [&](int tok0) {
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j)
            if (NT * j < a.split_cap) my_idx[j] = list[min(tok0 + tid + NT * j, a.topk - 1)];
    };
    fetch(guess.tile0 * T);
    const int act = a.act_seq[bi];
    // this sequence's page table -> LDS (saves one dependent global load per selected token); a table that fits LDS
    // has at most BT_PER_LANE entries per lane
    constexpr int BT_PER_LANE = BT_MAX / NT;
    const bool bt_cached = a.bt_cached != 0;
    int btv[BT_PER_LANE];
    if (bt_cached) {
#pragma unroll
        for (int j = 0; j < BT_PER_LANE; ++j)
            if (tid + NT * j < a.bt_stride) btv[j] = a.block_table[(int64_t)bi * a.bt_stride + tid + NT * j];
    }
    if (bt_cached) {
#pragma unroll
        for (int j = 0; j < BT_PER_LANE; ++j)
            if (tid + NT * j < a.bt_stride) bt_lds[tid + NT * j] = btv[j];
    }
    const SplitRange r = share_of(a, act, si, nsplit, sp);
    if (r.tile0 != guess.tile0) fetch(r.tile0 * T); // block-uniform
    const int tok0 = r.tile0 * T;
    const int ntiles_even = (r.ntiles + 1) & ~1; // whole wavefronts of entries
    // (as unsigned numbers: an unused entry, -1, is past every limit)
    const uint32_t max_logical = (uint32_t)min((int64_t)a.bt_stride * a.block_size, (int64_t)1 << 31);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        const int i = tid + NT * j;
        if (i >= ntiles_even * T) break; // wave-uniform: tiles are 32 wide, waves 64
        const uint32_t idx = (i < r.ntiles * T && tok0 + i < r.cur) ? (uint32_t)my_idx[j] : 0xffffffffu;
        int row = -1;
        if (idx < max_logical) {
            const uint32_t slot = (uint32_t)((uint64_t)idx * a.page_mul >> a.page_shift); // idx / block_size
            int page; // (two loads under a branch, not one load from a selected pointer: that would be a generic-address load)
            if (bt_cached)
                page = bt_lds[slot];
            else
                page = a.block_table[(int64_t)bi * a.bt_stride + slot];
            const int64_t pr = (int64_t)page * a.block_size + (idx - slot * a.block_size);
            if (page >= 0 && pr < a.n_rows) row = (int)pr;
        }
        rows[i] = max(row, 0);
        const uint64_t present = __ballot(row >= 0);
        if (lane == 0) {
            tmask[i >> 5] = (uint32_t)present;
            tmask[(i >> 5) + 1] = (uint32_t)(present >> 32);
        }
    }
    __syncthreads(); // rows[] / tmask[] ready
    return r;
}

// k-step of position i of 18: the two halves of the contraction one after the other, each its eight nope steps and its rope step
__host__ __device__ constexpr int kstep_at(int i) { return i < 8 ? i : i == 8 ? 16 : i < 17 ? i - 1 : i; }
// fragments of Q: 2 (position) + block of 16 heads
constexpr bool parked(int f) { return f % PARK_EVERY == PARK_EVERY - 1; }
// operand fragments read ahead of the matrix instructions that use them: K, V in the score wave, V in the value wave (more
// are registers that the waves do not have)
constexpr int KD = 4, VD_S = 3, VD_V = 2;
#define STEP_FENCE() __builtin_amdgcn_sched_barrier(0)

// (fmaxf has the compiler quiet every operand first; the scores are sums of products, which are no signalling NaN)
__device__ __forceinline__ float max3(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Over the four lanes of a wavefront that are 16 apart: the maxima of a and of b, in every one of them.  (Without a trip through LDS:
// v_permlane32_swap exchanges the upper half of its first operand with the lower half of its second, v_permlane16_swap the odd
// rows of 16 lanes of the first with the even rows of the second.  They need wait states behind an instruction that writes their
// operands, which the compiler leaves behind one that it knows: no inline assembly for those.)
__device__ __forceinline__ void max_over_rows(float a, float b, float& ma, float& mb)
{
    const auto h = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    const unsigned x = __builtin_bit_cast(unsigned, fmaxf(__builtin_bit_cast(float, (unsigned)h[0]), __builtin_bit_cast(float, (unsigned)h[1])));
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    const unsigned y = __builtin_bit_cast(unsigned, fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1])));
    const auto m = __builtin_amdgcn_permlane32_swap(y, y, false, false); // (lower half of y: a's maxima, upper: b's)
    ma = __builtin_bit_cast(float, (unsigned)m[0]);
    mb = __builtin_bit_cast(float, (unsigned)m[1]);
}

// O^T blocks DB0 .. DB0 + N - 1 of a pair's 32 heads, each 16 value columns x two blocks of 16 heads: V^T fragments of all 32 tokens of
// a tile by transposing reads, P~ in one fragment per block of heads.
template <int DB0, int N, int VD>
struct Values {
    f32x4 o[N][2];
    uint32_t off;       // this lane's place in a stage
    uint32_t at[4];     // the same in the stage in use, for the blocks n % 4
    s16x4 lo[VD], hi[VD];

    __device__ __forceinline__ void init(int lane)
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int b = 0; b < 2; ++b) o[i][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        // lane jj of row g of 16 lanes points at tile row 4 g + jj / 4 (+ 16: the same swizzle), columns 16 n + 4 (jj & 3) -> chunk 2 n +
        // (jj & 3) / 2, and gets column 16 n + jj of the rows 4 g .. 4 g + 3.  n % 4 is bits 1 and 2 of the chunk; a stage is a multiple
        // of 128 bytes, so that an exclusive or in these bits stays inside a row's group of eight chunks.
        const int jj = lane & 15, t = 4 * (lane >> 4) + (jj >> 2);
        off = t * KROW + ((((jj & 3) >> 1) ^ swz(t)) << 4) + (jj & 1) * 8;
    }
    template <int n>
    __device__ __forceinline__ void fetch(uint8_t* lds)
    {
        constexpr int db = DB0 + n, step = (db >> 2) * 128;
        lo[n % VD] = lds_read_tr(lds + at[db & 3] + step);
        hi[n % VD] = lds_read_tr(lds + at[db & 3] + step + 16 * KROW);
    }
    __device__ __forceinline__ void ahead(uint8_t* lds, int stage)
    {
        at[0] = off + stage;
        at[1] = at[0] ^ 32;
        at[2] = at[0] ^ 64;
        at[3] = at[0] ^ 96;
        unroll<VD>([&](auto n) { fetch<n>(lds); });
    }
    template <int n>
    __device__ __forceinline__ void step(uint8_t* lds, const u32x4 (&p)[2])
    {
        const bf16x8 v = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo[n % VD], hi[n % VD], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int b = 0; b < 2; ++b) o[n][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, __builtin_bit_cast(bf16x8, p[b]), o[n][b], 0, 0, 0);
        if constexpr (n + VD < N) fetch<n + VD>(lds);
    }
    // (fragments 0 .. VD - 1 have been requested)
    __device__ __forceinline__ void add(uint8_t* lds, const u32x4 (&p)[2])
    {
        unroll<N>([&](auto n) {
            step<n>(lds, p);
            STEP_FENCE();
        });
    }
    __device__ __forceinline__ void scale(float f0, float f1)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            o[i][0] *= f0;
            o[i][1] *= f1;
        }
    }
    // Epilogue.  Register e of o[i][b] holds dim 16 (DB0 + i) + 4 g + e of head 16 b + lane % 16.
    // A split's share, normalised by its own sum, in fp16 (|value| <= max |V| and 2^-11 relative rounding, a quarter
    // of the final bf16 rounding, half the bytes of fp32 for this kernel to write and the merge to read) where every token of the
    // call is split, in fp32 where only a last round's are.  It leaves
    // in fragment order, straight from the accumulators: [token][split][head group][column group dq 4][pair 4][i 4][block of
    // heads 2][lane 64] x 8 fp16, dims 4 g .. + 3 of column blocks 8 dq + 2 i and the next, or [column block 2][lane 64] x 4 fp32 in
    // place of the last two - every store instruction writes 1 KB of
    // consecutive bytes, and nothing is staged.  The merge kernel reads the same order and does the transposition to
    // rows once, for the output, instead of once per split here.  (Streaming stores: 34 MB leave the chip's 256
    // workgroups at once and are read back once.)
    __device__ __forceinline__ void store_partial(_Float16* base, const float (&mul)[2])
    {
#pragma unroll
        for (int i = 0; i < N / 2; ++i)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
                const int cb = DB0 / 2 + i;
                uint32_t x[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    x[k] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)(o[2 * i + (k >> 1)][b][2 * (k & 1)] * mul[b]),
                                                              (_Float16)(o[2 * i + (k >> 1)][b][2 * (k & 1) + 1] * mul[b])});
                __builtin_nontemporal_store(u32x4{x[0], x[1], x[2], x[3]}, reinterpret_cast<u32x4*>(base + (cb >> 2) * 16384 + ((cb & 3) * 2 + b) * 512));
            }
    }
    __device__ __forceinline__ void store_partial(float* base, const float (&mul)[2])
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int cb = (DB0 + i) / 2;
                __builtin_nontemporal_store(o[i][b] * mul[b], reinterpret_cast<f32x4*>(base + (cb >> 2) * 16384 + ((cb & 3) * 2 + b) * 512 + (i & 1) * 256));
            }
    }
    // One split: the output itself, bf16 rows [head][512] of 1024 bytes in LDS (orow: the pair's first).  v_permlane16_swap pairs up
    // four-dim pieces of neighbouring rows of lanes - an even row ends up with 8 dims of the first of two blocks, an odd one with
    // those of the second - so that a lane stores 16 bytes; the chunks of a row are XOR-swizzled with the head (16 rows of a store
    // meet all banks).
    __device__ __forceinline__ void stage_rows(uint8_t* orow, int l16, int g, const float (&mul)[2])
    {
#pragma unroll
        for (int i = 0; i < N; i += 2)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                uint32_t x[2][2]; // [block i, i + 1][pair of dims]
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int k = 0; k < 2; ++k) x[j][k] = pack_bf16x2(o[i + j][b][2 * k] * mul[b], o[i + j][b][2 * k + 1] * mul[b]);
                const auto e0 = __builtin_amdgcn_permlane16_swap(x[0][0], x[1][0], false, false);
                const auto e1 = __builtin_amdgcn_permlane16_swap(x[0][1], x[1][1], false, false);
                const int c = 2 * (DB0 + i + (g & 1)) + (g >> 1);
                *reinterpret_cast<u32x4*>(orow + (16 * b + l16) * OUT_ROW + ((c ^ l16) << 4)) = u32x4{(uint32_t)e0[0], (uint32_t)e1[0], (uint32_t)e0[1], (uint32_t)e1[1]};
            }
    }
};

// 64 lanes x 16 bytes from base + each lane's offset to 1 KB of LDS at d, in lane order, without registers in between; base and d are
// wave-uniform.  (Written out: the compiler would wait for it before every other LDS read.)
typedef __attribute__((address_space(3))) uint8_t lds_u8;
__device__ __forceinline__ void copy_to_lds(const void* base, uint32_t offset, uint8_t* d)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"((lds_u8*)d), "v"(offset), "s"(base) : "memory");
}

// The body of one wavefront.  SCORES: the pair's score wave (waves 0 .. 3), which holds Q and does the scores, the softmax and
// the values of the first NDB_S column blocks; else its value wave (waves 4 .. 7), which produces the tiles, eight rows of
// each, and does the values of the other blocks.
template <bool QUANT, bool SOME, bool SCORES>
__device__ __forceinline__ void sfa_wave(const SfaArgs& a, uint8_t* smem, uint32_t* tmask, int* rows, int* bt_lds, int tid)
{
    int tq = blockIdx.x, sp = blockIdx.y, nsplit = gridDim.y;
    const int hz = blockIdx.z;
    if constexpr (SOME) { // the tokens before t1 first, then the others, split by split
        const int w = tq - a.splits.t1, tokens = a.b * a.s1 - a.splits.t1;
        if (w >= 0) {
            nsplit = a.splits.n;
            sp = __builtin_amdgcn_readfirstlane(w / tokens); // (a division is vector code)
            tq -= sp * tokens;
        }
    }
    const int64_t part = (int64_t)(tq - (SOME ? a.splits.t1 : 0)) * nsplit; // (of a token with several splits: its first partial result)
    const int bi = tq / a.s1, si = tq - bi * a.s1;
    const int lane = tid & 63, pair = __builtin_amdgcn_readfirstlane(tid >> 6) & (PAIRS - 1); // (scalar: what follows from it is too)
    const int l16 = lane & 15, g = lane >> 4;
    const int head0 = hz * HEADS_PER_WG;
    const int hrow = pair * 32 + l16, head = head0 + hrow; // (and the ones 16 on)
    const bool active = head0 + pair * 32 < a.nq; // (a pair without heads works on copies of the last one, and stores nothing)

    // The start.  The score waves copy the query of their 32 heads to LDS, a head's nope columns to an instruction, and read their operand
    // fragments from there, while the value waves look up the share and gather the first two tiles: 8 K ticks until the first tile is
    // stored, where all waves did one after the other, the query through registers, 12 K.  (A load in operand layout would cost the
    // texture addresser a line per lane.)  The 16-byte chunks of a nope row are exchanged by the head's last four bits, of a rope row by
    // the three above the last: the 16 lanes that a read serves meet all banks.
    constexpr int NT = 64 * PAIRS;
    const int ht = tid & (NT - 1);
    bf16x8 q[SCORES ? NREG : 1];
    uint8_t* qpark = smem + QPARK_OFF + pair * (NPARK * 1024) + lane * 16;
    SplitRange share;
    RawTile<QUANT> raw0, raw;
    if constexpr (SCORES) {
        const int act = a.act_seq[bi];
        uint8_t* qrows = smem + pair * QPAIR;
        const int64_t qrow0 = (int64_t)tq * a.nq;
#pragma unroll
        for (int h = 0; h < 32; ++h)
            copy_to_lds(static_cast<const uint8_t*>(a.q_nope) + (qrow0 + min(head0 + 32 * pair + h, a.nq - 1)) * (DN * 2), (uint32_t)((lane ^ (h & 15)) * 16),
                        qrows + h * (DN * 2));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int h = 8 * i + (lane >> 3);
            copy_to_lds(static_cast<const uint8_t*>(a.q_rope) + qrow0 * (DR * 2),
                        (uint32_t)(min(head0 + 32 * pair + h, a.nq - 1) * (DR * 2) + (((lane & 7) ^ ((h >> 1) & 7)) * 16)), qrows + 32 * DN * 2 + i * 1024);
        }
        share = share_of(a, act, si, nsplit, sp);
        __syncthreads(); // (the look-up's)
        __syncthreads(); // rows[] / tmask[] ready
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // (a negative softmax_scale is applied as its magnitude to the negated query: the row statistics below are
        // taken on the raw scores, which needs a factor that commutes with max)
        const uint32_t f = a.softmax_scale < 0.f ? 0x80008000u : 0u;
        const u32x4 qflip = {f, f, f, f};
        // B operand layout: head = column, 8 consecutive k per row of 16 lanes
        u32x4 qa[QFRAGS];
#pragma unroll
        for (int i = 0; i < QFRAGS; ++i) {
            const int ks = kstep_at(i >> 1), h = 16 * (i & 1) + l16;
            qa[i] = *reinterpret_cast<const u32x4*>(ks < DN / 32 ? qrows + h * (DN * 2) + (((4 * ks + g) ^ l16) << 4)
                                                                 : qrows + 32 * DN * 2 + h * (DR * 2) + (((4 * (ks - DN / 32) + g) ^ ((h >> 1) & 7)) << 4)) ^ qflip;
        }
        __syncthreads(); // the score waves have their fragments: the rows' space is free for the parked fragments and the tiles
#pragma unroll
        for (int i = 0; i < QFRAGS; ++i) {
            const bf16x8 v = __builtin_bit_cast(bf16x8, qa[i]);
            if (parked(i))
                *reinterpret_cast<bf16x8*>(qpark + (i / PARK_EVERY) * 1024) = v;
            else
                q[SCORES ? i - i / PARK_EVERY : 0] = v;
        }
    } else {
        share = resolve_split<NT>(a, bi, si, tq, nsplit, sp, tmask, rows, bt_lds, ht, lane);
        if (share.ntiles > 0) {
            gather_tile<QUANT>(raw0, a, rows + 8 * pair, lane);
            gather_tile<QUANT>(raw, a, rows + min(1, share.ntiles - 1) * T + 8 * pair, lane);
        }
        __syncthreads(); // the score waves have their fragments
    }
    const int ntiles = share.ntiles, last = ntiles - 1;

    Values<SCORES ? 0 : NDB_S, SCORES ? NDB_S : NDB - NDB_S, SCORES ? VD_S : VD_V> val;
    if constexpr (SCORES) val.init(lane);
    // P~ of tile i lies in buffer i % 2, the order the S^T registers hold the tokens in, and the factor by which what was
    // summed before is to be multiplied, where the flag says so
    uint8_t* pbuf = smem + PBUF_OFF + pair * 2048; // (+ 16 lane)
    float* alpha_lds = reinterpret_cast<float*>(smem + ALPHA_OFF) + pair * 32;
    uint32_t* flag_lds = reinterpret_cast<uint32_t*>(smem + FLAG_OFF) + pair;
    float* lsum = reinterpret_cast<float*>(smem + LSUM_OFF) + pair * 32;
    // Between two barriers: the scores and the softmax of tile `it`, the values of tile it - 1, the production of tile it + 1
    // and the gather of tile it + 2.
    int st_old = 2 * STAGE, st = 0, st_new = STAGE; // stages of the tiles it - 1, it, it + 1
    auto turn = [&]() {
        const int t = st_old;
        st_old = st;
        st = st_new;
        st_new = t;
    };
    float l_tot[2], m_out[2] = {0.f, 0.f};
    if constexpr (SCORES) {
        // S operand (b128): tile rows l16 and 16 + l16 (the same swizzle), chunk 4 ks + g of k-step ks; swizzled offsets of the two
        // chunk positions inside a group of eight chunks
        uint32_t s_off[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) s_off[m] = l16 * KROW + (((4 * m + g) ^ swz(l16)) << 4);
        // fragment n of a tile: position n / 2, rows 16 (n % 2) ..
        bf16x8 kf[KD], qp;
        auto fetch_k = [&](auto nc) {
            constexpr int n = nc, ks = kstep_at(n >> 1);
            kf[n % KD] = *reinterpret_cast<const bf16x8*>(smem + st + s_off[ks & 1] + (ks >> 1) * 128 + (n & 1) * 16 * KROW);
            if constexpr (!(n & 1) && parked(n + 1)) qp = *reinterpret_cast<const bf16x8*>(qpark + (n / PARK_EVERY) * 1024);
        };
        static_assert(PARK_EVERY % 2 == 0 && KD < PARK_EVERY, "a parked fragment is its k-step's second, and out of use when the next one is read");
        float m_run[2] = {-INFINITY, -INFINITY}; // running max of S * scale * log2(e)
        float l_run[2] = {0.f, 0.f};             // this lane's share of sum exp
        float alpha[2] = {1.f, 1.f};
        bool rescale = false;
        // (never exactly zero: a masked score is -inf, and -inf * 0 would be NaN; 2^(s * 1e-30) is 1 for every finite s, so
        // a zero scale still gives every attended row the same weight)
        const float c_log2 = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, fmaxf(fabsf(a.softmax_scale) * 1.4426950408889634f, 1e-30f))));
        u32x4 p[2];
        auto tile = [&](int it) {
            f32x4 s0[2][2]; // [block of 16 rows][block of 16 heads]
            const uint32_t present = tmask[it];
            STEP_FENCE();
            unroll<QFRAGS>([&](auto nc) {
                constexpr int n = nc, i = n >> 1;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    constexpr int f = 2 * i;
                    const bf16x8 qi = b == 1 && parked(f + 1) ? qp : q[f + b - (f + b) / PARK_EVERY];
                    f32x4& s = s0[n & 1][b];
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[n % KD], qi, i == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s, 0, 0, 0);
                }
                if constexpr (n + KD < QFRAGS) fetch_k(std::integral_constant<int, n + KD>{});
                STEP_FENCE();
            });
            val.ahead(smem, st); // (this tile's values, behind the barrier)
            const uint32_t valid = __builtin_amdgcn_readfirstlane(present);
            if (valid != 0xffffffffu) {
                // register e of s0[rb][b] holds row 16 rb + 4 g + e for head 16 b + l16 (the lanes' shift first: the bit
                // positions left are compile-time constants)
                const uint32_t vh = valid >> (4 * g);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    f32x4& x = s0[r >> 3][(r >> 2) & 1];
                    x[r & 3] = ((vh >> (16 * (r >> 3) + (r & 3))) & 1u) ? x[r & 3] : -INFINITY;
                }
            }
            // P~ in the order the S^T registers hold the rows: k-slot s of lanes g is row 4 g + s % 4 + 16 (s / 4) - which is also how the
            // V^T fragments are read.  Relative to the running maximum as it was, while the maximum of this tile is on its way between
            // the lanes.
            float l_tile[2], mx[2], m_new[2];
            auto probabilities = [&](auto between) {
                unroll<2>([&](auto bc) {
                    constexpr int b = bc;
                    const float m_use = valid != 0u ? m_run[b] : 0.f; // (a tile without rows: every score is -inf, every P~ 0)
                    l_tile[b] = 0.f;
                    unroll<4>([&](auto rc) {
                        constexpr int r = 2 * rc;
                        const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[r >> 2][b][r & 3], c_log2, -m_use));
                        const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[r >> 2][b][(r & 3) + 1], c_log2, -m_use));
                        l_tile[b] += e0 + e1;
                        p[b][r >> 1] = pack_bf16x2(e0, e1);
                        between(std::integral_constant<int, 4 * b + r / 2>{});
                    });
                });
            };
            probabilities([&](auto ic) {
                constexpr int i = ic;
                // statistics on the raw scores (the factor is not negative, so it commutes with max)
                if constexpr (i == 0 || i == 1) {
                    const float x0 = max3(s0[0][i][0], s0[0][i][1], s0[0][i][2]), x1 = max3(s0[0][i][3], s0[1][i][0], s0[1][i][1]);
                    mx[i] = max3(x0, x1, max3(s0[1][i][2], s0[1][i][3], x0)) * c_log2;
                }
                if constexpr (i == 2) max_over_rows(mx[0], mx[1], m_new[0], m_new[1]);
            });
            // The reference exponent only follows the running maximum when it has grown by more than 2^8: until
            // then P~ = 2^(z - m_run) may exceed 1 (by at most 2^8, no issue for bf16 or the fp32 sums), which
            // makes the rescale of the accumulator registers a rare event.  Every P~, l and O stay relative to
            // the same m_run, so the result is unchanged.
#pragma unroll
            for (int b = 0; b < 2; ++b) m_new[b] = fmaxf(m_run[b], m_new[b]);
            rescale = __any(m_new[0] > m_run[0] + 8.f || m_new[1] > m_run[1] + 8.f);
            if (rescale) {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    alpha[b] = __builtin_amdgcn_exp2f(m_run[b] - m_new[b]); // 0 on the first tile (m_run = -inf)
                    l_run[b] *= alpha[b];
                    m_run[b] = m_new[b];
                    if (g == 0) alpha_lds[(it & 1) * (PAIRS * 32) + 16 * b + l16] = alpha[b];
                }
                probabilities([](auto) {});
            }
            if (lane == 0) flag_lds[(it & 1) * PAIRS] = rescale ? 1u : 0u;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                l_run[b] += l_tile[b];
                *reinterpret_cast<u32x4*>(pbuf + (it & 1) * (PAIRS * 2048) + b * 1024 + lane * 16) = p[b];
            }
        };
        __syncthreads(); // tile 0 stored, Q parked
        if (ntiles > 0) {
            unroll<KD>(fetch_k);
            tile(0);
            rescale = false; // (there is nothing to rescale yet)
            __syncthreads();
            turn();
            for (int it = 1; it < ntiles; ++it) {
                unroll<KD>(fetch_k);
                if (rescale) val.scale(alpha[0], alpha[1]);
                val.add(smem, p);
                tile(it);
                __syncthreads();
                turn();
            }
            if (rescale) val.scale(alpha[0], alpha[1]);
            val.add(smem, p);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const float l = l_run[b] + __shfl_xor(l_run[b], 16);
            l_tot[b] = l + __shfl_xor(l, 32);
            m_out[b] = m_run[b];
        }
    } else {
        Production<QUANT> prod;
        // Tile `tile` out of registers into a stage.  A load's registers are free as soon as their last pair is in hand: the
        // rows of the tile after are requested right behind that.
        constexpr int LOADS = RawTile<QUANT>::LOADS;
        constexpr int STEPS = NDB - NDB_S;
        auto produce = [&](RawTile<QUANT>& raw, auto regather, int tile, int stage, auto&& between) {
            constexpr bool GATHER = decltype(regather)::value;
            const uint32_t present = __builtin_amdgcn_readfirstlane(tmask[tile]);
            const int* next = rows + min(tile + 1, last) * T + 8 * pair;
            uint32_t row, row1;
            prod.begin(raw, present, stage, pair, lane);
            STEP_FENCE();
            unroll<PIECES>([&](auto ic) {
                constexpr int i = ic, per = 32 / LOADS, K = i / per;
                between(ic);
                prod.template piece<i>(raw, present, smem, stage, pair, lane);
                if constexpr (GATHER) {
                    if constexpr (i < 32 && i % per == per - 3) row = nope_row<QUANT, K>(next, lane);
                    if constexpr (i < 32 && i % per == per - 1) gather_nope<QUANT, K>(raw, row, a, lane);
                    if constexpr (i == 28) row1 = scale_row(next, lane);
                    if constexpr (i == 30) gather_scale<QUANT>(raw, row1, a, lane);
                    if constexpr (i == 32) row1 = rope_row(next, lane);
                }
                STEP_FENCE();
            });
            if constexpr (GATHER) gather_rope<QUANT>(raw, row1, a, lane);
            if constexpr (QUANT)
                if (__builtin_expect(prod.large, false)) plain_share(a, rows + tile * T + 8 * pair, present, smem + stage, pair, lane);
        };
        u32x4 p[2];
        auto values = [&](int it) {
            const uint8_t* pb = pbuf + (it & 1) * (PAIRS * 2048) + fresh(lane) * 16;
#pragma unroll
            for (int b = 0; b < 2; ++b) p[b] = *reinterpret_cast<const u32x4*>(pb + 1024 * b);
            if (__builtin_amdgcn_readfirstlane(flag_lds[(it & 1) * PAIRS])) {
                const float* al = alpha_lds + (it & 1) * (PAIRS * 32) + (fresh(lane) & 15);
                val.scale(al[0], al[16]);
            }
            STEP_FENCE();
        };
        auto value_step = [&](auto nc) {
            constexpr int n = nc;
            val.template step<n>(smem, p);
            STEP_FENCE();
        };
        auto nothing = [](auto) {};
        if (ntiles > 0) produce(raw0, std::false_type{}, 0, 0, nothing);
        __syncthreads(); // tile 0 stored, Q parked
        val.init(lane);  // (while the score wave has the first tile)
        if (ntiles > 0) {
            if (last > 0) produce(raw, std::true_type{}, 1, st_new, nothing);
            val.ahead(smem, st); // (this tile's values, behind the barrier)
            __syncthreads();
            turn();
            __builtin_amdgcn_s_setprio(1); // (the score wave is the older one of the SIMD and would take every slot)
            for (int it = 1; it < last; ++it) {
                values(it - 1);
                produce(raw, std::true_type{}, it + 1, st_new, [&](auto ic) {
                    constexpr int i = ic, n0 = i < 3 ? 0 : (i - 3) * STEPS / (PIECES - 3), n1 = i < 3 ? 0 : (i - 2) * STEPS / (PIECES - 3);
                    if constexpr (n1 > n0) value_step(std::integral_constant<int, n0>{});
                });
                val.ahead(smem, st);
                __syncthreads();
                turn();
            }
            if (last > 0) {
                values(last - 1);
                unroll<STEPS>(value_step);
                val.ahead(smem, st);
                __syncthreads();
                turn();
            }
            values(last);
            unroll<STEPS>(value_step);
        }
    }

    // The score waves publish the row sums; every wave normalises its own blocks.
    __syncthreads(); // nobody reads a tile, P~ or a factor any more
    if constexpr (SCORES) {
        if (g == 0) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                lsum[16 * b + l16] = l_tot[b];
                if (nsplit > 1 && head + 16 * b < a.nq) {
                    const int64_t prow = (part + sp) * a.nq + head + 16 * b;
                    a.part_ml[prow * 2] = m_out[b];
                    a.part_ml[prow * 2 + 1] = l_tot[b];
                }
            }
        }
    }
    __syncthreads();
    float mul[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        if constexpr (!SCORES) l_tot[b] = lsum[16 * b + l16];
        mul[b] = l_tot[b] > 0.f ? 1.f / l_tot[b] : 0.f;
    }
    if (nsplit > 1) {
        using P = typename std::conditional<SOME, float, _Float16>::type;
        const int64_t at = (((part + sp) * gridDim.z + hz) * 8 + (pair >> 1)) * 8192 + (pair & 1) * 4096;
        // (counted in fp16 up to the lane's 16 bytes: counted in P the int8 value wave had a gather's registers spilled in every tile)
        if (active) val.store_partial(reinterpret_cast<P*>(static_cast<_Float16*>(a.part_o) + at * (sizeof(P) / 2) + lane * 8), mul);
        return;
    }
    val.stage_rows(smem + pair * 32 * OUT_ROW, l16, g, mul);
    __syncthreads();
    // a wavefront copies whole rows, one per instruction
    const int row0 = pair * 32 + (SCORES ? 0 : 16);
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 8) {
        u32x4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = *reinterpret_cast<const u32x4*>(smem + (row0 + k0 + k) * OUT_ROW + ((lane ^ (k0 + k)) << 4));
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int oh = head0 + row0 + k0 + k;
            if (oh < a.nq) // (wave-uniform)
                *reinterpret_cast<u32x4*>(reinterpret_cast<uint8_t*>(a.out) + (((int64_t)tq * a.nq + oh) * DN + lane * 8) * 2) = v[k];
        }
    }
}

// grid (query tokens, KV splits, groups of 128 heads); SOME: where only the tokens from t1 on are split, (sum of the splits, 1, groups).
// Workgroups go to the XCDs round-robin in launch order, so with the
// token as the fastest dimension the splits of one token run on one XCD (when the token count is a multiple of 8)
// and share its L2 for the token's queries.
template <bool QUANT, bool SOME>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WAVES, 64 * WAVES), amdgpu_waves_per_eu(2, 2))) void sfa_decode_kernel(
    SfaArgs a)
{
    extern __shared__ __align__(16) uint8_t smem[];
    uint32_t* tmask = reinterpret_cast<uint32_t*>(smem + SPLIT_OFF);
    int* rows = reinterpret_cast<int*>(smem + SPLIT_OFF + tmask_bytes(a.split_cap));
    int* bt_lds = reinterpret_cast<int*>(smem + BT_OFF);
    // both roles run the same barrier sequence
    if (threadIdx.x < 64 * PAIRS)
        sfa_wave<QUANT, SOME, true>(a, smem, tmask, rows, bt_lds, threadIdx.x);
    else
        sfa_wave<QUANT, SOME, false>(a, smem, tmask, rows, bt_lds, threadIdx.x);
}

// attention_out <- 0 (cache without rows: every selected entry is absent)
__global__ void sfa_zero_kernel(uint32_t* out, int64_t n_words)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_words) out[i] = 0u;
}

// out[row, :] = sum_s (2^(m_s - M) l_s / L) o_s[row, :] with L = sum_s 2^(m_s - M) l_s and o_s the split's normalised
// output.  The partials lie in the fragment order the attention kernel's accumulators have (see its epilogue).  One
// workgroup merges, for one token, what the attention workgroups left for column group wv / 2 and pair 2 (wv % 2) + hb: 32 heads x
// 128 value columns; its wavefront i takes 16 of the heads and 64 columns, a lane owning for its head (16 (i % 2) + l16) the four
// 4-column runs at 16 j + 4 g of these.  G = 2, 4 or 8, the smallest that covers the split count: every split's loads are requested
// before any is used (splits past the last are the last again with weight 0).  That it is written as a loop over groups, of which there is one, is for the code that
// comes of it: without the loop the kernel takes longer, whether the loads are left to the compiler (by the profiler, with / without, 48 tokens 8.96 / 9.45 us, 96:
// 8.14 / 8.38) or kept in front by a fence (26: 7.65 / 7.78, 48: 8.96 / 9.13, 96: 8.14 / 8.38), the pairs (m, l) first or last.  More than eight splits:
// sfa_combine_many_launch.  The workgroup then turns its 32 x 128 block through LDS and writes the 256-byte row pieces, 16 lanes a piece.
// grid (tokens with several splits x head groups x 16), 256 lanes; token0: the first of these tokens.
constexpr int CROW = 128 * 2 + 16; // LDS row of the merge's transposition: 128 bf16 plus one 16-byte chunk of padding
template <int G, bool FP32>
__global__ __launch_bounds__(256) void sfa_combine_kernel(const void* __restrict__ partials, const float* __restrict__ part_ml, void* out, int nq,
                                                          int nsplit, int token0, int hgroups)
{
    using P = typename std::conditional<FP32, float, _Float16>::type;
    const P* part_o = static_cast<const P*>(partials); // (a plain pointer type keeps the symbol readable)
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    __shared__ __align__(16) uint8_t tr[32 * CROW];
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int i = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int task = blockIdx.x; // ((token - token0) * hgroups + hz) * 8 + wv) * 2 + hb
    const int hb = task & 1, wv = (task >> 1) & 7;
    const int th = task >> 4, hz = th % hgroups, tq = token0 + th / hgroups;
    const int64_t partial = (int64_t)(tq - token0) * nsplit;
    const int hh = wv & 1, dq = wv >> 1;
    const int head_base = hz * HEADS_PER_WG + 64 * hh + 32 * hb;
    if (head_base >= nq) return; // (a head block past the last head: nothing was written for it)
    float acc[2][8];
#pragma unroll
    for (int x = 0; x < 16; ++x) (&acc[0][0])[x] = 0.f;
    float M = -INFINITY, L = 0.f;
    const int b = i & 1, cb = i & 2; // the wavefront's block of 16 heads and first of two column blocks
    const int64_t split_stride = (int64_t)hgroups * 8 * 8192; // elements between two splits of a token
    const P* frag0 = part_o + ((partial * hgroups + hz) * 8 + wv) * 8192 + hb * 4096 + cb * 1024 + b * 512; // (the workgroup's four wavefronts read 8 or 16 KB in a row per split)
    const float2* ml0 = reinterpret_cast<const float2*>(part_ml) + partial * nq + min(head_base + 16 * b + l16, nq - 1);
    for (int s0 = 0; s0 < nsplit; s0 += G) {
        typename std::conditional<FP32, f32x8, f16x8>::type v[G][2];
        float2 ml[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int s = min(s0 + j, nsplit - 1);
            const P* base = frag0 + s * split_stride;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if constexpr (FP32) {
                    const f32x4 *lo = reinterpret_cast<const f32x4*>(base + h * 1024) + lane, *hi = lo + 64;
                    v[j][h] = __builtin_shufflevector(*lo, *hi, 0, 1, 2, 3, 4, 5, 6, 7);
                } else
                    v[j][h] = *reinterpret_cast<const f16x8*>(base + h * 1024 + lane * 8);
            }
            ml[j] = ml0[(int64_t)s * nq];
            if (s0 + j >= nsplit) ml[j].y = 0.f;
        }
        if constexpr (FP32) STEP_FENCE(); // (left alone, fewer of the loads are in flight: 44 tokens of 5 splits 13.4 us, so 13.0)
        // the group's maximum joins the running one: what was summed so far is rescaled once per group
        float Mg = M;
#pragma unroll
        for (int j = 0; j < G; ++j) Mg = ml[j].y > 0.f ? fmaxf(Mg, ml[j].x) : Mg;
        if (Mg != -INFINITY) { // (otherwise nothing attended in these splits)
            if (s0 > 0) {
                const float back = exp2f(M - Mg); // 0 while nothing has been summed (M = -inf)
                L *= back;
#pragma unroll
                for (int x = 0; x < 16; ++x) (&acc[0][0])[x] *= back;
            }
            M = Mg;
#pragma unroll
            for (int j = 0; j < G; ++j) {
                const float w = ml[j].y > 0.f ? exp2f(ml[j].x - M) * ml[j].y : 0.f;
                L += w;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[h][e] += (float)v[j][h][e] * w;
            }
        }
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float* x = &acc[h][4 * j];
            const u32x2 w = {pack_bf16x2(x[0] * inv, x[1] * inv), pack_bf16x2(x[2] * inv, x[3] * inv)};
            *reinterpret_cast<u32x2*>(tr + (16 * b + l16) * CROW + (32 * (cb + h) + 16 * j + 4 * g) * 2) = w;
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = 16 * k + (threadIdx.x >> 4), c = threadIdx.x & 15;
        const u32x4 w = *reinterpret_cast<const u32x4*>(tr + r * CROW + c * 16);
        if (head_base + r < nq)
            *reinterpret_cast<u32x4*>(reinterpret_cast<uint8_t*>(out) + (((int64_t)tq * nq + head_base + r) * DN + 128 * dq + 8 * c) * 2) = w;
    }
}

int num_cus()
{
    static std::atomic<int> cached[64]; // per device ordinal; 0 = not asked yet
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    n = cached[dev & 63].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev & 63].store(n, std::memory_order_relaxed);
    }
    return n;
}

} // namespace

// The KV splits.  One number for all tokens: one workgroup to a CU, and no more than share the tiles as well - nine splits of 64 tiles
// are eight tiles each like eight splits, but leave more partials, and a second group of them to the merge (26 tokens: 77.0 us a pass
// with nine, 73.9 with eight).  Where that is one split each and the tokens are some whole rounds of workgroups and a few more: as many
// splits of these few as fill the CUs once more, where the last round takes less so.  By the time that either should take, in ns:
// a tile (where more CUs work, the chip's clock falls: 150 workgroups 1700, 200: 1780, 256: 2030), the two ends of a workgroup, a
// partial result's way to memory and back, the merge's launch.
// 16 splits at most, but 32 of a single token, whose calls are launches and chains, where the tiles saved are more than the partial results to write and read
// cost, by heads x splits: a call of 2048 rows with 16 / 32, 128 heads 18.4 / 14.9 us, 256: 18.7 / 16.7, 384: 18.9 / 18.8, 512: 20.6 / 22.1, 1024: 24.5 / 27.2; of
// 1024 rows 14.9 / 14.1, 14.7 / 15.7, 15.1 / 17.5, 17.0 / 21.0; four tokens of 128 heads 20.2 / 21.5 (two of 2048 rows would gain, 18.2 / 16.9, not of 1024, 14.4 /
// 15.6).  Its distance from 64 bits is less with more of them (mean of 24 calls 2.07e-3 with 16, 1.96e-3 with 32; 1024 rows 2.01, 1.72: P~ is rounded relative to
// each split's own maximum).
// Prefill calls of 128 heads and 2048 rows a token, one split each and so, int8 cache: 257 tokens 239 -> 159 us, 300: 244 -> 177, 360:
// 246 -> 208, 384: 247 -> 218, 520: 370 -> 287, 640: 377 -> 348, 800: 500 -> 437; bf16 cache and packed rows within 1 us of these.
// (With fp16 partial results 300 take 170, and 129 in two splits each 102 instead of 118 - but calls of one split a token have fp32 sums
// to the end, and their range.  rms error of the last round's tokens against 64 bits, 300 tokens: one split 2.163e-3, so 2.141e-3.)
constexpr int64_t TILE_NS = 1550, TILE_FULL_NS = 480, ENDS_NS = 7000, PARTIAL_NS = 90, MERGE_NS = 2500;
SfaSplits sfa_pick_splits(int t, int nq, int topk, uint64_t scratch)
{
    const int hgroups = (nq + HEADS_PER_WG - 1) / HEADS_PER_WG, cus = std::max(1, num_cus() / hgroups); // (of a head group)
    const int tiles = (topk + T - 1) / T;
    const int most = t == 1 && hgroups <= 2 && 32 * hgroups <= tiles ? 32 : 16;
    auto even = [&](int n) { // no more splits than n, and no more than share the tiles as well
        n = std::max(1, std::min({n, tiles, most}));
        const int per = (tiles + n - 1) / n;
        return (tiles + per - 1) / per;
    };
    const int last = t % cus; // tokens of the last round, by one split each
    if (t < cus || last == 0) return {0, even(cus / std::max(t, 1))};
    auto round_ns = [&](int n) { // of the last round, its tokens in n splits each
        const int64_t w = (int64_t)last * n;
        return (tiles + n - 1) / n * (TILE_NS + TILE_FULL_NS * w * w / ((int64_t)cus * cus)) + ENDS_NS + (n > 1 ? w * hgroups * PARTIAL_NS + MERGE_NS : 0);
    };
    const SfaSplits some = {t - last, even(cus / last)};
    return some.n > 1 && round_ns(some.n) < round_ns(1) && sfa_workspace_bytes(t, nq, some) <= scratch ? some : SfaSplits{0, 1};
}

uint64_t sfa_partials_bytes(int t, int nq, const SfaSplits& splits)
{
    const int hgroups = (nq + HEADS_PER_WG - 1) / HEADS_PER_WG; // (whole 128-head groups: the partials lie in fragment order)
    return (uint64_t)splits.partials(t) * hgroups * HEADS_PER_WG * DN * (splits.fp32() ? sizeof(float) : sizeof(_Float16));
}

uint64_t sfa_workspace_bytes(int t, int nq, const SfaSplits& splits)
{
    return sfa_partials_bytes(t, nq, splits) + (uint64_t)splits.partials(t) * nq * 2 * sizeof(float);
}

// Scratch for callers that cannot allocate (sfa_static_scratch): one array per GPU the library runs on, held until the
// process ends.  In host code the array's name is only a handle for hipGetSymbolAddress - the device address it returns
// is what kernels and copies are given.
static __device__ __align__(256) unsigned char scratch[SFA_STATIC_SCRATCH_BYTES];

hipError_t sfa_static_scratch(void** ptr)
{
    static std::atomic<void*> cached[64]; // per device ordinal: every GPU has its own copy of the array at its own address
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    void* p = cached[dev & 63].load(std::memory_order_acquire);
    if (p == nullptr) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (p == nullptr) return hipErrorInvalidSymbol;
        cached[dev & 63].store(p, std::memory_order_release);
    }
    *ptr = p;
    return hipSuccess;
}

hipError_t sfa_launch(const SfaArgs& a, hipStream_t stream)
{
    const int t = a.b * a.s1;
    if (t == 0) return hipSuccess;
    if (a.n_rows == 0) {
        const int64_t words = (int64_t)t * a.nq * DN / 2;
        hipLaunchKernelGGL(sfa_zero_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, stream,
                           static_cast<uint32_t*>(a.out), words);
        return hipGetLastError();
    }
    SfaArgs args = a;
    const int tiles = (a.topk + T - 1) / T;
    // division of a 31-bit index by the page size as a multiplication: with 2^(l-1) < block_size <= 2^l and the multiplier
    // 2^(31+l) / block_size rounded up (less than 2^32), the excess of the product is less than 2^(31+l) / block_size
    int l = 0;
    while (((int64_t)1 << l) < a.block_size) ++l;
    args.page_mul = (uint32_t)((((uint64_t)1 << (31 + l)) + (uint32_t)a.block_size - 1) / (uint32_t)a.block_size);
    args.page_shift = 31 + l;
    const int t1 = a.splits.t1, n = a.splits.n, fewest = t1 > 0 ? 1 : n; // splits of a token
    args.split_cap = (((tiles + fewest - 1) / fewest + 1) & ~1) * T;
    const int smem_bytes = SPLIT_OFF + split_bytes(args.split_cap);
    args.bt_cached = a.bt_stride <= BT_MAX ? 1 : 0;
    static DeviceOnce attr_done[2][2];
    auto kern = t1 > 0 ? (a.quant ? sfa_decode_kernel<true, true> : sfa_decode_kernel<false, true>)
                       : (a.quant ? sfa_decode_kernel<true, false> : sfa_decode_kernel<false, false>);
    {
        hipError_t e = attr_done[t1 > 0][a.quant].run([&] {
            return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       LDS_LIMIT);
        });
        if (e != hipSuccess) return e;
    }
    const int hgroups = (a.nq + HEADS_PER_WG - 1) / HEADS_PER_WG;
    const dim3 grid = t1 > 0 ? dim3(t1 + (t - t1) * n, 1, hgroups) : dim3(t, n, hgroups);
    {
        ScopedKernelTimer tm(KID_SFA_DECODE, stream);
        hipLaunchKernelGGL(kern, grid, dim3(64 * WAVES), smem_bytes, stream, args);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (n > 1) {
        ScopedKernelTimer tm(KID_SFA_COMBINE, stream);
        if (n > 8) return sfa_combine_many_launch(a, n, t1, stream);
        const dim3 merges((t - t1) * hgroups * 16);
        auto merge = t1 > 0 ? (n <= 2 ? sfa_combine_kernel<2, true> : n <= 4 ? sfa_combine_kernel<4, true> : sfa_combine_kernel<8, true>)
                            : (n <= 2 ? sfa_combine_kernel<2, false> : n <= 4 ? sfa_combine_kernel<4, false> : sfa_combine_kernel<8, false>);
        hipLaunchKernelGGL(merge, merges, dim3(256), 0, stream, static_cast<const void*>(a.part_o), a.part_ml, a.out, a.nq, n, t1, hgroups);
        e = hipGetLastError();
    }
    return e;
}

} // namespace pto
