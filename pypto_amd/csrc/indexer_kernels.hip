// Lightning indexer (int8 index scores + top-k) - gfx950 kernels.
//
// Replaces the device side of lightning_indexer_decode_compute
// (models/deepseek_v32_exp/lightning_indexer_quant_impl.py:38-216); arithmetic follows the golden
// (models/deepseek_v32_exp/deepseekv32_lightning_indexer_quant.py:178-263):
//   w_scale[h] = fp16(q_scale[h] * weight[h])
//   y[h, n]    = fp16(relu(int32 dot(q[h], k[n])) * 2^-11)
//   score[n]   = (sum_h fp32(w_scale[h]) * fp32(y[h, n])) * fp32(k_scale[n])
//   top-k over score[0 : eff_seq), eff_seq = act_seq - (s1 - 1 - i); best first, equal scores by ascending
//   index (framework/src/interface/interpreter/calculator/calc_torch.cpp:2481-2494); unused slots = -1.
//
// indexer_score_kernel: v_mfma_i32_16x16x64_i8 with the query heads as rows (A, resident in registers)
// and 16 cached keys as columns (B, loaded from the paged cache straight in operand layout: lane l reads
// 16 bytes of key l%16).  The result has one key per lane and 16 heads per lane; relu, the 2^-11 scaling and
// the fp16 rounding are 4 VALU operations per (head, key), and the weighted head sum is a second MFMA
// (v_mfma_f32_16x16x32_f16: row 0 of A holds w_scale, B is the fp16 tile just produced; every product of two
// fp16 values is exact in fp32, so this is the golden's fp32 sum up to the order of additions).  Scores go to
// a dense fp32 row per query token, and their order-preserving keys into a 256-bin histogram in LDS (score_bin:
// quarter octaves).  Every workgroup owns a span of its sequence's keys and leaves its histogram in one or two slots of
// its own in the workspace (16-bit counts): plain stores, nothing to clear beforehand and no global atomics.
//
// Score rows of up to 32768 keys (by the page table's reach) are selected by one kernel (indexer_row_topk_kernel), without
// histograms; longer ones by two:
//
// indexer_select_kernel: every workgroup adds up the spans' histograms of its query token, finds the bin B that
// holds the k-th largest key, and files its 4096 scores: bins above B are winners, bin B goes to a tie list (both
// lists in the workspace, appended with one global atomic per workgroup; the counters are cleared by the score
// kernel).
//
// indexer_topk_kernel: one workgroup per query token takes the winners, picks the missing krem entries out of
// the tie list by radix-selecting on the 64-bit words (key << 32 | ~index) (so equal keys resolve to the
// smaller index), and puts the k words in order (order_words).  A tie list that overflowed its capacity (e.g. all scores
// equal) falls back to radix-selecting over the whole score row.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "timing.h"

namespace pto {
namespace {

constexpr int D = 128;          // index head dim
constexpr int CHUNK = 512;      // keys per pass of a workgroup of the score kernel (8 groups of 16 per wavefront)
constexpr int PASSES = 4;       // passes per workgroup (amortise the Q / w_scale set-up)
constexpr int MAX_K = 2048;     // top-k capacity
constexpr int NBINS = 2048;     // digit bins of the radix select and of the final ordering (11 bits)
constexpr int SBINS = 256;      // bins of the selection histogram (score_bin)
constexpr int SUBBINS = 64;     // second level inside the threshold bin: the next six key bits (tie_sub_bin)
constexpr int SUB_RANK_CAP = 128; // ties of one second-level step that are ranked by direct comparison (more: digit by digit)
constexpr int SEL_CHUNK = 4096; // scores per workgroup of the select kernel
constexpr int TIE_CAP = 8192;   // capacity of the per-row tie list
constexpr int INDEXER_ROW_MAX = 32768; // rows up to this length are selected by one kernel (indexer_row_topk_kernel)
constexpr int SCORE_GROUPS = 512; // workgroups of the paged score kernel below which its spans are made shorter
constexpr int SCORE_GROUPS_MIN = 384; // and below which they are made shorter because the contexts are (96 sequences of 1500 .. 16000 keys: 422
                                      // workgroups of four passes 33.6 us, 900 of two, more than fit the CUs at once, 39.4)
constexpr float SCORE_CACHED = 96e6f; // bytes of a batch's keys from which they are loaded past the last-level cache

__device__ __forceinline__ float f16_bits_to_f32(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
// A scale as it lies in memory (fp16 bits, or fp32 in the fp32-scale variant) and as the fp32 factor it stands for.
template <bool F32> struct ScaleOf { typedef uint16_t raw; static __device__ __forceinline__ float f32(raw v) { return f16_bits_to_f32(v); } };
template <> struct ScaleOf<true> { typedef float raw; static __device__ __forceinline__ float f32(raw v) { return v; } };
// fp16(fp32(a * b)): the product is rounded to fp32 first and that value to fp16, as the golden's tensor operations do.
// (The compiler would otherwise fuse the multiplication and the conversion into one mixed-precision instruction that
// rounds the exact product once - a different fp16 value about once in 8000 products.)
__device__ __forceinline__ _Float16 round_f32_product_to_f16(float a, float b)
{
    float p = a * b;
    asm volatile("" : "+v"(p));
    return (_Float16)p;
}
// w_scale = q_scale * weight rounded once to fp16: the fp16 product of two fp16 values, or - fp32 scales - the fp32
// product of the scale and the widened weight
template <bool F32>
__device__ __forceinline__ _Float16 w_scale_of(typename ScaleOf<F32>::raw q_scale, uint16_t weight)
{
    const _Float16 w = __builtin_bit_cast(_Float16, weight);
    if constexpr (F32)
        return round_f32_product_to_f16(q_scale, (float)w);
    else
        return (_Float16)(__builtin_bit_cast(_Float16, q_scale) * w);
}
__device__ __forceinline__ uint32_t score_key(float f) { return f32_to_ordered(f + 0.0f); } // -0 -> +0
// Bin of a score key in the selection histogram, non-decreasing in the key: quarter octaves (sign, exponent, two
// mantissa bits - the top 11 key bits) of the magnitudes 2^-20 .. 2^12, 128 bins for either sign; smaller and larger
// magnitudes fall into the first and last bin of their sign.  Keys of one interior bin share their top 11 bits.
__device__ __forceinline__ uint32_t score_bin(uint32_t key)
{
    constexpr int LO = (127 - 20) * 4; // exponent field and two mantissa bits of 2^-20
    const int t = (int)(key >> 21);
    return t >= 1024 ? 128u + (uint32_t)min(max(t - 1024 - LO, 0), 127) : (uint32_t)min(max(t - (1023 - LO - 127), 0), 127);
}
__device__ __forceinline__ bool score_bin_is_interior(uint32_t bin) { return (bin & 127u) != 0u && (bin & 127u) != 127u; }
// The keys of an interior bin share their top 11 bits; the next six split the bin into 64 equal steps, in key order.
__device__ __forceinline__ uint32_t tie_sub_bin(uint32_t key) { return (key >> 15) & (SUBBINS - 1u); }
// Smallest and largest key of a bin (the first and last bin of a sign reach to the end of the sign's keys).
__device__ __forceinline__ void score_bin_range(uint32_t bin, uint32_t& lo, uint32_t& hi)
{
    constexpr int LO = (127 - 20) * 4;
    const uint32_t j = bin & 127u;
    const uint32_t t = bin >= 128u ? 1024u + LO + j : j + (1023u - LO - 127u);
    lo = j == 0u ? (bin & 128u) << 24 : t << 21;
    hi = j == 127u ? ((bin & 128u) << 24) | 0x7fffffffu : (t << 21) | 0x1fffffu;
}

__device__ __forceinline__ uint64_t make_cand(uint32_t key, int idx)
{
    return ((uint64_t)key << 32) | (uint32_t)(0xffffffffu - (uint32_t)idx);
}

// One step of a wavefront scan in the vector unit's own lane network (no trip through LDS): the value of the lane
// CTRL names (row_shr:n = 0x110 + n within a row of 16 lanes, row_bcast15 = 0x142 / row_bcast31 = 0x143 across rows,
// limited to the rows of ROW_MASK), IDENT where there is no such lane.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_from(uint32_t v, uint32_t ident)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)ident, (int)v, CTRL, ROW_MASK, 0xf, false);
}

// wavefront-wide inclusive prefix sum: lane l gets v[0] + .. + v[l]
__device__ __forceinline__ uint32_t wave_prefix_sum(uint32_t v)
{
    v += dpp_from<0x111, 0xf>(v, 0u);
    v += dpp_from<0x112, 0xf>(v, 0u);
    v += dpp_from<0x114, 0xf>(v, 0u);
    v += dpp_from<0x118, 0xf>(v, 0u);
    v += dpp_from<0x142, 0xa>(v, 0u); // rows 1 and 3 add the totals of rows 0 and 2
    v += dpp_from<0x143, 0xc>(v, 0u); // rows 2 and 3 add the total of rows 0 and 1
    return v;
}

// wavefront-wide minimum / maximum, the same value in every lane
__device__ __forceinline__ uint32_t wave_min(uint32_t v)
{
    v = min(v, dpp_from<0x111, 0xf>(v, 0xffffffffu));
    v = min(v, dpp_from<0x112, 0xf>(v, 0xffffffffu));
    v = min(v, dpp_from<0x114, 0xf>(v, 0xffffffffu));
    v = min(v, dpp_from<0x118, 0xf>(v, 0xffffffffu));
    v = min(v, dpp_from<0x142, 0xa>(v, 0xffffffffu));
    v = min(v, dpp_from<0x143, 0xc>(v, 0xffffffffu));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    v = max(v, dpp_from<0x111, 0xf>(v, 0u));
    v = max(v, dpp_from<0x112, 0xf>(v, 0u));
    v = max(v, dpp_from<0x114, 0xf>(v, 0u));
    v = max(v, dpp_from<0x118, 0xf>(v, 0u));
    v = max(v, dpp_from<0x142, 0xa>(v, 0u));
    v = max(v, dpp_from<0x143, 0xc>(v, 0u));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The workgroup's histograms (S1 query tokens, `slots` runs of keys from slot `first` on) go to its own slots, as 16-bit counts (a
// slot has at most 2048 keys), two per lane.  The first workgroup of a sequence also clears the select kernel's list counters of
// its query tokens.  256 lanes.
template <int S1>
__device__ __forceinline__ void flush_span_hist(const IndexerArgs& a, const uint32_t (*hist)[S1][SBINS], int row0, int first, int slots, int tid)
{
    if (tid < SBINS / 2) {
        for (int h = 0; h < slots; ++h)
#pragma unroll
            for (int s = 0; s < S1; ++s) {
                const int64_t slot = (int64_t)(row0 + s) * a.pchunks + first + h;
                reinterpret_cast<uint32_t*>(a.span_hist + slot * SBINS)[tid] = hist[h][s][2 * tid] | (hist[h][s][2 * tid + 1] << 16);
            }
    }
    if (first == 0 && tid < 4 * S1) a.counters[(int64_t)row0 * 4 + tid] = 0u;
}

// S1 query tokens of one sequence share every key fragment.
// POW2: block_size is a power of two (page index by shift instead of an integer division per key).
template <int S1, bool POW2, bool F32>
__global__ __launch_bounds__(256) void indexer_score_kernel(IndexerArgs a)
{
    __shared__ __align__(16) uint32_t hist[1][S1][SBINS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const int bi = blockIdx.y;
    const int sgrp = blockIdx.z; // group of S1 consecutive query tokens of the sequence
    const int L = min(a.act_seq[bi], a.max_ctx); // keys past the page table's reach do not exist
    if (blockIdx.x * (CHUNK * PASSES) >= L) return;
    const int row0 = bi * a.s1 + sgrp * S1;

    for (int i = tid; i < S1 * SBINS; i += 256) (&hist[0][0][0])[i] = 0;

    // int8 A fragments: head hb*16 + l16, bytes 64*ks + 16*g .. +15
    i32x4 qf[S1][4][2];
    // fp16 A fragments of the head sum: row 0 (lanes with l16 == 0) holds w_scale, k-slot (g, e) of MFMA mm is
    // head 32*mm + 16*(e/4) + 4*g + e%4 - the head whose int32 result this lane group holds in that slot
    f16x8 wa[S1][2];
#pragma unroll
    for (int s = 0; s < S1; ++s) {
#pragma unroll
        for (int hb = 0; hb < 4; ++hb) {
            const int8_t* qp = a.q + ((int64_t)(row0 + s) * a.nh + hb * 16 + l16) * D + 16 * g;
            qf[s][hb][0] = *reinterpret_cast<const i32x4*>(qp);
            qf[s][hb][1] = *reinterpret_cast<const i32x4*>(qp + 64);
        }
#pragma unroll
        for (int mm = 0; mm < 2; ++mm)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t h = (int64_t)(row0 + s) * a.nh + 32 * mm + 16 * (e >> 2) + 4 * g + (e & 3);
                wa[s][mm][e] = l16 == 0 ? w_scale_of<F32>(static_cast<const typename ScaleOf<F32>::raw*>(a.q_scale)[h], a.weights[h]) : (_Float16)0.f; // one fp16 rounding
            }
    }
    __syncthreads(); // histogram zeroed

    for (int pass = 0; pass < PASSES; ++pass) {
    const int tok_begin = (blockIdx.x * PASSES + pass) * CHUNK;
    if (tok_begin >= L) break;
    const int tok_end = min(L, tok_begin + CHUNK);
    // Each wavefront owns 8 groups of 16 keys.  All page-table lookups are issued first, then all key loads
    // (absent keys read row 0 and get scale 0), so that 4 KB per wavefront are in flight before the first MFMA.
    constexpr int STEPS = CHUNK / 64;
    const int bs = a.block_size, bs_shift = __builtin_ctz(bs);
    int page[STEPS], tk[STEPS];
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        tk[j] = min(tok_begin + wave * 16 + 64 * j + l16, tok_end - 1);
        const int pi = POW2 ? tk[j] >> bs_shift : tk[j] / bs;
        page[j] = a.block_table[(int64_t)bi * a.bt_stride + pi];
    }
    int64_t krow[STEPS];
    bool present[STEPS];
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const int in_page = POW2 ? tk[j] & (bs - 1) : tk[j] % bs;
        present[j] = tok_begin + wave * 16 + 64 * j + l16 < tok_end && page[j] >= 0 && page[j] < a.n_blocks;
        krow[j] = present[j] ? (int64_t)page[j] * bs + in_page : 0;
    }
    i32x4 kf0[STEPS], kf1[STEPS];
    typename ScaleOf<F32>::raw ksb[STEPS];
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const int8_t* kp = a.k_cache + krow[j] * D + 16 * g;
        kf0[j] = *reinterpret_cast<const i32x4*>(kp);
        kf1[j] = *reinterpret_cast<const i32x4*>(kp + 64);
        ksb[j] = static_cast<const typename ScaleOf<F32>::raw*>(a.k_scale)[krow[j]];
    }
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const int tok = tok_begin + wave * 16 + 64 * j + l16;
        const bool ok = tok < tok_end;
#pragma unroll
        for (int s = 0; s < S1; ++s) {
            f16x8 y[2];
#pragma unroll
            for (int hb = 0; hb < 4; ++hb) {
                i32x4 acc = {0, 0, 0, 0};
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qf[s][hb][0], kf0[j], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qf[s][hb][1], kf1[j], acc, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    y[hb >> 1][4 * (hb & 1) + r] = (_Float16)((float)max(acc[r], 0) * (1.0f / 2048.0f));
            }
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
            sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[s][0], y[0], sum, 0, 0, 0);
            sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[s][1], y[1], sum, 0, 0, 0);
            // row 0 of the result: register 0 of lanes 0..15, one key each
            const int eff = L - (a.s1 - 1 - (sgrp * S1 + s));
            if (ok && g == 0) {
                const float sc = sum[0] * (present[j] ? ScaleOf<F32>::f32(ksb[j]) : 0.f);
                a.scores[(int64_t)(row0 + s) * a.score_stride + tok] = sc;
                if (a.use_hist && tok < eff) atomicAdd(&hist[0][s][score_bin(score_key(sc))], 1u);
            }
        }
    }
    } // pass
    __syncthreads();
    if (a.use_hist) flush_span_hist<S1>(a, hist, row0, (int)blockIdx.x, 1, tid);
}

// relu(a) * 2^-11 and relu(b) * 2^-11, each rounded once to fp16, packed (a in the low half).  The int32 sums arrive
// biased: the MFMA accumulators start at SCORE_BIAS = the bit pattern of the float 1.5 * 2^23, and since |a| < 2^21 the
// accumulator's bits, read as a float, are exactly 12582912 + a - the integer-to-float conversion costs nothing.  One
// fused multiply-add takes the bias off and scales (exact in fp32: a * 2^-11 has at most 21 significant bits); relu
// commutes with the rounding to fp16, so it is taken on the packed pair.  (Written in plain C on purpose: the
// compiler's hazard recognizer does not look inside inline assembly, and a hand-placed VALU write into a register that
// an MFMA is still writing goes wrong.)
constexpr int SCORE_BIAS = 0x4B400000;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t relu_scale_pack(int a, int b)
{
    f16x2 v = {(_Float16)__builtin_fmaf(__int_as_float(a), 0x1p-11f, -6144.0f),
               (_Float16)__builtin_fmaf(__int_as_float(b), 0x1p-11f, -6144.0f)};
    const f16x2 z = {(_Float16)0.f, (_Float16)0.f};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(v, z));
}

// Score kernel for block sizes that are multiples of 128: a wavefront owns 128 consecutive keys of one page per pass
// (one page-table entry; the entries of all its passes are fetched up front with one load, lane p holding pass p's).  Keys
// travel 64 at a time (8 KB, eight whole 128-byte rows to an instruction) through registers into the wavefront's own LDS,
// from where they are read in operand layout while the next 64 are on the way.  Results are filed 64 at a time: w_scale sits
// in every row of the head-sum operand, so every lane group holds the 16 scores of a key group and lane group g keeps those
// of key group g - after four key groups lane l holds the score of key l of the 64, next to that key's scale (loaded with one
// 128-byte instruction per 64 keys).
// A workgroup takes `passes` passes of 512 keys: PPASSES, pick_passes' choice for full page tables, or fewer, by the lengths, while
// there would be fewer than SCORE_GROUPS_MIN workgroups (where the selection needs histograms, no fewer than fill a slot).  Short
// contexts under wide tables would otherwise be few long workgroups (32 sequences of 8192 keys under 1024 columns: 24.7 us
// with spans of 4096 keys, 14.7 with 2048).
// MAY: loads past the caches' retention, where the batch's keys do not fit the last-level cache - which needs the whole-row
// loads: taken in operand layout, a row is two loads of half a cache line, and a line that is not kept in between is fetched
// twice (32 x 64 K keys, 272 MB: 56.8 us in operand layout, 65.0 with non-temporal loads; 57.8 and 52.7 this way).
constexpr int SCAN_SEQS = 256; // sequences whose lengths a wavefront looks at
template <int S1, bool F32, int PPASSES, bool MAY>
__global__ __launch_bounds__(256, S1 == 1 ? 3 : 2) void indexer_score_paged_kernel(IndexerArgs a)
{
    constexpr int SLOT = PPASSES < PASSES ? PPASSES : PASSES; // passes to a histogram slot
    __shared__ __align__(16) uint32_t hist[PPASSES / SLOT][S1][SBINS];
    __shared__ __align__(16) float s_sc[S1][CHUNK * PPASSES]; // the workgroup's scores, written out in one burst at the end
    __shared__ __align__(16) _Float16 s_w[S1][64];
    __shared__ __align__(16) uint8_t s_keys[4][64 * D];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const int sgrp = blockIdx.z;
    const int bs = a.block_size;
    // The (sequence, span of 512 passes keys) of this workgroup.  The workgroups that have work should be the first ones of the
    // launch order, so that they spread evenly over the CUs: workgroup w (its place in launch order, sequence-major) takes the
    // w-th span that holds keys.  Every wavefront finds it on its own from the sequence lengths (lane l holds sequences l, l +
    // 64, ..; a wavefront prefix sum of the spans per sequence), which are fetched together with the page-table entries of the
    // grid place; only if the span is another one (ragged lengths, other passes) are those fetched again.  Batches beyond
    // SCAN_SEQS sequences keep the grid place, the spans of a sequence turned by its number: workgroups go to the eight
    // dies in turn, and the first spans of all sequences, often the only ones with keys, would all meet on the same few (300
    // sequences of 3000 .. 9000 keys under 1024 columns: 426 us).
    // Lane p takes the page-table entry of pass p and the sequence's first entry, and picks once the length is known:
    // it then holds the first cache row of pass p (-1: unmapped page); a pass past the end re-reads the sequence's
    // first page and is discarded.
    const bool balanced = a.b <= SCAN_SEQS;
    const uint32_t w = blockIdx.x + gridDim.x * blockIdx.y;
    int bi = min((int)blockIdx.y, a.b - 1), span = balanced ? (int)blockIdx.x : (int)((blockIdx.x + blockIdx.y) % gridDim.x);
    int passes = PPASSES, passes_log2 = __builtin_ctz(PPASSES);
    int lens[SCAN_SEQS / 64];
    // (unconditional loads, so that they travel with the ones below; of more sequences SCAN_SEQS evenly spaced ones)
#pragma unroll
    for (int j = 0; j < SCAN_SEQS / 64; ++j) {
        const int i = lane + 64 * j;
        lens[j] = a.act_seq[balanced ? min(i, a.b - 1) : (int)((int64_t)i * a.b / SCAN_SEQS)];
    }
    int pg_mine, pg_first, L, mytok;
    auto fetch = [&]() {
        mytok = span * (CHUNK * passes) + wave * 128 + (lane < passes ? lane : 0) * CHUNK;
        const int32_t* bt = a.block_table + (int64_t)bi * a.bt_stride;
        pg_mine = bt[min(mytok / bs, a.bt_stride - 1)];
        pg_first = bt[0];
        L = min(a.act_seq[bi], a.max_ctx); // keys past the page table's reach do not exist
    };
    fetch();
    bool past_caches = false;
    if constexpr (PPASSES > 1 || MAY) {
        uint32_t groups = 0; // of one pass
#pragma unroll
        for (int j = 0; j < SCAN_SEQS / 64; ++j) {
            lens[j] = lane + 64 * j < a.b ? max(min(lens[j], a.max_ctx), 0) : 0;
            groups += (uint32_t)((lens[j] + CHUNK - 1) / CHUNK);
        }
        groups = (uint32_t)__builtin_amdgcn_readlane((int)wave_prefix_sum(groups), 63);
        if (balanced && PPASSES > 1) {
            while (passes > a.min_passes && (uint64_t)groups * (uint32_t)(a.s1 / S1) < (uint32_t)passes * SCORE_GROUPS_MIN) {
                passes >>= 1;
                --passes_log2;
            }
        }
        if constexpr (MAY) past_caches = (float)groups * (balanced ? 1.f : (float)a.b / SCAN_SEQS) * (CHUNK * D) > SCORE_CACHED;
    }
    if (balanced) {
        uint32_t base = 0;
        int fseq = -1, fspan = 0;
#pragma unroll
        for (int j = 0; j < SCAN_SEQS / 64; ++j) {
            if (64 * j >= a.b) break;
            const int len = min(lens[j], a.max_ctx);
            const uint32_t cnt = (lane + 64 * j < a.b && len > 0) ? ((uint32_t)((len - 1) / CHUNK) >> passes_log2) + 1u : 0u;
            const uint32_t incl = wave_prefix_sum(cnt), excl = incl - cnt;
            const uint64_t hit = __ballot(w >= base + excl && w < base + incl); // at most one lane, in one round
            if (hit != 0ull && fseq < 0) {
                const int l = __builtin_ctzll(hit);
                fseq = 64 * j + l;
                fspan = (int)(w - base - (uint32_t)__builtin_amdgcn_readlane((int)excl, l));
            }
            base += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
        if (fseq < 0) return; // more workgroups than spans with keys
        if (fseq != bi || fspan != span || passes != PPASSES) {
            bi = fseq;
            span = fspan;
            fetch();
        }
    }
    const int span_keys = CHUNK * passes;
    if (span * span_keys >= L) return;
    const int row0 = bi * a.s1 + sgrp * S1;
    const int wtok = span * span_keys + wave * 128; // first key of this wave's pass 0
    int64_t myrow;
    {
        const int tc = mytok < L ? mytok : 0;
        const int pg = mytok < L ? pg_mine : pg_first;
        myrow = (pg >= 0 && pg < a.n_blocks) ? (int64_t)pg * bs + tc % bs : -1;
    }
    auto pass_row = [&](int pass) {
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)myrow, pass);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(myrow >> 32), pass);
        return (int64_t)(((uint64_t)hi << 32) | lo);
    };

    // past: loads past the caches; halves: passes of 64 keys per wavefront (known to the compiler for PPASSES: 2 to 6 % faster)
    auto score = [&](auto past, auto halves) __attribute__((always_inline)) {
    // 64 keys on the way: load i holds chunk lane % 8 of key 8 i + lane / 8; in LDS the 16-byte chunks of a key are XOR-ed with
    // the key, so that both the row writes and the operand reads fall on all banks
    i32x4 raw[8];
    typename ScaleOf<F32>::raw ksc_next;
    auto load_half = [&](int hh) {
        const int64_t r = pass_row(hh >> 1);
        const int64_t rb = r < 0 ? 0 : r;
        const int8_t* kp = a.k_cache + (rb + 64 * (hh & 1)) * D + 16 * lane;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const i32x4* p = reinterpret_cast<const i32x4*>(kp + i * 8 * D);
            raw[i] = decltype(past)::value ? __builtin_nontemporal_load(p) : *p;
        }
        ksc_next = static_cast<const typename ScaleOf<F32>::raw*>(a.k_scale)[rb + 64 * (hh & 1) + lane];
    };
    uint8_t* keys = s_keys[wave];
    uint8_t* key_dst = keys + (lane >> 3) * D + (((lane & 7) ^ (lane >> 3)) << 4);
    const uint8_t* key_src0 = keys + l16 * D + ((g ^ (l16 & 7)) << 4);
    const uint8_t* key_src1 = keys + l16 * D + (((g + 4) ^ (l16 & 7)) << 4);
    // The query and its scales go through LDS too, whole rows to an instruction and once to a workgroup.  (Taken by every wavefront
    // in operand layout, neighbouring lanes in different rows, the 8 S1 loads of the query alone kept the load path busy for most of the
    // 4.5 us before the first product: now 3.0 with two query tokens.  13 sequences of 1000 .. 40000 keys, two query tokens, through
    // selection and attention 63.9 -> 59.9 us; 64 of them 153 -> 146.7; one sequence of 4096, a layer 62.1 -> 60.4.)
    // They are requested first, then the keys and their scales (memory operations complete in order).  Every memory operation from
    // here on is unconditional, so that the number in flight is the same on every path into the loop and the waits can count them.
    i32x4 qraw[2 * S1];
#pragma unroll
    for (int i = 0; i < 2 * S1; ++i)
        qraw[i] = *reinterpret_cast<const i32x4*>(a.q + ((int64_t)row0 * a.nh + (wave * 2 * S1 + i) * 8) * D + 16 * lane);
    // one head's w_scale to a lane, of query token wave % S1
    const int64_t w_at = (int64_t)(row0 + wave % S1) * a.nh + lane;
    const uint16_t w_raw = a.weights[w_at];
    const typename ScaleOf<F32>::raw qs_raw = static_cast<const typename ScaleOf<F32>::raw*>(a.q_scale)[w_at];
    load_half(0);
    for (int i = tid; i < PPASSES / SLOT * S1 * SBINS; i += 256) (&hist[0][0][0])[i] = 0;
    // (row r of s_keys: head r % 64 of query token r / 64; the chunks XOR-ed as the keys')
#pragma unroll
    for (int i = 0; i < 2 * S1; ++i)
        *reinterpret_cast<i32x4*>(&s_keys[0][0] + (wave * 2 * S1 + i) * 8 * D + (lane >> 3) * D + (((lane & 7) ^ (lane >> 3)) << 4)) = qraw[i];
    s_w[wave % S1][lane] = w_scale_of<F32>(qs_raw, w_raw);
    __syncthreads();
    // fp16 A fragments of the head sum, the same in every row: k-slot (g, e) of MFMA mm is head
    // 32*mm + 16*(e/4) + 4*g + e%4 - the head whose int32 result this lane group holds in that slot; the value is
    // q_scale * weights in one fp16 rounding
    f16x8 wa[S1][2];
#pragma unroll
    for (int s = 0; s < S1; ++s)
#pragma unroll
        for (int mm = 0; mm < 2; ++mm) {
            typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
            const _Float16* wp = &s_w[s][32 * mm + 4 * g];
            wa[s][mm] = __builtin_shufflevector(*reinterpret_cast<const f16x4*>(wp), *reinterpret_cast<const f16x4*>(wp + 16), 0, 1, 2, 3, 4, 5, 6, 7);
        }
    // int8 A fragments: head hb*16 + l16, bytes 64*ks + 16*g .. +15
    i32x4 qf[S1][4][2];
#pragma unroll
    for (int s = 0; s < S1; ++s)
#pragma unroll
        for (int hb = 0; hb < 4; ++hb) {
            const uint8_t* qp = &s_keys[0][0] + (s * 64 + hb * 16 + l16) * D;
            qf[s][hb][0] = *reinterpret_cast<const i32x4*>(qp + ((g ^ (l16 & 7)) << 4));
            qf[s][hb][1] = *reinterpret_cast<const i32x4*>(qp + (((g + 4) ^ (l16 & 7)) << 4));
        }
    __syncthreads();

    auto compute_half = [&](int hh, typename ScaleOf<F32>::raw ksc) {
        float res[S1];
#pragma unroll
        for (int s = 0; s < S1; ++s) res[s] = 0.f;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const i32x4 kf0 = *reinterpret_cast<const i32x4*>(key_src0 + jj * 16 * D);
            const i32x4 kf1 = *reinterpret_cast<const i32x4*>(key_src1 + jj * 16 * D);
#pragma unroll
            for (int s = 0; s < S1; ++s) {
                u32x4 y[2];
#pragma unroll
                for (int hb = 0; hb < 4; ++hb) {
                    i32x4 acc = {SCORE_BIAS, SCORE_BIAS, SCORE_BIAS, SCORE_BIAS};
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qf[s][hb][0], kf0, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qf[s][hb][1], kf1, acc, 0, 0, 0);
                    y[hb >> 1][2 * (hb & 1)] = relu_scale_pack(acc[0], acc[1]);
                    y[hb >> 1][2 * (hb & 1) + 1] = relu_scale_pack(acc[2], acc[3]);
                }
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
                sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[s][0], __builtin_bit_cast(f16x8, y[0]), sum, 0, 0, 0);
                sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[s][1], __builtin_bit_cast(f16x8, y[1]), sum, 0, 0, 0);
                res[s] = jj == g ? sum[0] : res[s];
            }
        }
        const int tok = wtok + (hh >> 1) * CHUNK + 64 * (hh & 1) + lane;
        const float ks = pass_row(hh >> 1) >= 0 ? ScaleOf<F32>::f32(ksc) : 0.f;
#pragma unroll
        for (int s = 0; s < S1; ++s) {
            const float sc = res[s] * ks;
            s_sc[s][tok - span * span_keys] = sc;
            const int eff = L - (a.s1 - 1 - (sgrp * S1 + s));
            if (a.use_hist && tok < eff) atomicAdd(&hist[hh / (2 * SLOT)][s][score_bin(score_key(sc))], 1u);
        }
    };

    // (past the end the last half is loaded again, a cache hit whose data is never used, so that the loads stay unconditional)
    for (int hh = 0; hh < halves; ++hh) {
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<i32x4*>(key_dst + i * 8 * D) = raw[i]; // (8 keys on: the same XOR)
        const typename ScaleOf<F32>::raw ksc = ksc_next;
        load_half(hh + 1 < halves ? hh + 1 : halves - 1);
        compute_half(hh, ksc);
    }
    };
    if (__builtin_expect(passes != PPASSES, 0)) {
        score(std::false_type{}, 2 * passes);
    } else if (past_caches) {
        asm volatile("; past the caches"); // (else the compiler merges the two sides' first loads, into plain ones)
        score(std::true_type{}, std::integral_constant<int, 2 * PPASSES>{});
    } else {
        score(std::false_type{}, std::integral_constant<int, 2 * PPASSES>{});
    }
    __syncthreads();
    // one contiguous 8 KB write per query token (256-byte stores from inside the loop, between the key loads, cost
    // 2 us more); score rows are padded to whole workgroup spans, so no bounds check
#pragma unroll
    for (int s = 0; s < S1; ++s) {
        float* dst = a.scores + (int64_t)(row0 + s) * a.score_stride + (int64_t)span * span_keys;
#pragma unroll
        for (int i = 0; i < (CHUNK * PPASSES + 1023) / 1024; ++i)
            if (4 * (tid + 256 * i) < span_keys)
                *reinterpret_cast<f32x4*>(dst + 4 * (tid + 256 * i)) = *reinterpret_cast<const f32x4*>(&s_sc[s][4 * (tid + 256 * i)]);
    }
    if (a.use_hist) flush_span_hist<S1>(a, hist, row0, span * passes / SLOT, max(passes / SLOT, 1), tid);
}

__global__ void indexer_fill_kernel(int32_t* p, int n, int32_t v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// inclusive suffix sum over a wavefront (lane l gets the sum of v[l .. 63]); all 64 lanes active
__device__ __forceinline__ uint32_t wave_suffix_sum(uint32_t v)
{
    const uint32_t incl = wave_prefix_sum(v);
    return (uint32_t)__builtin_amdgcn_readlane((int)incl, 63) - incl + v;
}

// block-wide inclusive suffix sum (lane t gets sum of v[t .. nthreads-1]); tmp holds one word per wavefront
template <int NWAVES>
__device__ __forceinline__ uint32_t block_suffix_sum(uint32_t v, uint32_t* tmp)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    {
        // suffix = wavefront total - exclusive prefix (unsigned arithmetic, exact)
        const uint32_t incl = wave_prefix_sum(v);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        v = total - incl + v;
    }
    __syncthreads();
    if (lane == 0) tmp[wave] = v;
    __syncthreads();
    // the totals of the wavefronts behind this one: one read, summed up between the lanes (up to 15 reads in a row took three times as
    // long as all the rest)
    static_assert(NWAVES == 4 || NWAVES == 16, "sums over lanes of a row that repeat");
    uint32_t add = tmp[lane & (NWAVES - 1)];
    add = (lane & (NWAVES - 1)) > wave ? add : 0u;
    if constexpr (NWAVES == 16) {
        add += dpp_from<0x128, 0xf>(add, 0u); // row_ror:8, 4
        add += dpp_from<0x124, 0xf>(add, 0u);
    }
    add += dpp_from<0x122, 0xf>(add, 0u); // row_ror:2, 1
    add += dpp_from<0x121, 0xf>(add, 0u);
    return v + add;
}

// Valid length of query token `row`'s score row: the sequence's length, cut to what the page table can address
// (the score kernels write no score beyond that), less the query tokens that come after this one.
__device__ __forceinline__ int row_length(const int32_t* act_seq, int row, int s1, int max_ctx)
{
    const int bi = row / s1, si = row - bi * s1;
    return max(min(act_seq[bi], max_ctx) - (s1 - 1 - si), 0);
}

// grid (chunks of SEL_CHUNK scores, query tokens), 256 lanes
__global__ __launch_bounds__(256) void indexer_select_kernel(IndexerArgs a)
{
    __shared__ uint32_t tmp[4];
    __shared__ uint32_t s_bin, s_base_gt, s_base_tie;
    __shared__ __align__(16) uint32_t s_hist[4][SBINS];
    const int tid = threadIdx.x, row = blockIdx.y;
    const int i_begin = blockIdx.x * SEL_CHUNK;
    // everything this workgroup reads is requested at once - the row's length, the histograms of the first GROUP spans
    // and the workgroup's 16 scores per lane (addresses clamped to the padded row) - one round trip.  The histograms
    // are read as they lie in memory, 16 bytes per lane: lane l takes bins 8 (l % 32) .. + 7 of spans l / 32,
    // l / 32 + 8, ..  A slot of a span without keys was never written: it is requested all the same (workspace
    // memory) and left out of the sum once the length is known.
    constexpr int GROUP = 32;
    const int sg = tid >> 5, oct = tid & 31;
    const uint16_t* sh = a.span_hist + (int64_t)row * a.pchunks * SBINS + 8 * oct;
    u32x4 cv[GROUP / 8];
#pragma unroll
    for (int j = 0; j < GROUP / 8; ++j) cv[j] = *reinterpret_cast<const u32x4*>(sh + (int64_t)min(sg + 8 * j, a.pchunks - 1) * SBINS);
    const float* x = a.scores + (int64_t)row * a.score_stride;
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const f32x4*>(x + min(i_begin + 4 * (j * 256 + tid), a.score_stride - 4));
    const int bi = row / a.s1;
    const int len = min(a.act_seq[bi], a.max_ctx);
    const int n = max(len - (a.s1 - 1 - (row - bi * a.s1)), 0);
    // (a workgroup past the row's end leaves further down, behind the first use of what was requested above: an exit
    // here would let the compiler move those requests behind the wait for the length - two round trips instead of one)
    const int slot_keys = CHUNK * a.min_passes;
    const int nsp = min((len + slot_keys - 1) / slot_keys, a.pchunks); // slots whose workgroup ran
    if (tid == 0) s_bin = 0xffffffffu; // n <= k: no threshold bin, everything is a winner

    uint32_t acc[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    for (int g0 = 0; g0 < nsp; g0 += GROUP) { // (one trip but for contexts beyond GROUP spans; block-uniform)
        if (g0 > 0) {
#pragma unroll
            for (int j = 0; j < GROUP / 8; ++j)
                cv[j] = *reinterpret_cast<const u32x4*>(sh + (int64_t)min(g0 + sg + 8 * j, a.pchunks - 1) * SBINS);
        }
#pragma unroll
        for (int j = 0; j < GROUP / 8; ++j) {
            const bool in = g0 + sg + 8 * j < nsp;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                acc[2 * c] += in ? cv[j][c] & 0xffffu : 0u;
                acc[2 * c + 1] += in ? cv[j][c] >> 16 : 0u;
            }
        }
    }
    // the two span groups of a wavefront (lanes l and l + 32 hold the same bins), then the four wavefronts through LDS
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const auto sw = __builtin_amdgcn_permlane32_swap(acc[c], acc[c], false, false);
        acc[c] = (uint32_t)sw[0] + (uint32_t)sw[1];
    }
    if ((tid & 32) == 0) {
        uint32_t* dst = &s_hist[tid >> 6][8 * oct];
        *reinterpret_cast<u32x4*>(dst) = u32x4{acc[0], acc[1], acc[2], acc[3]};
        *reinterpret_cast<u32x4*>(dst + 4) = u32x4{acc[4], acc[5], acc[6], acc[7]};
    }
    __syncthreads();
    if (i_begin >= n) return;
    // bin of the k-th largest key: lane t owns bin t
    const uint32_t own = s_hist[0][tid] + s_hist[1][tid] + s_hist[2][tid] + s_hist[3][tid];
    const uint32_t k = (uint32_t)a.k;
    {
        const uint32_t above = block_suffix_sum<4>(own, tmp) - own; // elements in the bins above
        if (above < k && k <= above + own) s_bin = (uint32_t)tid;
    }
    __syncthreads();
    const uint32_t bin = s_bin;

    // file this workgroup's scores: 16 per lane.  A score's side of the threshold bin is read off its key: winners lie
    // above the bin's largest key, ties between its smallest and largest.  Without a threshold bin every key is a winner.
    uint32_t key_lo = 0u, key_hi = 0u;
    const bool all_win = bin == 0xffffffffu;
    if (!all_win) score_bin_range(bin, key_lo, key_hi);
    uint32_t key[16];
    uint32_t c_gt = 0, c_tie = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int i = i_begin + 4 * (j * 256 + tid) + c;
            const uint32_t u = score_key(v[j][c]);
            key[4 * j + c] = u;
            const bool in = i < n;
            c_gt += in && (all_win || u > key_hi) ? 1u : 0u;
            c_tie += in && !all_win && u >= key_lo && u <= key_hi ? 1u : 0u;
        }
    const uint32_t packed = block_suffix_sum<4>(c_gt | (c_tie << 16), tmp);
    if (tid == 0) {
        uint32_t* cnt = a.counters + (int64_t)row * 4;
        s_base_gt = atomicAdd(cnt, packed & 0xffffu);
        s_base_tie = atomicAdd(cnt + 1, packed >> 16);
    }
    __syncthreads();
    uint32_t p_gt = s_base_gt + (packed & 0xffffu) - c_gt;
    uint32_t p_tie = s_base_tie + (packed >> 16) - c_tie;
    uint64_t* winners = a.winners + (int64_t)row * MAX_K;
    uint64_t* ties = a.ties + (int64_t)row * TIE_CAP;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int i = i_begin + 4 * (j * 256 + tid) + c;
            const uint32_t u = key[4 * j + c];
            const bool in = i < n;
            const bool gt = in && (all_win || u > key_hi), tie = in && !all_win && u >= key_lo && u <= key_hi;
            // (one store per element, to whichever list takes it)
            uint64_t* dst = gt ? winners + p_gt : ties + p_tie;
            if ((gt && p_gt < MAX_K) || (tie && p_tie < TIE_CAP)) *dst = make_cand(u, i);
            p_gt += gt ? 1u : 0u;
            p_tie += tie ? 1u : 0u;
        }
}

// Radix-select the `need` largest of the 64-bit words f enumerates (all share the bits above `top`), top-down
// in digits of 11 bits; every selected word is handed to emit().  Words are distinct, so the walk ends with a
// bin that is taken whole.  Workgroup of 1024 lanes; hist has 2048 words, tmp 16.
template <class Each, class Emit>
__device__ __forceinline__ void radix_select64(Each&& for_each, Emit&& emit, uint32_t need, int top, uint32_t* hist,
                                               uint32_t* tmp, uint32_t* s_bin, uint32_t* s_krem, uint32_t* s_cnt)
{
    const int tid = threadIdx.x;
    uint64_t prefix = 0, known = 0; // bits fixed so far and their mask
    while (need > 0 && top > 0) {
        const int bits = top >= 11 ? 11 : top;
        const int shift = top - bits;
        const uint64_t dmask = (1ull << bits) - 1ull;
        hist[tid] = 0;
        hist[tid + 1024] = 0;
        __syncthreads();
        for_each([&](uint64_t w) {
            if ((w & known) == prefix) atomicAdd(&hist[(uint32_t)((w >> shift) & dmask)], 1u);
        });
        __syncthreads();
        const uint32_t h_lo = hist[2 * tid], h_hi = hist[2 * tid + 1]; // lane t owns bins 2t and 2t+1
        const uint32_t incl = block_suffix_sum<16>(h_lo + h_hi, tmp);
        const uint32_t above_hi = incl - h_lo - h_hi, above_lo = above_hi + h_hi;
        if (above_hi < need && need <= above_hi + h_hi) {
            *s_bin = 2 * tid + 1;
            *s_krem = need - above_hi;
            *s_cnt = h_hi;
        } else if (above_lo < need && need <= above_lo + h_lo) {
            *s_bin = 2 * tid;
            *s_krem = need - above_lo;
            *s_cnt = h_lo;
        }
        __syncthreads();
        const uint64_t b = *s_bin;
        const uint32_t krem = *s_krem, cnt = *s_cnt;
        // everything in the bins above b is selected; bin b whole if it is exactly what is missing
        const bool whole = cnt == krem;
        for_each([&](uint64_t w) {
            if ((w & known) != prefix) return;
            const uint64_t d = (w >> shift) & dmask;
            if (d > b || (whole && d == b)) emit(w);
        });
        __syncthreads();
        if (whole) return;
        prefix |= b << shift;
        known |= dmask << shift;
        need = krem;
        top = shift;
    }
}

// A word's group for ordering: a non-decreasing function of its key with values 0 .. 2^BITS - 1.  `kind` 0 cuts the scores'
// range into equal steps (rounding is monotone: neither the difference nor the product turns two scores around), kind 1
// the range of their ordered keys - steps in proportion to the magnitude.
__device__ __forceinline__ float key_to_score(uint32_t key) { return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key); }
template <int BITS>
struct KeyGroups {
    static constexpr uint32_t LAST = (1u << BITS) - 1u;
    uint32_t kmin, kmax;
    float fmin, per;
    int shift;
    bool linear_ok; // the scores' range is finite and not empty
    __device__ __forceinline__ KeyGroups(uint32_t lo, uint32_t hi) : kmin(lo), kmax(hi)
    {
        fmin = key_to_score(lo);
        const float span = key_to_score(hi) - fmin;
        per = (float)LAST / span;
        shift = max(0, 32 - BITS - (int)__builtin_clz((hi - lo) | 1u));
        linear_ok = span > 0.f && span < __builtin_inff() && per < __builtin_inff();
    }
    __device__ __forceinline__ uint32_t of(uint32_t key, int kind) const
    {
        return kind == 0 ? min((uint32_t)((key_to_score(key) - fmin) * per), LAST) : (key - kmin) >> shift;
    }
};

// Ordering: word w[h] of a lane is real if tid + 1024 h < m (m <= 1024 PER); calls write(rank, word) for the k first of
// them in descending word order.  kmin / kmax bound the words' keys.  The words are grouped by KeyGroups, so a counting pass
// (histogram, suffix scan, scatter) puts every word within a few slots of its place - and then ranked inside their group by
// direct comparison.  Equal steps of the score come first: bell-shaped scores leave a few words in a step wherever the
// selection ends.  If those crowd (more than GROUP_CAP words in one), equal steps of the keys; if these do too (heavily tied
// scores), a bitonic sort.  (Steps of the keys alone crowd near zero, and a row whose selection reaches scores of both signs
// then paid for the sort: 18 us against 8.)
// 4096 groups: where the selection ends, which is where the scores of a bell are densest, 2048 hold 7 words on the average and up to 15
// (8192: as many ticks won in the comparisons as lost in the scan).
// Workgroup of 1024 lanes; buf has 1024 PER words, start ORDER_GROUPS (16-byte aligned), tmp 16.
constexpr uint32_t GROUP_CAP = 64;
constexpr int ORDER_BITS = 12, ORDER_GROUPS = 1 << ORDER_BITS;
template <int PER, class Write>
__device__ __forceinline__ void order_words(const uint64_t (&w)[PER], uint32_t m, uint32_t kmin, uint32_t kmax, uint64_t* buf, uint32_t* start,
                                            uint32_t* tmp, uint32_t* s_flag, int k, Write&& write)
{
    const int tid = threadIdx.x;
    const KeyGroups<ORDER_BITS> groups(kmin, kmax);
    uint32_t bin[PER];
    for (int kind = groups.linear_ok ? 0 : 1; kind < 2; ++kind) { // (block-uniform)
        __syncthreads();
        reinterpret_cast<u32x4*>(start)[tid] = u32x4{0u, 0u, 0u, 0u};
        if (tid == 0) *s_flag = 0;
        __syncthreads();
#pragma unroll
        for (int h = 0; h < PER; ++h) {
            bin[h] = groups.of((uint32_t)(w[h] >> 32), kind);
            if ((uint32_t)(tid + 1024 * h) < m) atomicAdd(&start[bin[h]], 1u);
        }
        __syncthreads();
        {
            const u32x4 c = reinterpret_cast<const u32x4*>(start)[tid]; // lane t owns groups 4 t .. 4 t + 3
            if (max(max(c[0], c[1]), max(c[2], c[3])) > GROUP_CAP) *s_flag = 1;
            const uint32_t incl = block_suffix_sum<16>((c[0] + c[1]) + (c[2] + c[3]), tmp);
            // slots taken by the higher groups
            const uint32_t s0 = incl - c[0], s1 = s0 - c[1], s2 = s1 - c[2];
            reinterpret_cast<u32x4*>(start)[tid] = u32x4{s0, s1, s2, s2 - c[3]};
        }
        __syncthreads();
        if (*s_flag == 0) {
#pragma unroll
            for (int h = 0; h < PER; ++h)
                if ((uint32_t)(tid + 1024 * h) < m) buf[atomicAdd(&start[bin[h]], 1u)] = w[h]; // (start ends up as the group's end)
            __syncthreads();
            // By place now, so that neighbouring lanes compare neighbouring words and write next to each other.  (A word's own lane
            // went all over LDS and the output for it: 5 K of the 32 K ticks of a row of 20000, this way 2 K.)
#pragma unroll
            for (int h = 0; h < PER; ++h) {
                const uint32_t i = (uint32_t)(tid + 1024 * h);
                if (i >= m) break;
                const uint64_t x = buf[i];
                const uint32_t b = groups.of((uint32_t)(x >> 32), kind);
                const uint32_t s0 = b + 1 < ORDER_GROUPS ? start[b + 1] : 0u, end = start[b]; // (a group begins where the next higher one ends)
                if ((int)s0 >= k) break;
                uint32_t rank = s0;
                for (uint32_t j = s0; j < end; ++j) rank += buf[j] > x ? 1u : 0u;
                if ((int)rank < k) write((int)rank, x);
            }
            return;
        }
    }
    // bitonic sort, descending, two words per lane and 2048 words.  A compare-exchange step of stride <= 64 stays inside
    // the 128 words owned by one wavefront (lane i of wave w handles the pair (128w + 2i - i%stride, + stride)),
    // so only the steps of stride >= 128 need a workgroup barrier; the others rely on LDS operations of one
    // wavefront completing in order.  The wait for them in front of the barrier that follows is written out: they come to it over
    // the loops' back edges, and left to __syncthreads the compiler drops it.
    __syncthreads();
#pragma unroll
    for (int h = 0; h < PER; ++h) buf[tid + 1024 * h] = (uint32_t)(tid + 1024 * h) < m ? w[h] : 0ull;
    __syncthreads();
    for (int size = 2; size <= 1024 * PER; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            if (stride >= 128) {
                __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
                __syncthreads();
            }
#pragma unroll
            for (int q = 0; q < PER / 2; ++q) {
                const int i = tid + 1024 * q;
                const int pos = 2 * i - (i & (stride - 1)); // lower index of the pair
                const bool desc = (pos & size) == 0;
                const uint64_t lo = buf[pos], hi = buf[pos + stride];
                if ((lo < hi) == desc) {
                    buf[pos] = hi;
                    buf[pos + stride] = lo;
                }
            }
            if (stride >= 128) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
    }
    __syncthreads();
    for (int j = tid; j < min((int)m, k); j += 1024) write(j, buf[j]);
}
__device__ __forceinline__ int word_index(uint64_t w) { return (int)(0xffffffffu - (uint32_t)(w & 0xffffffffull)); }

// smallest and largest key of the block, into (and out of) tmp[14] and tmp[15], which hold ~0 and 0 before; 1024 lanes
__device__ __forceinline__ void block_key_range(uint32_t& kmin, uint32_t& kmax, uint32_t* tmp)
{
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&tmp[14], kmin);
        atomicMax(&tmp[15], kmax);
    }
    __syncthreads();
    kmin = tmp[14];
    kmax = tmp[15];
}

__global__ __launch_bounds__(1024) void indexer_topk_kernel(IndexerArgs a)
{
    __shared__ uint32_t hist[NBINS];
    __shared__ uint64_t cand[MAX_K];
    __shared__ __align__(16) uint64_t tie[TIE_CAP];
    __shared__ uint32_t tmp[16];
    __shared__ uint32_t s_bin, s_krem, s_cnt, s_out;

    const int tid = threadIdx.x, row = blockIdx.x;
    // the winners and the first 2048 ties are requested together with the counts that say how many of them are real
    // (the lists are workspace memory: reading past their fill is harmless), one round trip instead of three
    const uint64_t* wsrc = a.winners + (int64_t)row * MAX_K;
    const uint64_t* tsrc = a.ties + (int64_t)row * TIE_CAP;
    static_assert(MAX_K == 2048 && TIE_CAP >= 2048, "two winners and two early ties per lane");
    const uint64_t w0 = wsrc[tid], w1 = wsrc[tid + 1024];
    const uint64_t t0 = tsrc[tid], t1 = tsrc[tid + 1024];
    const int n = row_length(a.act_seq, row, a.s1, a.max_ctx);
    const int k = a.k;
    // (the counters of a query token are cleared by its sequence's first score workgroup: a sequence without keys has none)
    const uint32_t c_gt = a.counters[(int64_t)row * 4], c_tie = a.counters[(int64_t)row * 4 + 1];
    const uint32_t n_gt = n > 0 ? min(c_gt, (uint32_t)MAX_K) : 0u;
    const uint32_t n_tie = n > 0 ? c_tie : 0u;
    const uint32_t need = (uint32_t)min(n, k) - min(n_gt, (uint32_t)min(n, k));

    cand[tid] = tid < (int)n_gt ? w0 : 0ull;
    cand[tid + 1024] = tid + 1024 < (int)n_gt ? w1 : 0ull;
    tie[tid] = t0;
    tie[tid + 1024] = t1;
    if (tid == 0) s_out = n_gt;
    __syncthreads();
    auto emit = [&](uint64_t w) {
        const uint32_t p = atomicAdd(&s_out, 1u);
        if (p < MAX_K) cand[p] = w;
    };

    if (need > 0 && n_tie <= TIE_CAP) {
        // the usual case: the tie list (one histogram bin) fits in LDS
        if (n_tie > 2048) { // block-uniform
            for (int i = tid + 2048; i < (int)n_tie; i += 1024) tie[i] = tsrc[i];
            __syncthreads();
        }
        auto each = [&](auto&& f) {
            for (int i = tid; i < (int)n_tie; i += 1024) f(tie[i]);
        };
        if (score_bin_is_interior(score_bin((uint32_t)(tie[0] >> 32)))) {
            // The ties of an interior bin share their top 11 key bits.  They are counted by the next six (64 steps in
            // key order, one LDS counter each); a suffix scan of the 64 counts by one wavefront finds the step that holds
            // the last wanted tie.  Ties in the steps above it are taken, those inside it (a few dozen) are set aside
            // and ranked against each other.  (Against a digit of the radix select: 64 counters instead of 2048 to clear
            // and scan, and no second digit.)
            uint32_t* subc = hist + NBINS - SUBBINS; // (the far end of hist: its front holds the ties set aside)
            if (tid < SUBBINS) subc[tid] = 0u;
            if (tid == 0) { // (overwritten below by the lane whose step it is)
                s_bin = 0u;
                s_krem = need;
                s_cnt = 0xffffffffu;
                tmp[0] = 0u;
            }
            __syncthreads();
            each([&](uint64_t w) { atomicAdd(&subc[tie_sub_bin((uint32_t)(w >> 32))], 1u); });
            __syncthreads();
            if (tid < SUBBINS) {
                const uint32_t c_sub = subc[tid];
                const uint32_t above = wave_suffix_sum(c_sub) - c_sub;
                if (above < need && need <= above + c_sub) {
                    s_bin = (uint32_t)tid;
                    s_krem = need - above;
                    s_cnt = c_sub;
                }
            }
            __syncthreads();
            const uint32_t sb = s_bin, krem = s_krem, cnt = s_cnt;
            const bool whole = cnt == krem, small = cnt <= SUB_RANK_CAP;
            uint64_t* aside = reinterpret_cast<uint64_t*>(hist);
            each([&](uint64_t w) {
                const uint32_t d = tie_sub_bin((uint32_t)(w >> 32));
                if (d > sb || (whole && d == sb))
                    emit(w);
                else if (d == sb && small) {
                    const uint32_t p = atomicAdd(&tmp[0], 1u);
                    if (p < SUB_RANK_CAP) aside[p] = w;
                }
            });
            __syncthreads();
            if (!whole && small) {
                // (words are distinct: the rank of one among the others is the number of larger ones)
                if (tid < (int)cnt) {
                    const uint64_t w = aside[tid];
                    uint32_t larger = 0;
                    for (uint32_t j = 0; j < cnt; ++j) larger += aside[j] > w ? 1u : 0u;
                    if (larger < krem) emit(w);
                }
            } else if (!whole) {
                // a crowded step (heavily tied scores): digit by digit over its 15 remaining key bits and the index
                __syncthreads();
                auto each_in = [&](auto&& f) {
                    each([&](uint64_t w) {
                        if (tie_sub_bin((uint32_t)(w >> 32)) == sb) f(w);
                    });
                };
                radix_select64(each_in, emit, krem, 47, hist, tmp, &s_bin, &s_krem, &s_cnt);
            }
        } else {
            // a first or last bin (magnitudes outside the histogram's range): its keys need not share any bits
            radix_select64(each, emit, need, 64, hist, tmp, &s_bin, &s_krem, &s_cnt);
        }
    } else if (need > 0) {
        // overflowed tie list: select over the whole row instead (winners are found again, so start empty)
        if (tid == 0) s_out = 0;
        __syncthreads();
        const float* x = a.scores + (int64_t)row * a.score_stride;
        auto each = [&](auto&& f) {
            for (int i0 = 4 * tid; i0 < n; i0 += 4096) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(x + i0);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (i0 + c < n) f(make_cand(score_key(v[c]), i0 + c));
            }
        };
        radix_select64(each, emit, (uint32_t)min(n, k), 64, hist, tmp, &s_bin, &s_krem, &s_cnt);
    }
    __syncthreads();

    // the indices of the selected words, best first, then -1
    int32_t* out = a.topk_res + (int64_t)row * k;
    const uint32_t m = (uint32_t)min(n, k);
    for (int j = (int)m + tid; j < k; j += 1024) out[j] = -1;
    uint64_t w[2];
    uint32_t kmin = 0xffffffffu, kmax = 0u;
    if (tid == 0) {
        tmp[14] = 0xffffffffu;
        tmp[15] = 0u;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        w[h] = cand[tid + 1024 * h];
        if ((uint32_t)(tid + 1024 * h) < m) {
            kmin = min(kmin, (uint32_t)(w[h] >> 32));
            kmax = max(kmax, (uint32_t)(w[h] >> 32));
        }
    }
    block_key_range(kmin, kmax, tmp);
    order_words<2>(w, m, kmin, kmax, cand, reinterpret_cast<uint32_t*>(tie), tmp, &s_bin, k,
                   [&](int rank, uint64_t word) { out[rank] = word_index(word); });
}

// Standalone top-k of fp32 rows (pypto.topk: python/pypto/op/comparison.py:302-344; order of equal values - smaller
// index first - framework/src/interface/interpreter/calculator/calc_torch.cpp:2481-2494,2734-2749): values and int32
// indices of the k largest (or smallest) elements of every row, best first.  One workgroup of 1024 lanes per row.
// Words are (key << 32 | ~index) with the order-preserving key of the value (of its negation for the smallest),
// so descending word order is the rule above; -0 and +0 count as equal.
// topk_sort_kernel sorts the whole row in LDS: k beyond MAX_K (rows of up to TOPK_SORT_CAP elements), and rows of up to
// TOPK_SORT_SMALL elements, where its 28 steps are fewer than the fixed steps of the other kernel.
// topk_select_kernel serves everything else: it finds the k largest words and orders only those.
constexpr int TOPK_SORT_CAP = 8192;
constexpr int TOPK_SORT_SMALL = 128;

// bitonic sort of a[0 .. p), p a power of two <= TOPK_SORT_CAP, descending; 1024 lanes
__device__ __forceinline__ void bitonic_desc(uint64_t* a, int p)
{
    const int tid = threadIdx.x;
    for (int size = 2; size <= p; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            for (int i = tid; i < p / 2; i += 1024) {
                const int pos = 2 * i - (i & (stride - 1)); // lower index of the pair
                const bool desc = (pos & size) == 0;
                const uint64_t lo = a[pos], hi = a[pos + stride];
                if ((lo < hi) == desc) {
                    a[pos] = hi;
                    a[pos + stride] = lo;
                }
            }
        }
    __syncthreads();
}

__global__ __launch_bounds__(1024) void topk_sort_kernel(const float* __restrict__ x, float* __restrict__ values,
                                                         int32_t* __restrict__ indices, int n, int k, int largest)
{
    __shared__ uint64_t buf[TOPK_SORT_CAP];
    const int tid = threadIdx.x;
    const float* row = x + (int64_t)blockIdx.x * n;
    int p = 2;
    while (p < n) p <<= 1;
    // (every real word is > 0: its index part is)
    for (int i = tid; i < p; i += 1024) buf[i] = i < n ? make_cand(score_key(largest ? row[i] : -row[i]), i) : 0ull;
    bitonic_desc(buf, p);
    for (int j = tid; j < k; j += 1024) {
        const int i = word_index(buf[j]);
        indices[(int64_t)blockIdx.x * k + j] = i;
        values[(int64_t)blockIdx.x * k + j] = row[i];
    }
}

// The k (<= MAX_K) first words of a row in descending word order, by one workgroup of 1024 lanes in one pass over the row:
// calls write(rank, word).  Bound by latency, not by bytes: a chain of memory round trips, LDS passes and barriers.
//   1. A sample, evenly spaced, is counted in equal steps of its scores' range; a suffix scan gives a pivot
//      that somewhat more than k elements of the row should reach (four standard deviations of the sample count more).  Where the
//      row is all in registers it is every fourth of a lane's elements, another fourth in each of four wavefronts: 4096 requested
//      from memory one by one, a line each, took the memory pipe 4 K of the 32 K ticks of a row of 20000.  Longer rows pay that:
//      four of a lane's (eight: 2 rows of 65536 24.6 us, not 23.0).
//   2. The row - requested before anything else - is filtered: the words that reach the pivot go to
//      LDS, a wavefront's with one counter update per 16 elements of a lane.  (16 wavefronts share four SIMDs: instructions bound
//      this, so the index is looked at only where the row ends and the smallest key is the pivot, not a minimum.)
//   3. If at least k and at most ROW_CAP did (else: row_select_exact), they are put in order by order_words, which drops
//      those behind the k-th.
// Rows of up to ROW_CAP elements skip 1 and keep everything.  NPT: elements per lane; 0: rows of any length, 32 elements per
// lane (128 KB) in flight.  `VEC` consecutive elements go to one lane (4: `load4(i)`, 16-byte aligned and readable up to the next
// multiple of 4096 elements, `cap`), so that the requests are wide.
constexpr int ROW_CAP = 4096;
struct RowLds {
    uint64_t buf[ROW_CAP];
    uint32_t hist[ORDER_GROUPS]; // (the sample's and the radix select's: the first NBINS)
    uint32_t tmp[16];
    uint32_t bin, krem, cnt, out;
};

// The same selection by counting passes over the row (11 key bits a pass, then the indices of equal keys): for rows whose
// sampled pivot misjudged - heavy ties, scores sorted by position in step with the samples, far outliers.  Leaves the k
// selected words in lds.buf.
template <class Load>
__device__ __forceinline__ void row_select_exact(RowLds& lds, int n, int k, Load&& load)
{
    const int tid = threadIdx.x;
    auto each = [&](auto&& f) {
        constexpr int AHEAD = 8; // (a lane's requests in flight)
        for (int base = tid; base < n; base += 1024 * AHEAD) {
            float v[AHEAD];
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) v[j] = load(min(base + 1024 * j, n - 1));
#pragma unroll
            for (int j = 0; j < AHEAD; ++j)
                if (base + 1024 * j < n) f(make_cand(score_key(v[j]), base + 1024 * j));
        }
    };
    __syncthreads();
    if (tid == 0) lds.out = 0u;
    __syncthreads();
    radix_select64(each, [&](uint64_t w) {
        const uint32_t p = atomicAdd(&lds.out, 1u);
        if (p < MAX_K) lds.buf[p] = w;
    }, (uint32_t)k, 64, lds.hist, lds.tmp, &lds.bin, &lds.krem, &lds.cnt);
    __syncthreads();
}

template <int NPT, int VEC, class Load, class Load4, class Length, class Write>
__device__ __forceinline__ void select_row(RowLds& lds, int cap, int k, Load&& load, Load4&& load4, Length&& length, Write&& write)
{
    constexpr int CH = NPT > 0 ? NPT : 16; // elements per lane filtered together
    constexpr int AHEAD = NPT > 0 ? 1 : 2; // such groups in flight
    const int tid = threadIdx.x, lane = tid & 63;
    // element j of this lane
    auto index = [&](int j) { return VEC == 4 ? 4 * (tid + 1024 * (j >> 2)) + (j & 3) : tid + 1024 * j; };
    float v[AHEAD][CH];
    auto request = [&](int j0, float (&to)[CH]) {
        if constexpr (VEC == 4) {
#pragma unroll
            for (int j = 0; j < CH; j += 4) {
                const f32x4 q = load4(min(index(j0 + j), cap - 4));
#pragma unroll
                for (int c = 0; c < 4; ++c) to[j + c] = q[c];
            }
        } else {
#pragma unroll
            for (int j = 0; j < CH; ++j) to[j] = load(min(index(j0 + j), cap - 1));
        }
    };
#pragma unroll
    for (int g = 0; g < AHEAD; ++g) request(g * CH, v[g]);
    const int n = length(); // (its loads travel with the row's)
    if (n <= 0) return;     // block-uniform
    k = min(k, n);
    lds.hist[tid] = 0u;
    lds.hist[tid + 1024] = 0u;
    if (tid == 0) {
        lds.out = 0u;
        lds.bin = 0u;
        lds.tmp[14] = 0xffffffffu;
        lds.tmp[15] = 0u;
    }
    uint32_t pivot = 0u;
    if (n > ROW_CAP) { // block-uniform
        float per_element; // samples
        constexpr int PER = AHEAD * CH / 4, FAR = PER < 4 ? PER : 4; // (of a lane: out of its registers, from memory)
        uint32_t key[PER], kmin = 0xffffffffu, kmax = 0u;
        if (NPT > 0 || n <= 1024 * AHEAD * CH) { // block-uniform
            // every fourth of the lane's elements, from one of the first four on in turn
            auto sample = [&](auto first) {
#pragma unroll
                for (int q = 0; q < PER; ++q) {
                    const int j = 4 * q + first;
                    key[q] = index(j) < n ? max(score_key(v[j / CH][j % CH]), 1u) : 0u; // (0: no element)
                }
            };
            switch (__builtin_amdgcn_readfirstlane(tid >> 6) & 3) {
            case 0: sample(std::integral_constant<int, 0>{}); break;
            case 1: sample(std::integral_constant<int, 1>{}); break;
            case 2: sample(std::integral_constant<int, 2>{}); break;
            default: sample(std::integral_constant<int, 3>{}); break;
            }
            per_element = 0.25f;
        } else {
            float sv[FAR];
#pragma unroll
            for (int q = 0; q < FAR; ++q) sv[q] = load((int)(((int64_t)(tid + 1024 * q) * n) / (1024 * FAR)));
#pragma unroll
            for (int q = 0; q < PER; ++q) key[q] = q < FAR ? max(score_key(sv[q < FAR ? q : 0]), 1u) : 0u;
            per_element = 1024.f * FAR / (float)n;
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            kmin = min(kmin, key[q] - 1u);
            kmax = max(kmax, key[q]);
        }
        __syncthreads();
        block_key_range(kmin, kmax, lds.tmp);
        const KeyGroups<11> groups(kmin + 1u, kmax);
        if (groups.linear_ok) {
#pragma unroll
            for (int q = 0; q < PER; ++q)
                if (key[q] != 0u) atomicAdd(&lds.hist[groups.of(key[q], 0)], 1u);
            __syncthreads();
            const float expect = (float)k * per_element;
            const uint32_t target = (uint32_t)(expect + 4.f * __builtin_sqrtf(expect)) + 2u;
            const uint32_t h_lo = lds.hist[2 * tid], h_hi = lds.hist[2 * tid + 1]; // lane t owns bins 2t and 2t+1
            const uint32_t incl = block_suffix_sum<16>(h_lo + h_hi, lds.tmp);
            // the highest step that `target` samples reach
            if (incl >= target && incl - h_lo - h_hi < target) lds.bin = incl - h_lo >= target ? 2 * tid + 1 : 2 * tid;
            __syncthreads();
            pivot = f32_to_ordered(groups.fmin + (float)lds.bin / groups.per);
        }
        __syncthreads();
        if (tid == 0) {
            lds.tmp[14] = 0xffffffffu;
            lds.tmp[15] = 0u;
        }
    }
    __syncthreads();
    uint32_t bottom = 0xffffffffu, top = 0u; // smallest and largest key that reached the pivot
    auto filter = [&](int j0, const float (&from)[CH]) { // elements j0 .. j0 + CH - 1 of the lane
        uint32_t key[CH], count = 0;
        bool in[CH];
#pragma unroll
        for (int j4 = 0; j4 < CH; j4 += 4) { // (block-uniform: past the row's end nothing, inside it without a look at the index)
            const int begin = 1024 * (j0 + j4);
#pragma unroll
            for (int j = j4; j < j4 + 4; ++j) in[j] = false;
            if (begin >= n) continue;
#pragma unroll
            for (int j = j4; j < j4 + 4; ++j) {
                key[j] = score_key(from[j]);
                in[j] = key[j] >= pivot;
            }
            if (begin + 4096 > n) {
#pragma unroll
                for (int j = j4; j < j4 + 4; ++j) in[j] = in[j] && index(j0 + j) < n;
            }
#pragma unroll
            for (int j = j4; j < j4 + 4; ++j) count += in[j] ? 1u : 0u;
        }
        const uint32_t incl = wave_prefix_sum(count);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        if (total == 0u) return; // wave-uniform
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&lds.out, total);
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
        if (at + total > ROW_CAP) return; // (wave-uniform; the row is selected exactly)
        at += incl - count;
#pragma unroll
        for (int j = 0; j < CH; ++j)
            if (in[j]) {
                lds.buf[at++] = make_cand(key[j], index(j0 + j));
                top = max(top, key[j]);
            }
        if (pivot == 0u) // (else the pivot bounds them: block-uniform)
#pragma unroll
            for (int j = 0; j < CH; ++j)
                if (in[j]) bottom = min(bottom, key[j]);
    };
    if constexpr (NPT > 0) {
        filter(0, v[0]);
    } else {
        for (int j0 = 0; 1024 * j0 < n; j0 += AHEAD * CH) { // block-uniform
#pragma unroll
            for (int g = 0; g < AHEAD; ++g) {
                filter(j0 + g * CH, v[g]);
                if (1024 * (j0 + (g + AHEAD) * CH) < n) request(j0 + (g + AHEAD) * CH, v[g]);
                __builtin_amdgcn_sched_barrier(0); // (no further look-ahead: it would cost registers)
            }
        }
    }
    bottom = wave_min(bottom);
    top = wave_max(top);
    if (lane == 0) {
        atomicMin(&lds.tmp[14], bottom);
        atomicMax(&lds.tmp[15], top);
    }
    __syncthreads();
    uint32_t m = lds.out, kmin = pivot == 0u ? lds.tmp[14] : pivot, kmax = lds.tmp[15];
    const bool exact = m < (uint32_t)k || m > ROW_CAP; // block-uniform
    if (exact) {
        row_select_exact(lds, n, k, load);
        m = (uint32_t)k;
    }
    uint64_t w[ROW_CAP / 1024];
#pragma unroll
    for (int h = 0; h < ROW_CAP / 1024; ++h) w[h] = lds.buf[tid + 1024 * h];
    if (exact) {
        if (tid == 0) {
            lds.tmp[14] = 0xffffffffu;
            lds.tmp[15] = 0u;
        }
        __syncthreads();
        kmin = 0xffffffffu;
        kmax = 0u;
#pragma unroll
        for (int h = 0; h < ROW_CAP / 1024; ++h)
            if ((uint32_t)(tid + 1024 * h) < m) {
                kmin = min(kmin, (uint32_t)(w[h] >> 32));
                kmax = max(kmax, (uint32_t)(w[h] >> 32));
            }
        block_key_range(kmin, kmax, lds.tmp);
    }
    order_words<ROW_CAP / 1024>(w, m, kmin, kmax, lds.buf, lds.hist, lds.tmp, &lds.cnt, k, write);
}

// The indexer's selection as one kernel over the score rows, for rows of at most INDEXER_ROW_MAX keys: no histograms, no
// lists in the workspace, one launch less.  Indices only, -1 behind the last.
template <int NPT>
__global__ __launch_bounds__(1024) void indexer_row_topk_kernel(IndexerArgs a)
{
    __shared__ __align__(16) RowLds lds;
    const int tid = threadIdx.x, row = blockIdx.x;
    const float* x = a.scores + (int64_t)row * a.score_stride;
    int32_t* out = a.topk_res + (int64_t)row * a.k;
    auto length = [&]() {
        const int n = row_length(a.act_seq, row, a.s1, a.max_ctx);
        for (int j = min(n, a.k) + tid; j < a.k; j += 1024) out[j] = -1;
        return n;
    };
    select_row<NPT, 4>(lds, a.score_stride, a.k, [&](int i) { return x[i]; },
                       [&](int i) { return *reinterpret_cast<const f32x4*>(x + i); }, length,
                       [&](int rank, uint64_t w) { out[rank] = word_index(w); });
}

// With the gather that uses it, k = 2048: 16 rows of 20000 20.6 us, 2 rows of 65536 23.0, 4 rows of 200000 47.1 (the sample always
// from memory, every index looked at, half the groups and each word compared by the lane that had read it: 23.5, 24.7, 53.8).
// Counting passes over the row and a bitonic sort of the selected words took the selection from 15 to 53 us for the first.
template <int NPT>
__global__ __launch_bounds__(1024) void topk_select_kernel(const float* __restrict__ x, float* __restrict__ values,
                                                           int32_t* __restrict__ indices, int n, int k, int largest)
{
    __shared__ __align__(16) RowLds lds;
    const float* row = x + (int64_t)blockIdx.x * n;
    auto load = [&](int i) { return largest ? row[i] : -row[i]; };
    int32_t* out_i = indices + (int64_t)blockIdx.x * k;
    float* out_v = values + (int64_t)blockIdx.x * k;
    select_row<NPT, 1>(lds, n, k, load, [&](int) { return f32x4{}; }, [&]() { return n; }, [&](int rank, uint64_t w) {
        const int i = word_index(w);
        float v = key_to_score((uint32_t)(w >> 32));
        v = largest ? v : -v;
        // (the key has lost the sign of a zero and may have lost a NaN's bits: those come from the row)
        if (!(fabsf(v) > 0.f)) v = row[i];
        out_i[rank] = i;
        out_v[rank] = v;
    });
}

} // namespace

bool topk_supported(int64_t n, int64_t k) { return n >= 1 && k >= 1 && k <= n && n <= (1 << 24) && (n <= TOPK_SORT_CAP || k <= MAX_K); }

hipError_t topk_launch(const float* x, float* values, int32_t* indices, int64_t rows, int n, int k, bool largest, hipStream_t stream)
{
    if (rows == 0) return hipSuccess;
    void (*kern)(const float*, float*, int32_t*, int, int, int) =
        n <= TOPK_SORT_SMALL || k > MAX_K ? topk_sort_kernel : n <= 4096 ? topk_select_kernel<4> :
        n <= 16384 ? topk_select_kernel<16> : topk_select_kernel<0>;
    hipLaunchKernelGGL(kern, dim3((unsigned)rows), dim3(1024), 0, stream, x, values, indices, n, k, largest ? 1 : 0);
    return hipGetLastError();
}

// workspace: scores [t, stride] f32 | span_hist [t, spans, 256] u16 | counters [t, 4] u32 | winners [t, 2048] u64 |
// ties [t, 8192] u64; spans: histogram slots
static uint64_t align256(uint64_t x) { return (x + 255) & ~(uint64_t)255; }

// Passes of 512 keys per workgroup of the paged score kernel: as many as leave SCORE_GROUPS workgroups, eight at most.  Where
// there are keys for that, few long streams serve best (32 x 64 K keys: 50 us with eight passes, 53 with four, 58 with two);
// a small batch needs short ones to reach every CU (a single 4 K context is 2 workgroups of four passes: 12 us, against 6).
// The kernel takes fewer where the contexts are shorter than the page tables.
static int pick_passes(int b, int s1, int64_t stride)
{
    const int64_t groups = (int64_t)b * (s1 % 2 == 0 ? s1 / 2 : s1) * (stride / CHUNK); // of one pass
    int p = 8;
    while (p > 1 && groups < p * SCORE_GROUPS) p >>= 1;
    return p;
}

uint64_t indexer_workspace_bytes(int b, int s1, int stride)
{
    const int t = b * s1;
    const int passes = pick_passes(b, s1, stride);
    const uint64_t spans = (uint64_t)stride / (CHUNK * std::min(passes, PASSES)); // (the unpaged kernel's spans: PASSES)
    return align256((uint64_t)t * stride * 4) + align256((uint64_t)t * spans * SBINS * 2) + align256((uint64_t)t * 4 * 4) +
           align256((uint64_t)t * (MAX_K + TIE_CAP) * 8);
}

void indexer_bind_workspace(IndexerArgs& a, void* ws)
{
    const int t = a.b * a.s1;
    a.span = a.block_size % 128 == 0 ? CHUNK * pick_passes(a.b, a.s1, a.score_stride) : CHUNK * PASSES;
    const uint64_t spans = (uint64_t)a.score_stride / std::min(a.span, CHUNK * PASSES);
    uint8_t* p = static_cast<uint8_t*>(ws);
    a.scores = reinterpret_cast<float*>(p);
    p += align256((uint64_t)t * a.score_stride * 4);
    a.span_hist = reinterpret_cast<uint16_t*>(p);
    p += align256((uint64_t)t * spans * SBINS * 2);
    a.counters = reinterpret_cast<uint32_t*>(p);
    p += align256((uint64_t)t * 4 * 4);
    a.winners = reinterpret_cast<uint64_t*>(p);
    a.ties = a.winners + (uint64_t)t * MAX_K;
    a.pchunks = (int32_t)spans;
}

template <int PPASSES>
static void launch_score_paged(const IndexerArgs& a, hipStream_t stream)
{
    const bool s2 = a.s1 % 2 == 0, f32 = a.scales_f32;
    // non-temporal where one call's keys take the last-level cache's better part (109 MB: 26.2 -> 24.8 us, 272 MB: 57.8 ->
    // 52.7; 68 MB, found there from one call to the next: 15.0 -> 16.4) and not more than two workgroups read them
    const bool nt = (double)a.b * a.max_ctx * D > SCORE_CACHED && a.s1 <= 2;
    auto kern = s2 ? (f32 ? (nt ? indexer_score_paged_kernel<2, true, PPASSES, true> : indexer_score_paged_kernel<2, true, PPASSES, false>)
                          : (nt ? indexer_score_paged_kernel<2, false, PPASSES, true> : indexer_score_paged_kernel<2, false, PPASSES, false>))
                   : (f32 ? (nt ? indexer_score_paged_kernel<1, true, PPASSES, true> : indexer_score_paged_kernel<1, true, PPASSES, false>)
                          : (nt ? indexer_score_paged_kernel<1, false, PPASSES, true> : indexer_score_paged_kernel<1, false, PPASSES, false>));
    // a workgroup for every span of the page tables' reach; fewer passes are taken with fewer than 2 SCORE_GROUPS workgroups
    // (in all query token groups) full and one more in every sequence
    const int64_t z = s2 ? a.s1 / 2 : a.s1, gx = (a.max_ctx + CHUNK * PPASSES - 1) / (CHUNK * PPASSES);
    const int64_t rows = a.b <= SCAN_SEQS && PPASSES > a.min_passes ? std::max<int64_t>(a.b, ((2 * SCORE_GROUPS + z - 1) / z + a.b + gx - 1) / gx) : a.b;
    hipLaunchKernelGGL(kern, dim3((unsigned)gx, (unsigned)rows, (unsigned)z), dim3(256), 0, stream, a);
}

hipError_t indexer_launch(const IndexerArgs& a, hipStream_t stream)
{
    const int t = a.b * a.s1;
    if (t == 0) return hipSuccess;
    const int max_ctx = a.bt_stride * a.block_size;
    if (max_ctx == 0 || a.n_blocks == 0) { // a page table without columns, or a cache without pages: no key exists, every slot is -1
        const int n = t * a.k;
        hipLaunchKernelGGL(indexer_fill_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, a.topk_res, n, -1);
        return hipGetLastError();
    }
    // one workgroup per span of keys the page table can address (a.pchunks slots per query token hold at least as many)
    IndexerArgs args = a;
    args.max_ctx = max_ctx;
    args.use_hist = max_ctx > INDEXER_ROW_MAX;
    args.min_passes = args.use_hist ? a.score_stride / a.pchunks / CHUNK : 1; // (no more spans than slots)
    {
        ScopedKernelTimer tm(KID_INDEXER_SCORE, stream);
        if (a.block_size % 128 == 0) {
            if (a.span == 8 * CHUNK) launch_score_paged<8>(args, stream);
            else if (a.span == 4 * CHUNK) launch_score_paged<4>(args, stream);
            else if (a.span == 2 * CHUNK) launch_score_paged<2>(args, stream);
            else launch_score_paged<1>(args, stream);
        } else {
            const bool pow2 = (a.block_size & (a.block_size - 1)) == 0;
            const bool s2 = a.s1 % 2 == 0, f32 = a.scales_f32;
            auto kern = s2 ? (pow2 ? (f32 ? indexer_score_kernel<2, true, true> : indexer_score_kernel<2, true, false>)
                                   : (f32 ? indexer_score_kernel<2, false, true> : indexer_score_kernel<2, false, false>))
                           : (pow2 ? (f32 ? indexer_score_kernel<1, true, true> : indexer_score_kernel<1, true, false>)
                                   : (f32 ? indexer_score_kernel<1, false, true> : indexer_score_kernel<1, false, false>));
            hipLaunchKernelGGL(kern, dim3((max_ctx + a.span - 1) / a.span, a.b, s2 ? a.s1 / 2 : a.s1), dim3(256), 0, stream, args);
        }
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (args.use_hist) {
        ScopedKernelTimer tm(KID_INDEXER_SELECT, stream);
        hipLaunchKernelGGL(indexer_select_kernel, dim3((max_ctx + SEL_CHUNK - 1) / SEL_CHUNK, t), dim3(256), 0, stream, args);
    }
    {
        ScopedKernelTimer tm(KID_INDEXER_TOPK, stream);
        auto kern = args.use_hist ? indexer_topk_kernel : max_ctx <= 4096 ? indexer_row_topk_kernel<4> :
                    max_ctx <= 16384 ? indexer_row_topk_kernel<16> : indexer_row_topk_kernel<0>;
        hipLaunchKernelGGL(kern, dim3(t), dim3(1024), 0, stream, args);
    }
    return hipGetLastError();
}

} // namespace pto
