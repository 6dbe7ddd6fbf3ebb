// Paged grouped-query decode attention for gfx950 (GLM-4.5 shape: 96 query heads, 8 KV heads, head dim 128, bf16).
// Reference: models/glm_v4_5/glm_attention.py:427-568 (ifa_func_kernel), golden ifa_flash_torch :1374-1483.
//
// The operator streams every cached K and V row of a sequence once (4096 bytes per token over all KV heads) and
// does 12 flop per byte, so it is bound by HBM bandwidth; the design goal is to keep enough 16-byte loads in flight
// and to touch every byte once.
//
// One workgroup per (KV chunk of a sequence, KV head, RT row tiles): a row tile is a query token of the sequence and up to 16
// of the KV head's query heads.  256 lanes = 4 wavefronts that free-run (no barrier in the main loop).  A wave owns every
// fourth 32-token sub-tile of the chunk (so the four waves together walk whole 128-token pages), moves it from registers to
// its own LDS, requests the next one and computes, and keeps its own online-softmax state (m, l, O) per row tile; the four
// states are merged through LDS at the end and written either as the final bf16 rows (one chunk per sequence) or as fp32
// partials that gqa_combine_kernel merges.
//   Loads take whole 256-byte cache rows, four to an instruction.  (K in the operand's layout straight from memory takes half
// cache lines, twice, from 16 rows: 868 us against 853 at 4.8 GB, and unusable without cache retention.)
//   Where the batch's keys do not fit the 256 MB last-level cache, they are loaded past it (non-temporal; a plain read
// stream reaches 6.3 TB/s on this card, a non-temporal one 7.1): 853 -> 800 us.  Where they fit, the caches serve part of it
// (197 MB, two query tokens a sequence: 42 us through the caches, 47 past them).  The lengths decide, not the page tables'
// reach; the whole sweep exists twice, since a choice at every sub-tile's loads costs 0.5 us at 33 MB (13.4 -> 14.0).
//   The page-table entries of 64 pages are held by a wavefront's lanes: a look-up from memory in front of every sub-tile
// waited for the sub-tile in flight as well (loads complete in order): 1077 -> 868 us.
//   Chunks are chosen on the device from the lengths (choose_chunk): as long as they can be while the workgroups fill the
// chip a whole number of times.  Two row tiles per workgroup (two query tokens of a sequence) share every K and V byte.
//   64 sequences of 4096 .. 32768 tokens, 96 / 8 heads: 1090 us with fixed chunks of 1024, 797 now (4.8 GB); 8
// sequences up to 8192, 12 / 1 heads: 19.5 us, 13 now, most of it the chain lengths - page table - keys - merge.
//
//   S^T[token, head] = K Q^T : v_mfma_f32_16x16x32_bf16, A = K rows (lane = token l%16, 8 dims at 8*(l/16) + 32*j), B = Q
//       (resident, heads padded to 16).
//   O^T[dim, head] += V^T P~^T : A = V^T by ds_read_b64_tr_b16, B = P~ rounded to bf16, which is exactly the register layout
//       S^T comes out in (lane = head l%16, 4 tokens per 16-token block), so P~ never leaves registers.  The contraction
//       index is visited in the order {4g..4g+3, 16+4g..16+4g+3} per lane group g on both operands.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include <stdint.h>

#include "common.h"
#include "kernels.h"
#include "timing.h"

namespace pto {
namespace {

constexpr int GD = 128;      // head dim
constexpr int GSUB = 32;     // tokens per wave sub-tile
constexpr int GWAVES = 4;
constexpr int GROW = GD * 2; // bytes per staged V row
constexpr float LOG2E = 1.4426950408889634f;
constexpr float GQA_CACHED = 256e6f; // bytes of keys and values that the last-level cache holds
constexpr int GQA_SLOTS = 256;   // one workgroup per CU (two fit; twice as many shorter ones measured 5 to 15 % slower on small batches)
constexpr int GQA_TARGET = 4096; // tokens a workgroup should have at most, where there are enough
constexpr int GQA_TARGET2 = 1024; // and with two row tiles (more only where that would be over GQA_MAX_SPLIT chunks): a wavefront's
                                  // running sums span 256 tokens, and there are no registers for PIECES (4096: 4 to 10 % faster)
// Workgroups of a launch at most (or one per KV head, query token and head group): the page tables may reach much further than
// the contexts do, and a workgroup for every unit they have room for costs 1 us on a CU only to find that it has none.  Then
// workgroups walk the units (64 sequences of 4096 tokens, 96 / 8 heads, 8192 columns: 234 us with a workgroup per unit, 179 so,
// 172 under tables of 32 columns; 300 sequences, 12 / 1 heads: 1434, 125 and 119).
// With two row tiles the chunks are shorter and a workgroup to each is the better way up to 8192 of them (32 sequences of 16000
// tokens, two query tokens, 96 / 8 heads, 4096 chunks: 400 us, 415 by a walk).
constexpr int GQA_GRID = 2048, GQA_GRID2 = 8192;
constexpr int GQA_MAX_SPLIT = 64; // chunks per sequence on average at most, beyond one round of GQA_SLOTS workgroups: the partials
                                  // take memory by the page table's reach (512 sequences, 96 / 8 heads, 1 M tokens: 1.6 GB)

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ __forceinline__ s16x4 lds_read_tr(uint8_t* p) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p); }

// byte offset inside a staged row of token t of 16-byte chunk c16: the 32-byte units of a row are XOR-ed with t % 8
__device__ __forceinline__ int vswz(int t, int c16) { return ((((c16 >> 1) ^ (t & 7)) << 5) | ((c16 & 1) << 4)); }

struct SubTile {
    u32x4 k[8], v[8]; // row 4*i + l/16, 16-byte chunk l%16
    bool mapped;   // the page exists
};

// wavefront-wide inclusive prefix sum in the lane network
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int gqa_dpp_add(int v)
{
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}
__device__ __forceinline__ int gqa_prefix_sum(int v)
{
    v = gqa_dpp_add<0x111, 0xf>(v);
    v = gqa_dpp_add<0x112, 0xf>(v);
    v = gqa_dpp_add<0x114, 0xf>(v);
    v = gqa_dpp_add<0x118, 0xf>(v);
    v = gqa_dpp_add<0x142, 0xa>(v); // rows 1 and 3 add the totals of rows 0 and 2
    return gqa_dpp_add<0x143, 0xc>(v);
}

// The lengths of up to GQA_SCAN sequences, by one wavefront: lane l holds those of sequences l, l + 64, ..  (cut to the page
// table's reach; -1 past the last sequence); of more, those of GQA_SCAN evenly spaced ones.
constexpr int GQA_SCAN = 256;
struct Lengths {
    int len[GQA_SCAN / 64];
    __device__ __forceinline__ void fetch(const GqaArgs& a, int lane)
    {
        const int reach = a.bt_stride * a.block_size;
#pragma unroll
        for (int j = 0; j < GQA_SCAN / 64; ++j) { // (requested together)
            const int i = lane + 64 * j;
            len[j] = 64 * j < a.b ? a.act_seq[a.b > GQA_SCAN ? (int)((int64_t)i * a.b / GQA_SCAN) : min(i, a.b - 1)] : 0;
        }
#pragma unroll
        for (int j = 0; j < GQA_SCAN / 64; ++j) len[j] = lane + 64 * j < a.b ? max(min(len[j], reach), 0) : -1;
    }
    // chunks of 128 c tokens of the lane's j-th sequence: an empty sequence has one too (its output rows are zero).  The
    // quotient by way of fp32 is off by at most one and put right (the counts of 128 tokens are below 2^24: exact).
    __device__ __forceinline__ int chunks(int j, int c, float inv_c) const
    {
        const int n = (len[j] + 127) >> 7;
        int q = (int)((float)(n + c - 1) * inv_c);
        const int r = n + c - 1 - q * c;
        q += r < 0 ? -1 : r >= c ? 1 : 0;
        return len[j] < 0 ? 0 : max(1, q);
    }
    // tokens, in units of 128 (256 sequences of 2^30 have 2^31: unsigned)
    __device__ __forceinline__ uint32_t sum() const
    {
        int n = 0;
#pragma unroll
        for (int j = 0; j < GQA_SCAN / 64; ++j) n += (max(len[j], 0) + 127) >> 7;
        return (uint32_t)__builtin_amdgcn_readlane(gqa_prefix_sum(n), 63);
    }
    // whether the batch's keys and values are to be loaded past the caches
    __device__ __forceinline__ bool past_caches(const GqaArgs& a) const
    {
        const float seqs = a.b > GQA_SCAN ? (float)a.b / GQA_SCAN : 1.f;
        return (float)sum() * seqs * (float)a.nkv * (128.f * 2 * GROW) > GQA_CACHED;
    }
    // chunks of all sequences
    __device__ __forceinline__ uint32_t units(const GqaArgs& a, int c) const
    {
        const float inv_c = 1.f / (float)c;
        int n = 0;
#pragma unroll
        for (int j = 0; j < GQA_SCAN / 64; ++j)
            if (64 * j < a.b) n += chunks(j, c, inv_c); // (uniform)
        return (uint32_t)__builtin_amdgcn_readlane(gqa_prefix_sum(n), 63);
    }
};

// The batch's chunk length: the smallest multiple of 128 tokens that cuts it into no more units than fill the chip's
// GQA_SLOTS workgroup slots a whole number of times - as many times as it takes to keep workgroups near GQA_TARGET tokens
// (fewer, longer ones pay less for starting up and for partials; more even out what the memory system serves unevenly).
// Depends on the lengths alone, so every wavefront finds the same one; the result never exceeds units_cap units.
__device__ __forceinline__ int choose_chunk(const GqaArgs& a, const Lengths& ls)
{
    int longest = 0;
#pragma unroll
    for (int j = 0; j < GQA_SCAN / 64; ++j) {
        if (64 * j >= a.b) break; // (uniform)
        longest = max(longest, ls.len[j]);
    }
    const uint32_t sum = ls.sum();
    // rounds of GQA_SLOTS workgroups with GQA_TARGET tokens (of at most 2^22, so that their slots fit 32 bits)
    const float slot = (float)min(a.longest, GQA_TARGET) * (GQA_SLOTS / 128.f);
    const int rounds = (int)fminf(fmaxf(ceilf((float)sum * (float)a.columns / slot), 1.f), 0x1p22f);
    const uint32_t target = (uint32_t)min(max(rounds * GQA_SLOTS / a.columns, a.b), (int)a.units_cap);
    int lo = max((int)((sum + target - 1) / target), 1); // (no shorter chunk can do)
    if (ls.units(a, lo) <= target) return lo * 128;
    longest = (int)wave_max_f32((float)longest) + 128; // the batch's (as a float it may be off by less than 128)
    int hi = max((longest + 127) / 128, lo + 1); // one chunk per sequence: at most a.b <= target units
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ls.units(a, mid) <= target) hi = mid;
        else lo = mid;
    }
    return hi * 128;
}

// Up to GQA_SCAN sequences: the (sequence, chunk) of unit u, and how many units there are; false: no such unit.  chunk: the
// chunk length, chosen if it is 0.
__device__ __forceinline__ bool gqa_unit(const GqaArgs& a, const Lengths& ls, int u, int& chunk, int& bi, int& split, int64_t& total)
{
    if (chunk == 0) chunk = min(choose_chunk(a, ls), a.longest);
    const float inv_c = 1.f / (float)(chunk >> 7);
    int base = 0;
    bi = -1;
#pragma unroll
    for (int j = 0; j < GQA_SCAN / 64; ++j) {
        if (64 * j >= a.b) break; // uniform
        const int cnt = ls.chunks(j, chunk >> 7, inv_c);
        const int incl = gqa_prefix_sum(cnt), excl = incl - cnt;
        const uint64_t hit = __ballot(u >= base + excl && u < base + incl); // at most one lane
        if (hit != 0ull) {
            const int l = __builtin_ctzll(hit);
            bi = 64 * j + l;
            split = u - base - __builtin_amdgcn_readlane(excl, l);
        }
        base += __builtin_amdgcn_readlane(incl, 63);
    }
    total = (uint32_t)base;
    return bi >= 0;
}

// More sequences: chunks of a fixed length, all sequences' first ones, then their second ones, .. (a walk in steps of a multiple of
// a sequence's chunks would meet the same chunk of every sequence).  Of the 64 units u, u + stride,
// .. those that have work, as a bit mask over the lanes: they lie inside their sequence, or are its first.
__device__ __forceinline__ uint64_t gqa_live_units(const GqaArgs& a, int64_t u, int64_t stride, int lane)
{
    const int64_t mine = u + lane * stride;
    const bool in = mine < a.units_cap;
    const int64_t split = in ? mine / a.b : 0;
    const int len = a.act_seq[in ? mine - split * a.b : 0];
    return __ballot(in && (split == 0 || split * a.chunk < len));
}

// grid: `stride` units x columns.  MAY: a batch that fills its page tables is loaded past the caches.  WALK: fewer units than there may be; a workgroup takes every stride-th, until there is none.
template <int RT, bool WALK, bool MAY>
__global__ __launch_bounds__(256, 2) void gqa_decode_kernel(GqaArgs a, int stride)
{
    // K and V staging, a pair of sub-tiles per wave; later the merge buffer (4 x 16 x 128 fp32)
    __shared__ __align__(16) uint8_t lds[2 * GWAVES * GSUB * GROW];
    __shared__ float s_ml[GWAVES][16][2];

    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Order of the workgroups: eight units (or stride, a power of two, if that is less) side by side, and behind each other
    // those that read the same keys, then the KV heads, whose rows lie beside each other in the cache.  Workgroups go to the
    // eight dies in turn, so the readers of the same keys share an L2.
    const int readers = a.s1 * a.hsub / RT;
    uint32_t first;
    int n2, rd;
    {
        const int sh = stride < 8 ? __builtin_ctz(stride) : 3;
        const uint32_t lin = blockIdx.x + gridDim.x * blockIdx.y, per = (uint32_t)(readers * a.nkv) << sh;
        const uint32_t o = lin / per, in = lin - o * per;
        first = (o << sh) + (in & ((1u << sh) - 1u));
        rd = (int)((in >> sh) % readers) * RT;
        n2 = (int)((in >> sh) / readers);
    }
    if (first >= (uint32_t)stride) return;
    const int g = a.nq / a.nkv;
    int chunk = a.chunk;
    int64_t at = first, total = a.units_cap; // the next unit to look at; units there are (at most)
    uint64_t live = 0; // beyond GQA_SCAN sequences: units at - 64 stride + l stride that have work
    for (bool again = false;; again = true) {
    int tid = threadIdx.x;
    if constexpr (WALK) asm volatile("" : "+v"(tid)); // (so that nothing derived from it is kept in registers from one unit to the next)
    const int lane = tid & 63, r16 = lane & 15, g4 = lane >> 4;
    Lengths ls;
    ls.fetch(a, lane);
    int bi, split;
    int64_t u; // the unit's place in the workspace
    if (a.b > GQA_SCAN) {
        while (live == 0) {
            if (at >= total) return;
            live = gqa_live_units(a, at, stride, lane);
            at += 64 * (int64_t)stride;
        }
        u = at + (__builtin_ctzll(live) - 64) * (int64_t)stride;
        live &= live - 1;
        split = (int)(u / a.b);
        bi = (int)(u - (int64_t)split * a.b);
        u = (int64_t)bi * a.nsplit + split;
    } else {
        u = at;
        if (at >= total || !gqa_unit(a, ls, (int)at, chunk, bi, split, total)) return;
        at += stride;
    }
    const bool past_caches = MAY && ls.past_caches(a); // uniform
    if (again) __syncthreads(); // (everyone is done with the last unit's merge buffer)
    if (a.part_o != nullptr && tid == 0 && rd == 0 && n2 == 0) { // for the combine kernel
        if (bi == 0 && split == 0) a.plan[0] = chunk;
        if (split == 0) a.plan[1 + bi] = (int32_t)u; // (read for up to GQA_SCAN sequences)
    }

    const int len = min(a.act_seq[bi], a.bt_stride * a.block_size);
    const int start = split * chunk;
    int tok_q[RT], hs[RT], end_r[RT], end = 0; // row tile r: its query token, head sub-group and end of the chunk
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int si = (rd + r) / a.hsub;
        hs[r] = rd + r - si * a.hsub;
        tok_q[r] = bi * a.s1 + si;
        end_r[r] = min(start + chunk, min(max(a.act_seq[bi] - (a.s1 - 1 - si), 0), max(len, 0)));
        end = max(end, end_r[r]);
    }
    uint16_t* out = static_cast<uint16_t*>(a.out);

    // Q fragments: B operand, lane = head r16 of the row tile, dims 8*g4 + 32*j
    u32x4 qf[RT][4];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int hloc = hs[r] * 16 + r16;
        const bool ok = hloc < g;
        const uint16_t* qp = static_cast<const uint16_t*>(a.q) + ((int64_t)tok_q[r] * a.nq + n2 * g + (ok ? hloc : 0)) * GD;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            qf[r][j] = *reinterpret_cast<const u32x4*>(qp + 8 * (g4 + 4 * j));
            if (!ok) qf[r][j] = u32x4{0u, 0u, 0u, 0u};
        }
    }

    const uint8_t* kbase = static_cast<const uint8_t*>(a.k) + (int64_t)n2 * GROW;
    const uint8_t* vbase = static_cast<const uint8_t*>(a.v) + (int64_t)n2 * GROW;
    const int64_t row_pitch = (int64_t)a.nkv * GROW;
    const uint32_t lane_at = (uint32_t)(g4 * (int)row_pitch + r16 * 16); // (nkv is below 2^15)
    const int32_t* bt = a.block_table + (int64_t)bi * a.bt_stride;
    uint8_t* myk = lds + 2 * w * (GSUB * GROW);
    uint8_t* myv = myk + GSUB * GROW;

    const int nsub = (max(end - start, 0) + GSUB - 1) / GSUB;
    const float sc = a.softmax_scale * LOG2E;

    // Sums of the last sub-tiles, up to PIECE of them, and of those before: a chain of the 32 sub-tiles that a wavefront has in
    // a chunk of 4096 tokens was 25 % further off in fp32 (times are the same).
    constexpr bool PIECES = RT == 1;
    constexpr int PIECE = 8;
    f32x4 o[RT][8], o_before[PIECES ? 8 : 1];
    float m_run[RT], l_run[RT], l_before = 0.f;
    int in_piece = 0;
    if constexpr (PIECES) {
#pragma unroll
        for (int i = 0; i < 8; ++i) o_before[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
        for (int i = 0; i < 8; ++i) o[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        m_run[r] = -INFINITY;
        l_run[r] = 0.f;
    }

    // Page-table entries: lane p holds that of page `window` + p (-1: none).  A sub-tile lies inside one page (block_size is a
    // multiple of 32 and chunks start on multiples of 128).
    int window = start / a.block_size;
    int entry = -1;
    auto fetch_entries = [&]() {
        const int e = bt[min(window + lane, a.bt_stride - 1)];
        entry = e >= 0 && e < a.n_blocks ? e : -1;
    };
    if (nsub > 0) fetch_entries();
    auto load = [&](int i, SubTile& t, auto past) __attribute__((always_inline)) {
        const int p0 = start + GSUB * i;
        const int page = p0 / a.block_size;
        if (page - window >= 64) { // (uniform; chunks of more than 64 pages)
            window = page;
            fetch_entries();
        }
        const int blk = __builtin_amdgcn_readlane(entry, page - window);
        t.mapped = blk >= 0; // an unmapped page is masked in compute(); its loads stay in bounds
        const int64_t at0 = ((int64_t)max(blk, 0) * a.block_size + (p0 - page * a.block_size)) * row_pitch; // uniform
        auto row = [&](const uint8_t* base, int i8) {
            const u32x4* p = reinterpret_cast<const u32x4*>(base + at0 + 4 * i8 * row_pitch + lane_at);
            return decltype(past)::value ? __builtin_nontemporal_load(p) : *p;
        };
#pragma unroll
        for (int i8 = 0; i8 < 8; ++i8) t.k[i8] = row(kbase, i8);
#pragma unroll
        for (int i8 = 0; i8 < 8; ++i8) t.v[i8] = row(vbase, i8);
    };
    auto stage = [&](const SubTile& t) __attribute__((always_inline)) {
#pragma unroll
        for (int i8 = 0; i8 < 8; ++i8) {
            const int tv = 4 * i8 + g4;
            *reinterpret_cast<u32x4*>(myk + tv * GROW + vswz(tv, r16)) = t.k[i8];
        }
#pragma unroll
        for (int i8 = 0; i8 < 8; ++i8) {
            const int tv = 4 * i8 + g4;
            *reinterpret_cast<u32x4*>(myv + tv * GROW + vswz(tv, r16)) = t.v[i8];
        }
    };

    auto compute = [&](int i, bool mapped) __attribute__((always_inline)) {
        const int p0 = start + GSUB * i;
        int krow = r16;
        if constexpr (RT > 1) asm volatile("" : "+v"(krow)); // (the reads' addresses anew for every sub-tile, not in registers)
        f32x4 s0[RT], s1[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) s0[r] = s1[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bf16x8 k0 = *reinterpret_cast<const bf16x8*>(myk + krow * GROW + vswz(krow, g4 + 4 * j));
            const bf16x8 k1 = *reinterpret_cast<const bf16x8*>(myk + (krow + 16) * GROW + vswz(krow, g4 + 4 * j));
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                s0[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, __builtin_bit_cast(bf16x8, qf[r][j]), s0[r], 0, 0, 0);
                s1[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, __builtin_bit_cast(bf16x8, qf[r][j]), s1[r], 0, 0, 0);
            }
        }
        if constexpr (RT > 1) __builtin_amdgcn_sched_barrier(0);
        u32x4 pf[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            float sv[8];
            float mt = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int tok = p0 + (e >> 2) * 16 + 4 * g4 + (e & 3);
                const float x = (e < 4 ? s0[r][e & 3] : s1[r][e & 3]) * sc;
                sv[e] = (tok < end_r[r] && mapped) ? x : -INFINITY;
                mt = fmaxf(mt, sv[e]);
            }
            mt = fmaxf(mt, __shfl_xor(mt, 16));
            mt = fmaxf(mt, __shfl_xor(mt, 32));
            const float m_new = fmaxf(m_run[r], mt);
            const float mref = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = exp2f(m_run[r] - mref);
            float p[8], psum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                p[e] = exp2f(sv[e] - mref);
                psum += p[e];
            }
            l_run[r] = l_run[r] * alpha + psum;
            m_run[r] = m_new;
            if constexpr (PIECES) l_before *= alpha;
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int db = 0; db < 8; ++db) {
                    o[r][db] *= alpha;
                    if constexpr (PIECES) o_before[db] *= alpha;
                }
            }
            pf[r] = u32x4{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])};
        }
        if constexpr (RT > 1) __builtin_amdgcn_sched_barrier(0);
        int tok_lo = 4 * g4 + (r16 >> 2);
        if constexpr (RT > 1) asm volatile("" : "+v"(tok_lo)); // (likewise)
#pragma unroll
        for (int db = 0; db < 8; ++db) {
            const s16x4 lo = lds_read_tr(myv + tok_lo * GROW + ((db ^ (tok_lo & 7)) << 5) + (r16 & 3) * 8);
            const s16x4 hi = lds_read_tr(myv + (tok_lo + 16) * GROW + ((db ^ (tok_lo & 7)) << 5) + (r16 & 3) * 8);
            const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int r = 0; r < RT; ++r)
                o[r][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, both),
                                                                   __builtin_bit_cast(bf16x8, pf[r]), o[r][db], 0, 0, 0);
        }
        if constexpr (PIECES) {
            if (++in_piece == PIECE) { // uniform
                in_piece = 0;
#pragma unroll
                for (int db = 0; db < 8; ++db) {
                    o_before[db] += o[0][db];
                    o[0][db] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                l_before += l_run[0];
                l_run[0] = 0.f;
            }
        }
    };

    auto sweep = [&](auto past) __attribute__((always_inline)) { // past: loads past the caches
        SubTile t;
        int i = w;
        load(i, t, past);
        for (; i + GWAVES < nsub; i += GWAVES) {
            const bool mapped = t.mapped;
            stage(t);
            load(i + GWAVES, t, past);
            compute(i, mapped);
        }
        stage(t);
        compute(i, t.mapped);
    };
    if (w < nsub) {
        if (past_caches) sweep(std::true_type{});
        else sweep(std::false_type{});
    }

    if constexpr (PIECES) {
#pragma unroll
        for (int db = 0; db < 8; ++db) o[0][db] += o_before[db];
        l_run[0] += l_before;
    }
    // merge the four waves
    float* mo = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        l_run[r] += __shfl_xor(l_run[r], 16);
        l_run[r] += __shfl_xor(l_run[r], 32);
        __syncthreads();
#pragma unroll
        for (int db = 0; db < 8; ++db)
            *reinterpret_cast<f32x4*>(mo + (w * 16 + r16) * GD + 16 * db + 4 * g4) = o[r][db];
        if (g4 == 0) {
            s_ml[w][r16][0] = m_run[r];
            s_ml[w][r16][1] = l_run[r];
        }
        __syncthreads();
        const int n = tid >> 4, d0 = (tid & 15) * 8;
        const int hloc = hs[r] * 16 + n;
        if (hloc >= g) continue;
        float M = -INFINITY;
#pragma unroll
        for (int ww = 0; ww < GWAVES; ++ww) M = fmaxf(M, s_ml[ww][n][0]);
        float L = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (M > -INFINITY) {
#pragma unroll
            for (int ww = 0; ww < GWAVES; ++ww) {
                const float wgt = exp2f(s_ml[ww][n][0] - M);
                L += wgt * s_ml[ww][n][1];
                const f32x4 x0 = *reinterpret_cast<const f32x4*>(mo + (ww * 16 + n) * GD + d0);
                const f32x4 x1 = *reinterpret_cast<const f32x4*>(mo + (ww * 16 + n) * GD + d0 + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[e] += wgt * x0[e];
                    acc[4 + e] += wgt * x1[e];
                }
            }
        }
        if (a.part_o == nullptr) {
            const int64_t head_row = (int64_t)tok_q[r] * a.nq + n2 * g + hloc;
            const float inv = L > 0.f ? 1.f / L : 0.f;
            const u32x4 pk = {pack_bf16x2(acc[0] * inv, acc[1] * inv), pack_bf16x2(acc[2] * inv, acc[3] * inv),
                              pack_bf16x2(acc[4] * inv, acc[5] * inv), pack_bf16x2(acc[6] * inv, acc[7] * inv)};
            *reinterpret_cast<u32x4*>(out + head_row * GD + d0) = pk;
        } else {
            const int64_t slot = (u * a.s1 + (tok_q[r] - bi * a.s1)) * a.nq + n2 * g + hloc;
            float* po = a.part_o + slot * GD + d0;
            *reinterpret_cast<f32x4*>(po) = f32x4{acc[0], acc[1], acc[2], acc[3]};
            *reinterpret_cast<f32x4*>(po + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
            if ((tid & 15) == 0) {
                float* pm = a.part_ml + slot * 2;
                pm[0] = M;
                pm[1] = L;
            }
        }
    }
    if constexpr (!WALK) break;
    } // units
}

// Merges the chunks that hold tokens of a query token: 32 lanes x 4 dims per head row and group of chunks, GROUPS such
// groups per row (merged through LDS) where there are many chunks - one group would walk them in too long a chain.
template <int GROUPS>
__global__ __launch_bounds__(256) void gqa_combine_kernel(GqaArgs a)
{
    constexpr int ROWS = 8 / GROUPS;
    __shared__ __align__(16) float s_acc[GROUPS > 1 ? 8 : 1][128];
    __shared__ float s_m[8], s_l[8];
    const int part = threadIdx.x >> 5, grp = part % GROUPS;
    const int64_t last_row = (int64_t)a.b * a.s1 * a.nq - 1;
    const int64_t want = (int64_t)blockIdx.x * ROWS + part / GROUPS;
    const int64_t head_row = want < last_row ? want : last_row; // (surplus groups redo the last row)
    const int d0 = (threadIdx.x & 31) * 4;
    const int tq = (int)(head_row / a.nq);
    const int bi = tq / a.s1, si = tq - bi * a.s1;
    int cur = a.act_seq[bi] - (a.s1 - 1 - si);
    cur = cur < 0 ? 0 : cur;
    const int reach = a.bt_stride * a.block_size;
    cur = cur > reach ? reach : cur;
    const int chunk = a.plan[0];
    const int nvalid = (cur + chunk - 1) / chunk;
    // the unit's partials lie [query token of the sequence, head]
    int64_t unit0 = a.plan[1 + bi];
    if (a.b > GQA_SCAN) unit0 = (int64_t)bi * a.nsplit; // (may leave 32 bits)
    const int64_t slot0 = (unit0 * a.s1 + si) * a.nq + (head_row - (int64_t)tq * a.nq), per = (int64_t)a.s1 * a.nq;
    const float* pm = a.part_ml + slot0 * 2;
    const float* po = a.part_o + slot0 * GD + d0;
    // eight chunks' loads in flight at a time (a chunk past the last valid one re-reads the last and is dropped): an online
    // merge, chunks grp, grp + GROUPS, .. in order
    constexpr int G = 8;
    float M = -INFINITY, L = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = grp; s0 < nvalid; s0 += G * GROUPS) {
        f32x4 v[G];
        float m[G], l[G], top = M;
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int s = min(s0 + j * GROUPS, nvalid - 1);
            m[j] = pm[2 * per * s];
            l[j] = pm[2 * per * s + 1];
            v[j] = *reinterpret_cast<const f32x4*>(po + per * s * GD);
        }
#pragma unroll
        for (int j = 0; j < G; ++j) top = fmaxf(top, m[j]);
        if (top > -INFINITY) {
            const float old = exp2f(M - top);
            L *= old;
            acc *= old;
            M = top;
#pragma unroll
            for (int j = 0; j < G; ++j) {
                if (s0 + j * GROUPS < nvalid) {
                    const float wgt = exp2f(m[j] - M);
                    L += wgt * l[j];
                    acc += v[j] * wgt;
                }
            }
        }
    }
    if constexpr (GROUPS > 1) {
        *reinterpret_cast<f32x4*>(&s_acc[part][d0]) = acc;
        if ((threadIdx.x & 31) == 0) {
            s_m[part] = M;
            s_l[part] = L;
        }
        __syncthreads();
        if (grp != 0) return;
        float top = -INFINITY;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) top = fmaxf(top, s_m[part + g]);
        L = 0.f;
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        if (top > -INFINITY) {
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) {
                const float wgt = exp2f(s_m[part + g] - top);
                L += wgt * s_l[part + g];
                acc += *reinterpret_cast<const f32x4*>(&s_acc[part + g][d0]) * wgt;
            }
        }
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const u32x2 pk = {pack_bf16x2(acc[0] * inv, acc[1] * inv), pack_bf16x2(acc[2] * inv, acc[3] * inv)};
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + head_row * GD + d0) = pk;
}

// attn_res <- 0 (cache without pages)
__global__ void gqa_zero_kernel(uint32_t* out, int64_t n_words)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_words) out[i] = 0u;
}

} // namespace

// units_cap: chunks of all sequences together.  One chunk per sequence and no second kernel where the sequences alone give
// GQA_SLOTS workgroups of at most GQA_TARGET tokens.
void gqa_plan(GqaArgs& a, int forced_chunk)
{
    const int64_t t = (int64_t)a.b * a.s1;
    const int64_t max_ctx = (int64_t)a.bt_stride * a.block_size;
    if (t == 0) { // (nothing to launch)
        a.chunk = 128;
        a.nsplit = a.row_tiles = a.columns = 1;
        a.units_cap = 0;
        return;
    }
    a.row_tiles = a.s1 * a.hsub % 2 == 0 ? 2 : 1;
    a.columns = (int32_t)((int64_t)a.nkv * a.s1 * a.hsub / a.row_tiles);
    const int64_t least = ((max_ctx + GQA_MAX_SPLIT - 1) / GQA_MAX_SPLIT + 127) / 128 * 128;
    a.longest = a.row_tiles == 1 ? INT32_MAX : (int32_t)std::max<int64_t>(GQA_TARGET2, least);
    if (forced_chunk > 0) {
        a.chunk = (forced_chunk + 127) / 128 * 128;
    } else if (a.b > GQA_SCAN) {
        a.chunk = a.row_tiles == 1 ? (int32_t)std::max<int64_t>(GQA_TARGET, least) : a.longest;
    } else {
        const int64_t round = (int64_t)GQA_SLOTS * (std::min(a.longest, GQA_TARGET) / 128);
        const int64_t work = (int64_t)a.b * ((max_ctx + 127) / 128) * a.columns;
        const int64_t rounds = (work + round - 1) / round;
        int64_t target = (rounds > 1 ? rounds : 1) * GQA_SLOTS / a.columns;
        const int64_t pages = (int64_t)a.b * ((max_ctx + 127) / 128);
        const int64_t one_round = std::min<int64_t>(GQA_SLOTS / a.columns, 2 * GQA_MAX_SPLIT * (int64_t)a.b);
        target = std::min(std::min(target, std::max(one_round, GQA_MAX_SPLIT * (int64_t)a.b)), pages);
        a.chunk = 0; // chosen on the device
        a.units_cap = std::max(target, a.b * std::max<int64_t>(1, (max_ctx + a.longest - 1) / a.longest));
        a.nsplit = a.units_cap > a.b ? 2 : 1;
        if (a.nsplit == 1) a.chunk = (int32_t)((max_ctx + 127) / 128 * 128);
    }
    if (a.chunk > 0) {
        const int64_t n = (max_ctx + a.chunk - 1) / a.chunk;
        a.nsplit = n < 1 ? 1 : (int32_t)n;
        a.units_cap = a.b * (int64_t)a.nsplit;
    }
    a.past_caches = (double)a.b * (double)max_ctx * a.nkv * 2 * GROW > GQA_CACHED;
}

static uint64_t gqa_align(uint64_t x) { return (x + 255) & ~(uint64_t)255; }

// partials [units_cap, s1, nq, 128] fp32 | (m, l) [units_cap, s1, nq, 2] fp32 | chunk length, first unit of every sequence
uint64_t gqa_workspace_bytes(const GqaArgs& a)
{
    if (a.nsplit == 1) return 0;
    const uint64_t rows = (uint64_t)a.units_cap * a.s1 * a.nq;
    return gqa_align(rows * GD * 4) + gqa_align(rows * 8) + gqa_align((1 + (uint64_t)a.b) * 4);
}

void gqa_bind_workspace(GqaArgs& a, void* workspace)
{
    const uint64_t rows = (uint64_t)a.units_cap * a.s1 * a.nq;
    uint8_t* p = static_cast<uint8_t*>(workspace);
    a.part_o = reinterpret_cast<float*>(p);
    a.part_ml = reinterpret_cast<float*>(p + gqa_align(rows * GD * 4));
    a.plan = reinterpret_cast<int32_t*>(p + gqa_align(rows * GD * 4) + gqa_align(rows * 8));
}

hipError_t gqa_launch(const GqaArgs& a, hipStream_t stream)
{
    const int64_t t = (int64_t)a.b * a.s1;
    if (t == 0 || a.nq == 0) return hipSuccess;
    if (a.n_blocks == 0) { // a cache without pages holds no token: every output row is zero (and no kernel reads the cache)
        const int64_t words = t * a.nq * 128 / 2;
        hipLaunchKernelGGL(gqa_zero_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, stream,
                           static_cast<uint32_t*>(a.out), words);
        return hipGetLastError();
    }
    {
        ScopedKernelTimer timer(KID_GQA_DECODE, stream);
        // as many units side by side as there can be, but no more than GQA_GRID workgroups
        int64_t stride = (a.units_cap + 7) / 8 * 8;
        const int64_t most = a.row_tiles == 1 ? GQA_GRID : GQA_GRID2;
        if (stride * a.columns > most) {
            stride = std::max<int64_t>(most / a.columns, 1);
            stride = stride >= 8 ? stride / 8 * 8 : stride >= 4 ? 4 : stride >= 2 ? 2 : 1;
        }
        const int64_t groups = stride * a.columns;
        const int64_t gx = groups < (1 << 22) ? groups : (1 << 22);
        auto kern = [&](auto walk) {
            constexpr bool W = decltype(walk)::value;
            return a.row_tiles == 2 ? (a.past_caches ? gqa_decode_kernel<2, W, true> : gqa_decode_kernel<2, W, false>)
                                    : (a.past_caches ? gqa_decode_kernel<1, W, true> : gqa_decode_kernel<1, W, false>);
        };
        hipLaunchKernelGGL((stride < a.units_cap ? kern(std::true_type{}) : kern(std::false_type{})),
                           dim3((unsigned)gx, (unsigned)((groups + gx - 1) / gx)), dim3(256), 0, stream, a, (int)stride);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.nsplit == 1) return e;
    {
        ScopedKernelTimer timer(KID_GQA_COMBINE, stream);
        const int64_t rows = t * a.nq;
        // (eight groups per row for few rows of many chunks: 16 chunks take one group 9 us where rows are few; with many rows the
        // second step costs more than it saves, 20 us against 6 at 6144 rows)
        if (a.units_cap > 12 * (int64_t)a.b && rows <= 2048)
            hipLaunchKernelGGL(gqa_combine_kernel<8>, dim3((unsigned)rows), dim3(256), 0, stream, a);
        else
            hipLaunchKernelGGL(gqa_combine_kernel<1>, dim3((unsigned)((rows + 7) / 8)), dim3(256), 0, stream, a);
    }
    return hipGetLastError();
}

} // namespace pto
