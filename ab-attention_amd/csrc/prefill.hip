// Weighted paged sparse prefill on gfx950 (bf16 MFMA flash attention).
//
// Computes, for every 128-query row of the plan and every valid query i,
//   z_t = q_i . k_t * log2(e)/sqrt(128) + w_j      (key t in KV4 block j)
//   o_i = sum_t 2^(z_t - m) v_t / sum_t 2^(z_t - m),  lse_i = m + log2(sum_t 2^(z_t - m))
// over exactly the row's S listed KV4 blocks (4S keys) of the head's K/V,
// which may be longer or shorter than Q (n_kv tokens). This is the
// ABSipAttention variant of the reference's FlashInfer prefill
// (ab_attention/flashinfer_backend.py:30-59): logits + w / (sm_scale*log2 e),
// then an online softmax in base 2 with scale sm_scale*log2 e.
//
// Kernel shape: one workgroup (4 waves) per row, two workgroups per CU; wave
// w owns queries 32w..32w+31. The row's pages are streamed in tiles of 8 KV4
// blocks (32 keys) through two rings of 4 LDS stages, one for K and one for
// V, that the hardware fills directly from global memory
// (global_load_lds_dwordx4: no staging registers). Each wave moves one
// quarter of every tile and waits only for its own transfers (s_waitcnt
// vmcnt) before the workgroup barrier that publishes them; every transfer
// has three steps to land. The page ids and weights of the row reach LDS the
// same way, 64 tiles at a time, so the loop issues no other global or scalar
// loads; ids and weights are read from LDS one step before their use.
// The loop is software pipelined (see step below): each step issues 16 MFMAs
// of two different tiles and places the softmax VALU work, the LDS operand
// reads and the transfers of other tiles between them, so the MFMA pipe of
// each SIMD is fed while LDS and the vector memory path are busy.
//   S^T = K Q^T  : v_mfma_f32_32x32x16_bf16, A = K rows from LDS, B = Q in VGPRs
//                  -> each lane holds one query and 16 keys, in 4-key groups
//                     that are exactly one KV4 block.
//   O^T += V^T P^T: A = V^T read from the row-major V tile with the
//                  transposing LDS read ds_read_b64_tr_b16, B = P straight
//                  from the S^T accumulators (bf16); the key order of each
//                  MFMA k-step is chosen so no cross-lane movement is needed.
// Softmax reference. A row first runs a fast pass: the reference m of each
// query is the maximum of its logits in the first tile (over both lanes that
// hold the query), and every later tile is exponentiated against it; the
// loop keeps only the running maximum of the logits. p = 2^(z - m) <= 2^64
// then keeps every sum of products far inside the float range, and a term
// more than 2^126 below m is below the resolution of a sum that holds a 1,
// so the result is the normalised softmax. If a query has no finite logit in
// the first tile, or a later logit exceeds m by more than 64, the workgroup
// (after a vote through LDS) discards the pass and runs the row again with a
// moving reference: lazy rescaling, where the reference moves only when a
// tile maximum exceeds it by more than 8. The fast loop carries no rescale
// branch and no per-step exchange between lanes, which leaves more of each
// step's issue slots to the MFMAs (5-6 % less time at the benchmark
// configurations). Where no later tile maximum passes the first tile's by
// more than 8, the lazy pass never moves its reference either, and the two
// passes give the same bits.
// LDS tiles are swizzled so that the operand reads are bank-conflict free. A
// transfer instruction writes 1 KiB contiguously (lane j at +16j), so the
// swizzle is realised by the choice of each lane's source address:
//   K: [key][16 chunks of 16 B], chunk position = chunk ^ (key & 15);
//   V: per page 8 blocks of 4 keys x 16 dims (128 B); inside block m the row
//      of key r sits at position r ^ ((m >> 1) & 3), so each 16-lane group of
//      a transposing read fetches one whole 128-byte block.
// Dense attention (every KV4 block at weight 0, no page list) runs on
// dense_kernel: the same rings, pipeline and two passes on
// v_mfma_f32_16x16x32_bf16 tiles (see there).
// Calls with too few rows to fill the chip split each row's tiles over several
// workgroups (kSplit, prefill_parts), whose float32 partial results
// combine_kernel adds up. In the fast pass the parts after the first take the
// row's reference, from the logits of its first tile (`lead` in the kernels), so
// that every p has the same bf16 bits however a row is split, and a split row
// differs from an unsplit one by the order of its float32 sums only. Rows that
// leave the fast pass round P against other references.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "layout.hpp"

namespace ab {
namespace {

constexpr int kPfThreads = 256;
constexpr int kRing = 4;                                       // stages per ring (K and V)
constexpr int kTilePages = 8;                                  // KV4 blocks per tile
constexpr int kPageBytes = kKvBlock * kHeadDim * 2;            // 1 KiB of K (or V)
constexpr int kTileBytes = kTilePages * kPageBytes;            // 8 KiB: K (or V) of one tile
constexpr int kKRing = 0;
constexpr int kVRing = kRing * kTileBytes;
constexpr int kBatchTiles = 64;                                // ids/weights per LDS batch
constexpr int kBatchBytes = kBatchTiles * kTilePages * 4;      // 2 KiB
constexpr int kIdsOffset = 2 * kRing * kTileBytes;             // 2 batch buffers of ids
constexpr int kWeightsOffset = kIdsOffset + 2 * kBatchBytes;   // 2 batch buffers of weights
constexpr int kVoteOffset = kWeightsOffset + 2 * kBatchBytes;  // 4 words: fast-pass votes
constexpr int kLdsBytes = kVoteOffset + 16;                    // 72 KiB + 16 B
// Split rows: ids and weights (32 bytes each) of the row's first tile, in a
// transfer's 1 KiB, and the stage that its K takes before the loop: V's last,
// which V(3) fills in step 0.
constexpr int kLeadOffset = kLdsBytes;
constexpr int kSplitLdsBytes = kLeadOffset + 1024;
constexpr int kLeadStage = 2 * kRing - 1;
constexpr int kGroupOps = 4;                                   // transfers per wave per step
constexpr int64_t kRowsPerLaunch = 11000;                      // see launch_prefill
// Limits of a split (prefill_parts): units that give each CU one workgroup (at
// most twice that many are made: 33 MiB of workspace), parts of a row and the
// fewest tiles of a part.
constexpr int64_t kPartUnits = 256;
constexpr int64_t kMaxParts = 64;
constexpr int64_t kMinPartTiles = 8;
// Largest p = 2^(y) allowed before the running reference is moved.
constexpr float kSlack = 8.0f;
// Largest logit above the first tile's maximum that the fast pass accepts:
// p <= 2^64 keeps every product and sum far from the float range.
constexpr float kFastRange = 64.0f;

// The dense kernel's LDS: the two rings and the votes.
constexpr int kDenseVoteOffset = 2 * kRing * kTileBytes;
constexpr int kDenseLdsBytes = kDenseVoteOffset + 16;          // 64 KiB + 16 B

static_assert(kSplitLdsBytes * 2 <= 160 * 1024, "two workgroups per CU must fit in LDS");
static_assert(kDenseLdsBytes * 2 <= 160 * 1024, "two dense workgroups per CU must fit in LDS");

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) unsigned char lds_u8;

// Transposing LDS read: within each 16-lane group, lane i receives element
// i%4 of the 8 bytes read by lanes 4r + i/4, for r = 0..3 (so the group reads
// a 4 x 16 tile of 16-bit values, row r from lanes 4r..4r+3, and each lane
// gets one column). lds is an absolute LDS byte address.
__device__ __forceinline__ i16x4 lds_read_tr16(uint32_t lds) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_i16x4*>(static_cast<uintptr_t>(lds)));
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes per lane from base + voffset straight into LDS: lane j writes LDS
// bytes [lds + 16j, lds + 16j + 16). The transfer is counted by vmcnt. The
// kernel holds nothing in m0 across these statements.
__device__ __forceinline__ void dma16(const void* base, uint32_t voffset, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voffset), "s"(base)
                 : "memory", "m0");
}
// The same from an address of its own in each lane.
__device__ __forceinline__ void dma16(const void* address, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(address) : "memory", "m0");
}
#pragma clang diagnostic pop

// s_waitcnt with vmcnt(N) and lgkmcnt(0) (expcnt left open), then a workgroup
// barrier that the compiler cannot move memory accesses across.
template <int N>
__device__ __forceinline__ void wait_and_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
    asm volatile("s_barrier" ::: "memory");
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// v_max_f32 without the NaN quieting the compiler adds around fmaxf of values
// it cannot prove canonical (logits are finite or -inf).
__device__ __forceinline__ float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
#pragma clang diagnostic pop

// Maxima of a (query 0) and b (query 1) over the four lanes i, 16 + i,
// 32 + i, 48 + i that hold a query in dense_kernel: three swaps of 16-lane
// rows (rows of the results: a01 b01 a23 b23, then a b a b, then all a / all b).
__device__ __forceinline__ void max_over_rows(float& a, float& b) {
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    const float m = vmax(__uint_as_float(s[0]), __uint_as_float(s[1]));
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    const float m2 = vmax(__uint_as_float(t[0]), __uint_as_float(t[1]));
    const auto u = __builtin_amdgcn_permlane16_swap(__float_as_uint(m2), __float_as_uint(m2), false, false);
    a = __uint_as_float(u[0]);
    b = __uint_as_float(u[1]);
}

// Bytes from one token's row of a head of K or V to the next. kPacked, for
// tensors whose tokens lie 256 bytes apart (contiguous ones and token slices
// of them), has it at compile time: with one kernel for every stride the c2
// prefill took 24.36 instead of 23.78 ms.
template <bool kPacked>
__device__ __forceinline__ uint32_t token_bytes(const TensorLayout& t) {
    return kPacked ? kHeadDim * 2u : t.token * 8u;
}
// Byte offset of a page. Both factors are under 2^24, so this and the lane's
// offset added to it are one instruction at any stride.
template <bool kPacked>
__device__ __forceinline__ uint32_t page_offset(uint32_t id, uint32_t page_bytes) {
    return kPacked ? id * kPageBytes : __umul24(id, page_bytes);
}

// XCD-aware row order of the prefill kernels. The hardware deals workgroups
// round-robin over the 8 XCDs, so workgroup w runs on XCD w % 8. Slot w / 8
// walks the heads in order: at any time all XCDs work on the same head (its
// K/V stay in the shared last-level cache), each on a contiguous eighth of its
// query blocks (neighbouring blocks share most sampled pages in the XCD's L2).
// Within an XCD, slots s and s + 32 of each full generation of 64 slots run
// on the same CU (two workgroups per CU), so they take adjacent query blocks:
// their sampled pages overlap and they sweep them in step, which turns part of
// the gathers into L1 hits. A launch covers the slots from slot_base (a
// multiple of 64) on, on every XCD. False for a slot past the rows.
struct RowSlot {
    uint32_t b, h;  // batch item and head
    int64_t bh, blk, row;
    __device__ __forceinline__ void set(uint32_t flat, uint32_t block, const Divisor& heads, int64_t qb) {
        b = heads.quotient(flat, h);
        bh = flat;
        blk = block;
        row = bh * qb + blk;
    }
};
// Rows of a call: query blocks per head, the same in one of 8 groups rounded
// up, flattened heads, first slot of the launch.
struct RowGrid {
    uint32_t qb;
    Divisor per_xcd;
    uint32_t bh, slot_base;
};
__device__ __forceinline__ bool row_slot(const RowGrid& g, const Divisor& heads, RowSlot& rs) {
    const uint32_t hw = blockIdx.x;
    const uint32_t xcd = hw & 7, slot0 = g.slot_base + (hw >> 3);
    const uint32_t generation = slot0 >> 6, s64 = slot0 & 63;
    const uint32_t slot = (generation + 1) * 64 <= g.per_xcd.d * g.bh ? generation * 64 + 2 * (s64 & 31) + (s64 >> 5) : slot0;
    uint32_t rest;
    const uint32_t flat = g.per_xcd.quotient(slot, rest), blk = xcd * g.per_xcd.d + rest;
    if (flat >= g.bh || blk >= g.qb) return false;
    rs.set(flat, blk, heads, g.qb);
    return true;
}

// The lists of a sparse call: row r's blocks, ids and log weights
// [rows][samples], then the `tail` blocks that every row attends to as well
// (a prompt behind the video; ids and weights [tail], tail 0 for none).
struct BlockLists {
    const int32_t* ids;
    const float* logw;
    int samples, tail;
    const int32_t* tail_ids;
    const float* tail_logw;
};

// row_slot for rows split into `parts` units each: unit (bh, part, blk), blk
// fastest, each XCD a contiguous eighth of the units. The units of one part
// of a head read the same stretch of its K/V (dense) or sweep the same range
// of their ascending page lists (sparse), so they share it in the XCD's L2.
// `unit` numbers the unit's partial result.
struct UnitSlot : RowSlot {
    int64_t unit;
    int part;
};
__device__ __forceinline__ bool unit_slot(const RowGrid& g, const Divisor& heads, uint32_t parts, UnitSlot& us) {
    const uint32_t units = g.qb * g.bh * parts, per_xcd = (units + 7) / 8;
    const uint32_t hw = blockIdx.x, unit = (hw & 7) * per_xcd + (hw >> 3);
    if ((hw >> 3) >= per_xcd || unit >= units) return false;
    const uint32_t head_part = unit / g.qb, flat = head_part / parts;
    us.set(flat, unit - head_part * g.qb, heads, g.qb);
    us.unit = unit;
    us.part = static_cast<int>(head_part - flat * parts);
    return true;
}
// Tiles [first, first + count) of part `part` of `parts` (parts <= tiles, so
// none is empty).
__device__ __forceinline__ void part_tiles(int tiles, int parts, int part, int& first, int& count) {
    first = static_cast<int>(int64_t(tiles) * part / parts);
    count = static_cast<int>(int64_t(tiles) * (part + 1) / parts) - first;
}

// Partial results of the split kernels, in the caller's workspace: per unit
// the unnormalised O of its 128 queries as 16 fragments of four consecutive
// dims per thread (fragment, thread), 64 KiB, so every store and load is a
// coalesced 16 bytes per lane; then per unit and query (reference m, sum l),
// m = -inf for a query without a finite logit in the unit.
constexpr int kFragments = 16;
constexpr int kCombineFragments = 2;  // fragments per workgroup of combine_kernel
struct Partials {
    f32x4* o;      // [units][kFragments][kPfThreads]
    float2* stat;  // [units][kQueryBlock]
    int parts;
};
struct NoPartials {};
template <bool kSplit>
using PartialsArg = std::conditional_t<kSplit, Partials, NoPartials>;

// The first thing each prefill kernel does: values from all three 64-byte lines
// of its arguments (in host memory) in scalar registers at once, so that the
// lines arrive together. Left to itself the compiler reads the last one, waits,
// then reads the others: 35.2 us against 35.7 at 24 heads x 3,496 tokens and 96
// blocks, 42.3 against 42.9 at 8 x 8,192 and 256.
__device__ __forceinline__ void touch_arguments(const void* q, const PrefillLayout& layout, const RowGrid& grid) {
    asm volatile("" ::"s"(q), "s"(layout.q.batch), "s"(grid.bh));
}

// The sparse prefill: the row's listed KV4 blocks, with their log weights.
// kSplit: one part of the row's tiles, its result left in `partials`. kTail:
// the shared blocks behind the row's own (at compile time: with the choice of
// list in the kernel every call runs, c2 took 23.12 instead of 22.74 ms).
template <bool kSplit, bool kPacked, bool kTail>
__global__ __launch_bounds__(kPfThreads, 2) void prefill_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    BlockLists lists, uint16_t* __restrict__ out,
    float* __restrict__ lse, PrefillLayout layout, int n, RowGrid grid, int fb, float scale_log2,
    const int32_t* __restrict__ order, PartialsArg<kSplit> partials) {
    extern __shared__ __align__(16) unsigned char smem[];
    touch_arguments(q, layout, grid);

    UnitSlot rs;
    int tile0 = 0, tiles = (lists.samples + (kTail ? lists.tail : 0)) / kTilePages;
    if constexpr (kSplit) {
        if (!unit_slot(grid, layout.heads, partials.parts, rs)) return;
        part_tiles(tiles, partials.parts, rs.part, tile0, tiles);
    } else {
        if (!row_slot(grid, layout.heads, rs)) return;
    }
    const int64_t bh = rs.bh, blk = rs.blk, row = rs.row;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qi = lane & 31, half = lane >> 5;
    const int token = static_cast<int>(blk) * kQueryBlock + wave * 32 + qi;
    const bool valid_q = token < n;
    // Row of Q / out / lse holding this token: the token itself, or
    // order[token] for a permuted token layout (clamped into the head).
    const int qrow_index = !valid_q ? 0 : order ? min(max(order[token], 0), n - 1) : token;

    // Q as the B operand of S^T = K Q^T: dims 16s + 8*half .. +8.
    bf16x8 bq[8];
    {
        const uint16_t* qrow = q + layout.q.at(rs.b, rs.h, qrow_index) + 8 * half;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            u32x4 val = {0u, 0u, 0u, 0u};
            if (valid_q) val = *reinterpret_cast<const u32x4*>(qrow + 16 * s);
            bq[s] = __builtin_bit_cast(bf16x8, val);
        }
    }

    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u8*)smem));
    const int32_t* row_ids = lists.ids + row * int64_t(lists.samples);
    const float* row_w = lists.logw + row * int64_t(lists.samples);
    const uint16_t* kbase = k + layout.k.at(rs.b, rs.h, 0);
    const uint16_t* vbase = v + layout.v.at(rs.b, rs.h, 0);
    const uint32_t k_token = token_bytes<kPacked>(layout.k), v_token = token_bytes<kPacked>(layout.v);

    // Batch b of ids and weights (tiles 64b .. 64b+63) into buffer b & 1, by
    // wave 0: two 1 KiB transfers each. Lanes past the row's end re-read its
    // last 16 bytes (those entries are never used). kTail: 16 bytes per lane
    // from the row's list or, past its end, from the tail.
    const uint32_t unit_bytes = static_cast<uint32_t>(tiles) * (kTilePages * 4u);
    auto issue_batch = [&](int b) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t at = min(uint32_t(b) * kBatchBytes + i * 1024u + 16u * lane, unit_bytes - 16u);
            if constexpr (kSplit) at += static_cast<uint32_t>(tile0) * (kTilePages * 4u);
            const uint32_t dst = (b & 1) * kBatchBytes + i * 1024u;
            if constexpr (kTail) {
                const uint32_t row_bytes = static_cast<uint32_t>(lists.samples) * 4u;
                const bool tail = at >= row_bytes;
                const uint32_t off = at - (tail ? row_bytes : 0u);
                dma16(reinterpret_cast<const char*>(tail ? lists.tail_ids : row_ids) + off, lds0 + kIdsOffset + dst);
                dma16(reinterpret_cast<const char*>(tail ? lists.tail_logw : row_w) + off, lds0 + kWeightsOffset + dst);
            } else {
                dma16(row_ids, at, lds0 + kIdsOffset + dst);
                dma16(row_w, at, lds0 + kWeightsOffset + dst);
            }
        }
    };

    // Transfers of this wave: pages 2w and 2w+1 of a K tile and of a V tile.
    // Source offsets inside a page (4 keys x 256 B) for lane j:
    //   K: key r = j/16 at LDS chunk position j%16 holds chunk pos ^ (key & 15);
    //   V: block m = j/8, row slot (j/2)%4 holds key slot ^ ((m>>1)&3), dims 16m + 8(j%2).
    uint32_t k_src[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int r = lane >> 4, pos = lane & 15;
        const int key = 4 * (2 * wave + e) + r;
        k_src[e] = uint32_t(r) * k_token + uint32_t(pos ^ (key & 15)) * 16u;
    }
    const uint32_t v_src = [&] {
        const int m = lane >> 3, sl = (lane >> 1) & 3, h = lane & 1;
        return uint32_t(sl ^ ((m >> 1) & 3)) * v_token + uint32_t(2 * m + h) * 16u;
    }();
    // This wave's two page ids of tile u, clamped into the head (a malformed
    // plan can never address outside it); tiles past the row's end read its
    // last tile (their transfers only keep the per-step count uniform).
    auto load_ids = [&](int u) {
        const int uc = min(u, tiles - 1);
        const u32x2 raw = *reinterpret_cast<const u32x2*>(smem + kIdsOffset + ((uc / kBatchTiles) & 1) * kBatchBytes +
                                                          ((uc % kBatchTiles) * kTilePages + 2 * wave) * 4);
        const u32x2 c = {uint32_t(min(max(static_cast<int>(raw[0]), 0), fb - 1)),
                         uint32_t(min(max(static_cast<int>(raw[1]), 0), fb - 1))};
        return c;
    };
    const uint32_t k_page = kKvBlock * k_token, v_page = kKvBlock * v_token;
    auto dma_k = [&](int u, uint32_t id, int e) {
        dma16(kbase, page_offset<kPacked>(id, k_page) + k_src[e], lds0 + kKRing + (u & (kRing - 1)) * kTileBytes + (2 * wave + e) * kPageBytes);
    };
    auto dma_v = [&](int u, uint32_t id, int e) {
        dma16(vbase, page_offset<kPacked>(id, v_page) + v_src, lds0 + kVRing + (u & (kRing - 1)) * kTileBytes + (2 * wave + e) * kPageBytes);
    };
    // The four block weights of this lane's keys in tile u: lane register r
    // holds key 8*(r/4) + 4*half + r%4, i.e. page 2(r/4) + half.
    auto load_weights = [&](int u, float (&wv)[4]) {
        const int uc = min(u, tiles - 1);
        const float* ws = reinterpret_cast<const float*>(smem + kWeightsOffset +
                                                         ((uc / kBatchTiles) & 1) * kBatchBytes) +
                          (uc % kBatchTiles) * kTilePages;
#pragma unroll
        for (int g = 0; g < 4; ++g) wv[g] = ws[2 * g + half];
    };

    // Operand-read offsets of this lane (stage-relative).
    int k_off[8];  // S^T A operand: key qi, chunk 2s + half
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) k_off[s8] = qi * 256 + 16 * ((2 * s8 + half) ^ (qi & 15));
    int v_off[4];  // PV A operand, transposing read: page half (+4ks + 2t), block 2dt + (lane>>4)&1
    {
        const int gd = (lane >> 4) & 1, r = (lane >> 2) & 3, q4 = lane & 3;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) v_off[dt] = half * 1024 + (2 * dt + gd) * 128 + 32 * (r ^ dt) + 8 * q4;
    }
    // The same as absolute LDS addresses, so every operand read is one
    // register plus the instruction's constant offset (the dynamic-LDS base
    // is not a compile-time constant and would cost an add per read).
    uint32_t k_abs[8], v_abs[4];
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) k_abs[s8] = lds0 + kKRing + k_off[s8];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) v_abs[dt] = lds0 + kVRing + v_off[dt];
    auto read_k = [&](int u, int j) {
        return *reinterpret_cast<const lds_u32x4*>(
            static_cast<uintptr_t>(k_abs[j] + (u & (kRing - 1)) * kTileBytes));
    };
    // PV A operand j of tile u: V^T for k-step j/4, dims 32(j%4) .. +31. MFMA
    // k-index 8*half + 4t + r of k-step ks is key r of tile page 4*ks + 2t +
    // half, on both operands. Lane (group g = lane/16, i = lane%16) does two
    // transposing reads; the source lane 4r + q addresses key r of that page,
    // dims 32dt + 16(g%2) + 4q .. +3, so lane i receives dim 32dt + 16(g%2) + i.
    auto read_v = [&](int u, int j) {
        const uint32_t a0 = v_abs[j & 3] + (u & (kRing - 1)) * kTileBytes + (j >> 2) * 4096;
        const i16x4 lo = lds_read_tr16(a0), hi = lds_read_tr16(a0 + 2048);
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    f32x16 o_acc[4];
    // Reference, running sum and state of this lane's query; mx is the same
    // in both lane halves of a query after the exchange, so they are too.
    float m_run, l_run;
    bool started;

    // Step t works on three tiles at once, so that every MFMA of the wave has
    // independent VALU and LDS work beside it. Entering step t, sc holds the
    // logits y = s*log2(e)/sqrt(d) + (w - m_run) of S(t).
    //   phase A: S(t+1) = K(t+1) Q^T (K(t+1) already in registers), beside
    //            p = 2^y of S(t), the reads of V(t) and this step's four
    //            transfers;
    //   phase B: O += V(t)^T P(t)^T, beside the logits of S(t+1) and the
    //            reads of K(t+2) for the next step.
    // Fast pass (kSafe false): the reference stays where the first tile put
    // it and mx is the running maximum of every logit of the lane, checked
    // after the loop. Safe pass: mx is the maximum of S(t) over this lane's
    // keys and the reference moves only when a tile maximum exceeds it by
    // more than kSlack (so p <= 2^kSlack), decided per wave at the start of
    // the step that exponentiates the tile.
    // Rings: K(u) is read in step u-2 and V(u) in step u. Step t transfers
    // K(t+5) into the stage of K(t+1) and V(t+3) into the stage of V(t-1),
    // both read in step t-1; the barrier at the top of step t retires those
    // reads and publishes K(t+2) and V(t) (transferred in step t-3), so every
    // transfer has three steps. Transfers past the row's end keep the count
    // uniform (4 per wave per step) and land in stages nobody reads again.
    auto step = [&](auto safe, int t, f32x16& sc, f32x16& sn, float& mx, u32x4 (&ka)[8], float (&wn)[4],
                    u32x2& idk, u32x2& idv) {
        constexpr bool kSafe = decltype(safe)::value;
        wait_and_barrier<2 * kGroupOps>();
        if (wave == 0 && t % kBatchTiles == kBatchTiles / 2 && (t / kBatchTiles + 1) * kBatchTiles < tiles)
            issue_batch(t / kBatchTiles + 1);
        if constexpr (kSafe) {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
            const bool was_started = started;
            const bool grow = was_started ? mx > kSlack : mx > -INFINITY;
            started = was_started || grow;
            if (__any(grow)) {
                const float shift = grow ? mx : 0.f;
                // l_run and O are still zero before the first move, so alpha is
                // left at 1 there (2^-mx could overflow for a very negative mx).
                const float alpha = was_started ? fast_exp2(-shift) : 1.f;
                m_run += shift;
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[dt][r] *= alpha;
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] -= shift;
            }
        }
        uint32_t pw[4][2];
        float psum = 0.f;
        bf16x8 va[8];
#pragma unroll
        for (int r = 0; r < 16; ++r) sn[r] = 0.f;
        __builtin_amdgcn_sched_barrier(0);
        // Phase A runs at wave priority 1, phase B at 0: when the SIMD's two
        // waves compete for issue, the one computing the next tile's logits
        // goes first (0.9 % faster at c2 than equal priorities; priority 3,
        // or raising it from the barrier on, was slower).
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ka[j]), bq[j], sn, 0, 0, 0);
            const float p0 = fast_exp2(sc[2 * j]), p1 = fast_exp2(sc[2 * j + 1]);
            psum = j == 0 ? p0 + p1 : (psum + p0) + p1;
            pw[j >> 1][j & 1] = pack_bf16(p0, p1);
            va[j] = read_v(t, j);
            if (j == 1) dma_k(t + 5, idk[0], 0);
            if (j == 3) dma_k(t + 5, idk[1], 1);
            if (j == 5) dma_v(t + 3, idv[0], 0);
            if (j == 7) dma_v(t + 3, idv[1], 1);
            if (j == 2) load_weights(t + 1, wn);
            __builtin_amdgcn_sched_barrier(0);
        }
        l_run += psum;
        float wm[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) wm[g] = wn[g] - m_run;
        if constexpr (kSafe) mx = -INFINITY;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int ks = j >> 2;
            const u32x4 bw = {pw[2 * ks][0], pw[2 * ks][1], pw[2 * ks + 1][0], pw[2 * ks + 1][1]};
            o_acc[j & 3] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[j], __builtin_bit_cast(bf16x8, bw), o_acc[j & 3], 0, 0, 0);
            ka[j] = read_k(t + 2, j);
            const float y0 = __builtin_fmaf(sn[2 * j], scale_log2, wm[j >> 1]);
            const float y1 = __builtin_fmaf(sn[2 * j + 1], scale_log2, wm[j >> 1]);
            sn[2 * j] = y0;
            sn[2 * j + 1] = y1;
            mx = fmaxf(fmaxf(mx, y0), y1);  // one v_max3_f32
            if (j == 6) idk = load_ids(t + 6);
            if (j == 7) idv = load_ids(t + 4);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // One pass over the row's tiles. The fast pass returns whether the
    // workgroup must run the safe pass instead (its result is then
    // discarded): a query with no finite logit in the first tile, or a logit
    // above its reference by more than kFastRange.
    auto pass = [&](auto safe) -> bool {
        constexpr bool kSafe = decltype(safe)::value;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[dt][r] = 0.f;
        m_run = 0.f;
        l_run = 0.f;
        started = false;
        // Prologue: batch 0 of ids/weights (this also completes the Q loads);
        // K(0..3) and V(0..2); S(0) and K(1) into registers once K(0) and K(1)
        // are in; K(4) goes into K(0)'s stage only after every wave has read
        // it. The last eight transfers before step 0 are then K(3), V(1), V(2),
        // K(4), as step 0's wait expects.
        const bool lead = kSplit && !kSafe && tile0 > 0;
        if (wave == 0) {
            if (lead)
                dma16(reinterpret_cast<const char*>(lane & 2 ? static_cast<const void*>(row_w) : row_ids) + 16 * (lane & 1),
                      lds0 + kLeadOffset);
            issue_batch(0);
        }
        wait_and_barrier<0>();
        if (lead) {
            const u32x2 raw = *reinterpret_cast<const u32x2*>(smem + kLeadOffset + 8 * wave);
#pragma unroll
            for (int e = 0; e < 2; ++e)
                dma16(kbase, page_offset<kPacked>(uint32_t(min(max(static_cast<int>(raw[e]), 0), fb - 1)), k_page) + k_src[e],
                      lds0 + kLeadStage * kTileBytes + (2 * wave + e) * kPageBytes);
        }
        {
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                const u32x2 ik = load_ids(u);
                dma_k(u, ik[0], 0);
                dma_k(u, ik[1], 1);
            }
            const u32x2 iv0 = load_ids(0);
            dma_v(0, iv0[0], 0);
            dma_v(0, iv0[1], 1);
            const u32x2 ik3 = load_ids(3);
            dma_k(3, ik3[0], 0);
            dma_k(3, ik3[1], 1);
            const u32x2 iv1 = load_ids(1), iv2 = load_ids(2);
            dma_v(1, iv1[0], 0);
            dma_v(1, iv1[1], 1);
            dma_v(2, iv2[0], 0);
            dma_v(2, iv2[1], 1);
        }
        f32x16 s0, s1;
        u32x4 ka[8];
        // S of the tile in a stage of K's ring (or, from kRing on, V's).
        auto compute_s = [&](int stage) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                ka[j] = *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(k_abs[j] + stage * kTileBytes));
#pragma unroll
            for (int r = 0; r < 16; ++r) s0[r] = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ka[j]), bq[j], s0, 0, 0, 0);
        };
        // The query's reference from its largest logit, over both lane halves; a
        // query without a finite one fails the pass.
        auto set_reference = [&](float mx) {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
            started = mx > -INFINITY;
            m_run = started ? mx : 0.f;
        };
        if (lead) {
            wait_and_barrier<14>();  // the leading tile is in; the 14 transfers after it may be in flight
            compute_s(kLeadStage);
            const float* ws = reinterpret_cast<const float*>(smem + kLeadOffset + 4 * kTilePages);
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, __builtin_fmaf(s0[r], scale_log2, ws[2 * (r >> 2) + half]));
            set_reference(mx);
        }
        const u32x2 ik4 = load_ids(4);
        u32x2 idk = load_ids(5), idv = load_ids(3);
        wait_and_barrier<10>();  // K(0), K(1) in; 10 newer transfers may be in flight
        compute_s(0);
#pragma unroll
        for (int j = 0; j < 8; ++j) ka[j] = read_k(1, j);
        wait_and_barrier<63>();  // every wave's reads of K(0) are done (no transfer wait)
        dma_k(4, ik4[0], 0);
        dma_k(4, ik4[1], 1);
        // Logits of S(0), against reference 0 or the leading tile's.
        float w0[4], mx = -INFINITY;
        load_weights(0, w0);
        if (lead) {
#pragma unroll
            for (int g = 0; g < 4; ++g) w0[g] -= m_run;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s0[r] = __builtin_fmaf(s0[r], scale_log2, w0[r >> 2]);
            mx = fmaxf(mx, s0[r]);
        }
        if constexpr (!kSafe) {
            if (!lead) {
                set_reference(mx);
#pragma unroll
                for (int r = 0; r < 16; ++r) s0[r] -= m_run;
                mx = -INFINITY;
            }
            if (!started) mx = INFINITY;
        }
        // Four steps per iteration: t is a multiple of 4 there, so every ring
        // stage (u & 3) is a compile-time constant and the LDS addresses fold
        // into the instructions' offsets.
        int t = 0;
        for (; t + 3 < tiles; t += 4) {
            step(safe, t, s0, s1, mx, ka, w0, idk, idv);
            step(safe, t + 1, s1, s0, mx, ka, w0, idk, idv);
            step(safe, t + 2, s0, s1, mx, ka, w0, idk, idv);
            step(safe, t + 3, s1, s0, mx, ka, w0, idk, idv);
        }
        for (; t + 1 < tiles; t += 2) {
            step(safe, t, s0, s1, mx, ka, w0, idk, idv);
            step(safe, t + 1, s1, s0, mx, ka, w0, idk, idv);
        }
        if (t < tiles) step(safe, t, s0, s1, mx, ka, w0, idk, idv);
        // No transfer may still be landing when the workgroup's LDS is
        // released or the rings are refilled.
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0)
        if constexpr (kSafe) return false;
        // Workgroup vote: every wave publishes its flag, then all read all.
        const uint32_t bad = __any(mx > kFastRange) ? 1u : 0u;
        uint32_t* votes = reinterpret_cast<uint32_t*>(smem + kVoteOffset);
        if (lane == 0) votes[wave] = bad;
        wait_and_barrier<0>();
        const u32x4 all = *reinterpret_cast<const u32x4*>(votes);
        return (all[0] | all[1] | all[2] | all[3]) != 0u;
    };
    if (pass(std::false_type{})) pass(std::true_type{});

    const auto lsw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    const float l_tot = __uint_as_float(lsw[0]) + __uint_as_float(lsw[1]);
    if constexpr (kSplit) {
        f32x4* dst = partials.o + rs.unit * (kFragments * kPfThreads) + tid;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                dst[(4 * dt + g) * kPfThreads] = f32x4{o_acc[dt][4 * g], o_acc[dt][4 * g + 1], o_acc[dt][4 * g + 2],
                                                       o_acc[dt][4 * g + 3]};
        if (half == 0)
            partials.stat[rs.unit * kQueryBlock + wave * 32 + qi] = float2{started ? m_run : -INFINITY, l_tot};
        return;
    }
    if (valid_q) {
        // A query whose every listed block has weight -inf gets o = 0 and
        // lse = -inf.
        const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
        uint16_t* orow = out + layout.out.at(rs.b, rs.h, qrow_index);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const u32x2 pk = {pack_bf16(o_acc[dt][4 * g] * inv, o_acc[dt][4 * g + 1] * inv),
                                  pack_bf16(o_acc[dt][4 * g + 2] * inv, o_acc[dt][4 * g + 3] * inv)};
                *reinterpret_cast<u32x2*>(orow + 32 * dt + 8 * g + 4 * half) = pk;
            }
        if (lse != nullptr && half == 0) lse[bh * int64_t(n) + qrow_index] = started ? m_run + log2f(l_tot) : -INFINITY;
    }
}

// Dense attention: every KV4 block of K/V in order (tile u holds blocks
// 8u .. 8u+7) at weight 0, blocks past the end at -inf, with no page list in
// memory. Every row of a head reads the same pages in the same order, so the
// gathers come from L2 and the MFMAs bound it; it runs on
// v_mfma_f32_16x16x32_bf16, which takes less energy per FLOP than the
// 32x32x16 form (the sparse kernel, bound by its gathers, keeps that one).
// Same rings, transfers, pipeline and two passes as prefill_kernel; the LDS
// holds the two rings and the votes (no page ids or weights).
//
// MFMA mapping (lane l = 16g + i, i < 16, g < 4): wave w owns queries
// 32w + 16j + i (j = 0, 1).
//   S^T = K Q^T : A = 16 keys x 32 dims (lane: key i, dims 8g..+7 of the
//                 k-step), B = 32 dims x 16 queries (lane: query i, the same
//                 dims); the lane gets keys 4g..4g+3 of each 16-key half kt of
//                 the tile for query i: one whole KV4 block, page 4kt + g.
//   O^T += V^T P^T: A = 16 dims x 32 keys, B = 32 keys x 16 queries; the
//                 MFMA k-index 8g + 4kt + r is key r of page 4kt + g on both
//                 operands, so P goes from the S^T accumulators to the B
//                 operand unmoved, and the A operand is two transposing reads
//                 (pages g and 4 + g).
// A query spans the four lanes i, 16 + i, 32 + i, 48 + i; its maximum and sum
// are combined over them with permlane swaps. V's dim blocks are placed by
// the page's parity (position m ^ (page & 1), through the transfer's source
// addresses): the four 16-lane groups of a transposing read fetch the same
// dim block of four different pages, which then fall in opposite halves of
// the banks.
template <bool kSplit, bool kPacked>
__global__ __launch_bounds__(kPfThreads, 2) void dense_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    uint16_t* __restrict__ out, float* __restrict__ lse, PrefillLayout layout, int n, RowGrid grid, int fb,
    int samples, float scale_log2, PartialsArg<kSplit> partials) {
    extern __shared__ __align__(16) unsigned char smem[];
    touch_arguments(q, layout, grid);
    UnitSlot rs;
    int tile0 = 0, tiles = samples / kTilePages;
    if constexpr (kSplit) {
        if (!unit_slot(grid, layout.heads, partials.parts, rs)) return;
        part_tiles(samples / kTilePages, partials.parts, rs.part, tile0, tiles);
    } else {
        if (!row_slot(grid, layout.heads, rs)) return;
    }
    const int64_t bh = rs.bh, blk = rs.blk;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    auto token_of = [&](int j) { return static_cast<int>(blk) * kQueryBlock + wave * 32 + 16 * j + li; };

    // Q as the B operand of S^T = K Q^T: query 16j + li, dims 32ks + 8lg .. +8.
    bf16x8 bq[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int token = token_of(j);
        const uint16_t* qrow = q + layout.q.at(rs.b, rs.h, min(token, n - 1)) + 8 * lg;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4 val = {0u, 0u, 0u, 0u};
            if (token < n) val = *reinterpret_cast<const u32x4*>(qrow + 32 * ks);
            bq[j][ks] = __builtin_bit_cast(bf16x8, val);
        }
    }

    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u8*)smem));
    const uint16_t* kbase = k + layout.k.at(rs.b, rs.h, 0);
    const uint16_t* vbase = v + layout.v.at(rs.b, rs.h, 0);
    const uint32_t k_token = token_bytes<kPacked>(layout.k), v_token = token_bytes<kPacked>(layout.v);

    // Transfers of this wave: pages 2w + e (e = 0, 1) of a K tile and of a V
    // tile. Source offsets inside a page (4 keys x 256 B) for lane j:
    //   K: key r = j/16 at LDS chunk position j%16 holds chunk pos ^ (key & 15);
    //   V: 128-byte position P = j/8 holds dim block m = P ^ e, key (j/2)%4,
    //      dims 16m + 8(j%2).
    uint32_t k_src[2], v_src[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int r = lane >> 4, pos = lane & 15;
        const int key = 4 * (2 * wave + e) + r;
        k_src[e] = uint32_t(r) * k_token + uint32_t(pos ^ (key & 15)) * 16u;
        const int P = lane >> 3, sl = (lane >> 1) & 3, h = lane & 1;
        v_src[e] = uint32_t(sl) * v_token + uint32_t(2 * (P ^ e) + h) * 16u;
    }
    // This wave's two pages of tile u, clamped into the head; tiles past the
    // row's end read its last tile (their transfers only keep the per-step
    // count uniform).
    auto load_ids = [&](int u) {
        const int id = (tile0 + min(u, tiles - 1)) * kTilePages + 2 * wave;
        const u32x2 c = {uint32_t(min(id, fb - 1)), uint32_t(min(id + 1, fb - 1))};
        return c;
    };
    const uint32_t k_page = kKvBlock * k_token, v_page = kKvBlock * v_token;
    auto dma_k = [&](int u, uint32_t id, int e) {
        dma16(kbase, page_offset<kPacked>(id, k_page) + k_src[e], lds0 + kKRing + (u & (kRing - 1)) * kTileBytes + (2 * wave + e) * kPageBytes);
    };
    auto dma_v = [&](int u, uint32_t id, int e) {
        dma16(vbase, page_offset<kPacked>(id, v_page) + v_src[e], lds0 + kVRing + (u & (kRing - 1)) * kTileBytes + (2 * wave + e) * kPageBytes);
    };
    // The weights of this lane's keys in tile u: pages lg and 4 + lg, 0 inside
    // K/V and -inf past its end.
    auto load_weights = [&](int u, float (&wv)[2]) {
        const int uc = tile0 + min(u, tiles - 1);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) wv[kt] = uc * kTilePages + 4 * kt + lg < fb ? 0.f : -INFINITY;
    };

    // Operand-read addresses of this lane, absolute in LDS, so every read is
    // one register plus the instruction's constant offset (ring stage, key
    // half, dim block). K (A of S^T): key 16kt + li, chunk 4ks + lg at
    // position chunk ^ li. V (A of O^T, transposing read): page lg (+4), dim
    // block dt at position dt ^ (lg & 1), key li/4, dims 4(li%4) .. +3, so
    // lane li receives dim 16dt + li of the page's four keys.
    uint32_t k_abs[4], v_abs[2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) k_abs[ks] = lds0 + kKRing + li * 256 + 16 * ((4 * ks + lg) ^ li);
    {
        const int par = lg & 1, base = kVRing + lg * kPageBytes + 32 * (li >> 2) + 8 * (li & 3);
        v_abs[0] = lds0 + base + par * 128;  // even dt: position dt + par
        v_abs[1] = lds0 + base - par * 128;  // odd dt: position dt - par
    }
    auto read_k = [&](int u, int f) {  // f = 4kt + ks
        return *reinterpret_cast<const lds_u32x4*>(
            static_cast<uintptr_t>(k_abs[f & 3] + (u & (kRing - 1)) * kTileBytes + (f >> 2) * 4096));
    };
    auto read_v_half = [&](int u, int dt, int h) {
        const uint32_t a = v_abs[dt & 1] + (u & (kRing - 1)) * kTileBytes + dt * 128 + h * 4 * kPageBytes;
        return lds_read_tr16(a);
    };

    // O^T accumulators: o[dt][j] holds dims 16dt + 4lg .. +3 of query 16j + li.
    f32x4 o_acc[8][2];
    // Reference, running sum and state of query j. thr[j] is -inf until the
    // query's first finite logit, kSlack after.
    float m_run[2], l_run[2], thr[2];

    // Step t, as in prefill_kernel: phase A computes S(t+1) beside p = 2^y of
    // S(t) (sc[2kt + j]: key half kt, query j), the reads of V(t) and this
    // step's four transfers; phase B computes O += V(t)^T P(t)^T beside the
    // logits of S(t+1) and the reads of K(t+2). Fast pass: mx[0] is the
    // running maximum of every logit of the lane. Safe pass: mx[j] is the
    // maximum of query j over this lane's keys of S(t), and the reference
    // moves lazily (kSlack). Rings and transfer lead as in prefill_kernel.
    auto step = [&](auto safe, int t, f32x4 (&sc)[4], f32x4 (&sn)[4], float (&mx)[2], u32x4 (&ka)[8],
                    float (&wn)[2], u32x2& idk, u32x2& idv) {
        constexpr bool kSafe = decltype(safe)::value;
        wait_and_barrier<2 * kGroupOps>();
        if constexpr (kSafe) {
            max_over_rows(mx[0], mx[1]);
            const bool grow0 = mx[0] > thr[0], grow1 = mx[1] > thr[1];
            if (__any(grow0 || grow1)) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const bool grow = j ? grow1 : grow0;
                    const bool was_started = thr[j] == kSlack;
                    const float shift = grow ? mx[j] : 0.f;
                    // l_run and O are still zero before the first move, so alpha
                    // is left at 1 there (2^-mx could overflow for a very
                    // negative mx).
                    const float alpha = was_started ? fast_exp2(-shift) : 1.f;
                    thr[j] = grow ? kSlack : thr[j];
                    m_run[j] += shift;
                    l_run[j] *= alpha;
#pragma unroll
                    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o_acc[dt][j][r] *= alpha;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) sc[2 * kt + j][r] -= shift;
                }
            }
        }
        uint32_t pw[2][4];
        float psum[2], p_prev = 0.f;
        bf16x8 va[8];
        i16x4 v_lo = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) sn[c][r] = 0.f;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const int ks = x >> 2, kt = (x >> 1) & 1, j = x & 1;
            sn[2 * kt + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ka[4 * kt + ks]),
                                                                     bq[j][ks], sn[2 * kt + j], 0, 0, 0);
            // p of element x of S(t): sc[c][r], c = x/4 = 2kt' + j', r = x%4.
            const int c = x >> 2, r = x & 3;
            const float p = fast_exp2(sc[c][r]);
            if (r == 0) psum[c & 1] = (c >> 1) == 0 ? p : psum[c & 1] + p;
            else psum[c & 1] += p;
            if (x & 1) pw[c & 1][2 * (c >> 1) + (r >> 1)] = pack_bf16(p_prev, p);
            p_prev = p;
            const i16x4 vh = read_v_half(t, x >> 1, x & 1);
            if (x & 1) va[x >> 1] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v_lo, vh, 0, 1, 2, 3, 4, 5, 6, 7));
            else v_lo = vh;
            if (x == 2) dma_k(t + 5, idk[0], 0);
            if (x == 6) dma_k(t + 5, idk[1], 1);
            if (x == 10) dma_v(t + 3, idv[0], 0);
            if (x == 14) dma_v(t + 3, idv[1], 1);
            if (x == 4) load_weights(t + 1, wn);
            __builtin_amdgcn_sched_barrier(0);
        }
        l_run[0] += psum[0];
        l_run[1] += psum[1];
        float wm[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) wm[c] = wn[c >> 1] - m_run[c & 1];
        if constexpr (kSafe) {
            mx[0] = -INFINITY;
            mx[1] = -INFINITY;
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const int dt = x >> 1, j = x & 1;
            const u32x4 bw = {pw[j][0], pw[j][1], pw[j][2], pw[j][3]};
            o_acc[dt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt], __builtin_bit_cast(bf16x8, bw), o_acc[dt][j], 0, 0, 0);
            // The K reads for the next step go out in the first half, so they
            // have landed by the next step's barrier (which waits for them).
            if (x < 8) ka[x] = read_k(t + 2, x);
            if (x & 1) {
                // Logits of elements x-1 and x of S(t+1): sn[c][r], c = x/4.
                const int c = x >> 2, r = x & 3;
                const float y0 = __builtin_fmaf(sn[c][r - 1], scale_log2, wm[c]);
                const float y1 = __builtin_fmaf(sn[c][r], scale_log2, wm[c]);
                sn[c][r - 1] = y0;
                sn[c][r] = y1;
                float& m = mx[kSafe ? (c & 1) : 0];
                m = fmaxf(fmaxf(m, y0), y1);  // one v_max3_f32
            }
            if (x == 12) idk = load_ids(t + 6);
            if (x == 14) idv = load_ids(t + 4);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // One pass over the row's tiles, as in prefill_kernel.
    auto pass = [&](auto safe) -> bool {
        constexpr bool kSafe = decltype(safe)::value;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) o_acc[dt][j][r] = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            m_run[j] = 0.f;
            l_run[j] = 0.f;
            thr[j] = -INFINITY;
        }
        // Prologue: K(0..3) and V(0..2); S(0) and K(1) into registers once
        // K(0) and K(1) are in; K(4) goes into K(0)'s stage only after every
        // wave has read it. The last eight transfers before step 0 are then
        // K(3), V(1), V(2), K(4), as step 0's wait expects. A leading tile comes
        // with Q, before them, so that its logits are computed while they are in
        // flight (4 heads x 256 queries over 4,000 keys: 18.25 us with its
        // transfers just before theirs, 18.15 now, 17.9 without the tile).
        const bool lead = kSplit && !kSafe && tile0 > 0;
        if (lead) {
#pragma unroll
            for (int e = 0; e < 2; ++e)
                dma16(kbase, page_offset<kPacked>(uint32_t(min(2 * wave + e, fb - 1)), k_page) + k_src[e],
                      lds0 + kLeadStage * kTileBytes + (2 * wave + e) * kPageBytes);
        }
        wait_and_barrier<0>();
        {
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                const u32x2 ik = load_ids(u);
                dma_k(u, ik[0], 0);
                dma_k(u, ik[1], 1);
            }
            const u32x2 iv0 = load_ids(0);
            dma_v(0, iv0[0], 0);
            dma_v(0, iv0[1], 1);
            const u32x2 ik3 = load_ids(3);
            dma_k(3, ik3[0], 0);
            dma_k(3, ik3[1], 1);
            const u32x2 iv1 = load_ids(1), iv2 = load_ids(2);
            dma_v(1, iv1[0], 0);
            dma_v(1, iv1[1], 1);
            dma_v(2, iv2[0], 0);
            dma_v(2, iv2[1], 1);
        }
        f32x4 s0[4], s1[4];
        u32x4 ka[8];
        // S of the tile in a stage of K's ring (or, from kRing on, V's).
        auto compute_s = [&](int stage) {
#pragma unroll
            for (int f = 0; f < 8; ++f)
                ka[f] = *reinterpret_cast<const lds_u32x4*>(
                    static_cast<uintptr_t>(k_abs[f & 3] + stage * kTileBytes + (f >> 2) * 4096));
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) s0[c][r] = 0.f;
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                const int ks = x >> 2, kt = (x >> 1) & 1, j = x & 1;
                s0[2 * kt + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ka[4 * kt + ks]),
                                                                         bq[j][ks], s0[2 * kt + j], 0, 0, 0);
            }
        };
        // Each query's reference from its largest logit, over its four lanes; a
        // query without a finite one fails the pass.
        auto set_reference = [&](float (&mx)[2]) {
            max_over_rows(mx[0], mx[1]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bool started = mx[j] > -INFINITY;
                m_run[j] = started ? mx[j] : 0.f;
                thr[j] = started ? kSlack : -INFINITY;
            }
        };
        if (lead) {
            compute_s(kLeadStage);
            float mx[2] = {-INFINITY, -INFINITY};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float w = 4 * (c >> 1) + lg < fb ? 0.f : -INFINITY;
#pragma unroll
                for (int r = 0; r < 4; ++r) mx[c & 1] = fmaxf(mx[c & 1], __builtin_fmaf(s0[c][r], scale_log2, w));
            }
            set_reference(mx);
        }
        const u32x2 ik4 = load_ids(4);
        u32x2 idk = load_ids(5), idv = load_ids(3);
        wait_and_barrier<10>();  // K(0), K(1) in; 10 newer transfers may be in flight
        compute_s(0);
#pragma unroll
        for (int f = 0; f < 8; ++f) ka[f] = read_k(1, f);
        wait_and_barrier<63>();  // every wave's reads of K(0) are done (no transfer wait)
        dma_k(4, ik4[0], 0);
        dma_k(4, ik4[1], 1);
        // Logits of S(0), against reference 0 or the leading tile's.
        float w0[2], mx[2] = {-INFINITY, -INFINITY};
        load_weights(0, w0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float w = lead ? w0[c >> 1] - m_run[c & 1] : w0[c >> 1];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s0[c][r] = __builtin_fmaf(s0[c][r], scale_log2, w);
                mx[c & 1] = fmaxf(mx[c & 1], s0[c][r]);
            }
        }
        if constexpr (!kSafe) {
            if (lead) {
                mx[0] = fmaxf(mx[0], mx[1]);
            } else {
                set_reference(mx);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s0[c][r] -= m_run[c & 1];
                mx[0] = -INFINITY;
            }
            if (thr[0] != kSlack || thr[1] != kSlack) mx[0] = INFINITY;
        }
        int t = 0;
        for (; t + 3 < tiles; t += 4) {
            step(safe, t, s0, s1, mx, ka, w0, idk, idv);
            step(safe, t + 1, s1, s0, mx, ka, w0, idk, idv);
            step(safe, t + 2, s0, s1, mx, ka, w0, idk, idv);
            step(safe, t + 3, s1, s0, mx, ka, w0, idk, idv);
        }
        for (; t + 1 < tiles; t += 2) {
            step(safe, t, s0, s1, mx, ka, w0, idk, idv);
            step(safe, t + 1, s1, s0, mx, ka, w0, idk, idv);
        }
        if (t < tiles) step(safe, t, s0, s1, mx, ka, w0, idk, idv);
        // No transfer may still be landing when the workgroup's LDS is
        // released or the rings are refilled.
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0)
        if constexpr (kSafe) return false;
        // Workgroup vote: every wave publishes its flag, then all read all.
        const uint32_t bad = __any(mx[0] > kFastRange) ? 1u : 0u;
        uint32_t* votes = reinterpret_cast<uint32_t*>(smem + kDenseVoteOffset);
        if (lane == 0) votes[wave] = bad;
        wait_and_barrier<0>();
        const u32x4 all = *reinterpret_cast<const u32x4*>(votes);
        return (all[0] | all[1] | all[2] | all[3]) != 0u;
    };
    if (pass(std::false_type{})) pass(std::true_type{});

#pragma unroll
    for (int j = 0; j < 2; ++j) {
        // Sum over the query's four lanes, in the same order in each of them.
        const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(l_run[j]), __float_as_uint(l_run[j]), false, false);
        const float l16 = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
        const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(l16), __float_as_uint(l16), false, false);
        const float l_tot = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
        const int token = token_of(j);
        if constexpr (kSplit) {
            f32x4* dst = partials.o + rs.unit * (kFragments * kPfThreads) + tid;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) dst[(2 * dt + j) * kPfThreads] = o_acc[dt][j];
            if (lg == 0)
                partials.stat[rs.unit * kQueryBlock + wave * 32 + 16 * j + li] =
                    float2{thr[j] == kSlack ? m_run[j] : -INFINITY, l_tot};
            continue;
        }
        if (token < n) {
            // A query whose every block has weight -inf (none here while K/V
            // is not empty) gets o = 0 and lse = -inf.
            const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
            uint16_t* orow = out + layout.out.at(rs.b, rs.h, token) + 4 * lg;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                const u32x2 pk = {pack_bf16(o_acc[dt][j][0] * inv, o_acc[dt][j][1] * inv),
                                  pack_bf16(o_acc[dt][j][2] * inv, o_acc[dt][j][3] * inv)};
                *reinterpret_cast<u32x2*>(orow + 16 * dt) = pk;
            }
            if (lse != nullptr && lg == 0) lse[bh * int64_t(n) + token] = thr[j] == kSlack ? m_run[j] + log2f(l_tot) : -INFINITY;
        }
    }
}

// Sum of a row's partial results: m = max over its parts, w_p = 2^(m_p - m),
// o = sum w_p o_p / sum w_p l_p, in float32, rounded to bf16 once. Bound by
// reading the partials (64 KiB per unit) or, for few rows, by the latency of
// its loads: workgroup (row, y) takes fragments 2y and 2y + 1, so one row
// spreads over eight workgroups, and the loads of eight parts are in flight
// together. Thread t holds the fragments thread t of the split kernel stored
// (kDense: its layout).
template <bool kDense>
__global__ __launch_bounds__(kPfThreads) void combine_kernel(Partials partials, PrefillLayout layout, uint32_t qb,
                                                             int64_t n, uint16_t* __restrict__ out,
                                                             float* __restrict__ lse,
                                                             const int32_t* __restrict__ order) {
    constexpr int kQueries = kDense ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    RowSlot rs;
    const uint32_t flat = blockIdx.x / qb;
    rs.set(flat, blockIdx.x - flat * qb, layout.heads, qb);
    const int64_t bh = rs.bh, blk = rs.blk;
    const int64_t unit0 = bh * partials.parts * int64_t(qb) + blk;  // part p: unit0 + p * qb
    const int f0 = blockIdx.y * kCombineFragments;
    // Query of the thread's fragment f: 16 (f % 2) + lane % 16 (dense) or lane % 32 of the wave's 32.
    int query[kQueries];
    float m[kQueries], total[kQueries];
#pragma unroll
    for (int j = 0; j < kQueries; ++j) {
        query[j] = wave * 32 + (kDense ? 16 * j + (lane & 15) : lane & 31);
        m[j] = -INFINITY;
        total[j] = 0.f;
    }
#pragma unroll 8
    for (int p = 0; p < partials.parts; ++p)
#pragma unroll
        for (int j = 0; j < kQueries; ++j)
            m[j] = fmaxf(m[j], partials.stat[(unit0 + p * int64_t(qb)) * kQueryBlock + query[j]].x);
    f32x4 acc[kCombineFragments];
#pragma unroll
    for (int e = 0; e < kCombineFragments; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int p = 0; p < partials.parts; ++p) {
        const int64_t unit = unit0 + p * int64_t(qb);
        const f32x4* src = partials.o + unit * (kFragments * kPfThreads) + f0 * kPfThreads + tid;
        f32x4 part[kCombineFragments];
#pragma unroll
        for (int e = 0; e < kCombineFragments; ++e) part[e] = src[e * kPfThreads];
        float w[kQueries];
#pragma unroll
        for (int j = 0; j < kQueries; ++j) {
            const float2 st = partials.stat[unit * kQueryBlock + query[j]];
            // A part without a finite logit for the query adds nothing.
            w[j] = st.x > -INFINITY ? fast_exp2(st.x - m[j]) : 0.f;
            total[j] = __builtin_fmaf(w[j], st.y, total[j]);
        }
#pragma unroll
        for (int e = 0; e < kCombineFragments; ++e)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[e][r] = __builtin_fmaf(w[kDense ? e & 1 : 0], part[e][r], acc[e][r]);
    }
#pragma unroll
    for (int j = 0; j < kQueries; ++j) {
        const int64_t token = blk * kQueryBlock + query[j];
        if (token >= n) continue;
        const int64_t at = order ? min<int64_t>(max(order[token], 0), n - 1) : token;
        uint16_t* orow = out + layout.out.at(rs.b, rs.h, at);
        const float inv = total[j] > 0.f ? 1.0f / total[j] : 0.f;
#pragma unroll
        for (int e = j; e < kCombineFragments; e += kQueries) {
            const int f = f0 + e;
            const int dim = kDense ? 16 * (f >> 1) + 4 * (lane >> 4) : 32 * (f >> 2) + 8 * (f & 3) + 4 * (lane >> 5);
            const u32x2 pk = {pack_bf16(acc[e][0] * inv, acc[e][1] * inv), pack_bf16(acc[e][2] * inv, acc[e][3] * inv)};
            *reinterpret_cast<u32x2*>(orow + dim) = pk;
        }
        if (lse != nullptr && f0 == 0 && lane < (kDense ? 16 : 32))
            lse[bh * n + at] = m[j] > -INFINITY ? m[j] + log2f(total[j]) : -INFINITY;
    }
}

// Plan ids of a permuted token layout -> KV4 pages of the stored layout:
// out[i] = map[clamp(ids[i])]. Bound by the ids' read and write (12.6 million
// ids, out of the caches: 34.0 us one id per thread, 20.5 four, at 4.9 TB/s) and,
// below about a million, by the launch and one load after another (14,336 ids
// 2.5 -> 1.9 us, 400,000 3.0 -> 2.0). Each thread takes 4 ids with 16-byte loads
// and stores where ids and out lie on 16 bytes; four such groups per thread left
// small calls with few workgroups (14,336 ids 2.4 us) and gained nothing on large
// ones (22.8).
template <bool kAligned>
__global__ __launch_bounds__(256) void remap_ids_kernel(const int32_t* __restrict__ ids, int64_t count,
                                                        const int32_t* __restrict__ map, int map_len,
                                                        int32_t* __restrict__ out) {
    typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
    const int64_t first = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
    auto mapped = [&](int32_t id) { return map[min(max(id, 0), map_len - 1)]; };
    if (kAligned && first + 4 <= count) {
        const i32x4 v = *reinterpret_cast<const i32x4*>(ids + first);
        const i32x4 r = {mapped(v[0]), mapped(v[1]), mapped(v[2]), mapped(v[3])};
        *reinterpret_cast<i32x4*>(out + first) = r;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (first + e < count) out[first + e] = mapped(ids[first + e]);
}

// Merge of two attention states over disjoint key sets (base-2 LSEs), as
// FlashInfer's merge_state: m = max(s_a, s_b), w = 2^(s - m),
// o = (o_a w_a + o_b w_b) / (w_a + w_b), s = m + log2(w_a + w_b), in fp32.
// One thread per 8 dims (16 bytes) of one query's 128-dim row.
__global__ __launch_bounds__(256) void merge_kernel(const uint16_t* __restrict__ oa, const float* __restrict__ sa,
                                                   const uint16_t* __restrict__ ob, const float* __restrict__ sb,
                                                   int64_t count, uint16_t* __restrict__ out,
                                                   float* __restrict__ s_out) {
    const int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t row = idx >> 4, part = idx & 15;
    if (row >= count) return;
    const float a = sa[row], b = sb[row];
    const float m = fmaxf(a, b);
    const float wa = fast_exp2(a - m), wb = fast_exp2(b - m);
    const float d = wa + wb, inv = 1.0f / d;
    const u32x4 va = reinterpret_cast<const u32x4*>(oa + row * kHeadDim)[part];
    const u32x4 vb = reinterpret_cast<const u32x4*>(ob + row * kHeadDim)[part];
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float lo = (bf16_lo(va[e]) * wa + bf16_lo(vb[e]) * wb) * inv;
        const float hi = (bf16_hi(va[e]) * wa + bf16_hi(vb[e]) * wb) * inv;
        r[e] = pack_bf16(lo, hi);
    }
    reinterpret_cast<u32x4*>(out + row * kHeadDim)[part] = r;
    if (s_out != nullptr && part == 0) s_out[row] = m + log2f(d);
}

}  // namespace

int launch_merge(const void* oa, const float* sa, const void* ob, const float* sb, int64_t count, void* out,
                 float* s_out, hipStream_t stream) {
    if (count == 0) return 0;
    const int64_t threads = count * 16;
    hipLaunchKernelGGL(merge_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const uint16_t*>(oa), sa, static_cast<const uint16_t*>(ob), sb, count,
                       static_cast<uint16_t*>(out), s_out);
    return check_launch("merge_kernel");
}

int launch_remap_ids(const int32_t* ids, int64_t count, const int32_t* map, int64_t map_len, int32_t* out,
                     hipStream_t stream) {
    if (count == 0) return 0;
    constexpr int64_t kPerBlock = 256 * 4;
    const bool aligned = ((reinterpret_cast<uintptr_t>(ids) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
    hipLaunchKernelGGL(aligned ? remap_ids_kernel<true> : remap_ids_kernel<false>,
                       dim3(static_cast<unsigned>((count + kPerBlock - 1) / kPerBlock)), dim3(256), 0, stream, ids,
                       count, map, static_cast<int>(map_len), out);
    return check_launch("remap_ids_kernel");
}

// Row slots per XCD that one prefill launch covers (a whole number of
// generations of 64 slots): the rows of a call are split into launches of
// about kRowsPerLaunch rows each.
int64_t prefill_launch_slots(int64_t bh, int64_t n) {
    const int64_t qb = (n + kQueryBlock - 1) / kQueryBlock;
    const int64_t rows = bh * qb;
    const int64_t generations = ((qb + 7) / 8 * bh + 63) / 64;
    const int64_t launches = std::max<int64_t>(1, (rows + kRowsPerLaunch - 1) / kRowsPerLaunch);
    return (generations + launches - 1) / launches * 64;
}

// Parts each row's tiles are split into: 1 unless the rows leave much of the
// chip idle. A call's units (rows * parts) run at once while there are at most
// 512 (two workgroups per CU); the time of a tile step then grows from 0.49 us
// (a few lone workgroups) over 0.58 (one on every CU) to 0.88 (two), measured
// on dense calls of 24 to 3,072 rows, and a unit costs its tiles plus a
// prologue and epilogue worth about 8, with the row's reference where it is
// split (0.1 to 0.3 us). Splitting adds combine_kernel (6 us)
// and its 128 KiB of traffic per unit (0.03 us); dense units cannot run faster
// than their K/V arrive (5.5 TB/s). More units than 512 lose: their rounds do
// not start together and share less of what they read (640 dense rows of 512
// tiles: 680 us, in 2 parts 618, but 640 sparse rows of 128: 211 and 238), so
// calls of more than 256 rows never split. Measured, unsplit and at the parts
// this picks: dense 24 rows x 3,715 tiles 1,874 -> 299 us, 48 x 3,721 1,815 ->
// 415, 4 x 1,024 504 -> 37, 256 x 512 282 -> 251; sparse 64 x 64 37.9 -> 24.7,
// 16 x 128 68.9 -> 21.7.
int prefill_parts(int64_t rows, int64_t tiles, int64_t kv_bytes) {
    constexpr double kSetupSteps = 8, kCombine = 6, kUnitTraffic = 0.03, kBytesPerUs = 5.5e6, kGain = 0.95;
    auto cost = [&](int64_t parts) {
        const double units = double(rows * parts), wide = double(kPartUnits);
        const double step = units <= wide ? 0.49 + 0.09 * units / wide : 0.58 + 0.30 * (units / wide - 1.0);
        const double run = step * (double((tiles + parts - 1) / parts) + kSetupSteps);
        return std::max(run, double(kv_bytes) / kBytesPerUs) + (parts > 1 ? kCombine + kUnitTraffic * units : 0.0);
    };
    int best = 1;
    if (rows > kPartUnits) return best;
    double best_cost = kGain * cost(1);
    for (int64_t parts = 2; parts <= kMaxParts && parts * kMinPartTiles <= tiles && rows * parts <= 2 * kPartUnits; ++parts)
        if (cost(parts) < best_cost) {
            best = static_cast<int>(parts);
            best_cost = cost(parts);
        }
    return best;
}

namespace {
int call_parts(bool dense, int64_t bh, int64_t n, int64_t n_kv, int64_t samples) {
    return prefill_parts(bh * ((n + kQueryBlock - 1) / kQueryBlock), samples / kTilePages,
                         dense ? bh * n_kv * kHeadDim * 4 : 0);
}
}  // namespace

size_t prefill_workspace_bytes(bool dense, int64_t bh, int64_t n, int64_t n_kv, int64_t samples) {
    const int parts = call_parts(dense, bh, n, n_kv, samples);
    const size_t units = size_t(bh) * ((n + kQueryBlock - 1) / kQueryBlock) * parts;
    return parts == 1 ? 0 : units * (kFragments * kPfThreads * sizeof(f32x4) + kQueryBlock * sizeof(float2));
}

int launch_prefill(const PrefillCall& c, hipStream_t stream) {
    const bool dense = c.dense;
    const int64_t bh = c.batch * c.layout.heads.d, n = c.q_tokens, n_kv = c.kv_tokens, samples = c.samples;
    const int64_t qb = (n + kQueryBlock - 1) / kQueryBlock;
    const int64_t rows = bh * qb;
    if (samples % kTilePages != 0 || c.tail_samples % kTilePages != 0)
        return set_error(1, "prefill: samples (%lld) must be a multiple of %d", (long long)samples, kTilePages);
    if (!dense)
        for (const void* p : {static_cast<const void*>(c.ids), static_cast<const void*>(c.log_weights),
                              static_cast<const void*>(c.tail_ids), static_cast<const void*>(c.tail_log_weights)})
            if (reinterpret_cast<uintptr_t>(p) & 15u)
                return set_error(1, "prefill: ids and log_weights must be 16-byte aligned");
    // The kernels address a head of K/V with 32-bit byte offsets made of 24-bit factors.
    for (const TensorLayout* t : {&c.layout.k, &c.layout.v})
        if (int64_t(t->token) * 8 * kKvBlock >= (1 << 24) || n_kv / kKvBlock >= (1 << 24) ||
            n_kv * t->token * 8 > int64_t(0xffffffff))
            return set_error(1, "prefill: one head of K/V must be under 4 GiB");
    const float scale_log2 = static_cast<float>(1.4426950408889634 / 11.313708498984761);  // log2(e)/sqrt(128)
    const int64_t per_xcd = (qb + 7) / 8;
    if (rows == 0) return 0;
    const int parts = c.workspace ? call_parts(dense, bh, n, n_kv, samples + c.tail_samples) : 1;
    const int lds_bytes = dense ? kDenseLdsBytes : parts > 1 ? kSplitLdsBytes : kLdsBytes;
    const int fb = static_cast<int>(n_kv / kKvBlock), s = static_cast<int>(samples);
    const dim3 block(kPfThreads);
    uint16_t* out = static_cast<uint16_t*>(c.out);
    const BlockLists lists{c.ids, c.log_weights, s, static_cast<int>(c.tail_samples), c.tail_ids, c.tail_log_weights};
    auto launch_as = [&](auto split, auto packed, int64_t workgroups, int64_t slot_base, auto partials) -> int {
        const RowGrid rows_of{static_cast<uint32_t>(qb), divisor(static_cast<uint32_t>(per_xcd)),
                              static_cast<uint32_t>(bh), static_cast<uint32_t>(slot_base)};
        constexpr bool kSplit = decltype(split)::value, kPacked = decltype(packed)::value;
        const auto dense_fn = dense_kernel<kSplit, kPacked>;
        const auto sparse_fn = c.tail_samples ? prefill_kernel<kSplit, kPacked, true> : prefill_kernel<kSplit, kPacked, false>;
        const void* kernel = dense ? reinterpret_cast<const void*>(dense_fn) : reinterpret_cast<const void*>(sparse_fn);
        if (int rc = ensure_lds_limit(kernel, lds_bytes)) return rc;
        const dim3 grid(static_cast<unsigned>(workgroups));
        if (dense)
            hipLaunchKernelGGL(dense_fn, grid, block, lds_bytes, stream,
                               static_cast<const uint16_t*>(c.q), static_cast<const uint16_t*>(c.k),
                               static_cast<const uint16_t*>(c.v), out, c.lse, c.layout, static_cast<int>(n), rows_of, fb, s, scale_log2,
                               partials);
        else
            hipLaunchKernelGGL(sparse_fn, grid, block, lds_bytes, stream,
                               static_cast<const uint16_t*>(c.q), static_cast<const uint16_t*>(c.k),
                               static_cast<const uint16_t*>(c.v), lists, out, c.lse, c.layout, static_cast<int>(n),
                               rows_of, fb, scale_log2, c.order, partials);
        return check_launch(dense ? "dense_kernel" : "prefill_kernel");
    };
    const bool packed = c.layout.k.token == kHeadDim / 4 && c.layout.v.token == kHeadDim / 4;
    auto launch = [&](auto split, int64_t workgroups, int64_t slot_base, auto partials) {
        return packed ? launch_as(split, std::true_type{}, workgroups, slot_base, partials)
                      : launch_as(split, std::false_type{}, workgroups, slot_base, partials);
    };
    if (parts > 1) {
        const int64_t units = rows * parts;
        Partials partials;
        partials.o = static_cast<f32x4*>(c.workspace);
        partials.stat = reinterpret_cast<float2*>(partials.o + units * kFragments * kPfThreads);
        partials.parts = parts;
        if (int rc = launch(std::true_type{}, (units + 7) / 8 * 8, 0, partials)) return rc;
        const dim3 grid(static_cast<unsigned>(rows), kFragments / kCombineFragments);
        if (dense)
            hipLaunchKernelGGL(combine_kernel<true>, grid, block, 0, stream, partials, c.layout, static_cast<uint32_t>(qb), n, out, c.lse,
                               nullptr);
        else
            hipLaunchKernelGGL(combine_kernel<false>, grid, block, 0, stream, partials, c.layout, static_cast<uint32_t>(qb), n, out, c.lse,
                               c.order);
        return check_launch("combine_kernel");
    }
    // The rows are launched in chunks of about kRowsPerLaunch, each a whole
    // number of generations (64 row slots per XCD; a generation is what the
    // chip holds at once, two workgroups per CU). The rows resident on an XCD
    // sweep their (ascending) page lists at the same pace only while they
    // started together; over a long launch their start times spread out, the
    // pages they touch at one moment spread over the whole head and the XCD's
    // L2 stops serving them. A new launch lines them up again (at c2, one
    // launch: 25.0 ms; five launches of whole heads: 23.9 ms, bit-identical),
    // and whole generations leave no half-empty generation in each launch.
    const int64_t slots = per_xcd * bh;                    // row slots per XCD
    const int64_t per_launch = prefill_launch_slots(bh, n);
    for (int64_t slot_base = 0; slot_base < slots; slot_base += per_launch) {
        const int64_t count = std::min(per_launch, slots - slot_base);
        if (int rc = launch(std::false_type{}, count * 8, slot_base, NoPartials{})) return rc;
    }
    return 0;
}

}  // namespace ab
