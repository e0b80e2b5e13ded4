// IBCS on gfx950: query clustering + key pooling, centroid/key pair-LSE with
// per-centroid normalisers, and population-weighted block masses.
//
// Dataflow (one head chunk, the caller's workspace holds every intermediate):
//   cluster_pool_kernel  Q,K -> scaled centroids [rows,8,128] bf16, populations
//                        [rows,8] f32, pooled keys [bh,fb,2,128] bf16
//   (lse.hip)            centroids x pooled keys (bf16 MFMA) -> fp16 pair-LSE
//                        [rows,8,ld] and (max, den) [rows,8]
//   masses_kernel        pair-LSE + normalisers + populations -> scores [rows,fb]
//
// Reference stages: csrc/ibcs.cu:106-238 (cluster), :244-266 (pool),
// :329-489 (LSE), :495-538 (scores). Exactness notes:
//   - cluster/pool follow the reference's fp32 operation order (lane-strided
//     fmaf chains, xor-butterfly sums, row-order centroid sums, IEEE division),
//     so they match the CPU oracle bit for bit;
//   - pair-LSE uses one exp2 and one log2 per (centroid, block):
//     exp2(a-mx) + exp2(b-mx) == 1 + exp2(min-mx) because exp2(0) == 1. The
//     reference's max(sum, 1e-20) floor never binds for finite inputs (sum >= 1);
//   - the normaliser D is accumulated tile by tile from the fp16-rounded values
//     (online max/rescale), matching the reference up to fp32 rounding order.
#include <cfloat>
#include <type_traits>

#include "common.hpp"
#include "layout.hpp"
#include "masses.hpp"

namespace ab {
namespace {

// ---------------------------------------------------------------------------
// Stage 1+2: clustering of one 128-query block and pooling of the same 128
// key tokens. One workgroup of 128 threads per (query block, head): thread i
// owns query i (its row kept in 128 VGPRs as f32); thread d owns dim d in the
// mean, which reads the block from LDS one 64-row half at a time (17 KB of LDS
// and 164 VGPRs: three waves per SIMD).
//
// Bound by VALU issue on a full chip (nine distance passes of 256 sub/fma per
// query are over half of it) and by the chain of passes, reductions and
// barriers of one workgroup (22 us) on a small call. Centre rows come through
// scalar loads instead of being published in LDS, the argmax stays in
// registers (DPP), and the member sums split the slots between the waves:
// 80 heads x 75,600 tokens 1,061 -> 887 us, 12 x 32,760 97 -> 81 us, 2 x 2,048
// 26.8 -> 21.7 us (18.3 with two lanes per query, below).

// Calls with few query blocks run the same with kLanes = 2 lanes per query
// (256 threads): lanes l and l + 32 of a wave hold one query, 16 of its 32
// chains each (the even and the odd ones: the two halves of the distance's
// tree).

constexpr int kHalfRows = 64;
constexpr int kRowWords = kHeadDim / 2 + 1;  // padded bf16 row: 65 dwords

// The reference's distance (csrc/ibcs.cu:143-155, :171-181) is 32 partial
// chains, chain l = fmaf over dims l, l+32, l+64, l+96, summed by the xor
// butterfly 16,8,4,2,1 (every lane of a butterfly ends with the pairwise
// tree). That tree is evaluated depth first here: its k-th leaf is chain
// bitrev5(k), and a leaf's value is added to the pending partial of each
// level its index completes, so one partial per level is live instead of
// 32. The additions are the tree's, so the bits are the same.
__host__ __device__ constexpr int leaf_chain(int k) {
    return ((k & 1) << 4) | ((k & 2) << 2) | (k & 4) | ((k & 8) >> 2) | ((k & 16) >> 4);
}
// Rows are held in leaf order, the four dims of a chain together: element
// [k][r] of a row is dim leaf_chain(k) + 32r. A query's row sits in 32 f32x4
// registers that way, and the mean's row in LDS (one 16-byte read or write
// per chain).
__device__ __forceinline__ int center_pos(int d) { return 4 * leaf_chain(d & 31) + (d >> 5); }

// Sum of the tree over this lane's 32 / kLanes leaves, leaf k being the chain
// over the differences delta(k, r), r = 0..3. With two lanes the halves meet in
// the last addition.
template <int kLanes, class Delta>
__device__ __forceinline__ float chain_tree(Delta delta) {
    constexpr int kLeaves = 32 / kLanes, kLevels = kLanes == 1 ? 5 : 4;
    float pending[kLevels + 1];
#pragma unroll
    for (int k = 0; k < kLeaves; ++k) {
        float acc = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float d = delta(k, r);
            acc = __builtin_fmaf(d, d, acc);
        }
        float v = acc;
        int level = 0;
#pragma unroll
        for (int b = 0; b < kLevels; ++b)
            if (((k >> b) & 1) && level == b) {
                v = pending[b] + v;
                level = b + 1;
            }
        pending[level] = v;
    }
    if constexpr (kLanes == 1) return pending[kLevels];
    const uint32_t half = __float_as_uint(pending[kLevels]);
    const auto both = __builtin_amdgcn_permlane32_swap(half, half, false, false);
    return __uint_as_float(both[0]) + __uint_as_float(both[1]);
}

// Distance of the lane's query to a row in LDS, leaf order (center: this
// lane's half of it).
template <int kLanes>
__device__ __forceinline__ float lane_distance(const f32x4 (&x)[32 / kLanes], const float* __restrict__ center) {
    f32x4 c;
    return chain_tree<kLanes>([&](int k, int r) {
        if (r == 0) c = *reinterpret_cast<const f32x4*>(center + 4 * k);
        return x[k][r] - c[r];
    });
}

// v_perm_b32 selector of four zero bytes.
constexpr uint32_t kZeroSelect = 0x0c0c0c0cu;

// The same to a query row that every lane shares, read through the scalar
// cache straight into scalar registers (packed: the row's 64 bf16 pairs in
// global memory, wave-uniform address): no LDS reads, and no store and barrier
// to publish the row first. With two lanes per query each picks its half of a
// pair with one v_perm_b32 (sel). Not inside: a zero row in its place, by the
// same instructions with zeros as their selector, mask and factor (a branch to
// code of its own took plans of 1,300 blocks from 112.3 to 112.9 us).
template <int kLanes>
__device__ __forceinline__ float lane_distance_to_row(const f32x4 (&x)[32 / kLanes],
                                                     const uint32_t* __restrict__ packed, uint32_t sel, bool inside) {
    const uint32_t hi_mask = inside ? 0xffff0000u : 0u, lo_factor = inside ? 0x10000u : 0u;
    if (!inside) sel = kZeroSelect;
    return chain_tree<kLanes>([&](int k, int r) {
        const int dim = leaf_chain(k);
        const uint32_t pair = packed[(dim >> 1) + 16 * r];
        const float c = kLanes == 2 ? __uint_as_float(__builtin_amdgcn_perm(pair, pair, sel))
                        : (dim & 1) ? __uint_as_float(pair & hi_mask)
                                    : __uint_as_float(pair * lo_factor);
        return x[k][r] - c;
    });
}

// Maximum over the wave's lanes, in every lane: DPP row shifts and row
// broadcasts leave it in lane 63 (a few cycles each; a shuffle goes through the
// LDS unit).
__device__ __forceinline__ float wave_max(float v) {
    // Lanes without a source take their own value.
    auto step = [&](auto ctrl, auto rows) {
        const int own = __float_as_int(v);
        v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(own, own, decltype(ctrl)::value, decltype(rows)::value,
                                                               0xf, false)));
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});  // row_shr:1
    step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});  // row_shr:2
    step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});  // row_shr:4
    step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});  // row_shr:8
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});  // row_bcast:15 into rows 1 and 3
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});  // row_bcast:31 into rows 2 and 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Block-wide argmax over the queries' values: largest value, lowest query on
// ties (cub::ArgMax semantics, csrc/ibcs.cu:94-102), valid in every thread.
// Per wave: the maximum (exact, whatever its order), then the lowest lane
// holding it from a ballot; the waves meet in LDS. One barrier: the caller
// places another barrier between this call and the next (the LDS slots are
// reused).
template <int kLanes>
__device__ __forceinline__ int block_argmax(float value, float* s_val, int* s_idx) {
    const float m = wave_max(value);
    const uint64_t hit = __ballot(value == m);  // empty only if every value is NaN
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s_val[wave] = m;
        s_idx[wave] = 64 / kLanes * wave + (hit != 0u ? static_cast<int>(__builtin_ctzll(hit)) : 0);
    }
    __syncthreads();
    // Queries 0-63 and 64-127; of equal values the first holds the lower index.
    float v[2];
    int idx[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        v[h] = s_val[kLanes * h];
        idx[h] = s_idx[kLanes * h];
        if constexpr (kLanes == 2) {
            const float other = s_val[2 * h + 1];
            // Only NaNs in a wave: any number of the other one wins.
            if (other > v[h] || (v[h] != v[h] && other == other)) {
                v[h] = other;
                idx[h] = s_idx[2 * h + 1];
            }
        }
    }
    return v[1] > v[0] ? idx[1] : idx[0];
}

// Byte selector of v_perm_b32 that moves the bf16 of dim `dim` of a packed
// pair into the high half of a float (low half zero): bytes 1,0 for an even
// dim, 3,2 for an odd one (0x0c selects a zero byte).
__device__ __forceinline__ uint32_t bf16_select(int dim) { return (dim & 1) ? 0x03020c0cu : 0x01000c0cu; }

// One dim of a staged row, with the selector precomputed: one v_perm_b32.
__device__ __forceinline__ float block_elem_sel(const uint32_t* block, int row, int word, uint32_t sel) {
    const uint32_t w = block[row * kRowWords + word];
    return __uint_as_float(__builtin_amdgcn_perm(w, w, sel));
}

template <int kLanes>
__global__ __launch_bounds__(kQueryBlock* kLanes) __attribute__((amdgpu_waves_per_eu(3, 3))) void cluster_pool_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    QkLayout layout, uint16_t* __restrict__ centroids, float* __restrict__ pops, uint16_t* __restrict__ pooled,
    int64_t n, int64_t qb, float qk_scale_log2, const int32_t* __restrict__ order) {
    __shared__ uint32_t half_block[(kHalfRows + 1) * kRowWords];  // 64 rows and a row of zeros
    __shared__ __align__(16) float center_row[kHeadDim];
    constexpr int kWaves = 2 * kLanes, kWaveQueries = 64 / kLanes, kLeaves = 32 / kLanes;
    __shared__ float s_val[kWaves];
    __shared__ int s_idx[kWaves];
    __shared__ uint32_t slot_mask[4][kCentroids];  // members among queries 32i .. 32i + 31

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The lane's query and its half of the dims (kLanes = 2: even or odd).
    const int query = kWaveQueries * wave + (lane & (kWaveQueries - 1));
    const int part = kLanes == 2 ? lane >> 5 : 0;
    const int64_t blk = blockIdx.x, bh = blockIdx.y;
    const int64_t base = blk * kQueryBlock;
    const int valid = static_cast<int>(min<int64_t>(kQueryBlock, n - base));
    const int64_t row = bh * qb + blk;

    // Loads, all issued before any is used: the key pairs this thread pools
    // (16 bytes of pairs tid/16 + 8i, i < 8) and this thread's own query row
    // (256 bytes). Token t of the head is stored row t, or order[t] for a
    // permuted token layout (clamped into the head); rows past the sequence
    // end are clamped and their data discarded. Offsets are in 16-byte units
    // from the head's base (32-bit, checked by the launcher).
    uint32_t h;
    const uint32_t b = layout.heads.quotient(layout.first_head + blockIdx.y, h);
    const u32x4* qhead = reinterpret_cast<const u32x4*>(q + layout.q.at(b, h, 0));
    const u32x4* khead = reinterpret_cast<const u32x4*>(k + layout.k.at(b, h, 0));
    const uint32_t q_row = layout.q.token / 2u, k_row = layout.k.token / 2u;
    const int c16 = tid & 15, r0 = tid >> 4;
    const int pairs = valid / 2;
    const int nm1 = static_cast<int>(n - 1), b32 = static_cast<int>(base);
    auto stored = [&](int t, uint32_t row) {  // t: token index inside the block; its offset
        const int tok = b32 + min(t, valid - 1);
        return uint32_t(__umul24(order ? min(max(order[tok], 0), nm1) : tok, row));
    };
    constexpr int kPairs = 8 / kLanes;  // key pairs per thread
    u32x4 ka[kPairs], kb[kPairs];
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
        const int p = r0 + 8 * kLanes * i;
        ka[i] = khead[stored(2 * p, k_row) + c16];
        kb[i] = khead[stored(2 * p + 1, k_row) + c16];
    }
    const uint32_t part_sel = bf16_select(part);
    f32x4 x[kLeaves];
    {
        const uint32_t qoff = stored(query, q_row);
        u32x4 qv[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) qv[j] = qhead[qoff + j];
        // Pool the keys: bf16(0.5 * (k_2r + k_2r+1)) (:244-266).
        u32x4* kdst = reinterpret_cast<u32x4*>(pooled + (bh * (n / 2) + base / 2) * kHeadDim);
#pragma unroll
        for (int i = 0; i < kPairs; ++i) {
            const int p = r0 + 8 * kLanes * i;
            if (p < pairs) {
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = 0.5f * (bf16_lo(ka[i][e]) + bf16_lo(kb[i][e]));
                    const float hi = 0.5f * (bf16_hi(ka[i][e]) + bf16_hi(kb[i][e]));
                    o[e] = pack_bf16(lo, hi);
                }
                kdst[p * 16 + c16] = o;
            }
        }
        // Queries past the sequence end are zero rows.
        const bool zero_row = query >= valid;
#pragma unroll
        for (int j = 0; j < 16; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t w = zero_row ? 0u : qv[j][e];
                const int d = 8 * j + 2 * e;
                if constexpr (kLanes == 1) {
                    x[leaf_chain(d & 31)][d >> 5] = bf16_lo(w);
                    x[leaf_chain((d + 1) & 31)][(d + 1) >> 5] = bf16_hi(w);
                } else {
                    x[leaf_chain(d & 31)][d >> 5] = __uint_as_float(__builtin_amdgcn_perm(w, w, part_sel));
                }
            }
    }

    if (tid < kRowWords) half_block[kHalfRows * kRowWords + tid] = 0u;  // read after the barriers below
    // The rows of half h (queries 64h .. 64h+63) into LDS, written by the waves
    // that hold them: v_perm_b32 takes the high halves of two floats, which
    // gives back the loaded bf16 pair bit for bit. With two lanes per query
    // they swap halves of words w and w + 32, and write one of them each.
    auto stage_half = [&](int h) {
        if (wave / kLanes == h) {
            uint32_t* dst = half_block + (query & 63) * kRowWords + 32 * part;
            auto value = [&](int d) { return __float_as_uint(x[leaf_chain(d & 31)][d >> 5]); };
            if constexpr (kLanes == 1) {
#pragma unroll
                for (int w = 0; w < kHeadDim / 2; ++w)
                    dst[w] = __builtin_amdgcn_perm(value(2 * w + 1), value(2 * w), 0x07060302u);
            } else {
#pragma unroll
                for (int w = 0; w < kHeadDim / 4; ++w) {
                    const auto s = __builtin_amdgcn_permlane32_swap(value(2 * w), value(2 * w + 64), false, false);
                    dst[w] = __builtin_amdgcn_perm(s[1], s[0], 0x07060302u);
                }
            }
        }
        __syncthreads();
    };

    // Per-dim mean over valid queries in row order (csrc/ibcs.cu:130-140):
    // thread d < 128 owns dim d, its word of a packed row and its half of that.
    {
        const int my_word = tid >> 1;
        const uint32_t my_sel = bf16_select(tid);
        float sum = 0.0f;
        for (int h = 0; h < 2; ++h) {
            stage_half(h);
            const int end = tid < kHeadDim ? min(valid - kHalfRows * h, kHalfRows) : 0;
            int i = 0;
            for (; i + 16 <= end; i += 16) {  // 16 reads in flight, adds in row order
                float v[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) v[e] = block_elem_sel(half_block, i + e, my_word, my_sel);
#pragma unroll
                for (int e = 0; e < 16; ++e) sum += v[e];
            }
            for (; i < end; ++i) sum += block_elem_sel(half_block, i, my_word, my_sel);
            __syncthreads();
        }
        if (tid < kHeadDim) center_row[center_pos(tid)] = __fdiv_rn(sum, static_cast<float>(valid));
    }
    __syncthreads();

    // Farthest-first centres with nearest-centre assignment (:158-197). A
    // centre is a query of the block: its row is read from global memory (in
    // the caches since the block's own loads) by scalar loads.
    const bool live = query < valid;
    const float mean_d = lane_distance<kLanes>(x, center_row + 4 * kLeaves * part);
    float min_d = live ? mean_d : -INFINITY;
    int center = block_argmax<kLanes>(min_d, s_val, s_idx);
    min_d = INFINITY;
    int assign = 0;
    for (int slot = 0; slot < kCentroids; ++slot) {
        center = __builtin_amdgcn_readfirstlane(center);
        const uint32_t coff = __builtin_amdgcn_readfirstlane(stored(center, q_row));
        // A query past the end (only if NaNs leave no other maximum) is a zero row.
        const float dist = lane_distance_to_row<kLanes>(x, reinterpret_cast<const uint32_t*>(qhead + coff), part_sel,
                                                        center < valid);
        if (live && dist < min_d) {
            min_d = dist;
            assign = slot;
        }
        if (slot + 1 < kCentroids) {
            __syncthreads();  // every thread has read the last argmax's slots
            center = block_argmax<kLanes>(live ? min_d : -INFINITY, s_val, s_idx);
        }
    }

    // Members of each slot: per wave, the ballot of the queries assigned to
    // it. Queries 32i + bit, walked word by word and bit by bit, come in query
    // order (the reference's member order).
#pragma unroll
    for (int s = 0; s < kCentroids; ++s) {
        const uint64_t m = __ballot(live && assign == s);
        if (lane == 0) {
            slot_mask[wave * (2 / kLanes)][s] = static_cast<uint32_t>(m);
            if constexpr (kLanes == 1) slot_mask[2 * wave + 1][s] = static_cast<uint32_t>(m >> 32);
        }
    }
    __syncthreads();
    auto members = [&](int s) {
        return __popc(slot_mask[0][s]) + __popc(slot_mask[1][s]) + __popc(slot_mask[2][s]) + __popc(slot_mask[3][s]);
    };
    if (tid < kCentroids) pops[row * kCentroids + tid] = static_cast<float>(members(tid));

    // Centroid = bf16(member sum / count), then the LSE pre-scale
    // bf16(centroid * 128^-0.5 * log2 e) (csrc/ibcs.cu:213-237, :293-295).
    // Each wave sums its share of the slots, lane l dims 2l and 2l + 1 (one word
    // of a row), each slot's members in query order (half 0, then half 1) from the
    // staged half that holds them. Two slots are walked together, four members
    // of each at a time, so eight reads are in flight; a slot that has run out
    // reads the zero row, whose +0.0 leaves a sum (never -0.0) as it is. The
    // member masks are wave-uniform, so finding the next member is scalar work.
    constexpr int kWaveSlots = kCentroids / kWaves;
    float sum_lo[kWaveSlots], sum_hi[kWaveSlots];
#pragma unroll
    for (int i = 0; i < kWaveSlots; ++i) sum_lo[i] = sum_hi[i] = 0.0f;
    for (int h = 0; h < 2; ++h) {
        stage_half(h);
#pragma unroll
        for (int i = 0; i < kWaveSlots; i += 2) {
            uint64_t m[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int s = kWaveSlots * wave + i + j;
                m[j] = (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(slot_mask[2 * h + 1][s]))) << 32) |
                       uint32_t(__builtin_amdgcn_readfirstlane(slot_mask[2 * h][s]));
            }
            while ((m[0] | m[1]) != 0u) {
                uint32_t w[2][4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int idx = m[j] != 0u ? static_cast<int>(__builtin_ctzll(m[j])) : kHalfRows;
                        m[j] &= m[j] - 1u;
                        w[j][e] = half_block[idx * kRowWords + lane];
                    }
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        sum_lo[i + j] += bf16_lo(w[j][e]);
                        sum_hi[i + j] += bf16_hi(w[j][e]);
                    }
            }
        }
        __syncthreads();
    }
    uint32_t* dst = reinterpret_cast<uint32_t*>(centroids) + row * (kCentroids * kHeadDim / 2) + lane;
#pragma unroll
    for (int i = 0; i < kWaveSlots; ++i) {
        const int s = kWaveSlots * wave + i;
        const int cnt = members(s);
        auto scaled = [&](float sum) {
            const uint32_t c = cnt > 0 ? f32_to_bf16(__fdiv_rn(sum, static_cast<float>(cnt))) : 0u;
            return f32_to_bf16(__uint_as_float(c << 16) * qk_scale_log2);
        };
        dst[s * (kHeadDim / 2)] = scaled(sum_lo[i]) | (scaled(sum_hi[i]) << 16);
    }
}

// ---------------------------------------------------------------------------
// Stage 4: population-weighted masses, one workgroup per row:
//   m_j = sum_s fmaf(n_s / D_s, exp2(l_sj - M_s), .) * (1 / sum_s n_s)
// (RowMasses in masses.hpp).

constexpr int kMassThreads = 256;

__global__ __launch_bounds__(kMassThreads) void masses_kernel(
    const _Float16* __restrict__ lse, const float* __restrict__ pops,
    const float* __restrict__ lse_max, const float* __restrict__ lse_den,
    float* __restrict__ scores, int fb, int64_t ld) {
    const int64_t row = blockIdx.x;
    RowMasses rm;
    rm.load(pops, lse_max, lse_den, row);
    const _Float16* src = lse + row * kCentroids * ld;
    float* dst = scores + row * int64_t(fb);
    for (int j0 = threadIdx.x * 8; j0 < fb; j0 += kMassThreads * 8) {
        f16x8 h[kCentroids];
#pragma unroll
        for (int s = 0; s < kCentroids; ++s) h[s] = *reinterpret_cast<const f16x8*>(src + s * ld + j0);
        float score[8];
        rm.eight(h, score);
        // Two 16-byte stores (rows start at any multiple of 4 bytes, which
        // global stores accept); the ragged end of the row element by element.
        typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
        if (j0 + 8 <= fb) {
            *reinterpret_cast<f32x4_u*>(dst + j0) = f32x4_u{score[0], score[1], score[2], score[3]};
            *reinterpret_cast<f32x4_u*>(dst + j0 + 4) = f32x4_u{score[4], score[5], score[6], score[7]};
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (j0 + e < fb) dst[j0 + e] = score[e];
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host launchers (validated by the C-ABI layer in api.hip).

int64_t lse_stride(int64_t fb) { return (fb + 63) / 64 * 64; }

// Lanes per query: two while the blocks leave most SIMDs to one workgroup, where
// the length of its chain of passes is the time (32 blocks 22.6 -> 18.3 us, 256
// 23.6 -> 20.1); from about 768 blocks (33.0 us both) the extra v_perm_b32s and
// waves cost more than they save (1,536 blocks 45 against 54 us).
int cluster_lanes(int64_t blocks) { return blocks <= 640 ? 2 : 1; }

int launch_cluster_pool(const void* q, const void* k, const QkLayout& layout, int64_t bh, int64_t n, void* centroids,
                        float* pops, void* pooled, float qk_scale_log2, const int32_t* order, hipStream_t stream) {
    // The kernel addresses a head with 32-bit offsets in 16-byte units, made of 24-bit factors.
    if (n <= 0 || n > kMaxKvBlocks * kKvBlock) return set_error(1, "ibcs: %lld tokens per head", (long long)n);
    for (const TensorLayout* t : {&layout.q, &layout.k})
        if (t->token / 2 >= (1u << 24) || n * int64_t(t->token / 2) > int64_t(0xffffffff))
            return set_error(1, "ibcs: token stride of %lld is too large", 4 * (long long)t->token);
    const int64_t qb = (n + kQueryBlock - 1) / kQueryBlock;
    dim3 grid(static_cast<unsigned>(qb), static_cast<unsigned>(bh));
    const int lanes = cluster_lanes(qb * bh);
    const auto kernel = lanes == 2 ? cluster_pool_kernel<2> : cluster_pool_kernel<1>;
    hipLaunchKernelGGL(kernel, grid, dim3(kQueryBlock * lanes), 0, stream, static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), layout,
                       static_cast<uint16_t*>(centroids), pops, static_cast<uint16_t*>(pooled), n, qb,
                       qk_scale_log2, order);
    return check_launch("cluster_pool_kernel");
}

int launch_masses(const void* lse, const float* pops, const float* lse_max, const float* lse_den,
                  int64_t rows, int64_t fb, float* scores, hipStream_t stream) {
    hipLaunchKernelGGL(masses_kernel, dim3(static_cast<unsigned>(rows)), dim3(kMassThreads), 0, stream,
                       static_cast<const _Float16*>(lse), pops, lse_max, lse_den, scores,
                       static_cast<int>(fb), lse_stride(fb));
    return check_launch("masses_kernel");
}

}  // namespace ab
