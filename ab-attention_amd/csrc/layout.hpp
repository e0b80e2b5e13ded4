// Where the tensors of a call lie in memory.
#pragma once

#include "common.hpp"

namespace ab {

// A [batch, heads, tokens, 128] bf16 tensor whose rows of 128 are contiguous;
// strides in units of 4 elements (rows start on 8 bytes, those of inputs on
// 16). Contiguous tensors, slices of their tokens and the transposed views of
// [batch, tokens, heads, 128] that linear projections leave are all of this
// form. 32-bit strides keep the kernels' arguments short: they lie in host
// memory, and each cache line of them costs a small call about half a
// microsecond.
struct TensorLayout {
    uint32_t batch, head, token;
    // Element offset of a token of head h of batch item b.
    __device__ __forceinline__ int64_t at(uint32_t b, uint32_t h, uint32_t t) const {
        return (int64_t(b) * batch + int64_t(h) * head + int64_t(t) * token) * 4;
    }
};

// Division of a wave-uniform number by a number of the call in a few scalar
// instructions (the compiler's 32-bit division is a chain of ~25 vector ones,
// its 64-bit one takes about a microsecond of a small call): with m =
// floor((2^32 - 1) / d), n * m / 2^32 is less than 1 below n / d, so its floor is
// the quotient or one less.
struct Divisor {
    uint32_t d, m;
    __device__ __forceinline__ uint32_t quotient(uint32_t n, uint32_t& rest) const {
        uint32_t q = __umulhi(n, m);
        rest = n - q * d;
        if (rest >= d) {
            ++q;
            rest -= d;
        }
        // Kept in scalar registers, and with them the addresses made of them.
        rest = __builtin_amdgcn_readfirstlane(rest);
        return __builtin_amdgcn_readfirstlane(q);
    }
};
inline Divisor divisor(uint32_t d) { return {d, 0xffffffffu / (d > 0 ? d : 1u)}; }

// The layout of a contiguous tensor (its size is checked by the caller: batch
// is only used past a first batch item).
inline TensorLayout contiguous_layout(int64_t tokens) {
    return {0u, static_cast<uint32_t>(tokens) * (kHeadDim / 4), kHeadDim / 4};
}

// Q and K of a plan: heads first_head, first_head + 1, ... of the flattened
// (batch, head) index.
struct QkLayout {
    TensorLayout q, k;
    Divisor heads;
    uint32_t first_head;
};

inline QkLayout contiguous_qk(int64_t batch_heads, int64_t tokens) {
    const TensorLayout t = contiguous_layout(tokens);
    return {t, t, divisor(static_cast<uint32_t>(batch_heads)), 0};
}

struct PrefillLayout {
    TensorLayout q, k, v, out;
    Divisor heads;
};

// One prefill call (see ab_prefill in include/ab_attention.h).
struct PrefillCall {
    const void *q, *k, *v;
    void* out;
    float* lse;
    PrefillLayout layout;
    int64_t batch, q_tokens, kv_tokens;
    bool dense;
    int64_t samples;
    const int32_t* ids;
    const float* log_weights;
    int64_t tail_samples;
    const int32_t* tail_ids;
    const float* tail_log_weights;
    const int32_t* order;
    void* workspace;
};

}  // namespace ab
