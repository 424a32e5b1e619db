// Merging the partial results of the split decodes: (m, l, O) per slot (a
// split, or a part of one) and query head, in the generic workspace layout
// ws_ml [slot][Hq][2], ws_acc [slot][Hq][D].
//
// The matrix-core split kernels end with finish_part: the only part of a
// sequence writes its output, otherwise the workgroup that counts in last for a
// (sequence, kv head) merges its parts in the same launch. A merge launch of its
// own runs behind the whole decode (2.4 us at its smallest and the gap before
// it; 64 sequences at head_dim 64: 37.3 against 35.2 us for both); it remains for
// calls that cannot count in (see paged_decode.hip), with the same arithmetic: factors 2^(m - M) against the
// largest m, l added in a fixed order, one fma per slot in slot order for every
// dim of O, so both give the same bits.
#pragma once

#include "decode_common.h"

namespace qvp {

constexpr int kMergeRows = 16;   // query heads merged at a time (a kv head's group)
constexpr int kMergeSlots = 64;  // slots per sequence merge_rows takes
constexpr int kMergeWg = 256;    // threads of every workgroup that merges
// Floats of LDS merge_rows uses.
constexpr int kMergeLds = kMergeRows * (kMergeSlots + 1);

struct SplitOutput {
    void* out;           // [num_seqs][Hq][D]
    uint32_t out_dtype;  // qvp_dtype
    int32_t* counters;   // [num_seqs][kv heads], zero between launches; NULL: a merge launch follows
};

// Slots of a sequence: first and count (slots past the context are not written).
struct SlotRange {
    uint64_t first;
    int count;
};
__device__ inline SlotRange slots_of(int first_split, int ctx, int split_tokens, int parts_shift) {
    const int full = (ctx - 1) / split_tokens;
    const int part_tokens = split_tokens >> parts_shift;
    return {static_cast<uint64_t>(first_split) << parts_shift,
            (full << parts_shift) + (ctx - full * split_tokens + part_tokens - 1) / part_tokens};
}

__device__ inline void store_output4(const SplitOutput& so, uint64_t at, const floatx4& x) {
    if (so.out_dtype == QVP_DTYPE_F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) static_cast<float*>(so.out)[at + e] = x[e];
    } else if (so.out_dtype == QVP_DTYPE_BF16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) static_cast<uint16_t*>(so.out)[at + e] = from_float<uint16_t>(x[e]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) static_cast<_Float16*>(so.out)[at + e] = from_float<_Float16>(x[e]);
    }
}

__device__ inline uint64_t pair_bits(float a, float b) {
    return static_cast<uint64_t>(__float_as_uint(b)) << 32 | __float_as_uint(a);
}
__device__ inline float low_float(uint64_t x) { return __uint_as_float(static_cast<uint32_t>(x)); }
__device__ inline float high_float(uint64_t x) { return __uint_as_float(static_cast<uint32_t>(x >> 32)); }
__device__ inline uint64_t load_agent(const void* p) {
    return __hip_atomic_load(static_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void store_agent(void* p, uint64_t x) {
    __hip_atomic_store(static_cast<uint64_t*>(p), x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A workgroup of kMergeWg threads merges query heads row0 .. row0 + rows - 1
// (of all Hq; rows <= kMergeRows) of sequence b over its slots (count <=
// kMergeSlots), head_dim a multiple of four. Agent-scope loads: the slots may
// come from other workgroups of the same launch.
__device__ inline void merge_rows(const SplitOutput& so, const float* ws_ml, const float* ws_acc, const SlotRange& slots,
                                  uint32_t b, uint32_t row0, int rows, uint32_t num_q_heads, int head_dim, float* lds) {
    const int ns = slots.count;
    float* f_s = lds;                              // [rows][ns]: factors
    float* sum_s = lds + kMergeRows * kMergeSlots;  // [rows]
    const int t = static_cast<int>(threadIdx.x);
    // Sixteen lanes per row: lane s holds slots s, s + 16, ...
    constexpr int kPer = kMergeSlots / 16;
    const int lr = t >> 4;
    const int ls = t & 15;
    uint64_t ml[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        ml[k] = pair_bits(-INFINITY, 0.f);
        if (lr < rows && ls + 16 * k < ns) {
            ml[k] = load_agent(ws_ml + ((slots.first + ls + 16 * k) * num_q_heads + row0 + lr) * 2);
        }
    }
    // The first item's accumulators are on their way before the factors are known.
    constexpr int kAhead = 8;
    const int d4 = head_dim / 4;
    const int items = rows * d4;
    auto acc_at = [&](int e, int s) {
        const int r = e / d4;
        return ws_acc + ((slots.first + s) * num_q_heads + row0 + r) * head_dim + 4 * (e - r * d4);
    };
    uint64_t a[kAhead][2];
    auto load_ahead = [&](int e, int s0) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            a[k][0] = a[k][1] = 0;
            if (e < items && s0 + k < ns) {
                const float* p = acc_at(e, s0 + k);
                a[k][0] = load_agent(p);
                a[k][1] = load_agent(p + 2);
            }
        }
    };
    load_ahead(t, 0);
    float m = low_float(ml[0]);
#pragma unroll
    for (int k = 1; k < kPer; ++k) m = fmaxf(m, low_float(ml[k]));
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 16));
    float l = 0.f;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (lr < rows && ls + 16 * k < ns) {
            const float f = fast_exp2(low_float(ml[k]) - m);
            f_s[lr * ns + ls + 16 * k] = f;
            l = fmaf(high_float(ml[k]), f, l);
        }
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) l += __shfl_xor(l, off, 16);
    if (lr < rows && ls == 0) sum_s[lr] = l;
    __syncthreads();
    for (int e = t; e < items; e += kMergeWg) {
        const int r = e / d4;
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < ns; s0 += kAhead) {
            if (s0 > 0 || e != t) load_ahead(e, s0);
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                if (s0 + k < ns) {
                    const float f = f_s[r * ns + s0 + k];
                    acc[0] = fmaf(low_float(a[k][0]), f, acc[0]);
                    acc[1] = fmaf(high_float(a[k][0]), f, acc[1]);
                    acc[2] = fmaf(low_float(a[k][1]), f, acc[2]);
                    acc[3] = fmaf(high_float(a[k][1]), f, acc[3]);
                }
            }
        }
        const float ls_r = sum_s[r];
        floatx4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = acc[i] / ls_r;
        store_output4(so, (static_cast<uint64_t>(b) * num_q_heads + row0 + r) * head_dim + 4 * (e - r * d4), x);
    }
}

// The end of a split kernel's workgroup: rows row0 .. row0 + rows - 1 of part
// `slot` of sequence b, whose merged waves' values come from value(row, d4, m,
// l). `heads_at` is b * kv heads + the kv head. lds: kMergeLds floats, free
// once every wave's values are in (value may read other LDS).
template <int kD, typename F>
__device__ inline void finish_part(const SplitOutput& so, float* ws_ml, float* ws_acc, const SlotRange& slots,
                                   uint64_t slot, uint32_t b, uint32_t row0, int rows, uint32_t num_q_heads,
                                   uint32_t counter, const F& value, float* lds, int* sm_last) {
    for (int e = static_cast<int>(threadIdx.x); e < rows * (kD / 4); e += kMergeWg) {
        const int r = e / (kD / 4);
        const int d4 = 4 * (e - r * (kD / 4));
        float m, l;
        const floatx4 acc = value(r, d4, m, l);
        if (slots.count == 1 && so.counters != nullptr) {
            floatx4 x;
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = acc[i] / l;
            store_output4(so, (static_cast<uint64_t>(b) * num_q_heads + row0 + r) * kD + d4, x);
            continue;
        }
        const uint64_t head = slot * num_q_heads + row0 + r;
        store_agent(ws_acc + head * kD + d4, pair_bits(acc[0], acc[1]));
        store_agent(ws_acc + head * kD + d4 + 2, pair_bits(acc[2], acc[3]));
        if (d4 == 0) store_agent(ws_ml + head * 2, pair_bits(m, l));
    }
    if (so.counters == nullptr || slots.count == 1) return;
    // The persistent decode's protocol: agent-scope stores, each wave's wait
    // for its own (a barrier alone does not wait for stores), a barrier, one
    // agent-scope increment; the last workgroup reads with agent-scope loads
    // and leaves the counter at zero.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const int done =
            __hip_atomic_fetch_add(so.counters + counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
        *sm_last = done == slots.count;
        if (done == slots.count) {
            __hip_atomic_store(so.counters + counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(*sm_last) == 0) return;
    merge_rows(so, ws_ml, ws_acc, slots, b, row0, rows, num_q_heads, kD, lds);
}

}  // namespace qvp
