// qvp_paged_prefill: causal attention of a step's new tokens over the paged
// cache. The reference defines prefill as paged_attention_decode<T> applied per
// prompt position p with context_len = p + 1 (include/qwenvl_paged/
// PagedAttention.h:43-44; tests/EndToEnd.test.cpp:252-256), so every output
// row here is the decode of its position.
//
// MFMA path (bf16 or fp16 cache, head_dim 128 or 64, GQA group <= 16,
// power-of-two tokens_per_block >= 16). The rows of (sequence b, kv head g) are its new
// positions times the G query heads of g's group, position-major, so row r is
// head r % G at position q_start + r / G; a work item is 128 consecutive rows
// (a cut may fall inside a position: every wave is full for any group).
// Its workgroup streams the tokens its last row sees in 32-token tiles: each
// tile is loaded once, straight into LDS, two steps ahead of its use, into a
// ring of four tiles that hold the K and V rows as in the frame (16-byte chunks
// XOR-permuted by row so the fragment reads spread over the banks; the PV
// operands come out of V transposed by ds_read_b64_tr_b16). Each of the four
// waves holds 32 of the rows in the MFMA columns, a column seeing the tokens up
// to its position (masks only on tiles that reach the item's first position).
// The tile loop is software-pipelined over three tiles: PV of tile t - 1 and QK
// of tile t + 1 run beside the softmax of tile t. Items past 1.25 x a CU's share
// are cut into pieces that the last one merges (piece_count), and are launched
// longest first so that the short ones fill the tail.
//
// Decode path (any other shape): one virtual sequence per new position (same
// frames, context p + 1), packed into a private batch and run through
// qvp_paged_decode, whose query and output rows are exactly the prefill's.
#include "mfma_tile.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>
#include <cstring>
#include <vector>

namespace qvp {
namespace {

constexpr int kPrefillWaves = 4;
constexpr int kPrefillThreads = kPrefillWaves * 64;
constexpr int kPrefillRows = kPrefillWaves * 32;  // rows per item: the 32 MFMA columns of each wave
// Block ids per virtual batch of the decode-kernel path.
constexpr size_t kMaxVirtualIds = size_t{1} << 20;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

// The tile math runs on 32x32x16 MFMAs, lane l = (c = l % 32, h = l / 32).
// Beside vector work one of them takes 6 cycles less than the two 16x16x32
// MFMAs it replaces (measured with four vector instructions per 16 cycles of
// matrix work: 41.6 against 47.8 cycles). S^T = K Q^T: A row c is token c of
// the tile, so score register r of lane (c, h) is token (r % 4) + 8 (r / 4) +
// 4h for column c. O^T += V^T P^T: the eight weights r = 8ks .. 8ks + 7 of a
// lane are the B operand of k-step ks as they are (k index 8h + e is token
// 16ks + 8 (e / 4) + 4h + e % 4), and row c of block n is dim 32n + c.
template <bool kF16>
__device__ inline floatx16 mfma32(const u32x4& a, const u32x4& b, floatx16 c) {
    if constexpr (kF16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                      0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                       c, 0, 0, 0);
    }
}

// K and V tiles in LDS: rows as in the frame (token-major), each in a ring of
// four tiles (tile t in slot t % 4). ds_read_b64_tr_b16 hands lane i of each 16-lane
// group element i % 4 of the 8 bytes that lane 4e + i / 4 of the group
// addressed, as element e: with the group's lanes on tokens t .. t + 3 (by
// i / 4) and 16 dims, lane i gets dim i of the four tokens, half of a PV
// operand.
constexpr int kRing = 4;
// The LDS rows hold their 16-byte chunks XOR-permuted by row, so that the 64
// lanes of a read spread over the banks: chunk x of row r lies at x ^ key(r).
// K is read a chunk of 32 rows at a time, V four neighbouring chunks of eight
// rows. (A 128-byte row covers half of the 256-byte bank period: its key has
// three bits and row pairs share it.)
template <int kD>
__device__ inline int k_key(int row) {
    return kD == 128 ? row & 15 : (row >> 1) & 7;
}
template <int kD>
__device__ inline int v_key(int row) {
    return kD == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

struct PrefillItem {
    int32_t b;      // sequence
    int32_t g;      // kv head
    int32_t start;  // the sequence's first new position
    int32_t r0;     // first row of the item
    int32_t nrows;  // rows of (b, g): new positions x G
    int32_t row0;   // query / output row of the first new position
    int32_t t0, t1;  // tiles of the rows' context
    // An item that holds all of its rows' tiles (nparts 1) writes their output.
    // Otherwise it is one of nparts pieces: its result goes to workspace slot
    // `slot`, the pieces' slots are slot0 .. slot0 + nparts - 1, and the
    // workgroup that completes counters[slot0] merges them.
    int32_t slot, slot0, nparts;
    int32_t pad;
};
static_assert(sizeof(PrefillItem) == 12 * sizeof(int32_t), "PrefillItem is twelve int32");

// Results of split items: per slot and wave, (m, l) of its 32 rows and their O
// as the lanes hold it, two dims per lane and store (512 contiguous bytes).
struct PrefillParts {
    int32_t* counters;
    uint64_t* ml;   // [slot][wave][32]
    uint64_t* acc;  // [slot][wave][kPv x 8][64 lanes]
};

template <typename T>
__device__ inline const __attribute__((address_space(4))) T* as_const(const T* ptr) {
    return (const __attribute__((address_space(4))) T*)(ptr);
}

// The running maximum of a row moves only when a score passes it by more than
// kLazy in log2 units, so O is rescaled on few tiles; weights then reach
// 2^(kLazy + kBias). fp16 weights carry 2^kBias so that small ones stay normal
// binary16 numbers, with the largest below 2^15.
template <bool kF16>
struct PrefillWeights {
    static constexpr float kLazy = kF16 ? 4.0f : kLazyMaxLog2;
    static constexpr float kBias = kF16 ? 11.0f : 0.0f;
};

// Largest of this lane's sixteen scores. maximum (not fmax) takes the MFMA
// results without a canonicalising instruction each; a NaN score makes its
// row's weights NaN either way.
__device__ inline float lane_max(const floatx16& s) {
    float m = s[0];
#pragma unroll
    for (int r = 1; r < 15; r += 2) {
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, s[r]), s[r + 1]);
    }
    return __builtin_elementwise_maximum(m, s[15]);
}

// P of one tile as the hi and lo B operands of the PV k-steps; returns this
// lane's sum of its sixteen weights. hi and lo = P - hi are both rounded to
// nearest even: 2^-18 of a weight at most for bf16 (2^-17 with hi truncated, at
// the same instruction count; no weight is exactly 1 here, as the largest is
// under a maximum that moves with every tile). v_dot2_f32_bf16 would give p - hi
// in one instruction, but holds the matrix core up: beside MFMAs it costs as
// much as three others.
template <bool kF16>
__device__ inline float prefill_weights(const floatx16& s, float scale_log2, float bias, u32x4 (&hi)[2],
                                        u32x4 (&lo)[2]) {
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
        const float p0 = fast_exp2(fmaf(s[r], scale_log2, bias));
        const float p1 = fast_exp2(fmaf(s[r + 1], scale_log2, bias));
        psum += p0 + p1;
        if constexpr (kF16) {
            const f16x2_t a = {static_cast<_Float16>(p0), static_cast<_Float16>(p1)};
            const f16x2_t b = {static_cast<_Float16>(p0 - static_cast<float>(a[0])),
                               static_cast<_Float16>(p1 - static_cast<float>(a[1]))};
            hi[r / 8][(r / 2) & 3] = __builtin_bit_cast(uint32_t, a);
            lo[r / 8][(r / 2) & 3] = __builtin_bit_cast(uint32_t, b);
        } else {
            const bf16x2_t a = {static_cast<__bf16>(p0), static_cast<__bf16>(p1)};
            const uint32_t x = __builtin_bit_cast(uint32_t, a);
            const bf16x2_t b = {static_cast<__bf16>(p0 - __uint_as_float(x << 16)),
                                static_cast<__bf16>(p1 - __uint_as_float(x & 0xffff0000u))};
            hi[r / 8][(r / 2) & 3] = x;
            lo[r / 8][(r / 2) & 3] = __builtin_bit_cast(uint32_t, b);
        }
    }
    return psum;
}

template <bool kF16, int kD, typename OutT>
__global__ __launch_bounds__(kPrefillThreads, 2) void prefill_mfma(DecodeGeometry p, const PrefillItem* items,
                                                                   PrefillParts parts, void* out_ptr) {
    constexpr int kQk = kD / 16;               // QK k-steps
    constexpr int kPv = kD / 32;               // PV row blocks
    constexpr int kHalf = kPv / 2;             // row blocks per half of PV
    constexpr int kChunks = kD / 8;            // 16-byte chunks per row
    constexpr int kLoadRows = 64 / kChunks;    // rows one direct load fills
    constexpr int kLoads = 8 / kLoadRows;      // direct loads per wave of a tile's K (and of its V)
    constexpr uint32_t kRow = 2 * kD;          // bytes
    constexpr uint32_t kTileBytes = kTileTokens * kRow;
    constexpr float kLazy = PrefillWeights<kF16>::kLazy;
    constexpr float kBias = PrefillWeights<kF16>::kBias;
    __shared__ __attribute__((aligned(256))) uint8_t sm[2 * kRing * kTileBytes];
    __shared__ int sm_bad[kPrefillWaves];

    const auto* itp = as_const(items) + blockIdx.x;
    const int b = itp->b;
    const int g = itp->g;
    const int start = itp->start;
    const int r0 = itp->r0;
    const int nrows = itp->nrows;
    const int row0 = itp->row0;
    const int t0 = itp->t0;
    const int t1 = itp->t1;
    const int nparts = itp->nparts;

    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int c = lane & 31;
    const int h = lane >> 5;
    const int G = static_cast<int>(p.group);
    const int pmin = start + r0 / G;
    const int last_tok = start + min(r0 + kPrefillRows - 1, nrows - 1) / G;
    // A wave past the last row only loads its share of the tiles.
    const bool active = r0 + 32 * wave < nrows;

    // Column c is row r0 + 32 wave + c; columns past the last row repeat it
    // (valid data, never written).
    const int row = min(r0 + 32 * wave + c, nrows - 1);
    const int pos = row / G;
    const int col_last = start + pos;
    const uint64_t qoff =
        (static_cast<uint64_t>(row0 + pos) * p.num_q_heads + static_cast<uint64_t>(g) * G + (row - pos * G)) * kD;
    u32x4 q[kQk];
#pragma unroll
    for (int i = 0; i < kQk; ++i) {
        q[i] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.query) + qoff + 16 * i + 8 * h);
    }

    // Tile loads go straight into LDS (global_load_lds_dwordx4): one
    // instruction fills kLoadRows rows (1 KiB), lane l landing at byte 16 l of
    // them -- row l / kChunks, physical chunk l % kChunks, which takes the
    // logical chunk the row's key puts there. Wave w loads rows 8w .. 8w + 7
    // of K and V; they lie in one 16-token half, and that in one block
    // (tokens_per_block is a power of two >= 16). Past the half of the item's
    // last token that half is loaded again, and its rows past the token load
    // the token's (finite data under weights of 0), so every address stays
    // inside a mapped frame.
    const auto* trow = as_const(p.tables) + static_cast<uint64_t>(b) * p.max_nb;
    const uint8_t* kbase = p.kv_base + p.k_off + static_cast<uint64_t>(g) * p.head_stride;
    const uint64_t kv_gap = p.v_off - p.k_off;
    const uint32_t tstride = static_cast<uint32_t>(p.token_stride);
    const uint32_t bstride = static_cast<uint32_t>(p.block_stride);
    const int half_off = 16 * (wave >> 1);
    const int last_half = last_tok & ~15;
    auto half_of = [&](int tile) { return min(tile * kTileTokens + half_off, last_half); };
    auto block_of = [&](int tile) { return trow[half_of(tile) >> p.tpb_shift]; };
    auto frame_of = [&](int tile, int blk) {
        return kbase + static_cast<uint64_t>(static_cast<uint32_t>(blk)) * bstride +
               static_cast<uint32_t>(half_of(tile) & (p.tpb - 1)) * tstride;
    };
    // The lane's offsets from that row; `end` for the last half.
    uint32_t off_k[kLoads], off_v[kLoads];
    auto offsets = [&](uint32_t (&off)[kLoads], bool v, int end) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int lr = 8 * wave + kLoadRows * i + lane / kChunks;
            const int key = v ? v_key<kD>(lr) : k_key<kD>(lr);
            off[i] = static_cast<uint32_t>(min(lr & 15, end)) * tstride + 16u * static_cast<uint32_t>((lane % kChunks) ^ key);
        }
    };
    typedef __attribute__((address_space(3))) uint8_t lds_byte;
    lds_byte* const lds = (lds_byte*)sm;
    const uint32_t lds_rows = static_cast<uint32_t>((uintptr_t)lds) + 8u * wave * kRow;
    // In assembly, as the compiler would wait for every direct load before any
    // transposed read of LDS, whichever ring slot either of them is in. The
    // loads write no register; the s_waitcnt before each barrier covers them.
    auto load_rows = [&](uint32_t at, const uint8_t* frame, const uint32_t (&off)[kLoads]) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(at), "v"(off[0]), "s"(frame)
                     : "memory");
        if constexpr (kLoads == 2) {
            asm volatile("s_add_u32 m0, %0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :
                         : "s"(at), "v"(off[kLoads - 1]), "s"(frame)
                         : "memory", "scc");
        }
    };
    auto load_k = [&](int tile, const uint8_t* frame) {
        load_rows(lds_rows + (tile & (kRing - 1)) * kTileBytes, frame, off_k);
    };
    auto load_v = [&](int tile, const uint8_t* frame) {
        load_rows(lds_rows + (kRing + (tile & (kRing - 1))) * kTileBytes, frame + kv_gap, off_v);
    };
    // Before the loads of a tile: its offsets if it reaches the last half.
    // (They stay: later tiles load that half again.)
    auto end_offsets = [&](int tile, uint32_t (&off)[kLoads], bool v) {
        if (tile * kTileTokens + half_off >= last_half) offsets(off, v, last_tok - last_half);
    };
    // Waits until all but the youngest 2 kLoads direct loads have landed.
    auto wait_older_loads = [&]() { __builtin_amdgcn_s_waitcnt(0x0070 | (2 * kLoads)); };
    // Fragment addresses: the chunks one lane reads of a tile differ by XOR of
    // constant bits (and rows 8 and 16 further), so one address serves them all.
    const uint32_t k_lane = static_cast<uint32_t>(c * kRow + 16 * (h ^ k_key<kD>(c)));
    const int vi = lane & 15;
    const int vrow = 4 * h + (vi >> 2);
    const uint32_t v_lane = static_cast<uint32_t>(
        kRing * kTileBytes + vrow * kRow + 16 * ((2 * ((lane >> 4) & 1) + ((vi & 3) >> 1)) ^ v_key<kD>(vrow)) +
        8 * (vi & 1));
    static_assert(kTileBytes % 256 == 0, "XOR of chunk bits must not carry");
    // K operands of k-steps x kQk / 2 .. (x + 1) kQk / 2 - 1.
    auto read_k = [&](int tile, int x, u32x4 (&kf)[kQk / 2]) {
        const uint32_t a = k_lane + static_cast<uint32_t>(tile & (kRing - 1)) * kTileBytes;
#pragma unroll
        for (int i = 0; i < kQk / 2; ++i) {
            kf[i] = *(const __attribute__((address_space(3))) u32x4*)(lds + (a ^ (32u * (i + x * kQk / 2))));
        }
    };
    // V operands of row blocks x kHalf .. (x + 1) kHalf - 1, both k-steps.
    auto read_v = [&](int tile, int x, u32x4 (&vf)[kHalf][2]) {
        const uint32_t a = v_lane + static_cast<uint32_t>(tile & (kRing - 1)) * kTileBytes;
#pragma unroll
        for (int n = 0; n < kHalf; ++n)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    // Eight rows further the key changes by 2 (both head dims).
                    const v4i16 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4i16 __attribute__((address_space(3)))*)(
                        lds + ((a ^ (64u * (n + x * kHalf)) ^ (32u * e)) + (16 * ks + 8 * e) * kRow)));
                    vf[n][ks][2 * e] = __builtin_bit_cast(uint2v, t)[0];
                    vf[n][ks][2 * e + 1] = __builtin_bit_cast(uint2v, t)[1];
                }
    };

    const int t_diag = (pmin + 1) / kTileTokens;  // first tile that needs masks
    const float lazy_raw = kLazy / p.scale_log2;
    floatx16 o[kPv];
    float lsum, m_run;

    // One pass over the item's tiles. `careful` (a second pass, taken when the
    // first left a non-finite output) multiplies the masked tiles' V column by
    // column with the values past the column's position cleared: V rows a row
    // does not see meet weights of 0, but 0 x inf would still poison it.
    auto run = [&](bool careful) {
        struct Weights { u32x4 hi[2], lo[2]; };
        // Running maximum m of the column as bias = kBias - m and thr, the raw
        // score past which it moves; thr is -inf until a score was seen.
        float thr = -INFINITY, bias = kBias, alpha = 1.0f, lm = -INFINITY;
        bool rescale_o = false;
        lsum = 0.f;
#pragma unroll
        for (int n = 0; n < kPv; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[n][r] = 0.f;
        auto qk = [&](const u32x4 (&kf)[kQk / 2], int x, floatx16& sc) {
            if (x == 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < kQk / 2; ++i) sc = mfma32<kF16>(kf[i], q[i + x * kQk / 2], sc);
        };
        auto pv = [&](const u32x4 (&vf)[kHalf][2], int x, const Weights& w) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
                for (int n = 0; n < kHalf; ++n) o[n + x * kHalf] = mfma32<kF16>(vf[n][ks], w.hi[ks], o[n + x * kHalf]);
#pragma unroll
                for (int n = 0; n < kHalf; ++n) o[n + x * kHalf] = mfma32<kF16>(vf[n][ks], w.lo[ks], o[n + x * kHalf]);
            }
        };
        auto pv_careful = [&](const u32x4 (&vf)[kHalf][2], int x, const Weights& w, int t) {
            for (int col = 0; col < 32; ++col) {
                const bool mine = c == col;
                const int lim = __builtin_amdgcn_readlane(col_last, col) - t * kTileTokens - 4 * h;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    u32x4 hi, lo, keep;
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const int tok = 16 * ks + 8 * (d >> 1) + 2 * (d & 1);  // of elements 2d, 2d + 1
                        hi[d] = mine ? w.hi[ks][d] : 0u;
                        lo[d] = mine ? w.lo[ks][d] : 0u;
                        keep[d] = (tok <= lim ? 0x0000ffffu : 0u) | (tok + 1 <= lim ? 0xffff0000u : 0u);
                    }
#pragma unroll
                    for (int m = 0; m < kHalf; ++m) {
                        const int n = m + x * kHalf;
                        const floatx16 a = mfma32<kF16>(vf[m][ks] & keep, lo, mfma32<kF16>(vf[m][ks] & keep, hi, o[n]));
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[n][r] = mine ? a[r] : o[n][r];
                    }
                }
            }
        };
        auto mask = [&](floatx16& sc, int t) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                sc[r] = t * kTileTokens + (r & 3) + 8 * (r >> 2) + 4 * h > col_last ? -INFINITY : sc[r];
            }
        };
        auto rescale = [&]() {
            if (rescale_o) {
#pragma unroll
                for (int n = 0; n < kPv; ++n) o[n] *= alpha;
            }
        };
        // Moves the maxima that a score of the tile passes by more than kLazy
        // (lm: this lane's largest). O still lacks the previous tile's product
        // then, so it is scaled at the next call.
        auto raise = [&]() {
            const uint64_t up = __builtin_amdgcn_ballot_w64(lm > thr);
            if (!rescale_o && up == 0) return;
            rescale();
            rescale_o = up != 0;
            const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(lm), __float_as_uint(lm), false, false);
            const float mt = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
            const bool move = mt > thr;
            const float to = kBias - mt * p.scale_log2;
            alpha = move && thr != -INFINITY ? fast_exp2(to - bias) : 1.0f;
            bias = move ? to : bias;
            thr = move ? mt + lazy_raw : thr;
            lsum *= alpha;
        };

        floatx16 sa, sb;
        Weights wa, wb;
        u32x4 va[kHalf][2];  // first half of the V operands the next PV takes
        // Loads run two steps ahead: step t issues K(t + 3) and V(t + 2) (past
        // the end the last tile again, into slots nothing reads any more, so
        // that the count of loads in flight stays the same) and at its end
        // waits for those of step t - 1 only. (A lone workgroup's step was as
        // long as one load's latency, 0.75 us, with loads one step ahead.) A
        // direct load has landed in LDS once vmcnt counts it done: each wave
        // waits for its own before the barrier that hands the tiles to the
        // other waves.
        const uint8_t* frame_v = frame_of(t0, block_of(t0));  // of the tile whose V goes next; its K went a step before
        const uint8_t* frame_k = frame_of(t0 + 1, block_of(t0 + 1));
        int blk = block_of(t0 + 2);
        offsets(off_k, false, 15);
        offsets(off_v, true, 15);
        end_offsets(t0, off_k, false);
        end_offsets(t0, off_v, true);
        load_k(t0, frame_v);
        load_v(t0, frame_v);
        end_offsets(t0 + 1, off_k, false);
        load_k(t0 + 1, frame_k);
        // The query loads end here too: left open, the compiler waits for them
        // (and with them for every tile load) in each step.
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        frame_v = frame_k;
        frame_k = frame_of(t0 + 2, blk);
        blk = block_of(t0 + 3);
        end_offsets(t0 + 2, off_k, false);
        load_k(t0 + 2, frame_k);
        end_offsets(t0 + 1, off_v, true);
        load_v(t0 + 1, frame_v);
        if (active) {
            u32x4 k0[kQk / 2], k1[kQk / 2];
            read_k(t0, 0, k0);
            read_k(t0, 1, k1);
            qk(k0, 0, sa);
            qk(k1, 1, sa);
            if (t_diag <= t0) mask(sa, t0);
            lm = lane_max(sa);
        }
        // Step t: the softmax of tile t (s -> w), with QK of tile t + 1 (-> s2)
        // and PV of tile t - 1 (w0) around it: none of the three depends on
        // another, so the matrix products run beside the vector work.
        auto step = [&](int t, const floatx16& s, Weights& w, floatx16& s2, const Weights& w0, auto first, auto masked) {
            constexpr bool kFirst = decltype(first)::value;
            constexpr bool kMasked = decltype(masked)::value;
            end_offsets(t + 3, off_k, false);
            end_offsets(t + 2, off_v, true);
            // Issued among the matrix products (see below): on their own the
            // address steps hold a lone wave up for a fifth of its step.
            auto load_ahead = [&]() {
                frame_v = frame_k;
                frame_k = frame_of(t + 3, blk);
                load_k(t + 3, frame_k);
                load_v(t + 2, frame_v);
                blk = block_of(t + 4);
            };
            if (!active) load_ahead();
            if (active) {
                raise();
                u32x4 k0[kQk / 2], k1[kQk / 2], vb[kHalf][2];
                read_k(t + 1, 0, k0);
                if constexpr (!kFirst) {
                    if (kMasked && careful) {
                        pv_careful(va, 0, w0, t - 1);
                    } else {
                        pv(va, 0, w0);
                    }
                }
                read_k(t + 1, 1, k1);
                load_ahead();
                qk(k0, 0, s2);
                if constexpr (!kFirst) read_v(t - 1, 1, vb);
                qk(k1, 1, s2);
                lsum += prefill_weights<kF16>(s, p.scale_log2, bias, w.hi, w.lo);
                if constexpr (!kFirst) {
                    if (kMasked && careful) {
                        pv_careful(vb, 1, w0, t - 1);
                    } else {
                        pv(vb, 1, w0);
                    }
                }
                read_v(t, 0, va);
                if constexpr (kMasked) mask(s2, t + 1);
                lm = lane_max(s2);
            }
            wait_older_loads();
            __syncthreads();
        };
        int t = t0;
        if (t + 1 < t1) {
            step(t, sa, wa, sb, wa, std::true_type{}, std::true_type{});
            sa = sb;
            for (++t; t + 2 < min(t_diag, t1); t += 2) {
                step(t, sa, wb, sb, wa, std::false_type{}, std::false_type{});
                step(t + 1, sb, wa, sa, wb, std::false_type{}, std::false_type{});
            }
            for (; t < t1 - 1; ++t) {
                step(t, sa, wb, sb, wa, std::false_type{}, std::true_type{});
                sa = sb;
                wa = wb;
            }
        }
        // Tile t = t1 - 1: PV of the tile before, its softmax and its own PV.
        if (active) {
            raise();
            u32x4 vb[kHalf][2];
            if (t > t0) {
                read_v(t - 1, 1, vb);
                if (careful) {
                    pv_careful(va, 0, wa, t - 1);
                    pv_careful(vb, 1, wa, t - 1);
                } else {
                    pv(va, 0, wa);
                    pv(vb, 1, wa);
                }
            }
            rescale();
            lsum += prefill_weights<kF16>(sa, p.scale_log2, bias, wa.hi, wa.lo);
            read_v(t, 0, va);
            read_v(t, 1, vb);
            if (careful) {
                pv_careful(va, 0, wa, t);
                pv_careful(vb, 1, wa, t);
            } else {
                pv(va, 0, wa);
                pv(vb, 1, wa);
            }
            const auto both =
                __builtin_amdgcn_permlane32_swap(__float_as_uint(lsum), __float_as_uint(lsum), false, false);
            lsum = __uint_as_float(both[0]) + __uint_as_float(both[1]);
            m_run = thr == -INFINITY ? -INFINITY : kBias - bias;
        }
    };
    run(false);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last loads land before LDS is used again
    float nonfinite = 0.f;
    if (active) {
#pragma unroll
        for (int n = 0; n < kPv; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) nonfinite = fmaf(o[n][r], 0.f, nonfinite);
    }
    const bool wave_bad = __builtin_amdgcn_ballot_w64(nonfinite != 0.f) != 0;
    if (lane == 0) sm_bad[wave] = wave_bad ? 1 : 0;
    __syncthreads();
    int bad = 0;
#pragma unroll
    for (int w = 0; w < kPrefillWaves; ++w) bad |= sm_bad[w];
    if (__builtin_amdgcn_readfirstlane(bad) != 0) {
        run(true);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    if (nparts > 1) {
        // The pieces' protocol is the persistent decode's: agent-scope stores,
        // each wave's wait for them, a barrier, one increment per piece; the
        // completing workgroup reads the slots with agent-scope loads, in piece
        // order, so the sum does not depend on who came last.
        const int slot0 = itp->slot0;
        if (active) {
            const uint64_t at = static_cast<uint64_t>(itp->slot) * kPrefillWaves + wave;
            if (h == 0) {
                const uint64_t ml = static_cast<uint64_t>(__float_as_uint(lsum)) << 32 | __float_as_uint(m_run);
                __hip_atomic_store(parts.ml + at * 32 + c, ml, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            uint64_t* acc = parts.acc + at * kPv * 8 * 64 + lane;
#pragma unroll
            for (int n = 0; n < kPv; ++n)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint64_t x = static_cast<uint64_t>(__float_as_uint(o[n][2 * k + 1])) << 32 |
                                       __float_as_uint(o[n][2 * k]);
                    __hip_atomic_store(acc + (n * 8 + k) * 64, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            const int done = __hip_atomic_fetch_add(parts.counters + slot0, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sm_bad[0] = done == nparts - 1;
            if (done == nparts - 1) {
                __hip_atomic_store(parts.counters + slot0, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(sm_bad[0]) == 0 || !active) return;
        const uint64_t first = static_cast<uint64_t>(slot0) * kPrefillWaves + wave;
        float m_all = -INFINITY;
        for (int i = 0; i < nparts; ++i) {
            const uint64_t ml = __hip_atomic_load(parts.ml + (first + i * kPrefillWaves) * 32 + c, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
            m_all = fmaxf(m_all, __uint_as_float(static_cast<uint32_t>(ml)));
        }
        lsum = 0.f;
#pragma unroll
        for (int n = 0; n < kPv; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[n][r] = 0.f;
        for (int i = 0; i < nparts; ++i) {
            const uint64_t at = first + i * kPrefillWaves;
            const uint64_t ml = __hip_atomic_load(parts.ml + at * 32 + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t* acc = parts.acc + at * kPv * 8 * 64 + lane;
            uint64_t x[kPv][8];
#pragma unroll
            for (int n = 0; n < kPv; ++n)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    x[n][k] = __hip_atomic_load(acc + (n * 8 + k) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            // A piece whose tokens a row does not see has m = -inf, l = 0, O = 0.
            const float f = fast_exp2(__uint_as_float(static_cast<uint32_t>(ml)) - m_all);
            lsum += __uint_as_float(static_cast<uint32_t>(ml >> 32)) * f;
#pragma unroll
            for (int n = 0; n < kPv; ++n)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    o[n][2 * k] += __uint_as_float(static_cast<uint32_t>(x[n][k])) * f;
                    o[n][2 * k + 1] += __uint_as_float(static_cast<uint32_t>(x[n][k] >> 32)) * f;
                }
        }
    }
    if (r0 + 32 * wave + c >= nrows) return;
    // C register r of PV block n in lane (c, h) is O[column c][dim 32n +
    // (r % 4) + 8 (r / 4) + 4h]: four contiguous outputs per r / 4, stored as
    // one vector (one 2-byte store per element took a fifth of the kernel).
    OutT* dst = static_cast<OutT*>(out_ptr) + qoff + 4 * h;
    const float inv = 1.0f / lsum;
#pragma unroll
    for (int n = 0; n < kPv; ++n) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            floatx4 x;
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = o[n][4 * k + r] * inv;
            OutT* at = dst + 32 * n + 8 * k;
            if constexpr (sizeof(OutT) == 4) {
                *reinterpret_cast<floatx4*>(at) = x;
            } else {
                uint2v a;
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    if constexpr (std::is_same_v<OutT, uint16_t>) {
                        const bf16x2_t y = {static_cast<__bf16>(x[2 * r]), static_cast<__bf16>(x[2 * r + 1])};
                        a[r] = __builtin_bit_cast(uint32_t, y);
                    } else {
                        const f16x2_t y = {static_cast<_Float16>(x[2 * r]), static_cast<_Float16>(x[2 * r + 1])};
                        a[r] = __builtin_bit_cast(uint32_t, y);
                    }
                }
                *reinterpret_cast<uint2v*>(at) = a;
            }
        }
    }
}

bool prefill_mfma_supported(const DecodeGeometry& g, uint32_t kv_dtype, uintptr_t query_addr, uintptr_t kv_base_addr,
                            uintptr_t out_addr) {
    const bool pow2 = g.tpb != 0 && (g.tpb & (g.tpb - 1)) == 0;
    const bool aligned = (g.block_stride % 16 == 0) && (g.k_off % 16 == 0) && (g.v_off % 16 == 0) &&
                         (g.token_stride % 16 == 0) && (g.head_stride % 16 == 0) && (kv_base_addr % 16 == 0) &&
                         (query_addr % 16 == 0) && (out_addr % 16 == 0);
    // Groups above 16 decode on the vector kernel, with fp32 weights, and so
    // prefill there. A lane's offset inside a block and the frame stride are
    // kept in 32 bits.
    return (kv_dtype == QVP_DTYPE_BF16 || kv_dtype == QVP_DTYPE_F16) && (g.head_dim == 128 || g.head_dim == 64) &&
           g.group >= 1 && g.group <= 16 && pow2 && g.tpb >= 16 && aligned &&
           g.token_stride * g.tpb <= 0x7fffffffu && g.block_stride <= 0xffffffffu;
}

template <bool kF16, int kD>
void launch_prefill(const DecodeGeometry& g, const PrefillItem* items, uint32_t count, const PrefillParts& parts,
                    uint32_t out_dtype, void* out, hipStream_t s) {
    const dim3 grid(count), block(kPrefillThreads);
    switch (out_dtype) {
        case QVP_DTYPE_F32:
            hipLaunchKernelGGL((prefill_mfma<kF16, kD, float>), grid, block, 0, s, g, items, parts, out);
            break;
        case QVP_DTYPE_BF16:
            hipLaunchKernelGGL((prefill_mfma<kF16, kD, uint16_t>), grid, block, 0, s, g, items, parts, out);
            break;
        default:
            hipLaunchKernelGGL((prefill_mfma<kF16, kD, _Float16>), grid, block, 0, s, g, items, parts, out);
            break;
    }
}

uint32_t log2_u32(uint32_t x) {
    uint32_t r = 0;
    while ((1u << r) < x) ++r;
    return r;
}

}  // namespace

void destroy_prefill_plan(qvp_prefill_plan& p) {
    if (p.staging_pending) (void)hipEventSynchronize(p.staging_done);
    if (p.staging != nullptr) (void)hipHostFree(p.staging);
    if (p.staging_done != nullptr) (void)hipEventDestroy(p.staging_done);
    if (p.device != nullptr) (void)hipFree(p.device);
    if (p.parts != nullptr) (void)hipFree(p.parts);
    if (p.virt != nullptr) (void)qvp_batch_destroy(p.virt);
    destroy_reader(p.reader);
    p = qvp_prefill_plan{};
}

namespace {

// Bytes of one workspace slot (head_dim 128), and the most slots a plan uses
// (64 MB): beyond them items stay whole.
constexpr size_t kPartBytes = kPrefillRows * (128 + 2) * sizeof(float);
constexpr uint32_t kMaxParts = 1024;

// How many pieces an item of nt tiles is cut into when a CU's share of the
// launch is `share` tiles: two workgroups share a CU and a lone one runs its
// tiles faster, so only items past 1.25 shares end late. Every piece costs its
// merger about three tiles' time (64 KB through the workspace), which makes
// sqrt(nt / 3) pieces the best for an item alone on the chip. (One item of 126
// tiles alone: 80.6 us whole, 28.8 us in 6 pieces; 63 tiles: 42.8 and 23.1 us;
// cutting to T / 512 tiles whatever the share put 4 prompts of up to 1024
// tokens at 46.5 us against 38.3 us whole, the workspace traffic being 75 MB.)
uint32_t piece_count(uint32_t nt, double share) {
    if (nt <= 1.25 * share) return 1;
    const uint32_t most = static_cast<uint32_t>(std::sqrt(nt / 3.0));
    return std::max<uint32_t>(1, std::min(most, static_cast<uint32_t>(std::ceil(nt / std::max(share, 1.0)))));
}

// The work list of one prefill, longest items first, so that the short ones
// fill the end. When all workgroups are resident at once (two per CU) none
// waits for another: the second half then goes shortest first, which puts the
// longest and the shortest on one CU.
std::vector<PrefillItem> plan_items(const std::vector<int32_t>& lens, const uint32_t* q_start, uint32_t group,
                                    uint32_t kv_heads, uint32_t cus, uint32_t* num_parts) {
    std::vector<PrefillItem> whole;
    uint64_t tiles = 0;
    uint32_t longest = 0;
    int32_t row = 0;
    for (size_t sq = 0; sq < lens.size(); ++sq) {
        const int32_t start = static_cast<int32_t>(q_start[sq]);
        const int32_t nrows = (lens[sq] - start) * static_cast<int32_t>(group);
        for (int32_t r0 = 0; r0 < nrows; r0 += kPrefillRows) {
            const int32_t last = start + (std::min(r0 + kPrefillRows, nrows) - 1) / static_cast<int32_t>(group);
            const int32_t nt = last / kTileTokens + 1;
            tiles += static_cast<uint64_t>(nt) * kv_heads;
            longest = std::max(longest, static_cast<uint32_t>(nt));
            for (uint32_t kv = 0; kv < kv_heads; ++kv) {
                whole.push_back(PrefillItem{static_cast<int32_t>(sq), static_cast<int32_t>(kv), start, r0, nrows, row, 0,
                                            nt, -1, -1, 1, 0});
            }
        }
        row += lens[sq] - start;
    }
    const double share = static_cast<double>(tiles) / cus;
    uint32_t used = 0;
    std::vector<PrefillItem> items;
    items.reserve(whole.size() + kMaxParts);
    for (const PrefillItem& it : whole) {
        const uint32_t nt = static_cast<uint32_t>(it.t1);
        const uint32_t n = piece_count(nt, share);
        if (n < 2 || used + n > kMaxParts) {
            items.push_back(it);
            continue;
        }
        for (uint32_t i = 0; i < n; ++i) {
            PrefillItem piece = it;
            piece.t0 = static_cast<int32_t>(nt * i / n);
            piece.t1 = static_cast<int32_t>(nt * (i + 1) / n);
            piece.slot = static_cast<int32_t>(used + i);
            piece.slot0 = static_cast<int32_t>(used);
            piece.nparts = static_cast<int32_t>(n);
            items.push_back(piece);
        }
        used += n;
    }
    *num_parts = used;
    // Longest first: a counting sort on the tile count (stable).
    std::vector<uint32_t> at(longest + 2, 0);
    for (const PrefillItem& it : items) ++at[longest - static_cast<uint32_t>(it.t1 - it.t0) + 1];
    for (size_t i = 1; i < at.size(); ++i) at[i] += at[i - 1];
    std::vector<PrefillItem> sorted(items.size());
    for (const PrefillItem& it : items) sorted[at[longest - static_cast<uint32_t>(it.t1 - it.t0)]++] = it;
    if (sorted.size() > cus && sorted.size() <= 2 * static_cast<size_t>(cus)) {
        std::reverse(sorted.begin() + cus, sorted.end());
    }
    return sorted;
}

// Grows a device buffer that earlier prefills on `s` or on the plan's last
// stream may still read.
int grow(void** ptr, size_t* cap, size_t need, const qvp_reader& reader, hipStream_t s) {
    if (*ptr != nullptr) {
        QVP_HIP(hipStreamSynchronize(s));
        if (reader.pending && reader.stream != s) QVP_HIP(hipStreamSynchronize(reader.stream));
        QVP_HIP(hipFree(*ptr));
    }
    *ptr = nullptr;
    *cap = 0;
    QVP_HIP(hipMalloc(ptr, need));
    *cap = need;
    return QVP_OK;
}

}  // namespace

}  // namespace qvp

extern "C" int qvp_paged_prefill(const qvp_prefill_args* a, void* stream) {
    using qvp::fail;
    if (a == nullptr) return fail(QVP_ERR_INVALID_ARGUMENT, "args is NULL");
    qvp_packed_view v{};
    QVP_TRY(qvp_batch_view(a->batch, &v));
    qvp_batch* batch = const_cast<qvp_batch*>(a->batch);
    if (a->query == nullptr || a->out == nullptr || a->kv_base == nullptr) {
        return fail(QVP_ERR_INVALID_ARGUMENT, "query, out or kv_base is NULL");
    }
    if (v.num_seqs > 0 && a->q_start == nullptr) return fail(QVP_ERR_INVALID_ARGUMENT, "q_start is NULL");
    const size_t esz = qvp::dtype_size(a->kv_dtype);
    const size_t osz = qvp::dtype_size(a->out_dtype);
    if (esz == 0 || osz == 0) return fail(QVP_ERR_INVALID_ARGUMENT, "unknown dtype");
    if (a->num_query_heads == 0 || a->num_kv_heads == 0 || a->num_query_heads % a->num_kv_heads != 0) {
        return fail(QVP_ERR_INVALID_ARGUMENT, "%u query heads do not group onto %u kv heads", a->num_query_heads,
                    a->num_kv_heads);
    }
    if (a->layer >= a->num_layers) {
        return fail(QVP_ERR_INVALID_ARGUMENT, "layer %u outside %u layers", a->layer, a->num_layers);
    }
    if (a->head_dim == 0) return fail(QVP_ERR_INVALID_ARGUMENT, "head_dim is 0");
    if (a->tokens_per_block != v.tokens_per_block) {
        return fail(QVP_ERR_INVALID_ARGUMENT, "batch packed for %u tokens per block, args say %u", v.tokens_per_block,
                    a->tokens_per_block);
    }
    if (a->head_stride < a->head_dim || a->token_stride == 0) {
        return fail(QVP_ERR_INVALID_ARGUMENT, "head vectors overlap");
    }
    const uint64_t last_elem = static_cast<uint64_t>(a->num_layers - 1) * a->layer_stride + a->stream_stride +
                               static_cast<uint64_t>(a->tokens_per_block - 1) * a->token_stride +
                               static_cast<uint64_t>(a->num_kv_heads - 1) * a->head_stride + a->head_dim;
    if (last_elem * esz > a->block_stride) {
        return fail(QVP_ERR_INVALID_ARGUMENT, "layout addresses %llu bytes but frames are %llu bytes",
                    static_cast<unsigned long long>(last_elem * esz),
                    static_cast<unsigned long long>(a->block_stride));
    }
    const std::vector<int32_t>& lens = batch->host_seq_lens;
    uint64_t total_new = 0;
    for (uint32_t s = 0; s < v.num_seqs; ++s) {
        if (a->q_start[s] >= static_cast<uint32_t>(lens[s])) {
            return fail(QVP_ERR_INVALID_ARGUMENT, "sequence %u: first new position %u is not below its context %d", s,
                        a->q_start[s], lens[s]);
        }
        total_new += static_cast<uint32_t>(lens[s]) - a->q_start[s];
    }
    if (total_new > 0x7fffffffu) return fail(QVP_ERR_INVALID_ARGUMENT, "too many new tokens");
    if (v.num_seqs == 0) return QVP_OK;

    qvp::DecodeGeometry g{};
    g.kv_base = static_cast<const uint8_t*>(a->kv_base);
    g.block_stride = a->block_stride;
    g.k_off = static_cast<uint64_t>(a->layer) * a->layer_stride * esz;
    g.v_off = g.k_off + a->stream_stride * esz;
    g.token_stride = a->token_stride * esz;
    g.head_stride = a->head_stride * esz;
    g.tables = v.block_tables;
    g.seq_lens = v.seq_lens;
    g.query = a->query;
    g.max_nb = v.max_blocks_per_seq;
    g.tpb = a->tokens_per_block;
    g.tpb_shift = qvp::log2_u32(a->tokens_per_block);
    g.num_q_heads = a->num_query_heads;
    g.num_kv_heads = a->num_kv_heads;
    g.group = a->num_query_heads / a->num_kv_heads;
    g.head_dim = a->head_dim;
    g.scale_log2 = a->scale * qvp::kLog2e;
    hipStream_t s = qvp::as_stream(stream);
    qvp_prefill_plan& plan = batch->prefill;
    // A pack left pending by qvp_pack_ahead is uploaded before its prefill.
    QVP_TRY(qvp::flush_own_upload(batch, s));

    // The MFMA kernel takes its running maximum on raw scores: scale > 0.
    if (!(a->scale > 0.0f) || !qvp::prefill_mfma_supported(g, a->kv_dtype, reinterpret_cast<uintptr_t>(a->query),
                                                            reinterpret_cast<uintptr_t>(a->kv_base),
                                                            reinterpret_cast<uintptr_t>(a->out))) {
        // One virtual sequence per new position, over the same frames, run in
        // chunks of at most kMaxVirtualIds block ids (a long prompt needs
        // about n^2 / (2 tokens_per_block) of them). Chunks are packed and
        // decoded in order on the stream; the query and output rows of a
        // chunk start at its first position's row.
        if (plan.virt == nullptr) QVP_TRY(qvp_batch_create(&plan.virt));
        qvp_decode_args d{};
        d.kv_base = a->kv_base;
        d.block_stride = a->block_stride;
        d.batch = plan.virt;
        d.kv_dtype = a->kv_dtype;
        d.out_dtype = a->out_dtype;
        d.layer = a->layer;
        d.num_layers = a->num_layers;
        d.num_query_heads = a->num_query_heads;
        d.num_kv_heads = a->num_kv_heads;
        d.head_dim = a->head_dim;
        d.tokens_per_block = a->tokens_per_block;
        d.head_stride = a->head_stride;
        d.token_stride = a->token_stride;
        d.stream_stride = a->stream_stride;
        d.layer_stride = a->layer_stride;
        d.scale = a->scale;
        const uint64_t row_elems = static_cast<uint64_t>(a->num_query_heads) * a->head_dim;
        std::vector<uint32_t> ids, cu{0}, ctx;
        uint64_t first_row = 0;
        auto flush = [&]() -> int {
            if (ctx.empty()) return QVP_OK;
            QVP_TRY(qvp_pack(plan.virt, static_cast<uint32_t>(ctx.size()), ids.data(), cu.data(), ctx.data(),
                             a->tokens_per_block, v.num_pool_blocks, v.split_tokens, stream));
            d.query = static_cast<const uint8_t*>(a->query) + first_row * row_elems * esz;
            d.out = static_cast<uint8_t*>(a->out) + first_row * row_elems * osz;
            QVP_TRY(qvp_paged_decode(&d, stream));
            first_row += ctx.size();
            ids.clear();
            cu.assign(1, 0);
            ctx.clear();
            return QVP_OK;
        };
        for (uint32_t sq = 0; sq < v.num_seqs; ++sq) {
            const uint32_t* row = batch->host_ids.data() + batch->host_cu_blocks[sq];
            for (uint32_t pos = a->q_start[sq]; pos < static_cast<uint32_t>(lens[sq]); ++pos) {
                const uint32_t nb = (pos + a->tokens_per_block) / a->tokens_per_block;
                if (ids.size() + nb > qvp::kMaxVirtualIds) QVP_TRY(flush());
                ids.insert(ids.end(), row, row + nb);
                cu.push_back(static_cast<uint32_t>(ids.size()));
                ctx.push_back(pos + 1);
            }
        }
        return flush();
    }

    // (Made and uploaded on every call, four prompts of 2048 tokens took 57 us
    // more alone than back to back; 28 us in the first call of a pack now.)
    // The plan depends on the pack (its context lengths), the first new
    // positions and the grouping: a call with the same ones (the next layer)
    // finds it on the device. Another stream than the last call's makes it
    // anew, after that call's kernel.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    QVP_HIP(hipStreamIsCapturing(s, &capture));
    const bool capturing = capture != hipStreamCaptureStatusNone;
    if (!capturing) QVP_TRY(qvp::wait_for_reader(plan.reader, s));
    const bool current = plan.valid && plan.generation == batch->generation && plan.stream == s &&
                         plan.group == g.group && plan.num_kv_heads == g.num_kv_heads &&
                         plan.q_start.size() == v.num_seqs &&
                         std::equal(plan.q_start.begin(), plan.q_start.end(), a->q_start);
    if (!current) {
        for (uint32_t sq = 0; sq < v.num_seqs; ++sq) {
            const uint64_t rows = static_cast<uint64_t>(static_cast<uint32_t>(lens[sq]) - a->q_start[sq]) * g.group;
            if (rows > 0x7fffffffu - qvp::kPrefillRows) return fail(QVP_ERR_INVALID_ARGUMENT, "too many new tokens");
        }
        int dev = 0, cus = 0;
        QVP_HIP(hipGetDevice(&dev));
        QVP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        uint32_t parts = 0;
        const std::vector<qvp::PrefillItem> items = qvp::plan_items(
            lens, a->q_start, g.group, g.num_kv_heads, static_cast<uint32_t>(std::max(cus, 1)), &parts);
        if (items.size() > 0x7fffffffu) return fail(QVP_ERR_INVALID_ARGUMENT, "too many prefill items");
        plan.valid = false;
        const size_t bytes = items.size() * sizeof(qvp::PrefillItem);
        // Host-side reuse of pinned staging only: no system-scope release.
        if (plan.staging_done == nullptr) {
            QVP_HIP(hipEventCreateWithFlags(&plan.staging_done, hipEventDisableTiming | hipEventDisableSystemFence));
        }
        if (plan.staging_pending) {
            QVP_HIP(hipEventSynchronize(plan.staging_done));
            plan.staging_pending = false;
        }
        if (plan.staging_cap < bytes) {
            if (plan.staging != nullptr) QVP_HIP(hipHostFree(plan.staging));
            plan.staging = nullptr;
            plan.staging_cap = 0;
            QVP_HIP(hipHostMalloc(&plan.staging, bytes, hipHostMallocCoherent));
            plan.staging_cap = bytes;
        }
        if (plan.device_cap < bytes) QVP_TRY(qvp::grow(&plan.device, &plan.device_cap, bytes, plan.reader, s));
        const size_t counter_bytes = qvp::round_up(parts * sizeof(int32_t), 256);
        if (parts > 0 && plan.parts_cap < counter_bytes + parts * qvp::kPartBytes) {
            const size_t need = counter_bytes + parts * qvp::kPartBytes;
            QVP_TRY(qvp::grow(&plan.parts, &plan.parts_cap, need, plan.reader, s));
            plan.parts_clean = false;
        }
        // Every launch leaves its counters at zero, but their number moves the
        // results behind them, which earlier plans wrote.
        if (parts > 0 && (!plan.parts_clean || plan.num_parts != parts)) {
            QVP_TRY(qvp_fill_bytes(plan.parts, 0, counter_bytes, s));
            plan.parts_clean = true;
        }
        if (parts > 0) plan.num_parts = parts;
        std::memcpy(plan.staging, items.data(), bytes);
        QVP_TRY(qvp::pull_from_pinned(plan.device, plan.staging, bytes, s));
        QVP_HIP(hipEventRecord(plan.staging_done, s));
        plan.staging_pending = true;
        plan.num_items = static_cast<uint32_t>(items.size());
        plan.stream = s;
        plan.generation = batch->generation;
        plan.group = g.group;
        plan.num_kv_heads = g.num_kv_heads;
        plan.q_start.assign(a->q_start, a->q_start + v.num_seqs);
        plan.valid = true;
    }

    const auto* dev_items = static_cast<const qvp::PrefillItem*>(plan.device);
    const uint32_t count = plan.num_items;
    qvp::PrefillParts parts{};
    if (plan.parts != nullptr) {
        uint8_t* base = static_cast<uint8_t*>(plan.parts);
        parts.counters = reinterpret_cast<int32_t*>(base);
        parts.ml = reinterpret_cast<uint64_t*>(base + qvp::round_up(plan.num_parts * sizeof(int32_t), 256));
        parts.acc = parts.ml + static_cast<uint64_t>(plan.num_parts) * qvp::kPrefillRows;
    }
    const bool f16 = a->kv_dtype == QVP_DTYPE_F16;
    if (g.head_dim == 128) {
        f16 ? qvp::launch_prefill<true, 128>(g, dev_items, count, parts, a->out_dtype, a->out, s)
            : qvp::launch_prefill<false, 128>(g, dev_items, count, parts, a->out_dtype, a->out, s);
    } else {
        f16 ? qvp::launch_prefill<true, 64>(g, dev_items, count, parts, a->out_dtype, a->out, s)
            : qvp::launch_prefill<false, 64>(g, dev_items, count, parts, a->out_dtype, a->out, s);
    }
    QVP_HIP(hipGetLastError());
    QVP_TRY(qvp::note_reader(plan.reader, s, s));
    // The kernel reads the packed block tables: a later pack into this slot
    // from another stream waits for it.
    return qvp::note_reader(batch->readers[batch->current], s, batch->upload_stream[batch->current]);
}
