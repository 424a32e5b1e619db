// Matrix-core split decode for bf16 and fp16 caches with head_dim 64, 96 or 256
// -- the reference's paged_attention_decode<T>
// (include/qwenvl_paged/PagedAttention.h:53-127) for T = bf16 or a two-byte
// half at those head dims, at batch scale.
//
// A workgroup takes one part of a sequence (the packer's fixed token splits,
// each cut into `parts` equal ranges) for one kv head; its four waves take the
// part's 32-token tiles round-robin. K and V of a tile sit in registers; the
// next tile's K is loaded as soon as QK has used this one's and its V after PV,
// so a wave always has between half a tile and a whole one in flight at
// the register cost of one. The tile math is the head_dim-128 decode's
// (mfma_tile.h): S^T = K Q^T per 16-token half (C register r of lane (c, j) is
// the score of token j + 4 (4u + r) for query head c), online softmax in base
// 2, O^T = V^T P^T. Lane (c, j) of V load q holds kD / 16 dims of token 4q + j
// (`lane_dim`), PV MFMA n takes element n of each of its loads, so C register r
// of MFMA n in lane (c, j) is O[head c][lane_dim(4j + r) + n]. The GQA group
// fills the MFMA columns, so each K/V byte is read once per group. P enters
// the MFMAs as hi + lo at head_dim 64 and for fp16, and as the three bf16 that
// make up its 24 bits for the other bf16 shapes, whose weights were kept in
// fp32 by the vector kernel (decode_grouped) that runs them otherwise.
//
// The waves merge through LDS and the parts in the launch (split_merge.h).
//
// HBM-bound. 28 query and 4 kv heads, contexts 512 .. 4096, with the merge: see
// split_parts in paged_decode.hip. Waves on four kv heads side by side (whole
// token rows per workgroup) were within 5% either way.
#include "decode_split16.h"
#include "mfma_tile.h"
#include "split_merge.h"

namespace qvp {
namespace {

constexpr int kS16Waves = 4;
constexpr int kS16Threads = kS16Waves * 64;

struct S16Args {
    const int32_t* split_seq;
    const int32_t* split_start;
    uint32_t split_tokens;
    uint32_t parts_shift;  // log2 of the ranges per split
    uint32_t part_tokens;  // split_tokens / parts, a multiple of 32
    SplitOutput so;
    float* ws_ml;          // [num_splits * parts][Hq][2]: running max (base 2), running sum
    float* ws_acc;         // [num_splits * parts][Hq][kD]
};

template <int kD>
struct S16Tile {
    u32x4 k[2][kD / 32];       // [half u][k-group i]: token 16u + (c >> 2) + 4 (c & 3), dims 32i + 8j .. + 7
    uint32_t v[8][kD / 32];    // [load q]: token 4q + j, dims of lane c in order
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3a __attribute__((ext_vector_type(3), aligned(4)));

template <typename T>
__device__ inline const __attribute__((address_space(4))) T* as_const(const T* ptr) {
    return (const __attribute__((address_space(4))) T*)(ptr);
}

// First dim of element n of lane-row x in a V load: contiguous runs of kD / 16
// dims, or at head_dim 256 two runs of eight (each 16-byte load instruction of
// a token then covers 256 contiguous bytes).
template <int kD>
__device__ inline int lane_dim(int x, int n) {
    return kD == 256 ? 8 * x + (n < 8 ? n : 120 + n) : (kD / 16) * x + n;
}

// Weights of one tile as B operands: fp16 and kTerms 2 as tile_weights; bf16
// with kTerms 3 exactly, as the truncations of p, p - hi and p - hi - mid.
template <bool kF16, int kTerms>
__device__ inline float split_weights(const floatx4 (&s)[2], float scale_log2, float m_use, u32x4 (&b)[kTerms]) {
    if constexpr (kTerms == 2) {
        return tile_weights<kF16>(s, scale_log2, m_use, b[0], b[1]);
    } else {
        float psum = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                uint32_t x0 = __float_as_uint(fast_exp2(fmaf(s[u][r], scale_log2, -m_use)));
                uint32_t x1 = __float_as_uint(fast_exp2(fmaf(s[u][r + 1], scale_log2, -m_use)));
                psum += __uint_as_float(x0) + __uint_as_float(x1);
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    b[k][2 * u + r / 2] = __builtin_amdgcn_perm(x1, x0, 0x07060302u);
                    if (k < 2) {
                        x0 = __float_as_uint(__uint_as_float(x0) - __uint_as_float(x0 & 0xffff0000u));
                        x1 = __float_as_uint(__uint_as_float(x1) - __uint_as_float(x1 & 0xffff0000u));
                    }
                }
            }
        }
        return psum;
    }
}

template <bool kF16, int kD>
__global__ __launch_bounds__(kS16Threads, 2) void decode_split16(DecodeGeometry p, S16Args sa) {
    constexpr int kK = kD / 32;
    constexpr int kN = kD / 16;
    constexpr int kTerms = kF16 || kD == 64 ? 2 : 3;
    using E = std::conditional_t<kF16, _Float16, uint16_t>;
    constexpr int kRowPad = kD + 4;  // LDS row of one merged output column (floats)
    constexpr int kLds = kS16Waves * 16 * kRowPad;  // floats
    static_assert(kLds >= kMergeLds, "the merge takes over the waves' LDS");
    __shared__ __attribute__((aligned(16))) float sm_o[kLds];  // [4][16][kRowPad]
    __shared__ int sm_last;
    __shared__ float sm_m[kS16Waves][16];
    __shared__ float sm_l[kS16Waves][16];

    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int c = lane & 15;
    const int j = lane >> 4;
    const int G = static_cast<int>(p.group);
    const int part = static_cast<int>(blockIdx.x / p.num_kv_heads);
    const int g = static_cast<int>(blockIdx.x - part * p.num_kv_heads);
    const int split = part >> sa.parts_shift;
    const int b = as_const(sa.split_seq)[split];
    const int first = as_const(sa.split_start)[split];
    const int ctx = as_const(p.seq_lens)[b];
    const int start = first + (part - (split << sa.parts_shift)) * static_cast<int>(sa.part_tokens);
    const int end = min(start + static_cast<int>(sa.part_tokens), ctx);
    if (start >= end) return;  // a range past the context: it has no slot
    const int ntile = (end - start + kTileTokens - 1) / kTileTokens;
    const auto* row = as_const(p.tables) + static_cast<uint64_t>(b) * p.max_nb;
    const uint32_t tmask = p.tpb - 1;
    const uint32_t tstride = static_cast<uint32_t>(p.token_stride);

    // Q operand of lane (c, j): query head g*G + c (columns past the group
    // repeat its last head and are never written), dims 32i + 8j .. + 7.
    // At head_dim 256 they are kept in LDS (rows 16 bytes apart in the banks):
    // 32 registers more would cost the second workgroup per CU or spill.
    constexpr bool kQLds = kD == 256;
    constexpr int kQRow = 2 * kD + 16;
    __shared__ __attribute__((aligned(16))) uint8_t sm_q[kQLds ? 16 * kQRow : 16];
    const uint16_t* const q0 = static_cast<const uint16_t*>(p.query) +
                               (static_cast<uint64_t>(b) * p.num_q_heads + static_cast<uint64_t>(g) * G) * kD;
    u32x4 qop[kQLds ? 1 : kK];
    if constexpr (kQLds) {
        for (int e = threadIdx.x; e < 16 * (kD / 8); e += kS16Threads) {
            const int hc = e / (kD / 8);
            const int x = e - hc * (kD / 8);
            *reinterpret_cast<u32x4*>(sm_q + hc * kQRow + 16 * x) =
                *reinterpret_cast<const u32x4*>(q0 + min(hc, G - 1) * kD + 8 * x);
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int i = 0; i < kK; ++i) {
            qop[i] = *reinterpret_cast<const u32x4*>(q0 + min(c, G - 1) * kD + 8 * j + 32 * i);
        }
    }
    auto q_of = [&](int i) {
        if constexpr (kQLds) {
            return *reinterpret_cast<const u32x4*>(sm_q + c * kQRow + 16 * j + 64 * i);
        } else {
            return qop[i];
        }
    };

    // Tile i holds tokens start + 32i .. + 31; each 16-token half lies in one
    // frame (start is a multiple of 32 and tokens_per_block a power of two >=
    // 16), a half past the part's end reads the last valid token's frame.
    // Tokens past the end read in-frame bytes: their scores are masked and
    // their values zeroed when the tile is computed.
    const uint8_t* kbase = p.kv_base + p.k_off + static_cast<uint64_t>(g) * p.head_stride;
    const uint64_t kv_gap = p.v_off - p.k_off;
    const uint32_t lane_k = static_cast<uint32_t>((c >> 2) + 4 * (c & 3)) * tstride + 16u * j;
    const uint32_t lane_v = static_cast<uint32_t>(j) * tstride + 2u * static_cast<uint32_t>(lane_dim<kD>(c, 0));
    struct Halves { const uint8_t* at[2]; };
    struct Blocks { int id[2]; };
    auto blocks_of = [&](int i) {
        Blocks r;
#pragma unroll
        for (int u = 0; u < 2; ++u) r.id[u] = row[min(start + kTileTokens * i + 16 * u, end - 1) >> p.tpb_shift];
        return r;
    };
    auto halves_of = [&](int i, const Blocks& blk) {
        Halves r;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t tok = static_cast<uint32_t>(start + kTileTokens * i + 16 * u) & tmask;
            r.at[u] = kbase + static_cast<uint64_t>(blk.id[u]) * p.block_stride + tok * tstride;
        }
        return r;
    };
    S16Tile<kD> t;
    auto load_k = [&](const Halves& at) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < kK; ++i) t.k[u][i] = load16(at.at[u] + lane_k + 64 * i);
    };
    // Each V load covers whole rows, so their lines are streamed (non-temporal:
    // head_dim 64 at 38.7 against 43.0 us with a merge launch, 256 at 76.5
    // against 79.7); a K row takes two or more loads, which meet in the caches
    // (non-temporal K loads too: 39.4 against 38.5 us and 75.9 against 69.3).
    auto load_v = [&](const Halves& at) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint8_t* vp = at.at[u] + kv_gap + 4u * q * tstride + lane_v;
                uint32_t(&v)[kD / 32] = t.v[4 * u + q];
                if constexpr (kD == 64) {
                    const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(vp));
                    v[0] = w[0];
                    v[1] = w[1];
                } else if constexpr (kD == 96) {
                    const u32x3a w = __builtin_nontemporal_load(reinterpret_cast<const u32x3a*>(vp));
#pragma unroll
                    for (int x = 0; x < 3; ++x) v[x] = w[x];
                } else {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const u32x4 w = load16_stream(vp + 256 * h);
#pragma unroll
                        for (int x = 0; x < 4; ++x) v[(4 * h + x) % (kD / 32)] = w[x];
                    }
                }
            }
    };

    floatx4 o[kN];
#pragma unroll
    for (int n = 0; n < kN; ++n) o[n] = floatx4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY;
    float l_run = 0.f;

    if (wave < ntile) {
        const Halves at = halves_of(wave, blocks_of(wave));
        load_k(at);
        load_v(at);
    }
    Blocks blk = blocks_of(min(wave + kS16Waves, ntile - 1));
    for (int i = wave; i < ntile; i += kS16Waves) {
        const int tok0 = start + kTileTokens * i;
        const bool more = i + kS16Waves < ntile;
        const Halves next = halves_of(i + kS16Waves, blk);
        blk = blocks_of(min(i + 2 * kS16Waves, ntile - 1));
        if constexpr (kQLds) asm volatile("" ::: "memory");  // read in every step, not held across them
        floatx4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int k = 0; k < kK; ++k) {
            const u32x4 qk = q_of(k);
#pragma unroll
            for (int u = 0; u < 2; ++u) s[u] = mfma16<kF16>(t.k[u][k], qk, s[u]);
        }
        if (more) load_k(next);
        if (tok0 + kTileTokens > end) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (tok0 + j + 16 * u + 4 * r >= end) s[u][r] = -INFINITY;
                }
            // Values of tokens past the part are not data (0 * NaN would poison O).
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (tok0 + 4 * q + j >= end) {
#pragma unroll
                    for (int x = 0; x < kD / 32; ++x) t.v[q][x] = 0u;
                }
            }
        }
        // Online softmax (softmax_p with its guard for columns without a score).
        const float mt = tile_max(s) * p.scale_log2;
        const float m_new = fmaxf(m_run, mt);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = fast_exp2(m_run - m_use);
        m_run = m_new;
        u32x4 w[kTerms];
        l_run = l_run * alpha + split_weights<kF16, kTerms>(s, p.scale_log2, m_use, w);
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
            for (int n = 0; n < kN; ++n) o[n] *= alpha;
        }
#pragma unroll
        for (int n = 0; n < kN; ++n) {
            u32x4 a;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                // Element n of tokens 2k and 2k + 1 of this lane's loads, token
                // 2k in the low half.
                a[k] = __builtin_amdgcn_perm(t.v[2 * k + 1][n >> 1], t.v[2 * k][n >> 1],
                                             (n & 1) ? 0x07060302u : 0x05040100u);
            }
#pragma unroll
            for (int x = 0; x < kTerms; ++x) o[n] = mfma16<kF16>(a, w[x], o[n]);
        }
        if (more) load_v(next);
    }
    l_run = sum_over_j(l_run);

    // Row r of the lane's column: runs of consecutive n are consecutive dims.
    auto write_row = [&](float* dst, int r) {
        constexpr int kRun = kD == 256 ? 8 : kN;
#pragma unroll
        for (int n = 0; n < kN; n += kRun) {
            float* at = dst + lane_dim<kD>(4 * j + r, n);
#pragma unroll
            for (int x = 0; x < kRun; x += 2) {
                *reinterpret_cast<float2*>(at + x) = float2{o[n + x][r], o[n + x + 1][r]};
            }
        }
    };
    // Merge the waves (one without tiles has m = -inf, l = 0, O = 0).
    if (j == 0) {
        sm_m[wave][c] = m_run;
        sm_l[wave][c] = l_run;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) write_row(sm_o + (wave * 16 + c) * kRowPad, r);
    __syncthreads();
    const int split_tokens = static_cast<int>(sa.split_tokens);
    const SlotRange slots = slots_of(split - as_const(sa.split_start)[split] / split_tokens, ctx, split_tokens,
                                     static_cast<int>(sa.parts_shift));
    auto value = [&](int hc, int d4, float& m, float& l) {
        m = sm_m[0][hc];
#pragma unroll
        for (int w = 1; w < kS16Waves; ++w) m = fmaxf(m, sm_m[w][hc]);
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
        l = 0.f;
#pragma unroll
        for (int w = 0; w < kS16Waves; ++w) {
            const float mw = sm_m[w][hc];
            const float f = mw == -INFINITY ? 0.f : fast_exp2(mw - m);
            acc += *reinterpret_cast<const floatx4*>(sm_o + (w * 16 + hc) * kRowPad + d4) * f;
            l += sm_l[w][hc] * f;
        }
        if constexpr (kD != 64) {
            // An infinite value meets a weight's terms one by one, and a zero or
            // negative lower term makes NaN of it where the whole weight gives
            // infinity. Such sums are taken again token by token.
            const bool nan = acc[0] != acc[0] || acc[1] != acc[1] || acc[2] != acc[2] || acc[3] != acc[3];
            if (nan && m > -INFINITY && m < INFINITY) {
                const float bias = (kF16 ? kF16WeightLog2 : 0.f) - m;
                acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int tok = start; tok < end; ++tok) {
                    const uint8_t* at = kbase + static_cast<uint64_t>(row[tok >> p.tpb_shift]) * p.block_stride +
                                        (static_cast<uint32_t>(tok) & tmask) * tstride;
                    const E* k = reinterpret_cast<const E*>(at);
                    const E* v = reinterpret_cast<const E*>(at + kv_gap) + d4;
                    const E* q = reinterpret_cast<const E*>(q0) + hc * kD;
                    float sc = 0.f;
#pragma unroll 1
                    for (int x = 0; x < kD; ++x) sc = fmaf(to_float<E>(q[x]), to_float<E>(k[x]), sc);
                    const float pw = fast_exp2(fmaf(sc, p.scale_log2, bias));
#pragma unroll
                    for (int x = 0; x < 4; ++x) acc[x] = fmaf(pw, to_float<E>(v[x]), acc[x]);
                }
            }
        }
        return acc;
    };
    finish_part<kD>(sa.so, sa.ws_ml, sa.ws_acc, slots, static_cast<uint64_t>(part), static_cast<uint32_t>(b),
                    static_cast<uint32_t>(g * G), G, p.num_q_heads,
                    static_cast<uint32_t>(b) * p.num_kv_heads + static_cast<uint32_t>(g), value, sm_o, &sm_last);
}

template <bool kF16, int kD>
void launch_for(const DecodeGeometry& g, const S16Args& sa, unsigned groups, hipStream_t stream) {
    hipLaunchKernelGGL((decode_split16<kF16, kD>), dim3(groups), dim3(kS16Threads), 0, stream, g, sa);
}

}  // namespace

bool split16_supported(const DecodeGeometry& g, uint32_t kv_dtype, uint32_t split_tokens, uintptr_t query_addr) {
    const bool pow2 = g.tpb != 0 && (g.tpb & (g.tpb - 1)) == 0;
    const bool aligned = (g.block_stride % 16 == 0) && (g.k_off % 16 == 0) && (g.v_off % 16 == 0) &&
                         (g.token_stride % 16 == 0) && (g.head_stride % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(g.kv_base) % 16 == 0) && (query_addr % 16 == 0);
    // A lane's offset inside a block is kept in 32 bits.
    return (kv_dtype == QVP_DTYPE_BF16 || kv_dtype == QVP_DTYPE_F16) &&
           (g.head_dim == 64 || g.head_dim == 96 || g.head_dim == 256) && g.group >= 1 && g.group <= 16 &&
           g.scale_log2 > 0.0f && pow2 && g.tpb >= 16 && split_tokens % kTileTokens == 0 && aligned &&
           g.token_stride * g.tpb <= 0x7fffffffu;
}

int launch_split16_decode(const DecodeGeometry& g, const qvp_packed_view& v, uint32_t parts, int32_t* counters,
                          uint32_t kv_dtype, uint32_t out_dtype, void* out, void* workspace, hipEvent_t split_event,
                          hipStream_t stream) {
    const uint64_t heads = static_cast<uint64_t>(v.num_splits) * parts * g.num_q_heads;
    S16Args sa{};
    sa.split_seq = v.split_seq;
    sa.split_start = v.split_start;
    sa.split_tokens = v.split_tokens;
    while ((1u << sa.parts_shift) < parts) ++sa.parts_shift;
    sa.part_tokens = v.split_tokens / parts;
    sa.so = SplitOutput{out, out_dtype, counters};
    sa.ws_ml = static_cast<float*>(workspace);
    sa.ws_acc = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + round_up(heads * 2 * sizeof(float), 256));
    const uint64_t groups = static_cast<uint64_t>(v.num_splits) * parts * g.num_kv_heads;
    if (groups > 0x7fffffffu) return fail(QVP_ERR_INVALID_ARGUMENT, "too many (split, kv head) pairs");
    const unsigned n = static_cast<unsigned>(groups);
    if (kv_dtype == QVP_DTYPE_F16) {
        g.head_dim == 64   ? launch_for<true, 64>(g, sa, n, stream)
        : g.head_dim == 96 ? launch_for<true, 96>(g, sa, n, stream)
                           : launch_for<true, 256>(g, sa, n, stream);
    } else {
        g.head_dim == 64   ? launch_for<false, 64>(g, sa, n, stream)
        : g.head_dim == 96 ? launch_for<false, 96>(g, sa, n, stream)
                           : launch_for<false, 256>(g, sa, n, stream);
    }
    QVP_HIP(hipGetLastError());
    if (split_event != nullptr) QVP_HIP(hipEventRecord(split_event, stream));
    if (counters != nullptr) return QVP_OK;
    return launch_merge_splits(g, v, parts, out_dtype, out, sa.ws_ml, sa.ws_acc, stream);
}

}  // namespace qvp
