// Online self-attention on bf16 parts for grids that fill the chip, rows of
// 16-byte multiples (dim % 4 == 0): O = softmax(Q K^T / sqrt(dim)) V over
// [heads, seq, dim], the contract of attention_f32.hip
// (src/runtime/metal_attention.rs:1-8, 64-137), in the same transposed form:
//   S^T[key, q] = sum_d K[key, d] Q[q, d]         (A = K, B = Q^T)
//   O^T[d, q]  += sum_key V^T[d, key] P^T[key, q]  (A = V^T, B = P^T)
// Every FP32 operand (Q, K, V and the probabilities) is held exactly as three
// bf16 parts and multiplied as six products of parts with FP32 sums
// (split_bf16.hpp). The score tile leaves a lane with query l % 32 of 16 keys;
// V's keys are laid out in LDS in that order, so the probabilities are split
// where they are and never leave registers.
//
// What bounds it: the bf16 matrix cores (12 * dim / 16 MFMAs of 32 cycles per 32
// queries and 32 keys), and beside them the VALU: the softmax, splitting the
// probabilities, and splitting each K and V element once per block. Eight
// waves share a tile, two per SIMD, so that one wave's softmax runs beside the
// other's MFMAs. Measured (us, one box, N(0, 1) operands) against the FP32-MFMA
// kernel: H128 S4096 D128 causal 4076 -> 2508 (219 TFLOP/s), H64 S2048 D128
// noncausal 996 -> 610, H128 S4096 D64 causal 2239 -> 1439, H24 S1531 D80
// noncausal 410 -> 160 (dims pad to 96 instead of 128, and 144 blocks of 256
// queries run in one round where 288 of 128 took two), H32 S1000 D96 noncausal
// 149 -> 97. A sequence of one to three key tiles gains least: H512 S64 D128
// causal 46.5 -> 21.9, H2 S64 D32 4.8 -> 4.8, and H304 S31 D128 noncausal
// loses, 17.1 -> 18.0 (one block a CU where that kernel has two). Error against
// FP64 (2-norm, relative): 4.0e-7 where that kernel had 5.4e-7 (H128 S4096 D128
// causal), 6.3e-7 for 7.8e-7 (H24 S1531 D80).
//
// Head dim 128 with four waves and a causal mask fills a SIMD's 512 registers
// and keeps 17 more in scratch: Q's operands, three of which it reloads a tile.
//
// V is scaled before it is split and the outputs are scaled back, Q is scaled
// up and K down, so every finite V and Q is carried exactly (split_bf16.hpp).
// What the parts do not carry is noticed and done again from global memory
// with FP32 MFMAs, per wave: non-finite sums (infinities, NaN or overflow among
// the operands) and queries past 2^64 in log2 units. With such queries out of
// the way the bits that a K below 2^-78 loses move no score by more than 2^-38
// a dim. Weights below 2^-100 of the reference weight keep fewer than 24 bits.
#include <type_traits>
#include <utility>

#include "attention_flash.hpp"
#include "split_bf16.hpp"

namespace jade {
namespace hipk {
namespace {

namespace flash {
using namespace split;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kKeys = 32;      // keys per tile
// The running maximum is a lazy reference: it moves only when a tile exceeds it
// by more than this (log2 units), so the accumulators are rarely rescaled.
constexpr float kLazyMax = 8.0f;
constexpr uint32_t kRawBuffer = 0x00020000;   // buffer descriptor word 3: raw buffer, 32-bit data format
constexpr uint32_t kDeadOffset = 0x80000000u;  // past every head of at most 2 GiB: reads zero
// Scaled Q past this takes the FP32 path: then no product of a part of Q with a
// part of a tiny K loses more than an FP32 score's rounding.
constexpr float kMostQ = 0x1p64f * kScaleQ;

__device__ inline float halves_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float halves_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// f(0), f(1), ... f(N - 1) with compile-time arguments: the interleaved
// schedules below are chosen by the compiler's front end, not by its unroller.
template <class F, int... I>
__device__ inline void each(std::integer_sequence<int, I...>, F &&f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ inline void each(F &&f) {
    each(std::make_integer_sequence<int, N>{}, f);
}
// Event E of ALL, spread evenly over the slots, belongs to slot N of SLOTS
// when first<N> <= E < first<N + 1>.
template <int N, int ALL, int SLOTS>
constexpr int kFirstEvent = N >= SLOTS ? ALL : (N * ALL + SLOTS - 1) / SLOTS;

// (head, query block) of workgroup `id` in a launch over heads x blocks. The
// hardware hands ids to the XCDs in turn. Each XCD takes kHeadGroup heads at a
// time, longest causal rows first within the group, so that most of its
// workgroups stream the same few heads' K and V through its L2.
constexpr int kHeadGroup = 4;
__device__ inline void block_of(int id, int heads, int blocks, int &head, int &qb) {
    if (heads % 8 != 0) {
        head = id % heads;
        qb = blocks - 1 - id / heads;
        return;
    }
    const int xcd = id % 8, at = id / 8, span = kHeadGroup * blocks;
    const int group = at / span, size = min(kHeadGroup, heads / 8 - group * kHeadGroup), rest = at - group * span;
    head = 8 * (group * kHeadGroup + rest % size) + xcd;
    qb = blocks - 1 - rest / size;
}

template <int DP, int NW>
struct Shape {
    static constexpr int kWide = DP <= 64 ? 64 : 128;            // dims staged (padding reads zero)
    static constexpr int kSteps = DP / 16, kBlocks = DP / 32;    // score steps, output blocks
    static constexpr int kChunks = kKeys * kWide / 8 / (64 * NW);  // K chunks (eight dims) per thread: 1 or 2
    static constexpr uint32_t kPartK = kKeys * kWide * 2, kPartV = kWide * kKeys * 2;
    static constexpr uint32_t kTileK = kParts * kPartK, kTileV = kParts * kPartV;
    static constexpr uint32_t kTiles = 2 * (kTileK + kTileV);
    // Eight waves share a SIMD's registers by two: Q's third part lives in LDS
    // at head dim 128.
    static constexpr bool kPlain = kChunks == 1;  // two waves per SIMD; else one, with its own overlap
    static constexpr bool kQInLds = NW == 8 && DP == 128;
    static constexpr uint32_t kLdsBytes = kTiles + (kQInLds ? uint32_t(NW) * kSteps * 1024u : 0u);
    static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");
};
}  // namespace flash

template <int DP, int NW, bool CAUSAL>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DP <= 64 || NW == 8 ? 2 : 1, DP <= 64 || NW == 8 ? 2 : 1))) void
attention_flash(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V,
                float *__restrict__ O, int seq, int dim, float qscale) {
    using namespace flash;
    using S = Shape<DP, NW>;
    constexpr int KS = S::kSteps, NB = S::kBlocks, WIDE = S::kWide, CH = S::kChunks, VROWS = 4 * CH;
    __shared__ __attribute__((aligned(1024))) char lds[S::kLdsBytes];
    const int tid = int(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c = lane & 31;
    constexpr int kBQ = 32 * NW;
    int head, qb;
    block_of(int(blockIdx.x) + int(gridDim.x) * int(blockIdx.y), int(gridDim.x), int(gridDim.y), head, qb);
    const size_t base = size_t(head) * size_t(seq) * size_t(dim);
    const int q0 = qb * kBQ + wave * 32, qi = q0 + c;
    const int t_end = ((CAUSAL ? min(seq, qb * kBQ + kBQ) : seq) + kKeys - 1) / kKeys;

    const uint32_t head_bytes = uint32_t(seq) * uint32_t(dim) * 4u, row_bytes = uint32_t(dim) * 4u;
    // Q^T operand: step s holds dims 16s + 8h + e of query qi, in log2 units.
    // Rows past seq and dims past dim read zero.
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(Q + base), 0, int(head_bytes), int(kRawBuffer));
    f32x4 qraw[KS][2];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int d = 16 * s + 8 * h + 4 * x;
            const uint32_t at = qi < seq && d < dim ? uint32_t(qi) * row_bytes + uint32_t(d) * 4u : kDeadOffset;
            qraw[s][x] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, int(at), 0, 0));
        }
    bf16x8 qp[KS][kParts];
    const uint32_t qplace = S::kTiles + uint32_t(wave * KS * 64 + lane) * 16u;  // third part, kQInLds
    float most_q = 0.f;  // largest |Q| scaled; NaN shows in the sums
    auto convert_q = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            u32x4 p[kParts];
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    f32x2 r = f32x2{qraw[s][x][2 * u], qraw[s][x][2 * u + 1]} * (qscale * kScaleQ);
                    most_q = fmaxf(most_q, fmaxf(fabsf(r.x), fabsf(r.y)));
#pragma unroll
                    for (int w = 0; w < kParts; ++w) {
                        const uint32_t k = pack(r.x, r.y);
                        p[w][2 * x + u] = k;
                        r = rest_of(r, k);
                    }
                }
#pragma unroll
            for (int w = 0; w < kParts; ++w) {
                if (S::kQInLds && w == 2)
                    *reinterpret_cast<u32x4 *>(lds + qplace + uint32_t(s) * 1024u) = p[w];
                else
                    qp[s][w] = __builtin_bit_cast(bf16x8, p[w]);
            }
        }
        asm volatile("" : "+v"(most_q));  // taken here, not after the loop from the 8 KS values
    };

    // Staging. K chunk i of a thread: row (tid + 64 NW i) / (WIDE / 8), eight
    // dims. V: two dims of VROWS keys.
    const __amdgpu_buffer_rsrc_t rk =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(K + base), 0, int(head_bytes), int(kRawBuffer));
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(V + base), 0, int(head_bytes), int(kRawBuffer));
    auto swz_k = [](int row) { return WIDE == 128 ? row & 15 : (row >> 1) & 7; };
    uint32_t koff[CH][2], kwrite[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int id = tid + 64 * NW * i, row = id / (WIDE / 8), q = id % (WIDE / 8);
#pragma unroll
        for (int x = 0; x < 2; ++x)
            koff[i][x] = 8 * q + 4 * x < dim ? uint32_t(row) * row_bytes + uint32_t(8 * q + 4 * x) * 4u : kDeadOffset;
        kwrite[i] = uint32_t(row * WIDE * 2 + ((q ^ swz_k(row)) << 4));
    }
    // LDS row of V dim 2l + j: the even dims, then the odd ones (so a wave's
    // writes go to adjacent rows and a lane ends up with adjacent dims), dims
    // past DP after them. Chunk 2s + x of a row holds keys 16s + 4x + {0-3, 8-11}:
    // the keys whose probabilities a lane of half x holds.
    const int vl = WIDE == 128 ? lane : c, vq = WIDE == 128 ? wave : 2 * wave + h;  // dim pair; octet (CH 2) or quad of keys
    const int vs = CH == 2 ? vq >> 1 : vq >> 2, vx = vq & 1, vhalf = CH == 2 ? 0 : (vq >> 1) & 1;
    const int vrow = vl < DP / 2 ? vl : DP / 2 + vl;  // dims past DP: rows DP + l - DP / 2 on
    const int vstep = vl < DP / 2 ? DP / 2 : (WIDE - DP) / 2;
    const uint32_t vdims = 2 * vl < dim ? uint32_t(8 * vl) : kDeadOffset;
    const uint32_t voff = uint32_t(16 * vs + 4 * vx + 8 * vhalf) * row_bytes + vdims;
    uint32_t vwrite[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = vrow + j * vstep;
        vwrite[j] = 2 * S::kTileK + uint32_t(row * 64 + (((2 * vs + vx) ^ ((row >> 2) & 3)) << 4) + 8 * vhalf);
    }
    f32x4 kraw[CH][2];
    f32x2 vraw[VROWS];
    auto load_k = [&](int i, int x, int t) {
        kraw[i][x] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, int(koff[i][x] + uint32_t(t * kKeys) * row_bytes), 0, 0));
    };
    auto load_v = [&](int e, int t) {
        const uint32_t key = uint32_t(t * kKeys + (e & 3) + (e >> 2) * 8);
        vraw[e] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rv, int(voff + key * row_bytes), 0, 0));
    };
    // Conversion: K pair (i, u), V pair (column j, u), in three pieces.
    constexpr int kPairsV = VROWS / 2;
    uint32_t kparts[CH][kParts][4], vparts[2][kParts][kPairsV];
    f32x2 rest;
    auto piece_of = [&](uint32_t &out, int piece, f32x2 x) {
        const f32x2 from = piece == 0 ? x : rest;
        out = pack(from.x, from.y);
        if (piece < 2) rest = rest_of(from, out);
    };
    auto convert_k = [&](int i, int u, int piece) {
        const f32x4 k = kraw[i][u >> 1];
        piece_of(kparts[i][piece][u], piece, (u & 1 ? f32x2{k.z, k.w} : f32x2{k.x, k.y}) * kScaleK);
    };
    auto convert_v = [&](int j, int u, int piece) {
        const f32x2 k0 = vraw[2 * u], k1 = vraw[2 * u + 1];
        piece_of(vparts[j][piece][u], piece, (j ? f32x2{k0.y, k1.y} : f32x2{k0.x, k1.x}) * kScaleV);
    };
    auto write_k = [&](int i, int p, uint32_t buf) {
        *reinterpret_cast<u32x4 *>(lds + (kwrite[i] + buf * S::kTileK) + uint32_t(p) * S::kPartK) =
            u32x4{kparts[i][p][0], kparts[i][p][1], kparts[i][p][2], kparts[i][p][3]};
    };
    auto write_v = [&](int j, int p, uint32_t buf) {
        char *to = lds + (vwrite[j] + buf * S::kTileV) + uint32_t(p) * S::kPartV;
        if constexpr (CH == 2)
            *reinterpret_cast<u32x4 *>(to) = u32x4{vparts[j][p][0], vparts[j][p][1], vparts[j][p][kPairsV - 2],
                                                   vparts[j][p][kPairsV - 1]};
        else
            *reinterpret_cast<u32x2 *>(to) = u32x2{vparts[j][p][0], vparts[j][p][1]};
    };
    // Operand reads.
    uint32_t kread[KS], vread[2];
#pragma unroll
    for (int s = 0; s < KS; ++s) kread[s] = uint32_t(c * WIDE * 2 + (((2 * s + h) ^ swz_k(c)) << 4));
#pragma unroll
    for (int s = 0; s < 2; ++s) vread[s] = 2 * S::kTileK + uint32_t(c * 64 + (((2 * s + h) ^ ((c >> 2) & 3)) << 4));
    bf16x8 kf[2][kParts], q2[2], vf[2][NB][kParts];
    auto read_k = [&](int s, int p, uint32_t buf) {
        kf[s & 1][p] = *reinterpret_cast<const bf16x8 *>(lds + (kread[s] + buf * S::kTileK) + uint32_t(p) * S::kPartK);
    };
    auto read_q = [&](int s) {
        if (S::kQInLds) q2[s & 1] = *reinterpret_cast<const bf16x8 *>(lds + qplace + uint32_t(s) * 1024u);
    };
    auto q_part = [&](int s, int p) { return S::kQInLds && p == 2 ? q2[s & 1] : qp[s][p]; };
    auto read_v = [&](int s, int b, int p, uint32_t buf) {
        vf[s][b][p] = *reinterpret_cast<const bf16x8 *>(lds + (vread[s] + buf * S::kTileV) + uint32_t(b) * 2048u +
                                                        uint32_t(p) * S::kPartV);
    };
    auto publish = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    f32x16 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f32x16{};
    float row_max = -INFINITY, row_sum = 0.f;  // row_sum: this lane's half of the keys

    const bool rows = q0 < seq;
    auto live = [&](int t) { return rows && t < t_end && (!CAUSAL || t * kKeys <= q0 + 31); };
    f32x16 st;  // scores, then probabilities, of the tile being weighted
    auto mask = [&](int t, f32x16 &s) {
        const int kt = t * kKeys;
        if (kt + kKeys <= seq && (!CAUSAL || kt + kKeys - 1 <= q0)) return;  // wave-uniform
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int key = kt + 8 * (v >> 2) + 4 * h + (v & 3);
            if (key >= seq || (CAUSAL && key > qi)) s[v] = -INFINITY;
        }
    };

    // Prologue: K of the first tile (two when pipelined) and V of it in LDS, the
    // next of each in flight. Every load is issued before the first is waited
    // for: a short sequence is little more than this (against each load waited
    // for in its turn, Q's behind branches: H304 S31 D128 noncausal 20.6 -> 18.1
    // us, H1 S64 D128 causal 14.3 -> 12.9, H512 S64 D128 causal 26.9 -> 23.7).
    constexpr int kAhead = S::kPlain ? 1 : 2;
    f32x4 kfirst[kAhead][CH][2];
#pragma unroll
    for (int w = 0; w < kAhead; ++w)
#pragma unroll
        for (int i = 0; i < CH; ++i)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                load_k(i, x, w);
                kfirst[w][i][x] = kraw[i][x];
            }
#pragma unroll
    for (int e = 0; e < VROWS; ++e) load_v(e, 0);
    __builtin_amdgcn_sched_barrier(0);
    convert_q();
#pragma unroll
    for (int w = 0; w < kAhead; ++w) {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
#pragma unroll
            for (int x = 0; x < 2; ++x) kraw[i][x] = kfirst[w][i][x];
#pragma unroll
            for (int x = 0; x < 12; ++x) convert_k(i, x / 3, x % 3);
#pragma unroll
            for (int p = 0; p < kParts; ++p) write_k(i, p, uint32_t(w));
        }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int x = 0; x < 2; ++x) load_k(i, x, kAhead);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int x = 0; x < 3 * kPairsV; ++x) convert_v(j, x / 3, x % 3);
#pragma unroll
        for (int p = 0; p < kParts; ++p) write_v(j, p, 0);
    }
#pragma unroll
    for (int e = 0; e < VROWS; ++e) load_v(e, 1);
    publish();
    if (!S::kPlain && live(0)) {
        st = f32x16{};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int p = 0; p < kParts; ++p) read_k(s, p, 0);
#pragma unroll
            for (int p = 0; p < kProducts; ++p)
                st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s & 1][kPartA[p]], qp[s][kPartB[p]], st, 0, 0, 0);
        }
        mask(0, st);
    }
    // The first tile's own staging overwrites the K this score product read.
    if (!S::kPlain) publish();
    if (!S::kPlain && live(1))
#pragma unroll
        for (int p = 0; p < kParts; ++p) read_k(0, p, 1);

    // One wave per SIMD (four waves, more than 64 dims) overlaps its own work:
    // scores of tile t + 1 (SCORE) beside the softmax of tile t
    // (WEIGH), then tile t's P V beside the conversion of K of t + 2 and V of
    // t + 1. The barrier lies inside the second half: by then this tile's
    // conversions are written and its V operands read, and the next tile's
    // first K operands are read after it.
    auto tile = [&](int t, auto sc, auto wc) __attribute__((always_inline)) {
        constexpr bool SCORE = decltype(sc)::value, WEIGH = decltype(wc)::value;
        const uint32_t cur = uint32_t(t) & 1u, other = cur ^ 1u;
        f32x16 sn[2] = {};
        bf16x8 pp[2][kParts];
        uint32_t pw[kParts][8];
        float top = -INFINITY, next_max = 0.f, old_weight = 1.f, lane_sum = 0.f;
        constexpr int kSoft = WEIGH ? 45 : 0, kEvents = kSoft + 12, kSlots1 = 6 * KS;
        auto event = [&](auto ec) __attribute__((always_inline)) {
            constexpr int e = decltype(ec)::value;
            if constexpr (e < kSoft) {
                if constexpr (e < 4) {
#pragma unroll
                    for (int v = 4 * e; v < 4 * e + 4; ++v) top = fmaxf(top, st[v]);
                } else if constexpr (e == 4) {
                    top = halves_max(top);
                    next_max = top > row_max + kLazyMax ? top : row_max;
                    // Scores that are all -inf leave the reference finite.
                    if (next_max == -INFINITY) next_max = 0.f;
                    old_weight = __builtin_amdgcn_exp2f(row_max - next_max);
                } else {
                    constexpr int u = (e - 5) / 5, w = (e - 5) % 5;
                    if constexpr (w < 2) {
                        constexpr int v = 2 * u + w;
                        st[v] = __builtin_amdgcn_exp2f(st[v] - next_max);
                        lane_sum += st[v];
                    } else {
                        piece_of(pw[w - 2][u], w - 2, f32x2{st[2 * u], st[2 * u + 1]});
                    }
                }
            } else {
                constexpr int x = e - kSoft;
                convert_k(0, x / 3, x % 3);
                if constexpr (x % 6 == 5) load_k(0, x / 6, t + 3);
                if constexpr (x == 11)
#pragma unroll
                    for (int p = 0; p < kParts; ++p) write_k(0, p, cur);
            }
        };
        each<kSlots1>([&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value, s = n / 6, p = n % 6;
            if constexpr (SCORE) {
                __builtin_amdgcn_sched_barrier(0);
                sn[s & 1] =
                    __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s & 1][kPartA[p]], qp[s][kPartB[p]], sn[s & 1], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (s + 1 < KS && (p & 1) == 0) read_k(s + 1, p == 0 ? 2 : p == 2 ? 0 : 1, other);
            }
            if constexpr (WEIGH) {
                // P V's first operands, over the last slots.
                constexpr int r = n - (kSlots1 - 3 * NB);
                if constexpr (r >= 0) read_v(0, r % NB, r / NB == 0 ? 2 : r / NB == 1 ? 0 : 1, cur);
            }
            constexpr int lo = kFirstEvent<n, kEvents, kSlots1>, hi = kFirstEvent<n + 1, kEvents, kSlots1>;
            each<hi - lo>([&](auto ec) __attribute__((always_inline)) {
                event(std::integral_constant<int, lo + decltype(ec)::value>{});
            });
            if constexpr (SCORE) __builtin_amdgcn_sched_barrier(0);
        });
        if (WEIGH) {
            row_sum = row_sum * old_weight + lane_sum;
            row_max = next_max;
            if (__any(old_weight != 1.0f)) {
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[b] *= old_weight;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int p = 0; p < kParts; ++p)
                    pp[s][p] = __builtin_bit_cast(
                        bf16x8, u32x4{pw[p][4 * s], pw[p][4 * s + 1], pw[p][4 * s + 2], pw[p][4 * s + 3]});
        }
        constexpr int kSlots2 = 12 * NB, kEvents2 = 12 * (CH - 1) + 6 * kPairsV, kGate = kSlots2 * 5 / 6 < kSlots2 - kParts ? kSlots2 * 5 / 6 : kSlots2 - kParts;
        auto event2 = [&](auto ec) __attribute__((always_inline)) {
            constexpr int e = decltype(ec)::value;
            if constexpr (e < 6 * kPairsV) {
                constexpr int j = e / (3 * kPairsV), u = e / 3 % kPairsV, x = e % 3;
                convert_v(j, u, x);
                if constexpr (x == 2) {
                    if constexpr (j == 1) {
                        load_v(2 * u, t + 2);
                        load_v(2 * u + 1, t + 2);
                    }
                    if constexpr (u == kPairsV - 1)
#pragma unroll
                        for (int p = 0; p < kParts; ++p) write_v(j, p, other);
                }
            } else {
                constexpr int x = e - 6 * kPairsV;
                convert_k(CH - 1, x / 3, x % 3);
                if constexpr (x % 6 == 5) load_k(CH - 1, x / 6, t + 3);
                if constexpr (x == 11)
#pragma unroll
                    for (int p = 0; p < kParts; ++p) write_k(CH - 1, p, cur);
            }
        };
        each<kSlots2>([&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value, s = n / (6 * NB), p = n / NB % 6, b = n % NB;
            if constexpr (n == kGate) publish();
            if constexpr (WEIGH) {
                __builtin_amdgcn_sched_barrier(0);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[s][b][kPartA[p]], pp[s][kPartB[p]], acc[b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (s == 0 && n % 2 == 0) {
                    constexpr int r = n / 2;  // 3 NB reads over 6 NB slots
                    read_v(1, r % NB, r / NB == 0 ? 2 : r / NB == 1 ? 0 : 1, cur);
                }
            }
            if constexpr (SCORE && n >= kGate && n < kGate + kParts) read_k(0, n - kGate, cur);
            constexpr int lo = kFirstEvent<n, kEvents2, kGate - 1>, hi = kFirstEvent<n + 1, kEvents2, kGate - 1>;
            each<hi - lo>([&](auto ec) __attribute__((always_inline)) {
                event2(std::integral_constant<int, lo + decltype(ec)::value>{});
            });
            if constexpr (WEIGH) __builtin_amdgcn_sched_barrier(0);
        });
        if (SCORE) {
            st = sn[0] + sn[1];
            mask(t + 1, st);
        }
    };
    // Two waves per SIMD: a wave's scores, softmax and P V follow each other and
    // the other wave's matrix work covers its softmax (against the schedule
    // above at H64 S2048 noncausal: D128 641 us for 768, D64 357 for 359). K of tile
    // t + 1 is converted beside the scores, V beside P V; the block's last tile
    // stages nothing (without STAGE H2 S64 D32 takes 5.1 us for 4.8, H256 S64
    // D32 6.0 for 5.6, H256 S300 D72 55.8 for 52.1; the schedule above spills
    // with such a form).
    auto plain_tile = [&](int t, auto wc, auto gc) __attribute__((always_inline)) {
        constexpr bool WORK = decltype(wc)::value, STAGE = decltype(gc)::value;
        const uint32_t cur = uint32_t(t) & 1u, other = cur ^ 1u;
        f32x16 sn[2] = {};
        if constexpr (WORK) {
            read_q(0);
            read_k(0, 2, cur);
            read_k(0, 0, cur);
            read_k(0, 1, cur);
        }
        constexpr int kSlots1 = 6 * KS;
        each<kSlots1>([&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value, s = n / 6, p = n % 6;
            if constexpr (WORK) {
                __builtin_amdgcn_sched_barrier(0);
                sn[s & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s & 1][kPartA[p]], q_part(s, kPartB[p]), sn[s & 1], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (s + 1 < KS && (p & 1) == 0) read_k(s + 1, p == 0 ? 2 : p == 2 ? 0 : 1, cur);
                if constexpr (s + 1 < KS && p == 1) read_q(s + 1);
            }
            constexpr int lo = kFirstEvent<n, 12, kSlots1>, hi = kFirstEvent<n + 1, 12, kSlots1>;
            each<STAGE ? hi - lo : 0>([&](auto ec) __attribute__((always_inline)) {
                constexpr int x = lo + decltype(ec)::value;
                convert_k(0, x / 3, x % 3);
                if constexpr (x % 6 == 5) load_k(0, x / 6, t + 2);
                if constexpr (x == 11)
#pragma unroll
                    for (int w = 0; w < kParts; ++w) write_k(0, w, other);
            });
            if constexpr (WORK) __builtin_amdgcn_sched_barrier(0);
        });
        bf16x8 pp[2][kParts];
        bf16x8 va[2][kParts];
        auto read_pair = [&](int step, int p) {  // step: (key half, pair of blocks)
            constexpr int kPairs = (NB + 1) / 2;
            const int s = step / kPairs, b = 2 * (step % kPairs);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (b + j < NB)
                    va[j][p] = *reinterpret_cast<const bf16x8 *>(lds + (vread[s] + cur * S::kTileV) + uint32_t(b + j) * 2048u +
                                                                 uint32_t(p) * S::kPartV);
        };
        if constexpr (WORK) {
            read_pair(0, 2);
            read_pair(0, 0);
            read_pair(0, 1);
            st = sn[0] + sn[1];
            mask(t, st);
            float top = st[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) top = fmaxf(top, st[v]);
            top = halves_max(top);
            float next_max = top > row_max + kLazyMax ? top : row_max;
            if (next_max == -INFINITY) next_max = 0.f;
            const float old_weight = __builtin_amdgcn_exp2f(row_max - next_max);
            float lane_sum = 0.f;
            uint32_t pw[kParts][8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                st[2 * u] = __builtin_amdgcn_exp2f(st[2 * u] - next_max);
                st[2 * u + 1] = __builtin_amdgcn_exp2f(st[2 * u + 1] - next_max);
                lane_sum += st[2 * u];
                lane_sum += st[2 * u + 1];
                f32x2 r = {st[2 * u], st[2 * u + 1]};
#pragma unroll
                for (int w = 0; w < kParts; ++w) {
                    pw[w][u] = pack(r.x, r.y);
                    r = rest_of(r, pw[w][u]);
                }
            }
            row_sum = row_sum * old_weight + lane_sum;
            row_max = next_max;
            if (__any(old_weight != 1.0f)) {
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[b] *= old_weight;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int p = 0; p < kParts; ++p)
                    pp[s][p] = __builtin_bit_cast(
                        bf16x8, u32x4{pw[p][4 * s], pw[p][4 * s + 1], pw[p][4 * s + 2], pw[p][4 * s + 3]});
        }
        // P V by pairs of output blocks: 12 MFMAs a pair (six for a lone block).
        constexpr int kPairs = (NB + 1) / 2, kSlots2 = 24 * kPairs;
        each<kSlots2>([&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value, step = n / 12, p = n % 12 / 2, j = n & 1;
            constexpr int s = step / kPairs, b = 2 * (step % kPairs) + j;
            if constexpr (WORK) {
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (b < NB)
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[j][kPartA[p]], pp[s][kPartB[p]], acc[b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (step + 1 < 2 * kPairs) {
                    if constexpr (p == 0 && j == 1) read_pair(step + 1, 2);
                    if constexpr (p == 3 && j == 1) read_pair(step + 1, 1);
                    if constexpr (p == 5 && j == 1) read_pair(step + 1, 0);
                }
            }
            constexpr int lo = kFirstEvent<n, 6 * kPairsV, kSlots2 - 4>, hi = kFirstEvent<n + 1, 6 * kPairsV, kSlots2 - 4>;
            each<STAGE ? hi - lo : 0>([&](auto ec) __attribute__((always_inline)) {
                constexpr int e = lo + decltype(ec)::value, v = e / (3 * kPairsV), u = e / 3 % kPairsV, x = e % 3;
                convert_v(v, u, x);
                if constexpr (x == 2) {
                    if constexpr (v == 1) {
                        load_v(2 * u, t + 2);
                        load_v(2 * u + 1, t + 2);
                    }
                    if constexpr (u == kPairsV - 1)
#pragma unroll
                        for (int w = 0; w < kParts; ++w) write_v(v, w, other);
                }
            });
            if constexpr (WORK) __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (STAGE) publish();
    };
    if constexpr (S::kPlain) {
        for (int t = 0; t < t_end - 1; ++t) {
            if (live(t))
                plain_tile(t, std::true_type{}, std::true_type{});
            else
                plain_tile(t, std::false_type{}, std::true_type{});
        }
        if (live(t_end - 1)) plain_tile(t_end - 1, std::true_type{}, std::false_type{});
    } else {
        for (int t = 0; t < t_end; ++t) {
            if (live(t + 1))
                tile(t, std::true_type{}, std::true_type{});
            else if (live(t))
                tile(t, std::false_type{}, std::true_type{});
            else
                tile(t, std::false_type{}, std::false_type{});
        }
    }

    // What the parts do not carry: see the file's head.
    float total = row_sum * 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) total += acc[b][v] * 0.f;
    float unscale = kUnscaleV;
    if (rows && __any(most_q > kMostQ || total != 0.f)) {
        unscale = 1.f;
        row_max = -INFINITY;
        row_sum = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = f32x16{};
        const bool mine = qi < seq;
        const float *qrow = Q + base + size_t(mine ? qi : 0) * dim;
        for (int t = 0; t < t_end && live(t); ++t) {
            const int key = t * kKeys + c;
            const float *krow = K + base + size_t(min(key, seq - 1)) * dim;
            st = f32x16{};
            for (int d0 = 0; d0 < DP; d0 += 8) {
                const int d = d0 + 4 * h;
                f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
                if (d < dim) {
                    if (key < seq) a = *reinterpret_cast<const f32x4 *>(krow + d);
                    if (mine) b = *reinterpret_cast<const f32x4 *>(qrow + d);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    st = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e] * qscale, st, 0, 0, 0);
            }
            mask(t, st);
            float top = row_max;
#pragma unroll
            for (int v = 0; v < 16; ++v) top = fmaxf(top, st[v]);
            top = halves_max(top);
            if (top == -INFINITY) top = 0.f;
            const float old_weight = __builtin_amdgcn_exp2f(row_max - top);
            float lane_sum = 0.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                st[v] = __builtin_amdgcn_exp2f(st[v] - top);
                lane_sum += st[v];
            }
            row_sum = row_sum * old_weight + lane_sum;
            row_max = top;
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[b] *= old_weight;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int k = t * kKeys + 8 * (v >> 2) + 4 * h + (v & 3);
                const float *vr = V + base + size_t(min(k, seq - 1)) * dim;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const int r = 32 * b + c, d = r < DP / 2 ? 2 * r : 2 * r - DP + 1;
                    const float x = k < seq && d < dim ? vr[d] : 0.f;
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, st[v], acc[b], 0, 0, 0);
                }
            }
        }
    }

    row_sum = halves_sum(row_sum);
    if (qi < seq) {
        const float inv = unscale / row_sum;
        float *orow = O + base + size_t(qi) * dim;
        // LDS row r of V is dim 2r (r < DP / 2) or 2 (r - DP / 2) + 1, and a
        // lane holds rows 32b + 8 (v >> 2) + 4h + (v & 3): r, r + 1 and their
        // odd partners are four adjacent dims.
#pragma unroll
        for (int x = 0; x < NB * 16; x += 2) {
            const int b = x / 16, v = x % 16, r = 32 * b + 8 * (v >> 2) + (v & 3);
            if (r >= DP / 2) continue;
            const int r2 = r + DP / 2, b2 = r2 / 32, v2 = 4 * (r2 % 32 / 8) + r2 % 4;
            const int d = 2 * (r + 4 * h);
            if (d < dim) {
                const f32x4 out = {acc[b][v] * inv, acc[b2][v2] * inv, acc[b][v + 1] * inv, acc[b2][v2 + 1] * inv};
                *reinterpret_cast<f32x4 *>(orow + d) = out;
            }
        }
    }
}

template <int DP, int NW>
hipError_t launch(hipStream_t stream, const FlashArgs &a) {
    const uint32_t bq = 32 * NW;
    const dim3 grid(a.heads, (a.seq + bq - 1) / bq), block(64 * NW);
    if (a.causal)
        hipLaunchKernelGGL((attention_flash<DP, NW, true>), grid, block, 0, stream, a.q, a.k, a.v, a.out, int(a.seq),
                           int(a.dim), a.qscale);
    else
        hipLaunchKernelGGL((attention_flash<DP, NW, false>), grid, block, 0, stream, a.q, a.k, a.v, a.out, int(a.seq),
                           int(a.dim), a.qscale);
    return hipGetLastError();
}

template <int DP>
hipError_t launch_dim(hipStream_t stream, const FlashArgs &a) {
    if constexpr (DP > 64)
        if (a.waves == 8) return launch<DP, 8>(stream, a);
    return launch<DP, 4>(stream, a);
}

}  // namespace

uint32_t attention_flash_lds_bytes(uint32_t dim, int waves) {
    using namespace flash;
    if (dim <= 64) return Shape<64, 4>::kLdsBytes;
    if (waves != 8) return Shape<128, 4>::kLdsBytes;
    return dim <= 96 ? Shape<96, 8>::kLdsBytes : Shape<128, 8>::kLdsBytes;
}

hipError_t launch_attention_flash(hipStream_t stream, const FlashArgs &a) {
    if (a.dim % 4 != 0 || a.dim > 128) return hipErrorInvalidValue;
    if (a.dim <= 32) return launch_dim<32>(stream, a);
    if (a.dim <= 64) return launch_dim<64>(stream, a);
    if (a.dim <= 96) return launch_dim<96>(stream, a);
    return launch_dim<128>(stream, a);
}

}  // namespace hipk
}  // namespace jade
