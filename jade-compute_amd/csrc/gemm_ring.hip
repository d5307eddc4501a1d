// FP32 GEMM on persistent 128x128 tiles for large products whose grid
// covers every CU: C[M,N] = A[M,K] * B[K,N], packed row-major, the same
// contract as gemm_f32.hip (src/runtime/ir.rs:21-32).
#include <type_traits>

#include "gemm_tiles.hpp"
#include "ops.hpp"
#include "split_bf16.hpp"

namespace jade {
namespace hipk {
namespace {

// ---- Persistent 128x128 tiles: one workgroup per CU, products on bf16 parts ----
// What bounds it: the bf16 matrix cores (six v_mfma_f32_32x32x16_bf16 per
// FP32 product block, split_bf16.hpp), at 1.8-2.0 GHz: a chip full of them
// runs 1.81 PFLOP/s with one wave per SIMD and 1.98 with two, so 300-330
// TFLOP/s of FP32 products. v_mfma_f32_32x32x2_f32, which this kernel ran on
// before, tops out at 157 and this kernel reached 150 with it.
// Measured (us, one box, against that kernel): 4096^3 934 -> 691 a call, 2048^3
// 121 -> 91, 4096x11008x4096 2525 -> 1865 a call. With the staging taken out of a
// copy (MFMAs and operand reads alone) 4096^3 runs 437 us; global loads, the
// conversion and the LDS writes each add 60-90 us of issue and waiting that
// the two waves of a SIMD do not hide. Neither the order of that work (spread
// one piece per MFMA as here 672, all before the MFMAs 701, after 730, left to
// the compiler 706) nor a third stage buffer with the writes a whole stage
// ahead of their barrier (735) changes it much; four waves of 64x64 (one per
// SIMD) ran 716, and 256x128 tiles spill.
//
// A launch of at most one workgroup per CU; workgroup b takes the tiles
// pos(b), pos(b) + G, pos(b) + 2G, ... of the XCD-grouped order (G workgroups,
// pos the XCD-contiguous position), so each XCD's 32 workgroups work on a
// block of 8 tile rows x 4 tile columns at a time. The workgroup's 32-k stages
// form one sequence over all its tiles: loads and conversions run ahead
// across tile boundaries.
//
// Eight waves of 32x64 (two 32x32 blocks each, two waves per SIMD). Each
// element of a stage is loaded and split once per workgroup: FP32 from global
// memory into registers two stages ahead, three bf16 parts into LDS (48 KiB a
// stage, two stages). A row (and B column) of a part is 64 bytes of LDS, k
// contiguous, its four 16-byte chunks XORed with (row >> 2) & 3, so that an
// operand read (16 rows at one chunk) covers all banks. B column 64w + 2c + j
// of the tile is LDS row 64w + 32j + c: a lane's outputs of blocks 0 and 1 are
// then adjacent columns, and the lanes that write B write adjacent rows.
//
// Accumulation is two-level: runs of kFoldRun stages (256 k) sum in the MFMA
// accumulators, small products first, and are folded into the running sums
// with VALU adds. Error against FP64 (2-norm, relative, uniform [-1, 1)):
// 4096^3 2.5e-7 (the FP32 MFMAs 3.0e-7), 2048^3 2.4e-7 (3.0e-7).
//
// The operands are scaled before they are split, so that every finite value is
// carried exactly, subnormals among them (split_bf16.hpp), and the sums are
// scaled back before they are stored. An infinity minus its own first part is
// NaN, and values past 2^111 and sums past 2^96 overflow once scaled: a wave whose
// sums are not all finite computes its outputs again from global memory with
// FP32 MFMAs and takes those in the place of the sums that are not, so
// infinities, NaN and overflow come out as FP32 arithmetic gives them, at about
// a third of the speed (4096^3 with one infinity in B, or with every sum past
// 2^96, 2200 us; four k steps of loads kept ahead of these products spilled 289
// registers and ran between 1985 and 2807). Which way an output is computed
// thus depends on its own row and column alone, not on its tile's other
// outputs: every form of this kernel gives it the same bits.
//
// Requires M, N multiples of 128 (N of 64 for DUAL), K a multiple of 256,
// 16-byte aligned operands, 32-bit load offsets inside a tile.
namespace ring_local {
using namespace ring;
using namespace split;

// One half-stage's operands (16 k) for one lane: part p of the A row block and
// of B column block j, eight consecutive k each.
struct Operands {
    bf16x8 a[kParts], b[2][kParts];
};

constexpr uint32_t kRawBuffer = 0x00020000;  // buffer descriptor word 3: raw buffer, 32-bit data format

__device__ inline int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ inline const float *uniform(const float *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v)), hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
    return reinterpret_cast<const float *>((uint64_t(hi) << 32) | lo);
}
// Position of logical 16-byte chunk j (eight k) in a 64-byte LDS row.
__device__ inline int swz(int row) { return (row >> 2) & 3; }
}  // namespace ring_local

// Plain stores single floats; Pairs stores each lane's two adjacent outputs as
// 8 bytes (C, residual and sum 8-byte aligned). Both store sum = C + residual
// as well where sum is not null (the stream kernel's FP32 add, so `sum` is
// bit-identical to an Add launched after the product). Dual computes 128x64
// tiles of two products of one A (B into C, B2 into C2), the operand columns
// of both side by side, and their SwiGLU into sum; every output takes the
// steps over k that its product takes alone.
enum class RingForm { Plain, Pairs, Dual };

template <RingForm FORM>
__global__ __launch_bounds__(ring::kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_f32_ring(
    const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ B2, float *__restrict__ C,
    float *__restrict__ C2, int N, int K, int tiles_m, int tiles_n, const float *__restrict__ residual,
    float *__restrict__ sum) {
    using namespace ring;
    using namespace ring_local;
    constexpr bool DUAL = FORM == RingForm::Dual;
    __shared__ __attribute__((aligned(1024))) char lds[kLdsBytes];
    const int tid = int(threadIdx.x), lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int h = lane >> 5, c = lane & 31, wm = wave >> 1, wn = wave & 1;
    const int nwg = int(gridDim.x), tiles = tiles_m * tiles_n;
    const int pos = xcd_order(int(blockIdx.x), nwg);
    const int mine = (tiles - pos + nwg - 1) / nwg;  // tiles pos, pos + nwg, ...
    const int nk = K / kBK;
    constexpr int kTileN = DUAL ? kBN / 2 : kBN;

    // Staging, per thread: one A chunk (row tid / 4, k 8 (tid % 4) on) and
    // four k (4 wave on) of two B columns.
    const int ar = tid >> 2, aq = tid & 3;
    const uint32_t va = uint32_t((ar * K + 8 * aq) * 4);
    const uint32_t vb = uint32_t((4 * wave * N + (DUAL ? lane : 2 * lane)) * 4), vbk = uint32_t(N) * 4u;
    const uint32_t wa = uint32_t(ar * 64 + ((aq ^ swz(ar)) << 4));
    const int br = (lane >> 5) * 64 + c;  // LDS row of the first column; the second is 32 rows on
    const uint32_t wb = uint32_t(kBRegion + br * 64 + (((wave >> 1) ^ swz(br)) << 4) + (wave & 1) * 8);
    // Operand reads: A row 32 wm + c, B row 64 wn + 32 j + c, chunk 2 half + h.
    uint32_t ra[2], rb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        ra[s] = uint32_t((32 * wm + c) * 64 + (((2 * s + h) ^ swz(c)) << 4));
        rb[s] = uint32_t(kBRegion + (64 * wn + c) * 64 + (((2 * s + h) ^ swz(c)) << 4));
    }

    auto tile_origin = [&](int j, int &m0, int &n0) {
        int tm, tn;
        grouped_tile(min(j, mine - 1) * nwg + pos, tiles_m, tiles_n, tm, tn);
        m0 = uniform(tm * kBM);
        n0 = uniform(tn * kTileN);
    };
    // Load cursors: the stage of the next A and of the next B load. Each
    // wraps to the next tile; past the last tile they run over it again, in
    // bounds, and those stages are never multiplied.
    int sa = 0, sb = 0;
    const float *pa, *pb, *pb2 = nullptr, *next_a, *next_b, *next_b2 = nullptr;
    {
        int m0, n0;
        tile_origin(0, m0, n0);
        pa = uniform(A + size_t(m0) * size_t(K));
        pb = uniform(B + n0);
        if (DUAL) pb2 = uniform(B2 + n0);
    }
    auto aim_next = [&](int tile) {
        int m0, n0;
        tile_origin(tile, m0, n0);
        next_a = uniform(A + size_t(m0) * size_t(K));
        next_b = uniform(B + n0);
        if (DUAL) next_b2 = uniform(B2 + n0);
    };
    aim_next(1);
    auto buffer = [](const float *base) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, -1, int(kRawBuffer));
    };
    f32x4 rawa[2][2];
    f32x2 rawb[2][4];
    auto load_a = [&](int set, int x) {  // the chunk's float4 x; the last one advances the cursor
        rawa[set][x] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer(pa), int(va), 16 * x, 0));
        if (x == 1) {
            const bool wrap = ++sa == nk;
            pa = wrap ? next_a : pa + kBK;
            sa = wrap ? 0 : sa;
        }
    };
    auto load_b = [&](int set, int e) {  // k row e of the thread's four
        if constexpr (DUAL) {
            rawb[set][e].x = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(buffer(pb), int(vb), int(uint32_t(e) * vbk), 0));
            rawb[set][e].y = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(buffer(pb2), int(vb), int(uint32_t(e) * vbk), 0));
        } else {
            rawb[set][e] = __builtin_bit_cast(
                f32x2, __builtin_amdgcn_raw_buffer_load_b64(buffer(pb), int(vb), int(uint32_t(e) * vbk), 0));
        }
        if (e == 3) {
            const bool wrap = ++sb == nk;
            const size_t step = size_t(kBK) * size_t(N);
            pb = wrap ? next_b : pb + step;
            if (DUAL) pb2 = wrap ? next_b2 : pb2 + step;
            sb = wrap ? 0 : sb;
        }
    };
    // Conversion of pair u of the A chunk (k 2u, 2u + 1) or of B (column
    // u / 2, k 2 (u % 2) on), in three pieces.
    uint32_t parts[2][kParts][4];
    f32x2 rest;
    auto convert = [&](int is_b, int set, int u, int piece) {
        if (piece == 0) {
            f32x2 x;
            if (is_b) {
                const f32x2 k0 = rawb[set][2 * (u & 1)], k1 = rawb[set][2 * (u & 1) + 1];
                x = u < 2 ? f32x2{k0.x, k1.x} : f32x2{k0.y, k1.y};
            } else {
                x = f32x2{rawa[set][u >> 1][2 * (u & 1)], rawa[set][u >> 1][2 * (u & 1) + 1]};
            }
            x *= kScale;
            const uint32_t p = pack(x.x, x.y);
            parts[is_b][0][u] = p;
            rest = f32x2{x.x - low_part(p), x.y - high_part(p)};
        } else if (piece == 1) {
            const uint32_t p = pack(rest.x, rest.y);
            parts[is_b][1][u] = p;
            rest = f32x2{rest.x - low_part(p), rest.y - high_part(p)};
        } else {
            parts[is_b][2][u] = pack(rest.x, rest.y);
        }
    };
    auto write_a = [&](int p, int buf) {
        *reinterpret_cast<u32x4 *>(lds + wa + uint32_t(p) * kPart + uint32_t(buf) * kStageB) =
            u32x4{parts[0][p][0], parts[0][p][1], parts[0][p][2], parts[0][p][3]};
    };
    auto write_b = [&](int col, int p, int buf) {
        *reinterpret_cast<u32x2 *>(lds + wb + uint32_t(col) * 2048u + uint32_t(p) * kPart + uint32_t(buf) * kStageB) =
            u32x2{parts[1][p][2 * col], parts[1][p][2 * col + 1]};
    };
    // Read r of a half-stage's nine, in the order the products take them.
    auto read_operand = [&](int r, int half, int buf, Operands &o) {
        constexpr int kPartOf[9] = {2, 0, 0, 0, 2, 2, 1, 1, 1}, kBlock[9] = {-1, 0, 1, -1, 0, 1, -1, 0, 1};
        const int p = kPartOf[r], j = kBlock[r];
        const uint32_t from = (j < 0 ? ra[half] : rb[half] + uint32_t(j) * 2048u) + uint32_t(p) * kPart +
                              uint32_t(buf) * kStageB;
        (j < 0 ? o.a[p] : o.b[j][p]) = *reinterpret_cast<const bf16x8 *>(lds + from);
    };
    auto publish = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // Prologue: stage 0 whole and the A chunk of stage 1 converted; A of
    // stages 2 and 3 and B of stages 1 and 2 in flight.
    auto fetch_a = [&](int set) {
#pragma unroll
        for (int x = 0; x < 2; ++x) load_a(set, x);
    };
    auto fetch_b = [&](int set) {
#pragma unroll
        for (int e = 0; e < 4; ++e) load_b(set, e);
    };
    auto convert_a = [&](int set, int buf) {
#pragma unroll
        for (int x = 0; x < 12; ++x) convert(0, set, x / 3, x % 3);
#pragma unroll
        for (int p = 0; p < kParts; ++p) write_a(p, buf);
    };
    auto convert_b = [&](int set, int buf) {
#pragma unroll
        for (int x = 0; x < 12; ++x) convert(1, set, x / 3, x % 3);
#pragma unroll
        for (int p = 0; p < kParts; ++p) {
            write_b(0, p, buf);
            write_b(1, p, buf);
        }
    };
    fetch_a(0);
    fetch_b(0);
    fetch_a(1);
    fetch_b(1);
    convert_a(0, 0);
    fetch_a(0);
    convert_b(0, 0);
    fetch_b(0);
    convert_a(1, 1);
    fetch_a(1);
    publish();
    Operands cur;
#pragma unroll
    for (int r = 0; r < 9; ++r) read_operand(r, 0, 0, cur);

    f32x16 acc[2] = {}, part[2] = {};

    // One half-stage: twelve MFMAs. HALF 0 multiplies k 0-15 of stage g (buffer
    // P), reads k 16-31 and converts B of stage g + 1 into buffer P ^ 1; HALF
    // 1 multiplies k 16-31, reads k 0-15 of stage g + 1 and converts A of stage
    // g + 2 into buffer P, which no wave reads any more.
    auto half_stage = [&](auto hc, auto pc, auto sc) __attribute__((always_inline)) {
        constexpr int HALF = decltype(hc)::value, P = decltype(pc)::value;
        constexpr bool START = decltype(sc)::value;
        constexpr int set = HALF == 0 ? P ^ 1 : P, out = set;
        Operands nxt;
        if constexpr (HALF == 1) publish();
#pragma unroll
        for (int n = 0; n < 12; ++n) {
            const int p = n >> 1, j = n & 1;
            __builtin_amdgcn_sched_barrier(0);
            if (START && p == 0) {
                acc[j] += part[j];
                part[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur.a[kPartA[p]], cur.b[j][kPartB[p]], f32x16{}, 0, 0, 0);
            } else {
                part[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur.a[kPartA[p]], cur.b[j][kPartB[p]], part[j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (n < 9) read_operand(n, HALF ^ 1, HALF == 0 ? P : P ^ 1, nxt);
#pragma unroll
            for (int x = 0; x < 12; ++x) {
                if (x * 10 / 12 != n) continue;
                const int u = x / 3, piece = x % 3;
                convert(HALF == 0, set, u, piece);
                if (piece == 2) {
                    if (HALF == 0) {
                        if (u == 2) {
                            load_b(set, 0);
                            load_b(set, 1);
                        }
                        if (u == 3) {
                            load_b(set, 2);
                            load_b(set, 3);
                        }
                        if (u & 1)
#pragma unroll
                            for (int w = 0; w < kParts; ++w) write_b(u >> 1, w, out);
                    } else {
                        if (u & 1) load_a(set, u >> 1);
                        if (u == 3)
#pragma unroll
                            for (int w = 0; w < kParts; ++w) write_a(w, out);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        cur = nxt;
    };
    auto stage = [&](auto pc, auto sc) __attribute__((always_inline)) {
        half_stage(std::integral_constant<int, 0>{}, pc, sc);
        half_stage(std::integral_constant<int, 1>{}, pc, std::false_type{});
    };
    const std::integral_constant<int, 0> even{};
    const std::integral_constant<int, 1> odd{};

    // Output row 8 (v >> 2) + (v & 3) of the lane's rows, columns 2c, 2c + 1
    // of the wave's (DUAL: column c of each product).
    const uint32_t out_lane = uint32_t((wm * 32 + 4 * h) * N + (DUAL ? wn * 32 + c : wn * 64 + 2 * c));
    auto store = [&](int m0, int n0) {
        m0 = uniform(m0);
        n0 = uniform(n0);
        // No address is computed ahead of the K loop, which would hold the
        // sixteen rows' offsets in registers across it.
        uint32_t from = out_lane, row = uint32_t(N);
        asm volatile("" : "+s"(m0), "+s"(n0), "+s"(row), "+v"(from));
        const size_t tile = size_t(m0) * row + n0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const size_t o = tile + size_t(8 * (v >> 2) + (v & 3)) * row + from;
            const float x0 = acc[0][v], x1 = acc[1][v];
            if constexpr (DUAL) {
                C[o] = x0;
                C2[o] = x1;
                sum[o] = swiglu(x0, x1);
            } else if constexpr (FORM == RingForm::Pairs) {
                *reinterpret_cast<float2 *>(C + o) = make_float2(x0, x1);
                if (sum) {  // block-uniform
                    const float2 r = *reinterpret_cast<const float2 *>(residual + o);
                    *reinterpret_cast<float2 *>(sum + o) = make_float2(x0 + r.x, x1 + r.y);
                }
            } else {
                C[o] = x0;
                C[o + 1] = x1;
                if (sum) {
                    sum[o] = x0 + residual[o];
                    sum[o + 1] = x1 + residual[o + 1];
                }
            }
        }
    };

    // The wave's outputs of the tile at (m0, n0) that are not finite, again in
    // FP32 from global memory: lane (h, c) takes k 4h on of every eight, for A
    // row c and B columns 2c, 2c + 1 (DUAL: column c of each product).
    auto again = [&](int m0, int n0) __attribute__((always_inline)) {
        const float *a = A + size_t(m0 + 32 * wm + c) * size_t(K) + 4 * h;
        const size_t col = size_t(4 * h) * size_t(N) + n0 + (DUAL ? 32 * wn + c : 64 * wn + 2 * c);
        const float *b0 = B + col, *b1 = DUAL ? B2 + col : B + col + 1;
        f32x16 run[2] = {}, whole[2] = {};
        for (int k = 0; k < K; k += 8) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(a + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const size_t row = size_t(k + e) * size_t(N);
                run[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], b0[row], run[0], 0, 0, 0);
                run[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], b1[row], run[1], 0, 0, 0);
            }
            if ((k & 127) == 120) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    whole[j] += run[j];
                    run[j] = f32x16{};
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (acc[j][v] * 0.f != 0.f) acc[j][v] = whole[j][v];
    };

    for (int t = 0; t < mine; ++t) {
        if (t > 0) aim_next(t + 1);
        for (int it = 0; it < nk / kUnroll; ++it) {
            stage(even, std::true_type{});
            stage(odd, std::false_type{});
            for (int r = 1; r < kUnroll / 2; ++r) {
                stage(even, std::false_type{});
                stage(odd, std::false_type{});
            }
        }
        int m0, n0;
        tile_origin(t, m0, n0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[j] += part[j];
            part[j] = f32x16{};
        }
        float total = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) total += acc[0][v] * 0.f + acc[1][v] * 0.f;  // 0, or NaN
        acc[0] *= kUnscale;
        acc[1] *= kUnscale;
        if (__any(total != 0.f)) again(m0, n0);
        store(m0, n0);
        acc[0] = acc[1] = f32x16{};
    }
}

}  // namespace

hipError_t launch_gemm_ring(hipStream_t stream, const float *a, const float *b, float *c, uint32_t n, uint32_t k,
                            int tiles_m, int tiles_n, unsigned grid, const float *residual, float *sum) {
    const dim3 block(ring::kThreads);
    const bool pairs = ((reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(residual) |
                         reinterpret_cast<uintptr_t>(sum)) & 7u) == 0;
    if (pairs)
        hipLaunchKernelGGL((gemm_f32_ring<RingForm::Pairs>), dim3(grid), block, 0, stream, a, b, nullptr, c, nullptr,
                           int(n), int(k), tiles_m, tiles_n, residual, sum);
    else
        hipLaunchKernelGGL((gemm_f32_ring<RingForm::Plain>), dim3(grid), block, 0, stream, a, b, nullptr, c, nullptr,
                           int(n), int(k), tiles_m, tiles_n, residual, sum);
    return hipGetLastError();
}

hipError_t launch_gemm_ring_swiglu(hipStream_t stream, const float *a, const float *bg, const float *bu, float *g,
                                   float *u, float *act, uint32_t n, uint32_t k, int tiles_m, int tiles_n,
                                   unsigned grid) {
    hipLaunchKernelGGL((gemm_f32_ring<RingForm::Dual>), dim3(grid), dim3(ring::kThreads), 0, stream, a, bg, bu, g, u,
                       int(n), int(k), tiles_m, tiles_n, nullptr, act);
    return hipGetLastError();
}

}  // namespace hipk
}  // namespace jade
