// FP32 GEMM for at most 16 rows and short K: C[M,N] = A[M,K] * B[K,N], packed
// row-major, any alignment (the contract of gemm_f32.hip,
// src/runtime/ir.rs:21-32).
//
// A product this small is latency: a load, a chain of products, a reduction.
// One workgroup of G waves computes 32 columns; wave g takes the 32-deep K
// slices g and g + G, whose loads all go out at once, on
// v_mfma_f32_16x16x4_f32 (16 rows pad half as many products as the 64x64 and
// 32x32 tiles' MFMAs), and the waves meet in LDS in wave order. Lane 16g + i
// loads k 8g .. 8g + 7 of A row i (two 16-byte loads a slice) and of B columns
// 2i, 2i + 1 (eight 8-byte loads, each four rows of 128 bytes).
//
// Measured (us, replayed) against the 64x64 tiles with two K groups, split
// over K with a second, reducing launch from K = 256: 8x256x128 5.1 -> 2.8,
// 8x128x256 6.9 -> 2.9, 16x512x512 8.1 -> 3.6, 4x1000x333 8.8 -> 3.2. A loop
// over more slices (a wave's loads waiting on one another) took the gain back:
// 16x64x1024 8.4 -> 8.5 with eight waves of four slices.
#include "gemm_rows16.hpp"

namespace jade {
namespace hipk {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kRawBuffer = 0x00020000;  // buffer descriptor word 3: raw buffer, 32-bit data format
constexpr int kSliceK = 32, kCols = 32, kRows = 16, kSlices = 2;

// sum != nullptr: also sum = C + residual (both [M, N]), the stream kernel's
// FP32 add.
template <int G>
__device__ inline void rows16(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int M,
                              int N, int K, const float *__restrict__ residual, float *__restrict__ sum) {
    __shared__ float sums[G][kRows][kCols];
    const int lane = int(threadIdx.x) & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int g = lane >> 4, i = lane & 15, n0 = int(blockIdx.x) * kCols;
    // Rows of A past M and rows of B past K lie past the buffers and read
    // zero; a run of A past K reads the next row and is zeroed below.
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(A), 0, int(uint32_t(M) * uint32_t(K) * 4u), int(kRawBuffer));
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(B), 0, int(uint32_t(K) * uint32_t(N) * 4u), int(kRawBuffer));
    f32x4 a[kSlices][2];
    f32x2 b[kSlices][8];
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
        const uint32_t k = uint32_t((wave + s * G) * kSliceK + 8 * g);
#pragma unroll
        for (int q = 0; q < 2; ++q)
            a[s][q] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, int((uint32_t(i) * uint32_t(K) + k + 4u * q) * 4u), 0, 0));
#pragma unroll
        for (int e = 0; e < 8; ++e)
            b[s][e] = __builtin_bit_cast(
                f32x2, __builtin_amdgcn_raw_buffer_load_b64(rb, int(((k + e) * uint32_t(N) + uint32_t(n0 + 2 * i)) * 4u), 0, 0));
    }
    f32x4 acc[2] = {};
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
        const int k = (wave + s * G) * kSliceK + 8 * g;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x = k + e < K ? a[s][e >> 2][e & 3] : 0.f;
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, b[s][e].x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, b[s][e].y, acc[1], 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        *reinterpret_cast<f32x2 *>(&sums[wave][4 * g + r][2 * i]) = f32x2{acc[0][r], acc[1][r]};
    __syncthreads();
    for (int o = int(threadIdx.x); o < M * kCols; o += 64 * G) {
        const int row = o / kCols, col = o % kCols;
        float x = sums[0][row][col];
#pragma unroll
        for (int w = 1; w < G; ++w) x += sums[w][row][col];
        if (n0 + col < N) {
            const size_t at = size_t(row) * size_t(N) + n0 + col;
            C[at] = x;
            if (sum) sum[at] = x + residual[at];
        }
    }
}

template <int G>
__global__ __launch_bounds__(64 * G) void gemm_f32_rows16(const float *A, const float *B, float *C, int M, int N,
                                                          int K, const float *residual, float *sum) {
    rows16<G>(A, B, C, M, N, K, residual, sum);
}

// Two independent products of one shape, one in each row of the grid. A kernel
// of its own: with the choice of pointers in the one above, a launch of one
// product took 0.05-0.08 us more (1x1000x512 3.09 -> 3.17).
template <int G>
__global__ __launch_bounds__(64 * G) void gemm_f32_rows16_pair(const float *A0, const float *B0, float *C0,
                                                               const float *A1, const float *B1, float *C1, int M,
                                                               int N, int K) {
    const bool second = blockIdx.y == 1;
    rows16<G>(second ? A1 : A0, second ? B1 : B0, second ? C1 : C0, M, N, K, nullptr, nullptr);
}

bool takes(int waves, uint32_t m, uint32_t k) {
    return (waves == 4 || waves == 8) && m <= uint32_t(kRows) && k <= uint32_t(kSlices * kSliceK * waves);
}

}  // namespace

hipError_t launch_gemm_rows16(hipStream_t stream, int waves, const float *a, const float *b, float *c, uint32_t m,
                              uint32_t n, uint32_t k, const float *residual, float *sum) {
    if (!takes(waves, m, k)) return hipErrorInvalidValue;
    const dim3 grid((n + kCols - 1) / kCols), block(64 * waves);
    hipLaunchKernelGGL(waves == 4 ? gemm_f32_rows16<4> : gemm_f32_rows16<8>, grid, block, 0, stream, a, b, c, int(m),
                       int(n), int(k), residual, sum);
    return hipGetLastError();
}

hipError_t launch_gemm_rows16_pair(hipStream_t stream, int waves, const float *a0, const float *b0, float *c0,
                                   const float *a1, const float *b1, float *c1, uint32_t m, uint32_t n, uint32_t k) {
    if (!takes(waves, m, k)) return hipErrorInvalidValue;
    const dim3 grid((n + kCols - 1) / kCols, 2), block(64 * waves);
    hipLaunchKernelGGL(waves == 4 ? gemm_f32_rows16_pair<4> : gemm_f32_rows16_pair<8>, grid, block, 0, stream, a0, b0,
                       c0, a1, b1, c1, int(m), int(n), int(k));
    return hipGetLastError();
}

}  // namespace hipk
}  // namespace jade
