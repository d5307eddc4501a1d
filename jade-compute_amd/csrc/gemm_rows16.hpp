// Host interface of the GEMM for at most 16 rows and short K (gemm_rows16.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace jade {
namespace hipk {

// C[m,n] = A[m,k] B[k,n], m at most 16, k at most 64 * waves (4 or 8); with
// `sum` non-null also sum = C + residual. A and B below 2 GiB.
hipError_t launch_gemm_rows16(hipStream_t stream, int waves, const float *a, const float *b, float *c, uint32_t m,
                              uint32_t n, uint32_t k, const float *residual, float *sum);
// c0 = a0 b0 and c1 = a1 b1, of one shape, in one launch; the same bits.
hipError_t launch_gemm_rows16_pair(hipStream_t stream, int waves, const float *a0, const float *b0, float *c0,
                                   const float *a1, const float *b1, float *c1, uint32_t m, uint32_t n, uint32_t k);

}  // namespace hipk
}  // namespace jade
