// Host interface of the flash attention kernel on bf16 parts
// (attention_flash.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace jade {
namespace hipk {

struct FlashArgs {
    const float *q, *k, *v;
    float *out;
    uint32_t heads, seq, dim;
    bool causal;
    float qscale;  // scale * log2(e)
    int waves;     // waves of 32 queries per block: 4, or 8 (dim over 64)
};

// Needs dim % 4 == 0 and at most 128, 16-byte aligned tensors and heads below
// 2 GiB.
hipError_t launch_attention_flash(hipStream_t stream, const FlashArgs &args);
uint32_t attention_flash_lds_bytes(uint32_t dim, int waves);

}  // namespace hipk
}  // namespace jade
