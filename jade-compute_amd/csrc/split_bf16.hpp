// FP32 products on the bf16 matrix cores: device helpers.
//
// An FP32 value is held exactly as the sum of three bf16 parts, each the
// round-to-nearest-even of what the parts before it leave (8 significant bits
// apiece: 24 in all; the residuals are exact FP32 subtractions). A product of
// two such values is the sum of nine products of parts; the six of the three
// largest orders are taken on v_mfma_f32_32x32x16_bf16, whose products are
// exact and whose sums are FP32, and the three left out are below 2^-26 of the
// product, a quarter of an FP32 product's own rounding.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace jade {
namespace hipk {
namespace {
namespace split {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kParts = 3;
constexpr int kProducts = 6;
// The six products as (part of A, part of B), smallest order first: in one
// accumulator the small ones are then added while the step's own large one is
// still missing.
constexpr int kPartA[kProducts] = {2, 0, 1, 1, 0, 0};
constexpr int kPartB[kProducts] = {0, 2, 1, 0, 1, 0};

__device__ inline uint32_t pack(float x, float y) {
    const bf16x2 p = __builtin_convertvector(f32x2{x, y}, bf16x2);
    return __builtin_bit_cast(uint32_t, p);
}
__device__ inline float low_part(uint32_t p) { return __uint_as_float(p << 16); }
__device__ inline float high_part(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// The smallest magnitudes seen, as (2 * bf16 bits - 1) per 16-bit half: zero
// wraps to the largest value, so it never counts. Parts of a value of at least
// 2^-100 (kSmallest) lose nothing to bf16's smallest subnormal.
constexpr uint16_t kSmallest = uint16_t(2 * ((127 - 100) << 7) - 1);
__device__ inline u16x2 doubled_less_one(uint32_t p) {
    return __builtin_bit_cast(u16x2, p) * u16x2{2, 2} + u16x2{0xffff, 0xffff};
}
__device__ inline bool lossy(u16x2 smallest) {
    return smallest.x < kSmallest || smallest.y < kSmallest;
}

}  // namespace split
}  // namespace
}  // namespace hipk
}  // namespace jade
