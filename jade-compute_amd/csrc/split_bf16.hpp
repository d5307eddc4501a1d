// FP32 products on the bf16 matrix cores: device helpers.
//
// An FP32 value is held exactly as the sum of three bf16 parts, each the
// round-to-nearest-even of what the parts before it leave (8 significant bits
// apiece: 24 in all; the residuals are exact FP32 subtractions). A product of
// two such values is the sum of nine products of parts; the six of the three
// largest orders are taken on v_mfma_f32_32x32x16_bf16, whose products are
// exact and whose sums are FP32. The three left out come to less than 2^-24 of
// the product at worst (0.995 of that, over all mantissas), as much as an FP32
// product's own rounding, and to 2^-27.5 in the root mean square, so a single
// product can be off by an ulp where FP32's is off by half of one, and a sum
// of many is closer than FP32 products with FP32 sums leave it.
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
// What the part pair `p` leaves of x, exactly, one v_dot2_f32_bf16 an element
// (p.lo * -1 + p.hi * 0 + x) in place of a shift or mask and a subtraction.
// Bit-identical to those on 13 million pairs from 2^-100 to 2^126, zeros and
// values that round up to the next binade among them. An infinite part makes
// its neighbour's rest NaN as well as its own: pairs are two k of one row,
// column or query, whose sums are not finite then anyway. The constants are
// kept in registers: the instruction takes an inline -1.0 as FP32's. Flash
// attention runs faster with it (H128 S4096 D128 causal 2673 -> 2575 us);
// the ring GEMM, whose MFMAs leave the VALU less room, slower (4096^3 728 ->
// 765) and keeps the shifts.
__device__ inline f32x2 rest_of(f32x2 x, uint32_t p) {
    uint32_t lo, hi;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(lo));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(hi));
    const bf16x2 part = __builtin_bit_cast(bf16x2, p);
    return f32x2{__builtin_amdgcn_fdot2_f32_bf16(part, __builtin_bit_cast(bf16x2, lo), x.x, false),
                 __builtin_amdgcn_fdot2_f32_bf16(part, __builtin_bit_cast(bf16x2, hi), x.y, false)};
}

// Operands are scaled by kScale before they are split: FP32's smallest
// subnormal, 2^-149, becomes 2^-133, bf16's, so every finite value splits
// exactly as long as it stays below 2^111 (v_cvt_pk_bf16_f32 and the matrix
// cores keep subnormal parts; past 2^111 a first part may round to infinity).
// Products and their sums then carry kScale^2, and one past 2^96 overflows,
// which shows in the sum. The multiplication takes the two instructions a pair
// that noticing small values would take.
constexpr float kScale = 0x1p16f, kUnscale = 0x1p-32f;
// Attention's V meets weights that are not scaled. 2^24 keeps V's parts normal
// numbers, whatever v_dot2_f32_bf16 (rest_of) makes of subnormal ones; sums past
// 2^103 may overflow. Its Q is scaled up by as much and its K down, so the
// scores are as they are without.
constexpr float kScaleV = 0x1p24f, kUnscaleV = 0x1p-24f, kScaleQ = 0x1p24f, kScaleK = 0x1p-24f;

}  // namespace split
}  // namespace
}  // namespace hipk
}  // namespace jade
