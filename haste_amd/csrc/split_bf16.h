// Floats as sums of three bfloat16: 8 + 8 + 8 bits of significand hold a float's 24 exactly, the products
// of such parts are exact in fp32, and of the nine the six that can reach a float's 24 bits run on the bf16
// matrix cores, sixteen times as fast as the fp32 ones (Henry, Tang and Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations", 2019).
#pragma once

#include <hip/hip_runtime.h>

namespace haste_hip {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned int pack_bf16(float a, float b) {
  const float2_t v = {a, b};
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, bf16x2_t));
}

__device__ __forceinline__ float bf16_low(unsigned int u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_high(unsigned int u) { return __uint_as_float(u & 0xffff0000u); }

// What operands are multiplied with before they are split, and the product's scale that comes of it.  A
// bfloat16 holds nothing below 2^-133, a float goes down to 2^-149: unscaled, operands below 2^-110 would
// lose their last part and those below 2^-134 all three.  Scaled, every part of every float is a normal
// bfloat16; in exchange operands from 2^104 and results from 2^80 on are infinite, which the users of the
// parts look out for.
constexpr float kSplitScale = 0x1p24f, kProductScale = 0x1p-48f;

// The parts, largest first, of two scaled floats side by side.
__device__ __forceinline__ void split_pair(float a, float b, unsigned int& hi, unsigned int& mid, unsigned int& lo) {
  hi = pack_bf16(a, b);
  a -= bf16_low(hi);
  b -= bf16_high(hi);
  mid = pack_bf16(a, b);
  a -= bf16_low(mid);
  b -= bf16_high(mid);
  lo = pack_bf16(a, b);
}

}  // namespace haste_hip
