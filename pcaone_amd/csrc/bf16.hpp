// BF16 / FP16 / FP8 rounding helpers shared by the operand-split kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace pcaone {

// Round-to-nearest-even FP32 -> BF16 bits (inputs are finite).
__device__ __forceinline__ uint16_t bf16_bits(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_value(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Round-to-nearest-even FP64 -> FP16 bits, and back.
__device__ __forceinline__ uint16_t fp16_bits(double x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }
__device__ __forceinline__ double fp16_value(uint16_t b) { return (double)__builtin_bit_cast(_Float16, b); }

// Round-to-nearest-even FP64 -> FP8 E4M3 (the OCP format: exponent bias 7,
// largest finite 448 = 0x7E, subnormal step 2^-9), larger values to 448; *val
// receives the value of the returned bits.  Each binade [2^E, 2^(E+1)) holds
// 8 steps of 2^(E-3); below 2^-6 the step stays 2^-9.  Adding and taking off
// 1.5 2^52 steps rounds to whole steps, ties to even; the exponent and the
// three leading fraction bits of the result are the E4M3 bits.
__host__ __device__ __forceinline__ uint8_t e4m3_bits(double y, double* val) {
  const double a = fmin(fmax(fabs(y), 0.0), 448.0);
  const uint32_t ex = (uint32_t)(__builtin_bit_cast(uint64_t, a) >> 52);
  const uint32_t em = ex < 1017u ? 1017u : ex;  // E = em - 1023 >= -6
  const double c = __builtin_bit_cast(double, (uint64_t)(em + 49) << 52 | 1ull << 51);
  const double r = (a + c) - c;
  const bool sub = r < 0x1p-6;  // as if one binade up, whose code is 8 larger
  const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, sub ? r + 0x1p-6 : r) >> 32);
  const uint32_t bits = (hi >> 17) - (sub ? (1016u << 3) + 8u : 1016u << 3);
  *val = y < 0.0 ? -r : r;
  return (uint8_t)(bits | (y < 0.0 && bits ? 0x80u : 0u));
}

}  // namespace pcaone
