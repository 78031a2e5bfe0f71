// Register decode of packed genotype codes for the GEMM kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace pcaone {
namespace {

// code -> top byte of v in BF16/FP32/FP64: 00 -> +2 (0x40), 01 -> 0, 10 -> 0, 11 -> -2 (0xC0)
constexpr uint32_t kLutTopByte = 0xC0000040u;

__device__ __forceinline__ uint32_t spread(uint32_t w, int t) { return (w >> (2 * t)) & 0x03030303u; }
__device__ __forceinline__ uint32_t top_bytes(uint32_t codes4) { return __builtin_amdgcn_perm(0u, kLutTopByte, codes4); }

// Top 32 bits of the FP32/FP64 value of byte e of `tb` (other bytes zero).
__device__ __forceinline__ uint32_t top_word(uint32_t tb, int e) {
  return __builtin_amdgcn_perm(tb, tb, ((uint32_t)(4 + e) << 24) | 0x0C0C0Cu);
}

}  // namespace
}  // namespace pcaone
