// 64-bit keys whose maximum is the first largest fp16 value (torch.argmax: NaN counts as the largest, -0 == +0).
#pragma once
#include "common.h"

namespace omni {

__device__ __forceinline__ unsigned long long argmax_key(uint32_t h16, uint32_t idx) {
  uint32_t h = h16 & 0xFFFFu;
  if (h == 0x8000u) h = 0;                                   // -0 == +0
  if ((h & 0x7FFFu) > 0x7C00u) h = 0x7FFFu;                  // every NaN, whatever its sign
  const uint32_t k = (h & 0x8000u) ? (~h & 0xFFFFu) : (h | 0x8000u);
  return ((unsigned long long)k << 32) | (unsigned long long)(0xFFFFFFFFu - idx);
}

__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)v, m, 64), hi = __shfl_xor((uint32_t)(v >> 32), m, 64);
    const unsigned long long o = ((unsigned long long)hi << 32) | lo;
    v = o > v ? o : v;
  }
  return v;
}

}  // namespace omni
