// Rows of 1024 .. 8192 channels held as the reference's virtual threads hold them, thread p of 512 with channels 2 p and 2 p + 1 of every 1024: the order of additions
// that norm_rows.hip and norm_product.hip share (act_product.hip the sums).
#pragma once
#include "common.h"

namespace omni {

typedef int v2i __attribute__((ext_vector_type(2)));

// One row's array behind a scalar descriptor: an access is one instruction with the lane's bytes and a scalar offset, and no address arithmetic
// in vector registers (global loads of this many arrays got two additions each).
struct RowArray {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ explicit RowArray(const void* base) : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xFFFFFFFFu, 0x00020000)) {}
  __device__ __forceinline__ v2h pair(uint32_t lane, uint32_t scalar) const {
    return __builtin_bit_cast(v2h, __builtin_amdgcn_raw_buffer_load_b32(r, lane, scalar, 0));
  }
  __device__ __forceinline__ v2i two(uint32_t lane, uint32_t scalar) const {
    return __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r, lane, scalar, 0));
  }
  __device__ __forceinline__ void put(uint32_t lane, uint32_t scalar, v2h v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, lane, scalar, 0);
  }
  __device__ __forceinline__ void put16(uint32_t lane, uint32_t scalar, uint16_t v) const { __builtin_amdgcn_raw_buffer_store_b16(v, r, lane, scalar, 0); }
};

// The sum over lanes l ^ 8, ^ 4, ^ 2, ^ 1 of a row of 16, in this order (behind the first addition the values repeat every 8 lanes, so that a
// rotation by 4 finds the partner), in every lane
__device__ __forceinline__ float row16_sum(float v) {
  v = v + dpp_mov<0x128>(v);      // row_ror:8
  v = v + dpp_mov<0x124>(v);      // row_ror:4
  v = v + lane_xor2(v);
  return v + lane_xor1(v);
}

// LDS is published, stores to memory are not waited for (__syncthreads waits for the residual's here)
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The statistics and codes of a row in the reference's order of additions (layernorm_kernels.cu:58-331: 1024 virtual threads, thread t adds up channels t, t + 1024, ..; a
// butterfly over a virtual warp, one over the 32 sums of those), 512 threads, one row or several in turn between the barriers: pair_sums | lds_barrier | pair_normalise |
// lds_barrier | pair_top, pair_total, pair_codes.
constexpr int PAIR_RED = 104;      // words of LDS a row: [16][sum, sum, square, square], [16][2] sums of the normalised values, 8 maxima

struct PairPlace {
  int lane, wave, vw;      // vw: the virtual warp; its sums lie beside those of vw ^ 16
  __device__ __forceinline__ explicit PairPlace(int tid) : lane(tid & 63), wave(__builtin_amdgcn_readfirstlane(tid >> 6)), vw(4 * wave + (lane >> 4)) {}
};

// sum and sum of squares: the virtual thread's, the virtual warp's
template <int C>
__device__ __forceinline__ void pair_sums(const float (&x)[C][2], float* red, const PairPlace& p) {
  float s[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      s[0][e] = s[0][e] + x[c][e];
      s[1][e] = s[1][e] + x[c][e] * x[c][e];
    }
  const float w0 = row16_sum(s[0][0]) + row16_sum(s[0][1]), w1 = row16_sum(s[1][0]) + row16_sum(s[1][1]);
  if ((p.lane & 15) == 0) {
    red[(p.vw & 15) * 4 + (p.vw >> 4)] = w0;
    red[(p.vw & 15) * 4 + 2 + (p.vw >> 4)] = w1;
  }
}

// x becomes the normalised row; its maxima, and with SUM the sums of its fp16 values (the reference adds these up in fp16)
template <int C, bool SUM>
__device__ __forceinline__ void pair_normalise(float (&x)[C][2], const v2h (&g)[C], float eps, float* red, const PairPlace& p) {
  constexpr int H = 1024 * C;
  const v4f q4 = *reinterpret_cast<const v4f*>(red + (p.lane & 15) * 4);
  const float mean = row16_sum(q4[0] + q4[1]) / (float)H;
  const float rstd = 1.0f / __builtin_sqrtf(row16_sum(q4[2] + q4[3]) / (float)H + eps);
  float amax = (float)(half_t)1e-6f, hs[2] = {0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      float y = (x[c][e] - mean) * rstd;
      y = rounded_f32(y * (float)g[c][e]);
      x[c][e] = y;
      const float yh = (float)(half_t)y;
      amax = __builtin_fmaxf(amax, __builtin_fabsf(yh));
      if constexpr (SUM) hs[e] = (float)(half_t)(hs[e] + yh);
    }
  amax = wave_max64(amax);
  if (p.lane == 0) red[96 + p.wave] = amax;
  if constexpr (SUM) {
    const float w = row16_sum(hs[0]) + row16_sum(hs[1]);
    if ((p.lane & 15) == 0) red[64 + (p.vw & 15) * 2 + (p.vw >> 4)] = w;
  }
}
__device__ __forceinline__ float pair_top(const float* red, const PairPlace& p) {
  float amax = red[96 + (p.lane & 7)];
  amax = __builtin_fmaxf(amax, lane_xor1(amax));
  amax = __builtin_fmaxf(amax, lane_xor2(amax));
  return __builtin_fmaxf(amax, dpp_mov<0x141>(amax));      // the other half of 8 lanes, mirrored
}
__device__ __forceinline__ half_t pair_total(const float* red, const PairPlace& p) {
  return (half_t)row16_sum(red[64 + (p.lane & 15) * 2] + red[64 + (p.lane & 15) * 2 + 1]);
}
// the two codes of a pair; q: 127 / pair_top
__device__ __forceinline__ uint16_t pair_codes(const float (&x)[2], float q) {
  return (uint16_t)((uint32_t)(uint8_t)rni_sat_s8(x[0] * q) | ((uint32_t)(uint8_t)rni_sat_s8(x[1] * q) << 8));
}

}  // namespace omni
