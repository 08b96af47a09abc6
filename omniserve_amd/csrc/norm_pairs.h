// Rows of 1024 .. 8192 channels held as the reference's virtual threads hold them, thread p of 512 with channels 2 p and 2 p + 1 of every 1024: what
// norm_rows.hip and norm_product.hip share.
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

}  // namespace omni
