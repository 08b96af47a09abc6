// Matrix instructions of a wave that has its SIMD to itself and 256 accumulator registers.
//
//  * The accumulators are pinned to accumulation registers ("+a"): left to the compiler, 64 tiles of a lone wave move between the register
//    files inside the loop (100 moves per 64 products).
//  * A lone wave issues an instruction every four cycles and a product takes sixteen: at most three others fit between two products.
//    OMNI_MFMA3_DMA16 is three products with one LDS-DMA request in their shadow.
//  * The compiler does not see a matrix instruction here: accumulators_settle() stands between the last of them and a read of the results.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define OMNI_MFMA_PINNED(OP, c, a, b) asm volatile(OP " %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b))

// c = a b
#define OMNI_MFMA_FRESH(OP, c, a, b) asm volatile(OP " %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b))

// ADDR: "%10" with a scalar base and src a 32-bit offset from it, "off" with src an address (base is then ignored).  M0 is the compiler's:
// saved and restored.
#define OMNI_MFMA3_DMA16(OP, ADDR, c0, c1, c2, a0, a1, a2, b, src, base, lds_dst)                                            \
  do {                                                                                                                      \
    uint32_t keep_m0;                                                                                                       \
    asm volatile(OP " %1, %4, %7, %1\n\ts_mov_b32 %0, m0\n\ts_mov_b32 m0, %9\n\t" OP " %2, %5, %7, %2\n\t"                   \
                 "global_load_lds_dwordx4 %8, " ADDR "\n\t" OP " %3, %6, %7, %3\n\ts_mov_b32 m0, %0"                         \
                 : "=&s"(keep_m0), "+a"(c0), "+a"(c1), "+a"(c2)                                                             \
                 : "v"(a0), "v"(a1), "v"(a2), "v"(b), "v"(src), "s"(lds_dst), "s"(base)                                      \
                 : "memory");                                                                                               \
  } while (0)

// The lines at 32 lanes' addresses (the first 32's) into the XCD's L2: a dword of each goes to 128 bytes of LDS that nobody reads, as one piece of vmcnt.
// For tiles that many compute units of an XCD read at about the same time: their requests come half a stage before they are needed, enough for what the L2
// holds and not for what it has to fetch; ahead of them each unit touches its share of what they have in common.  Whole waves only.  (No gain where a stage
// takes longer for its operands to be unpacked: the 4-bit group-wise tiles, 320 us of 28672 x 4096 and 2331 rows without, 322 with.)
__device__ __forceinline__ void touch_lines32(const void* src, uint32_t lds_sink) {
  uint32_t keep_m0;      // (M0 is the compiler's)
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_mov_b32 exec_hi, 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 exec_hi, -1\n\ts_mov_b32 m0, %0"
               : "=&s"(keep_m0)
               : "v"(src), "s"(lds_sink)
               : "memory");
}

// a value the optimiser knows nothing about: what is computed from it is computed where it stands, not kept across a loop
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
// the lane, computed where it stands: no register holds it, or what is computed from it, across a loop
__device__ __forceinline__ int lane_here() {
  int v;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(v));
  return v;
}
// at the start of a block behind a branch: the accumulators come into it where they are (a value that is read in other blocks than its own is moved to vector registers in
// front of the branch)
template <typename V, int N, int M>
__device__ __forceinline__ void accumulators_stay(V (&c)[N][M]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) asm volatile("" : "+a"(c[i][j])::"memory");
}
template <typename V, int N, int M>
__device__ __forceinline__ void accumulators_settle(V (&c)[N][M]) {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) asm volatile("" : "+a"(c[i][j]));      // (a later value: no read of it moves up)
}
