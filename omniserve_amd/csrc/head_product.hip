// The output head of a greedy step: fp16 hidden rows x fp16 [vocab, hidden] -> logits, rounded to fp16, -> index of each row's first largest one
// (llama_w4a8_unpad.py:556-563 and the sampler's argmax).  Few rows: a stream of weights, 262 MB for 32000 x 4096.
//
// Both operands arrive by LDS-DMA in pieces of 8 rows x 128 bytes (operand fragments loaded straight into registers read 64 bytes of each of 16 rows, which
// the address path takes at 15 bytes a clock).  A workgroup has 64 channels; a stage is 128 bytes of k of them and of the rows, consumed behind one
// barrier while as many more as 64 KiB hold are on their way; two workgroups to a compute unit.  The logits stay inside: a workgroup leaves one key a row.
//
// MI355X, with the argmax, against the vendor's product and omni_argmax_f16: 32000 x 4096 61.0 - 62.5 -> 42.8 us (1 - 16 rows; 6.4 TB/s without the launch that
// finishes), 61.9 -> 53.4 (64 rows); 16000 x 8192 55 - 56 -> 49, at 64 rows no faster.
//
// f32 sums of 256 products each, added up in the order of k: no further from 64 bits than one chain, and the same for equal weights wherever they stand, so that the first
// of equal rows is the one that is found.
#include "qgemm_kernel.h"
#include "argmax_key.h"

namespace omni {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int HEAD_CHANNELS = 64, HEAD_STAGE_K = 64, HEAD_CHAIN = 4;

struct HeadArgs {
  const half_t* x;
  const half_t* w;
  unsigned long long* part;      // [M][workgroups]
  int M, V, K;
};

template <bool STREAM>
__device__ __forceinline__ void head_dma16(uint32_t src, const void* base, uint32_t lds_dst) {
  uint32_t keep;
  if constexpr (STREAM)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3 nt\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(src), "s"(lds_dst), "s"(base) : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(src), "s"(lds_dst), "s"(base) : "memory");
}

// EIGHTS: M in pieces of 8 rows
template <int EIGHTS>
__global__ __launch_bounds__(256) void head_argmax_kernel(HeadArgs p) {
  constexpr int MB = (EIGHTS + 1) / 2, W_BYTES = HEAD_CHANNELS * 128, STAGE = W_BYTES + EIGHTS * 1024;
  constexpr int XP = (EIGHTS + 3) / 4, P = 2 + XP;            // pieces of x, and all, that a wave requests for a stage (some of x twice: the same bytes)
  constexpr int R = (64 << 10) / STAGE;
  constexpr int EARLY = MB <= 2 ? 15 : 7;                     // as the registers have room
  static_assert((R - 2) * P <= 63, "vmcnt");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[R * STAGE];
  __shared__ unsigned long long best[4][16 * MB];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, l4 = lane >> 4;
  const int n0 = blockIdx.x * HEAD_CHANNELS, nst = p.K / HEAD_STAGE_K;
  const uint32_t pitch = 2u * (uint32_t)p.K;

  uint32_t wsrc[2], xsrc[XP], xdst[XP];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * i + (lane >> 3);
    wsrc[i] = (uint32_t)min(16 * wave + r, p.V - 1 - n0) * pitch + (((lane & 7) ^ tiles_swizzle(r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int piece = (4 * i + wave) % EIGHTS, r = 8 * piece + (lane >> 3);
    xsrc[i] = (uint32_t)min(r, p.M - 1) * pitch + (((lane & 7) ^ tiles_swizzle(r & 15)) << 4);
    xdst[i] = W_BYTES + 1024 * piece;
  }
  const uint8_t* const wbase = reinterpret_cast<const uint8_t*>(p.w + (size_t)n0 * p.K);
  const uint8_t* const xbase = reinterpret_cast<const uint8_t*>(p.x);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds);
  // Rows lie whole KiBs apart: workgroups in step would all ask the same channels of the memory, so they begin with different numbers (`early`) of K's last chains,
  // whose sums wait for those in front of them.  (MI355X, 1 and 16 rows, at most 1, 4, 8, 15 chains: 32000 x 4096 50.7, 44 - 47, 43 - 46, 42 - 45 us, 128256 x 4096
  // 186 - 192, 174 - 179, 169 - 172, 164; beginning 640 bytes apart with orders of their own 44 and 166.  64 rows, 7 and 15 chains: 52 and 61.)
  const int chains = (nst + HEAD_CHAIN - 1) / HEAD_CHAIN, early = max(0, min((int)(blockIdx.x >> 3) % (EARLY + 1), chains - 3));
  const int turn = early ? HEAD_CHAIN * (chains - early) : 0, first = early ? nst - turn : 0;      // first: stages of those chains
  auto stage = [&](int t) {
    const size_t at = (size_t)(t + turn < nst ? t + turn : t + turn - nst) * 128;
    const uint32_t dst = lds0 + (uint32_t)(t % R) * STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) head_dma16<true>(wsrc[i], wbase + at, dst + 2048 * wave + 1024 * i);
#pragma unroll
    for (int i = 0; i < XP; ++i) head_dma16<false>(xsrc[i], xbase + at, dst + xdst[i]);
  };
  uint32_t off[2];                                            // of a fragment inside 16 rows
#pragma unroll
  for (int h = 0; h < 2; ++h) off[h] = (uint32_t)l15 * 128 + (((4 * h + l4) ^ tiles_swizzle(l15)) << 4);
  // (8 rows: the operand's columns 8 .. 15 are 0 .. 7 again)
  uint32_t xoff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) xoff[h] = EIGHTS == 1 ? (uint32_t)(l15 & 7) * 128 + (((4 * h + l4) ^ tiles_swizzle(l15 & 7)) << 4) : off[h];
  v4f acc[MB], total[MB], later[EARLY][MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) acc[m] = total[m] = (v4f){0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int t) {
    const uint8_t* const wt = lds + (t % R) * STAGE + 2048 * wave;
    const uint8_t* const xt = lds + (t % R) * STAGE + W_BYTES;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f16x8 a = *reinterpret_cast<const f16x8*>(wt + off[h]);
#pragma unroll
      for (int m = 0; m < MB; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, *reinterpret_cast<const f16x8*>(xt + 2048 * m + xoff[h]), acc[m], 0, 0, 0);
    }
  };
#pragma unroll
  for (int t = 0; t < R - 1; ++t)
    if (t < nst) stage(t);
  int t = 0;
  auto step = [&] {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((R - 2) * P) : "memory");
    __builtin_amdgcn_s_barrier();                             // stage t is there for every wave, everyone has left stage t - 1
    asm volatile("" ::: "memory");
    stage(t + R - 1);
    multiply(t);
    ++t;
  };
#pragma unroll
  for (int c = 0; c < EARLY; ++c) {
    const int end = c < early ? min(t + HEAD_CHAIN, first) : t;
    while (t < end) step();                                   // (more than R - 1 stages follow)
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      later[c][m] = acc[m];
      acc[m] = (v4f){0.f, 0.f, 0.f, 0.f};
    }
  }
  auto end_chain = [&] {                                      // ... behind stage t - 1
    if (((t - first) & (HEAD_CHAIN - 1)) != 0) return;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      total[m] += acc[m];
      acc[m] = (v4f){0.f, 0.f, 0.f, 0.f};
    }
  };
  while (t + R - 1 < nst) {
    step();
    end_chain();
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();                               // the rest is there
  asm volatile("" ::: "memory");
  while (t < nst) {
    multiply(t++);
    end_chain();
  }
#pragma unroll
  for (int m = 0; m < MB; ++m) total[m] += acc[m];
#pragma unroll
  for (int c = 0; c < EARLY; ++c) {
    for (int m = 0; m < MB; ++m)
      if (c < early) total[m] += later[c][m];
  }

  // the lane's four channels of row l15 of each block
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    unsigned long long key = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = n0 + 16 * wave + 4 * l4 + e;
      const half_t h = (half_t)total[m][e];
      const unsigned long long k = n < p.V ? argmax_key(__builtin_bit_cast(uint16_t, h), n) : 0;
      key = k > key ? k : key;
    }
#pragma unroll
    for (int x = 16; x < 64; x *= 2) {
      const uint32_t lo = __shfl_xor((uint32_t)key, x, 64), hi = __shfl_xor((uint32_t)(key >> 32), x, 64);
      const unsigned long long o = ((unsigned long long)hi << 32) | lo;
      key = o > key ? o : key;
    }
    if (l4 == 0) best[wave][16 * m + l15] = key;
  }
  __syncthreads();
  if ((int)threadIdx.x < p.M) {
    unsigned long long key = best[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < 4; ++w) key = best[w][threadIdx.x] > key ? best[w][threadIdx.x] : key;
    p.part[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = key;
  }
}

__global__ __launch_bounds__(256) void head_argmax_final_kernel(const unsigned long long* part, int n, long long* out) {
  __shared__ unsigned long long red[4];
  unsigned long long key = 0;
  for (int i = threadIdx.x; i < n; i += 256) {
    const unsigned long long k = part[(size_t)blockIdx.x * n + i];
    key = k > key ? k : key;
  }
  key = wave_max_u64(key);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = key;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) key = red[w] > key ? red[w] : key;
    out[blockIdx.x] = (long long)(0xFFFFFFFFu - (uint32_t)key);
  }
}

}  // namespace omni
using namespace omni;

static int head_groups(int V) { return (V + HEAD_CHANNELS - 1) / HEAD_CHANNELS; }

// 0: not its size (more rows have enough products a byte for the vendor's)
extern "C" size_t omni_head_argmax_workspace_bytes(int M, int V, int K) {
  if (M < 1 || M > 64 || V < 1 || K < 64 || K % 64 || 2ull * K * HEAD_CHANNELS >= 1ull << 32) return 0;
  return (size_t)M * head_groups(V) * sizeof(unsigned long long);
}

// Where this measured faster than the vendor's product and omni_argmax_f16 (MI355X, 13 vocabularies of 500 - 64000 x 9 K of 512 - 8192, us, this | those).  A workgroup
// alone takes 5 us for 1024 of K, whatever V: 500 x 4096 21 | 13, 8000 x 4096 23 | 22 at 1 row, 31 | 24 at 64; 10000 x 4096 23 | 25 and 31 | 32; 4000 x 2048 14 | 14.  The
// vendor's product loses where rows lie whole 4 KiBs apart and is good where they do not: 17 rows and more, 32000 x 5120 61 | 63 and 71 | 65, 50000 x 5120 108 | 96 and
// 129 | 102, 24000 x 3072 41 | 38 at 64 rows; x 4096 54 | 60, 94 | 87, 50 | 54.
extern "C" int omni_head_argmax_faster(int M, int V, int K) {
  if (omni_head_argmax_workspace_bytes(M, V, K) == 0) return 0;
  const bool many = M > 32;
  if (M > 16 && K % 2048 != 0 && K > (many ? 1024 : 4096)) return 0;
  if (K <= (many ? 1024 : 2048)) return V >= (many ? 2 : 1) * K;
  return V >= (many ? (K <= 2048 ? 10000 : 16000) : (K <= 4096 ? 10000 : 12000));
}

extern "C" int omni_head_argmax_f16(void* out_i64, const void* x_f16, const void* w_f16, int M, int V, int K, void* workspace, size_t workspace_bytes,
                                    void* stream) {
  const size_t need = omni_head_argmax_workspace_bytes(M, V, K);
  if (!out_i64 || !x_f16 || !w_f16 || need == 0 || ((reinterpret_cast<uintptr_t>(x_f16) | reinterpret_cast<uintptr_t>(w_f16)) & 15)) return OMNI_EINVAL;
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 7)) return OMNI_ENOMEM;
  const HeadArgs p{(const half_t*)x_f16, (const half_t*)w_f16, (unsigned long long*)workspace, M, V, K};
  const dim3 grid(head_groups(V)), block(256);
  hipStream_t st = (hipStream_t)stream;
  if (M <= 8) hipLaunchKernelGGL((head_argmax_kernel<1>), grid, block, 0, st, p);
  else if (M <= 16) hipLaunchKernelGGL((head_argmax_kernel<2>), grid, block, 0, st, p);
  else if (M <= 32) hipLaunchKernelGGL((head_argmax_kernel<4>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((head_argmax_kernel<8>), grid, block, 0, st, p);
  hipLaunchKernelGGL(head_argmax_final_kernel, dim3(M), block, 0, st, p.part, head_groups(V), (long long*)out_i64);
  return omni_launch_status();
}
