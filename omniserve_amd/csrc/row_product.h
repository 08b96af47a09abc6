// The product of one or two rows of int8 codes in LDS with a workgroup's share of a weight matrix (norm_product.hip, act_product.hip): 8 waves, wave w
// with the w-th eighth of the workgroup's K, weights through registers, K parts meeting in LDS.
//
//  * GATE: gate channels and the up channels that belong to them, 8 of each in a 16-row operand block (gate_up with silu_and_mul).
//  * ROWS32: 32 channels.  A packed 32-channel tile row fills only half of the matrix instruction's operand: the other eight operand rows carry the
//    same channels 64 k further, the codes of which lie in the neighbouring column of the activations; the two meet when the K parts do.
//  * ROWS64: 64 channels.
//
// int8 weights come as rows: both 64-byte halves of a row's 128 bytes are requested one after the other.
#pragma once
#include "qgemm_kernel.h"
#include "norm_pairs.h"

namespace omni {

constexpr int RP_WAVES = 8, RP_THREADS = 64 * RP_WAVES;
enum RowLayout { LAYOUT_GATE, LAYOUT_ROWS32, LAYOUT_ROWS64 };

// byte of k among a row's codes: as the packed tiles hold k (qgemm_kernel.h), or in its own order
template <int MODE>
__device__ __forceinline__ uint32_t code_place(uint32_t k) {
  if constexpr (MODE == MODE_W8) return k;
  return (k & ~63u) + ((k >> 2) & 3) * 16 + ((k >> 5) & 1) * 8 + ((k >> 4) & 1) * 4 + (k & 3);
}

// BLOCKS: 16-row operand blocks of the workgroup (packed weights: whole tile rows, 4 blocks to a pair).  KPART: k of a wave.  RING: units (of UNIT k) that
// fly together.  NT: packed weights load non-temporally (false: they lie in L2).
template <int MODE, int LAYOUT, int BLOCKS, int KPART, int RING_MAX, int ROWS, bool NT = true>
struct RowProduct {
  static constexpr bool W8 = MODE == MODE_W8, PAIRED = !W8 && LAYOUT == LAYOUT_ROWS32;
  static constexpr int PAIRS = BLOCKS / 4;                                  // tile-row pairs (ROWS32: the one tile row)
  static_assert(W8 || BLOCKS % 4 == 0, "whole tile rows");
  static constexpr int UNIT = (PAIRED || W8) && KPART % 128 == 0 ? 128 : 64, UNITS = KPART / UNIT;
  static_assert(KPART % UNIT == 0 && (!PAIRED || UNIT == 128), "whole units");
  static constexpr int HALVES = W8 ? UNIT / 64 : 1;
  static constexpr int LOADS = W8 ? HALVES * BLOCKS : 2 * PAIRS;            // 16-byte loads of a unit
  static constexpr int RING = UNITS < RING_MAX ? UNITS : RING_MAX;
  static constexpr int COLS = ROWS * (PAIRED ? 2 : 1);
  static constexpr int PART_BYTES = RP_WAVES * BLOCKS * 4 * COLS * 16;
  static constexpr int PER = KPART % 128 ? 1 : 128 / UNIT;                  // units that share their group's parameters
  static constexpr int GROUPS = MODE == MODE_GRP ? UNITS / PER : 1;

  uint4 wq[RING][LOADS];
  uint32_t gs[PAIRS ? PAIRS : 1][GROUPS], gz[PAIRS ? PAIRS : 1][GROUPS];
  v4i acc[BLOCKS];
  const uint8_t* base;      // of the lane
  long long step;           // packed: from a tile-row pair to the next; int8: from a block of rows to the next
  int turn;                 // the unit that this workgroup begins with

  __device__ __forceinline__ int place(int u) const {      // of the u-th unit in the wave's K
    const int v = u + turn;
    return v < UNITS ? v : v - UNITS;
  }

  // first: the workgroup's first operand block of all; k0: the wave's first k
  __device__ __forceinline__ void open(const uint8_t* W, const uint8_t* s2s, const uint8_t* s2z, int N, int K, int first, int k0) {
    const int lane = threadIdx.x & 63, lx = (lane >> 3) & 1, lc = lane & 7, le = lane >> 4;
// (workgroups in step ask the same channels of the memory: gate_up W8A8 28.9 us, turned 27.6, W4A8 14.3 and 13.8.  Not per-group weights, 16.2 and 17.6, and not
    // ROWS64: W8A8 down_proj 12.3 and 13.5, o_proj behind its prefetch 4.1 and 4.7)
    turn = MODE == MODE_GRP || LAYOUT == LAYOUT_ROWS64 ? 0 : (int)(blockIdx.x >> 3) % UNITS;
    if constexpr (W8) {
      if constexpr (LAYOUT == LAYOUT_GATE) {
        base = W + (size_t)(lx * (N / 2) + first * 8 + lc) * K + le * 16 + k0;
        step = 8LL * K;
      } else {
        base = W + (size_t)(first * 16 + (lane & 15)) * K + le * 16 + k0;
        step = 16LL * K;
      }
    } else {
      int trow, pair;      // the lane's tile row of the first pair; from a pair to the next
      if constexpr (LAYOUT == LAYOUT_GATE) trow = (lx ? N / 64 : 0) + first / 4, pair = 1;
      else if constexpr (PAIRED) trow = first / 4, pair = 1;
      else trow = first / 2 + lx, pair = 2;
      base = W + ((size_t)trow * (K / 32) + k0 / 32 + (PAIRED ? 2 * lx : 0)) * 512 + (lc * 4 + le) * 16;
      step = 512LL * pair * (K / 32);
      if constexpr (MODE == MODE_GRP) {
#pragma unroll
        for (int t = 0; t < PAIRS; ++t)
#pragma unroll
          for (int i = 0; i < GROUPS; ++i) {
            const size_t off = (size_t)((k0 + i * PER * UNIT) / 128) * N + (trow + t * pair) * 32 + lc * 4;
            gs[t][i] = *reinterpret_cast<const uint32_t*>(s2s + off);
            gz[t][i] = *reinterpret_cast<const uint32_t*>(s2z + off);
          }
      }
    }
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) acc[b] = (v4i){0, 0, 0, 0};
  }
  __device__ __forceinline__ void request(int u) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const uint8_t* src = base + (W8 ? j / HALVES : j >> 1) * step + (W8 ? place(u) * UNIT + (j % HALVES) * 64 : (place(u) * (UNIT / 32) + (j & 1)) * 512);
      v4i v;
      if constexpr (W8 || !NT) v = *reinterpret_cast<const v4i*>(src);             // (non-temporal, a line's second half is fetched again: 31 us, not 28)
      else v = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(src));
      wq[u % RING][j] = make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
    }
  }
  // codes: row 0's, at the wave's first k; the units behind the ring are requested as it empties
  __device__ __forceinline__ void multiply(const uint8_t* codes, int pitch) {
    const int lane = threadIdx.x & 63, col = lane & 15, row = min(PAIRED ? col >> 1 : col, ROWS - 1);      // (columns beyond: never read)
    const uint8_t* src = codes + row * pitch + (PAIRED ? (col & 1) * 64 : 0) + (lane >> 4) * 16;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      v4i wa[HALVES][BLOCKS];
      if constexpr (W8) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
          const uint4 w = wq[u % RING][j];
          wa[j % HALVES][j / HALVES] = (v4i){(int)w.x, (int)w.y, (int)w.z, (int)w.w};
        }
      } else {
#pragma unroll
        for (int t = 0; t < PAIRS; ++t) {
          const uint4 t0 = wq[u % RING][2 * t], t1 = wq[u % RING][2 * t + 1];
          const uint32_t d[2][4] = {{t0.x, t0.z, t1.x, t1.z}, {t0.y, t0.w, t1.y, t1.w}};
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              uint32_t w[4];
#pragma unroll
              for (int q = 0; q < 4; ++q) w[q] = (d[j][q] >> (4 * i)) & 0x0F0F0F0Fu;
              if constexpr (MODE == MODE_GRP) {
                const uint32_t sc = (gs[t][u / PER] >> (8 * (i * 2 + j))) & 0xFFu;
#pragma unroll
                for (int q = 0; q < 4; ++q) w[q] = w[q] * sc;
                vadd4_zbyte_x4(w, gz[t][u / PER], i * 2 + j);
              }
              wa[0][4 * t + i * 2 + j] = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
            }
        }
        if (u + RING < UNITS) request(u + RING);
      }
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        const v4i b = *reinterpret_cast<const v4i*>(src + place(u) * UNIT + h * 64);
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[h][i], b, acc[i], 0, 0, 0);
      }
      if constexpr (W8) {
        if (u + RING < UNITS) request(u + RING);
      }
    }
  }
  __device__ __forceinline__ void leave(uint8_t* parts, int wave) const {
    const int lane = threadIdx.x & 63, col = lane & 15;
    if (col < COLS) {
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b) *reinterpret_cast<v4i*>(parts + (((wave * BLOCKS + b) * 4 + (lane >> 4)) * COLS + col) * 16) = acc[b];
    }
  }
  // the sum of the K parts [w0, w1) in operand row r of block b, column c
  static __device__ __forceinline__ int total(const uint8_t* parts, int b, int r, int c, int w0 = 0, int w1 = RP_WAVES) {
    int sum = 0;
#pragma unroll
    for (int w = w0; w < w1; ++w) sum += *reinterpret_cast<const int*>(parts + (((w * BLOCKS + b) * 4 + (r >> 2)) * COLS + c) * 16 + (r & 3) * 4);
    return sum;
  }
};

}  // namespace omni
