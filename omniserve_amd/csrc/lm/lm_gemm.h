// What the products' kernels share: lm_gemm.hip and, in a file of their own, the 256 x 128 tiles.
#pragma once
#include "lm_common.h"
#include "omniserve_lm.h"

namespace lm {

template <int N> struct Int { static constexpr int value = N; };
template <int J, typename F>
__device__ __forceinline__ void countdown(F&& f) {      // f(J), f(J - 1), ..., f(0)
  f(Int<J>{});
  if constexpr (J > 0) countdown<J - 1>(f);
}

struct Part {        // a family of equally shaped groups
  const elem_t* w;   // [groups][n][k]
  const elem_t* x; int64_t ldx;
  void* y; int64_t ldy;
  int n, k;
  int64_t gx, gy;            // without perm: columns of x / y between neighbouring groups
  const float* bias;         // [n] added to the products of a gated unit (or null)
  const elem_t* gate;        // LM_EPI_GATE: the factor's argument, laid out like y
  int64_t ldg;
};

// What all kernels take: a field for one of them moves the arguments behind it for all.  (16 bytes more, and the gated unit of half tiles loads some of its arguments
// later: 130 tokens of 64 experts, 8 each, 256 x 2048 37.5 -> 40.0 us, 300 tokens of 1280 x 2048 101 -> 107.)
struct GemmArgs {
  Part a, b;                  // a: groups 0 .. groups - 1 (rows by perm / off), b: one group over rows 0 .. rows_b - 1
  int groups;
  const int* perm;            // row of y for every sorted place (null: identity, rows_a rows)
  const int* off;             // [groups + 1] sorted places of each group; chosen form (perm null): the expert of each of rows_a (token, choice) pairs
  int rows_a, rows_b;
  int x_div;                  // x row = y row / x_div (tokens of (token, choice) pairs)
  const int* tiles;           // lm_gemm_tiles with perm: (group, first place, rows, 0) of every row tile, behind them (0, 0, 0, how many; 0: not said)
  float scale;
  int act;                    // of the gated unit
};

__device__ __forceinline__ f32x4 glu(const Part& pt, int act, int c, f32x4 gate, f32x4 up) {      // c: gate channel's row in w, a multiple of 4
  if (pt.bias) {
    gate += *(const f32x4*)(pt.bias + c);
    up += *(const f32x4*)(pt.bias + c + 16);
  }
  f32x4 r;
  if (act == LM_ACT_GELU_TANH) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = gelu_tanh(gate[e]) * up[e];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = silu(gate[e]) * up[e];
  }
  return r;
}

template <int EPI>
__device__ __forceinline__ void store4(const Part& pt, int64_t row, int c, int64_t y0, f32x4 v, float scale) {
  if constexpr (EPI == LM_EPI_ELEM || EPI == LM_EPI_GLU) {
    *(quad_t*)((elem_t*)pt.y + row * pt.ldy + y0 + c) = to_quad(v);
  } else if constexpr (EPI == LM_EPI_F32) {
    *(f32x4*)((float*)pt.y + row * pt.ldy + y0 + c) = v * scale;
  } else {
    const f32x4 z = from_quad(*(const quad_t*)(pt.gate + row * pt.ldg + y0 + c));
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= sigmoid(z[e]);
    *(quad_t*)((elem_t*)pt.y + row * pt.ldy + y0 + c) = to_quad(v);
  }
}

constexpr int TM = LM_TILE_ROWS;                            // rows of a tile
static_assert(TM == 256, "the wave layouts");
constexpr int HTN = 128;                                    // channels of a half tile

// Row tiles with rows in them: experts fill fewer than the host has to reckon with (lm_route_max_tiles), and the tail without rows, of a tenth of the tiles with 32 experts and 8000 tokens, a sixth
// with 64 of fewer, would be the last XCD's alone, the others' rounds the longer for it (us, whole tiles, 7999 tokens, 6 of 32 experts of 1792, width 4096, up 1612 -> 1593, down 888 -> 840; 900 tokens
// 400 -> 314; 8 of 64 experts of 640, width 2048, 5800 tokens, up, 327 -> 277.  The half tiles, a workgroup each, wait for the entry: 1 - 2 % longer, and keep their order).  The last entry says how many, if it has no rows itself.
__device__ __forceinline__ int row_tiles(const int* tiles, int max_tiles) {
  const i32x4 last = *(const i32x4*)(tiles + 4 * (max_tiles - 1));
  return last[2] > 0 || last[3] <= 0 ? max_tiles : min(last[3], max_tiles);
}

// gemm_half_tiles_kernel<epi> over `wgs` workgroups; mt_a, mt_b: row tiles of both parts
__attribute__((visibility("hidden"))) void launch_half_tiles(const GemmArgs& a, int epi, unsigned wgs, int mt_a, int mt_b, hipStream_t s);

}  // namespace lm
