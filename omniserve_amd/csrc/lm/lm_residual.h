// Residual and norms of one token's row: what lm_residual_norm and the expert choice of few tokens share.
#pragma once
#include "lm_common.h"
#include "omniserve_lm.h"

namespace lm {

template <int TH>
struct Row {      // workgroup-wide sums
  float* red;     // [2][TH / 64]
  int phase = 0;
  __device__ __forceinline__ float sum(float v) {
    v = wave_sum(v);
    float* r = red + TH / 64 * (phase & 1);      // two areas in turn: one barrier per sum
    ++phase;
    if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < TH / 64; i += 4) t += (r[i] + r[i + 1]) + (r[i + 2] + r[i + 3]);
    return t;
  }
};

// v (columns 4 * (TH i + tid) .. + 3, zero from n on) -> normalised in place; kind 0: layer norm, 1: RMS norm
template <int TH, int NV>
__device__ __forceinline__ void normalise(f32x4 (&v)[NV], Row<TH>& row, int n, int kind, float eps, const float* w, const float* b) {
  float mean = 0.f;
  if (kind == LM_NORM_LAYER) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
    mean = row.sum(s) / (float)n;
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = 4 * (TH * i + (int)threadIdx.x);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[i][e] = c + e < n ? v[i][e] - mean : 0.f;
      ss += v[i][e] * v[i][e];
    }
  }
  const float r = 1.0f / sqrtf(row.sum(ss) / (float)n + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = 4 * (TH * i + (int)threadIdx.x);
    if (c >= n) continue;
    const f32x4 ww = *(const f32x4*)(w + c);
    f32x4 bb = zero4();
    if (b) bb = *(const f32x4*)(b + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[i][e] = c + e < n ? v[i][e] * r * ww[e] + bb[e] : 0.f;
  }
}

struct ResidualArgs {
  float* x; int64_t ldx;                     // residual stream
  const int* tokens; const elem_t* embed;    // tokens: the residual starts as these rows of the table [vocab][ldx] ...
  float embed_scale;                         // ... times this
  const elem_t* y; int64_t ldy;              // sublayer output (or null): added to the residual
  const float* sums; int slices;             // ... or the f32 sums of its product's K slices, [slices][sum_rows][ldy]
  int64_t sum_rows;
  const float* y_bias;                       // added to y (or null)
  const float* pair_w; int top, pairs0, shared;   // top > 0: y holds expert outputs by (token, choice), see moe_sum
  const float *post_w, *post_b;              // norm of the sublayer output before it is added (or null)
  const float *next_w, *next_b;              // norm of the new residual for the next sublayer (or null: as it is) -> h
  elem_t* h; int64_t ldh;
  const int* rows;                           // row r of the launch works on token rows[r] (or null: r) and writes h[r]
  int n, kind, store_x;
  float eps;
};

// Token t's row, by a workgroup of TH threads: the residual with what is added to it (stored), then, for p.h, the input of the next sublayer in x: columns 4 (TH i + thread) .. + 3
template <int TH, int NV>
__device__ __forceinline__ void residual_row(const ResidualArgs& p, Row<TH>& row, int t, f32x4 (&x)[NV]) {
  const int tid = threadIdx.x;
  f32x4 y[NV];
  float* xr = p.x + (int64_t)t * p.ldx;
  const elem_t* er = p.tokens ? p.embed + (int64_t)p.tokens[t] * p.ldx : nullptr;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = 4 * (TH * i + tid);
    x[i] = y[i] = zero4();
    if (c >= p.n) continue;
    x[i] = er ? p.embed_scale * from_quad(*(const quad_t*)(er + c)) : *(const f32x4*)(xr + c);
  }
  if (p.y || p.sums) {
    if (p.sums) {         // added up and rounded as gemm_reduce_kernel does
      constexpr int B = NV == 1 ? 4 : NV == 2 ? 2 : 1;      // slices in flight
      const float* sr = p.sums + (int64_t)t * p.ldy;
      const int64_t next = p.sum_rows * p.ldy;
      for (int k0 = 0; k0 < p.slices; k0 += B) {
        f32x4 v[B][NV];
#pragma unroll
        for (int k = 0; k < B; ++k)
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            const int c = 4 * (TH * i + tid);
            v[k][i] = c < p.n && k0 + k < p.slices ? *(const f32x4*)(sr + (k0 + k) * next + c) : zero4();
          }
#pragma unroll
        for (int k = 0; k < B; ++k)
#pragma unroll
          for (int i = 0; i < NV; ++i) y[i] += v[k][i];
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) y[i] = from_quad(to_quad(y[i]));
    }
    if (p.top > 0) {      // weighted sum of the chosen experts' rows (+ the shared expert's)
      const int64_t p0 = (int64_t)t * p.top;
      constexpr int B = NV >= 8 ? 1 : NV >= 4 ? 2 : 4;      // rows in flight
      for (int k0 = 0; k0 < p.top; k0 += B) {
        quad_t v[B][NV];
        float w[B];
        uint32_t some = 0;
#pragma unroll
        for (int b = 0; b < B; ++b) {
          const int k = min(k0 + b, p.top - 1);
          const float pw = p.pair_w[p0 + k];
          some |= __builtin_bit_cast(uint32_t, pw) ^ LM_NO_EXPERTS_BITS;
          w[b] = k0 + b < p.top ? pw : 0.f;
          const elem_t* yr = p.y + (p0 + k) * p.ldy;
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            const int c = 4 * (TH * i + tid);
            v[b][i] = c < p.n ? *(const quad_t*)(yr + c) : to_quad(zero4());
          }
        }
        // (behind the requests, which bring the weights, too; TH > 256: the forms of few rows, for which lm_norm_choose is)
        if (TH > 256 && some == 0) continue;
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int i = 0; i < NV; ++i) y[i] += w[b] * from_quad(v[b][i]);
      }
    }
    if (!p.sums && (p.top == 0 || p.shared)) {
      const elem_t* yr = p.y + (int64_t)(p.top > 0 ? p.pairs0 + t : t) * p.ldy;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = 4 * (TH * i + tid);
        if (c < p.n) y[i] += from_quad(*(const quad_t*)(yr + c));
      }
    }
    if (p.y_bias) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = 4 * (TH * i + tid);
        if (c < p.n) y[i] += *(const f32x4*)(p.y_bias + c);
      }
    }
    if (p.post_w) normalise<TH, NV>(y, row, p.n, p.kind, p.eps, p.post_w, p.post_b);
#pragma unroll
    for (int i = 0; i < NV; ++i) x[i] += y[i];
  }
  if (p.store_x) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = 4 * (TH * i + tid);
      if (c < p.ldx) *(f32x4*)(xr + c) = x[i];
    }
  }
  if (p.next_w) normalise<TH, NV>(x, row, p.n, p.kind, p.eps, p.next_w, p.next_b);
}

}  // namespace lm
