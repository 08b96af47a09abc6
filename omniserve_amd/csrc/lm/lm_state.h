// What the single-token kernels of the recurrent layers share: one workgroup owns one head's state [dk][dv] (f32), thread =
// 4 value columns x dk / 16 rows, all of them in registers; sums over the rows meet in LDS.
#pragma once
#include "lm_common.h"

namespace lm {

// Heads or places of the batch first over the grid.  Heads first, neighbouring workgroups take neighbouring states, where places first have them a slot apart, on the
// same memory channels at a time; but while all workgroups are on the chip at once, places first are as fast or faster.  (MI355X, heads of 128 x 128 in the steps of a
// model, us, gated / delta rule, places | heads first: 128 heads in all 7.4 | 7.4 / 9.1 | 9.1, 256 9.1 | 9.2 / 10.2 | 10.8, 384 11.8 | 13.1 / 12.6 | 12.2, 512 14.2 | 14.0 / 15.2 |
// 15.6, 768 21.8 | 19.8 / 23.7 | 20.4, 1536 45 | 40.6 / 44 | 40.6.)
static inline bool heads_first(int64_t B, int H) { return B * H > 512; }
template <typename Args>
static inline dim3 state_grid(const Args& a, int places) { return a.heads_first ? dim3(a.H, places) : dim3(places, a.H); }

// A grid's second dimension, which may be the places of the batch, ends at 65535: more go in launches of their own (a third dimension and its test in the kernel: a step of one
// sequence 4.1 -> 4.3 us).  a: the kernel's arguments, of which x, o, slot and pos go from place to place.
constexpr int STATE_PLACES = 32768;
template <typename Args, typename Launch>
static void in_places(Args a, int B, Launch launch) {
  for (; B > 0; B -= STATE_PLACES) {
    launch(a, min(B, STATE_PLACES));
    a.x += STATE_PLACES * a.ld;
    a.o += STATE_PLACES * a.ldo;
    a.slot += STATE_PLACES;
    a.pos += STATE_PLACES;
  }
}

// The recurrent state of a decode step, read and written once.  From 16 MB on (half of the L2s) it is not kept there: what it would push out is read
// again.  (MI355X, heads of 128 x 128, kept / not, 300 MB of other reads in front: 8 MB 10.1 / 9.6 us gated, 12.7 / 12.1 delta rule; 16 MB 12.7 / 11.4 and
// 15.4 / 13.7; 32 MB 20.2 / 17.0 and 23.1 / 19.7; 64 MB 34.1 / 29.0 and 39.3 / 35.6; a state still in the caches, heads of 256 x 256: 4 MB 10.2 / 12.1,
// 12 MB 12.2 / 13.8, 16 MB 13.0 / 14.1, but 32.1 / 31.4 with the reads behind it.  One sequence, 2 MB, 7.6 / 7.9 then, so small states stay.)
__host__ __device__ constexpr bool streams_state(int64_t sequences, int heads, int dk, int dv) {
  return sequences * heads * dk * dv * (int64_t)sizeof(float) >= (16 << 20);
}
template <bool STREAM>
__device__ __forceinline__ f32x4 load_state(const f32x4* p) {
  if constexpr (STREAM) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool STREAM>
__device__ __forceinline__ void store_state(f32x4* p, f32x4 v) {
  if constexpr (STREAM) __builtin_nontemporal_store(v, p);
  else *p = v;
}

constexpr int STATE_GROUPS = 16;                 // row groups

struct HeadOut {                                 // RMS norm over n of dv columns, times w, times silu(gate)
  const elem_t* gate;                            // of this head
  const float* w;
  int n;
  float eps;
};

// acc: this thread's part of sum_rows q S; the first wave returns with the sums of its 4 columns (lane < dv / 4)
template <int DV>
__device__ __forceinline__ f32x4 over_groups(f32x4 acc, f32x4 (*red)[DV / 4], int grp, int col) {
  red[grp][col] = acc;
  __syncthreads();
  f32x4 y = red[0][col];
#pragma unroll
  for (int g = 1; g < STATE_GROUPS; ++g) y += red[g][col];
  return y;
}

template <int DV>
__device__ __forceinline__ void head_out(f32x4 y, const HeadOut& p, elem_t* o) {      // threads 0 .. DV / 4 - 1, one wave
  const int col = threadIdx.x;
  float ss = (y[0] * y[0] + y[1] * y[1]) + (y[2] * y[2] + y[3] * y[3]);
#pragma unroll
  for (int m = DV / 8; m > 0; m >>= 1) ss += __shfl_xor(ss, m, 64);
  const float r = 1.0f / sqrtf(ss / (float)p.n + p.eps);
  const f32x4 g = from_quad(*(const quad_t*)(p.gate + 4 * col)), w = *(const f32x4*)(p.w + 4 * col);
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] *= r * w[e] * silu(g[e]);
  *(quad_t*)(o + 4 * col) = to_quad(y);
}

}  // namespace lm
