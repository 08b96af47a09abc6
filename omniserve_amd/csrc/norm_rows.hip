// rms_norm_general[_fuse_sum] with per-token quantisation for rows of 1024 .. 8192 channels in whole 1024s, fewer than ROWS_MANY of them (reference:
// kernels/csrc/layernorm_kernels.cu:58-331).  Everything else stays on general_norm_v2_kernel (row_kernels.h), to whose bits this kernel keeps.
//
// At these sizes a row is one compute unit's serial chain -- requests, two reductions, codes -- and the launch lasts as long as that chain.
// The reference's order of additions (1024 virtual threads, thread t adds up channels t, t + 1024, ..; a butterfly over 32 threads, one over
// their 32 sums) is what general_norm_v2_kernel replays out of an LDS copy of the row, by two of its eight waves, behind a barrier, twice.  Here the
// threads own the channels as the virtual threads do: thread p holds 2 p and 2 p + 1 of every 1024, so that
//
//  * the per-thread sums are formed in registers as the values appear: no copy, no replay, no barrier in front of them;
//  * a virtual warp is a row of 16 lanes: its butterfly is four DPP additions; the one over the 32 sums reads 16 bytes of LDS and is four more;
//  * the row maximum and the sum of the normalised values cross the workgroup together: two barriers in all instead of seven.
//
// MI355X, inside the captured step of the 8B model (4096 channels), general_norm_v2_kernel -> this one, us: 1 row, 8 slabs 8.3 -> 6.5; 16 rows, 8 slabs 8.0
// -> 6.3; first layer, no slabs, 6.3 -> 5.5.  What is left: the first load (the slabs come from other XCDs' launches; 128 KiB of them into one compute
// unit) and a launch's ends.  Rows alone, at 1, 128, 512 and 1023 of them: 4096 channels, no slabs, 4.3, 4.9, 6.3, 10.8 -> 3.0, 3.4, 4.2, 6.7; 4 slabs 6.3, 6.9, 15.7, 28.8
// -> 4.4, 4.9, 11.3, 21.1; 8192 channels, 8 slabs 9.0, 11.2, 32.5, 68 -> 8.1, 9.2, 27.3, 59.  Many slabs take a second trip: behind the product of 28672 x 8192 with its
// 14 slabs the two 32.5 -> 32.2, behind the int8 one with 28 72.3 -> 75.5 (16 slabs of int8 products, 1 and 16 rows: 4096 channels -0.1 and -0.2, 8192 +1.9 and +1.1).
#include "norm_pairs.h"
#include "norm_rows.h"

namespace omni {

// of more than 8 slabs, those whose requests are in flight together
template <int C>
constexpr int MANY_SLABS = C <= 4 ? 16 : 12;

// The norm's weights, requested first, are waited for here, in front of the residual's stores: a wait behind those would be for them, too
template <int C>
__device__ __forceinline__ void arrived(v2h (&g)[C]) {
#pragma unroll
  for (int c = 0; c < C; ++c) asm volatile("" : "+v"(g[c]));
}

// residual += h(epilogue(sum of the K slabs)); ZP: ((acc * sw) * sa) - (sz * as), else acc * (sw * sa)
template <bool ZP>
struct PairSlabs {
  NormSlabs s;
  __device__ __forceinline__ void pin() const {
    asm volatile("" ::"s"(s.res), "s"(s.slab), "s"(s.sstride), "s"(s.sk), "s"(s.wscales), "s"(s.wsz), "s"(s.ascales), "s"(s.asum));
  }
  // SK: slabs whose requests all go out in front of the first addition (those beyond s.sk read slab 0 again); a form of its own for each, to the
  // end: joined before the additions, hipcc waits for every load at the join
  template <int C, int SK>
  __device__ __forceinline__ void values_of(int row, uint32_t at, v2h (&g)[C], float (&x)[C][2]) const {
    const half_t sa_h = s.ascales[row];
    half_t as_h = (half_t)0.0f;
    if constexpr (ZP) as_h = s.asum[row];
    const RowArray res(s.res + (size_t)row * (1024 * C)), slab(s.slab + (size_t)row * (1024 * C)), ws(s.wscales), wz(s.wsz);
    const uint32_t step = (uint32_t)(s.sstride * 4);
    v2i t[SK][C];
#pragma unroll
    for (int k = 0; k < SK; ++k)
#pragma unroll
      for (int c = 0; c < C; ++c) t[k][c] = slab.two(2 * at, (SK <= 8 || k < s.sk ? k * step : 0) + 4096 * c);
    v2h a[C], sw[C], sz[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      a[c] = res.pair(at, 2048 * c);
      sw[c] = ws.pair(at, 2048 * c);
      if constexpr (ZP) sz[c] = wz.pair(at, 2048 * c);
    }
    __builtin_amdgcn_sched_barrier(0);      // every request in front of the first wait
    arrived(g);
    v2i acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = t[0][c];      // integers: any order is exact
#pragma unroll
    for (int k = 1; k < SK; ++k)
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] += SK <= 8 || k < s.sk ? t[k][c] : (v2i){0, 0};
    if constexpr (SK > 8)
      for (int k = SK; k < s.sk; ++k)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] += slab.two(2 * at, k * step + 4096 * c);
    const float sa = (float)sa_h, as = (float)as_h;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      v2h o;
#pragma unroll
      for (int e = 0; e < 2; ++e) {      // the product's own epilogue (qgemm_kernel.h), each step rounded to f32
        half_t ep;
        if constexpr (ZP) {
          float v = (float)acc[c][e] * (float)sw[c][e];
          v = v * sa;
          const float z = (float)sz[c][e] * as;
          ep = (half_t)rounded_f32(v - z);
        } else {
          const float sc = (float)sw[c][e] * sa;
          ep = (half_t)rounded_f32((float)acc[c][e] * sc);
        }
        o[e] = (half_t)((float)a[c][e] + (float)ep);
        x[c][e] = (float)o[e];
      }
      res.put(at, 2048 * c, o);
    }
  }
  template <int C>
  __device__ __forceinline__ void values(int row, int p, v2h (&g)[C], float (&x)[C][2]) const {
    const uint32_t at = 4 * p;      // bytes of a pair of halves
    switch (s.sk) {
      case 1: return values_of<C, 1>(row, at, g, x);
      case 2: return values_of<C, 2>(row, at, g, x);
      case 3: return values_of<C, 3>(row, at, g, x);
      case 4: return values_of<C, 4>(row, at, g, x);
      case 5: return values_of<C, 5>(row, at, g, x);
      case 6: return values_of<C, 6>(row, at, g, x);
      case 7: return values_of<C, 7>(row, at, g, x);
      case 8: return values_of<C, 8>(row, at, g, x);
      default: return values_of<C, MANY_SLABS<C>>(row, at, g, x);
    }
  }
};

struct PairAdd {      // residual += delta
  half_t* res;
  const half_t* delta;
  __device__ __forceinline__ void pin() const { asm volatile("" ::"s"(res), "s"(delta)); }
  template <int C>
  __device__ __forceinline__ void values(int row, int p, v2h (&g)[C], float (&x)[C][2]) const {
    const RowArray r(res + (size_t)row * (1024 * C)), d(delta + (size_t)row * (1024 * C));
    const uint32_t at = 4 * p;
    v2h a[C], b[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      a[c] = r.pair(at, 2048 * c);
      b[c] = d.pair(at, 2048 * c);
    }
    arrived(g);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      v2h o;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        o[e] = (half_t)((float)a[c][e] + (float)b[c][e]);
        x[c][e] = (float)o[e];
      }
      r.put(at, 2048 * c, o);
    }
  }
};

struct PairPlain {
  const half_t* in;
  __device__ __forceinline__ void pin() const { asm volatile("" ::"s"(in)); }
  template <int C>
  __device__ __forceinline__ void values(int row, int p, v2h (&g)[C], float (&x)[C][2]) const {
    const RowArray r(in + (size_t)row * (1024 * C));
    v2h a[C];
#pragma unroll
    for (int c = 0; c < C; ++c) a[c] = r.pair(4 * p, 2048 * c);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int e = 0; e < 2; ++e) x[c][e] = (float)a[c][e];
  }
};

template <int C, bool FUSE_SUM, typename Src>
__global__ __launch_bounds__(512) void norm_pairs_kernel(int8_t* __restrict__ out, Src src, const half_t* __restrict__ gamma, half_t* __restrict__ sum_out,
                                                         half_t* __restrict__ scale_out, float eps, PrefetchArgs pf) {
  constexpr int H = 1024 * C;
  __shared__ __attribute__((aligned(16))) float lds[8 * 256];      // 1 KiB a wave for fetching workgroups; a row's uses the first PAIR_RED words
  // one batch of scalar loads for the test below and the row's path
  src.pin();
  asm volatile("" ::"s"(out), "s"(gamma), "s"(sum_out), "s"(scale_out), "s"(eps), "s"(pf.blocks), "s"(pf.first_block));
  if (pf.blocks > 0 && (int)blockIdx.x >= pf.first_block) {      // extra workgroups: the next product's weights into L2
    prefetch_weights_to_l2(pf, lds);
    return;
  }
  const int p = threadIdx.x, row = blockIdx.x;
  const RowArray gains(gamma);
  v2h g[C];
#pragma unroll
  for (int c = 0; c < C; ++c) g[c] = gains.pair(4 * p, 2048 * c);
  float x[C][2];
  src.template values<C>(row, p, g, x);

  const PairPlace place(p);
  pair_sums<C>(x, lds, place);
  lds_barrier();
  pair_normalise<C, FUSE_SUM>(x, g, eps, lds, place);
  lds_barrier();
  const float amax = pair_top(lds, place);
  if (p == 0) scale_out[row] = (half_t)(amax / 127.0f);
  const float q = 127.0f / amax;
  const RowArray codes(out + (size_t)row * H);
#pragma unroll
  for (int c = 0; c < C; ++c) codes.put16(2 * p, 1024 * c, pair_codes(x[c], q));
  if constexpr (FUSE_SUM) {
    const half_t tot = pair_total(lds, place);
    if (p == 0) sum_out[row] = tot;
  }
}

template <bool FUSE_SUM, typename Src>
static void launch_pairs(const NormOut& o, const Src& src, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st) {
  const dim3 grid(tokens + pf.blocks), block(512);
  switch (hidden >> 10) {
#define OMNI_NORM_PAIRS(C_) \
  case C_: hipLaunchKernelGGL((norm_pairs_kernel<C_, FUSE_SUM, Src>), grid, block, 0, st, o.out, src, o.gamma, o.sum, o.scale, o.eps, pf); break
    OMNI_NORM_PAIRS(1);
    OMNI_NORM_PAIRS(2);
    OMNI_NORM_PAIRS(3);
    OMNI_NORM_PAIRS(4);
    OMNI_NORM_PAIRS(5);
    OMNI_NORM_PAIRS(6);
    OMNI_NORM_PAIRS(7);
    OMNI_NORM_PAIRS(8);
#undef OMNI_NORM_PAIRS
  }
}
template <typename Src>
static void launch_pairs(const NormOut& o, const Src& src, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st) {
  if (o.sum) launch_pairs<true>(o, src, tokens, hidden, pf, st);
  else launch_pairs<false>(o, src, tokens, hidden, pf, st);
}

void norm_pairs_slabs(const NormOut& o, const NormSlabs& s, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st) {
  if (s.wsz) launch_pairs<true>(o, PairSlabs<true>{s}, tokens, hidden, pf, st);
  else launch_pairs(o, PairSlabs<false>{s}, tokens, hidden, pf, st);
}
void norm_pairs_add(const NormOut& o, half_t* res, const half_t* delta, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st) {
  launch_pairs(o, PairAdd{res, delta}, tokens, hidden, pf, st);
}
void norm_pairs_plain(const NormOut& o, const half_t* in, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st) {
  launch_pairs(o, PairPlain{in}, tokens, hidden, pf, st);
}

}  // namespace omni
