// o_proj / down_proj of one or two rows from fp16 activations and their row maxima to int32 K slabs: what omni_*_gemm_partial_f16 (the few-row GEMV's A16
// form, qgemm_kernel.h) does for up to 16, in other slices.
//
// A row or two leave the matrix instructions idle and the GEMV is a stream of weights; what bounds it is how evenly the compute units stream.  Its plan for
// 16 rows gives down_proj of the 8B model 448 workgroups of 64 x 2048 (W8A8: 896 of 64 x 1024) -- 1.75 (3.5) for a compute unit -- and a slab for
// each K slice, which the norm behind it reads back.  Here a workgroup is 64 channels of 8 waves (row_product.h) and as many K slices as make the
// grid the chip: 256 workgroups of 64 x 3584, half as many slabs.  The activations' part of a slice becomes codes once for all waves, in front of the weights.
//
// One more workgroup a row leaves its scale and, with zero points, its sum in the reference's order of additions (fused_kernels.cu:108-127: 1024 virtual
// threads; norm_pairs.h).
//
// MI355X, 8B model, 1 row, the GEMV -> this: down_proj W4A8 8.7 -> 7.5 us, W8A8 15.3 -> 13.4 (its 4 slabs instead of 14: qkv behind them 11.7 -> 10.1);
// o_proj W8A8 5.8 -> 5.2.
#include "row_product.h"

namespace omni {

template <int MODE, int UNITS, int ROWS, bool NT>
__global__ __launch_bounds__(RP_THREADS, 2) void act_product_kernel(GemmArgs p, int slices) {
  constexpr int KS = 512 * UNITS, KPART = 64 * UNITS, PITCH = KS + 64;
  typedef RowProduct<MODE, LAYOUT_ROWS64, 4, KPART, 8, ROWS, NT> Product;      // a wave's whole part flies
  constexpr int LDS_PARTS = ROWS * PITCH;
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_PARTS + Product::PART_BYTES];
  asm volatile("" ::"s"(p.A16), "s"(p.W), "s"(p.amax), "s"(p.N), "s"(p.K), "s"(p.slab), "s"(slices));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int groups = p.N / 64, id = blockIdx.x;

  if (id >= groups * slices) {      // a row's scale and sum
    const int row = id - groups * slices;
    const float top = amax_rows_wave(p.amax);
    if (tid == row) p.scale_out[row] = (half_t)(top / 127.0f);
    if (!p.sum_out) return;
    const RowArray x(p.A16 + (size_t)row * p.K);
    float s[2] = {0.0f, 0.0f};
#pragma unroll 4
    for (int c = 0; c < p.K / 1024; ++c) {
      const v2h v = x.pair(4 * tid, 2048 * c);
#pragma unroll
      for (int e = 0; e < 2; ++e) s[e] = s[e] + (float)v[e];
    }
    const int vw = 4 * wave + (lane >> 4);
    float* const red = reinterpret_cast<float*>(lds);
    const float w = row16_sum(s[0]) + row16_sum(s[1]);
    if ((lane & 15) == 0) red[(vw & 15) * 2 + (vw >> 4)] = w;
    lds_barrier();
    const float tot = row16_sum(red[(lane & 15) * 2] + red[(lane & 15) * 2 + 1]);
    if (tid == 0) p.sum_out[row] = (half_t)tot;
    return;
  }

  const int slice = id / groups, ng = id - slice * groups, k0 = slice * KS;
  const AmaxRaw raw = amax_rows_issue(p.amax);
  constexpr int PIECES = ROWS * KS / 8, PER = (PIECES + RP_THREADS - 1) / RP_THREADS;      // of 8 values
  uint4 x[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = min(tid + i * RP_THREADS, PIECES - 1), m = at / (KS / 8);
    x[i] = *reinterpret_cast<const uint4*>(p.A16 + (size_t)m * p.K + k0 + 8 * (at - m * (KS / 8)));
  }
  Product product;
  product.open(p.W, p.s2s, p.s2z, p.N, p.K, 4 * ng, k0 + wave * KPART);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < Product::RING; ++u) product.request(u);
  __builtin_amdgcn_sched_barrier(0);
  const float q_row = quant_multiplier(amax_rows_finish(raw));      // of row (lane & 15)
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = tid + i * RP_THREADS, m = at / (KS / 8), k = 8 * (at - m * (KS / 8));
    const float q = ROWS == 1 ? __shfl(q_row, 0, 64) : __shfl(q_row, min(m, ROWS - 1), 64);
    if (at < PIECES) {
      uint8_t* const c = lds + m * PITCH;
      *reinterpret_cast<uint32_t*>(c + code_place<MODE>(k)) = quant4_f16(x[i].x, x[i].y, q);
      *reinterpret_cast<uint32_t*>(c + code_place<MODE>(k + 4)) = quant4_f16(x[i].z, x[i].w, q);
    }
  }
  lds_barrier();
  product.multiply(lds + wave * KPART, PITCH);
  uint8_t* const parts = lds + LDS_PARTS;
  product.leave(parts, wave);
  lds_barrier();
  if (wave < ROWS) {
    const int b = lane >> 4, r = lane & 15;
    const int n = MODE == MODE_W8 ? lane : (r >> 3) * 32 + b * 8 + (r & 7);
    p.slab[((size_t)slice * ROWS + wave) * p.N + ng * 64 + n] = Product::total(parts, b, r, wave);
  }
}

template <int MODE, int UNITS, bool NT>
static void launch(const GemmArgs& p, int slices, hipStream_t st) {
  const dim3 grid(p.N / 64 * slices + p.M), block(RP_THREADS);
  if constexpr (MODE != MODE_W8) {
    if (p.M == 2) {
      hipLaunchKernelGGL((act_product_kernel<MODE, UNITS, 2, NT>), grid, block, 0, st, p, slices);
      return;
    }
  }
  hipLaunchKernelGGL((act_product_kernel<MODE, UNITS, 1, NT>), grid, block, 0, st, p, slices);
}
template <int MODE, bool NT>
static void launch(const GemmArgs& p, int slices, hipStream_t st) {
  switch (p.K / (512 * slices)) {
    case 1: launch<MODE, 1, NT>(p, slices, st); break;
    case 2: launch<MODE, 2, NT>(p, slices, st); break;
    case 3: launch<MODE, 3, NT>(p, slices, st); break;
    case 4: launch<MODE, 4, NT>(p, slices, st); break;
    case 5: launch<MODE, 5, NT>(p, slices, st); break;
    case 6: launch<MODE, 6, NT>(p, slices, st); break;
    case 7: launch<MODE, 7, NT>(p, slices, st); break;
    default: launch<MODE, 8, NT>(p, slices, st); break;
  }
}

// Slices: of whole 512s (8 waves of whole k-steps), eight k-steps a wave at most, so many that the workgroups of 64 channels are the chip's 256 or come
// nearest below, but 8 KiB of weights a wave at least: more slices cost the norm behind them more than they gain here (o_proj of the 8B model, W4A8, in
// 4 slices 4.6 us and gate_up 14.7, in 2 4.7 and 13.7).  Rows of whole 1024s (the order of a row's sum).
int act_product_slices(int M, int N, int K, int mode) {
  if (mode < 0 || mode > 2 || M < 1 || M > (mode == MODE_W8 ? 1 : 2) || N % 64 || N < 64 || N > 64 * 256 || K < 1024 || K % 1024) return 0;
  const int least = mode == MODE_W8 ? 2 : 4;
  for (int s = std::min(256 / (N / 64), 16); s >= 1; --s)
    if (K % (512 * s) == 0 && (s == 1 || K / (512 * s) >= least)) return K / (512 * s) <= 8 ? s : 0;
  return 0;
}

}  // namespace omni
using namespace omni;

extern "C" int omni_act_product_slices(int M, int N, int K, int mode) { return act_product_slices(M, N, K, mode); }

extern "C" int omni_act_product(int mode, const void* act_f16, const void* amax_slots_u32, const void* weight, const void* zeros_i8, const void* scales_i8,
                                void* slab_i32, size_t slab_bytes, void* sum_f16, void* scale_f16, int M, int N, int K, void* stream) {
  const int slices = act_product_slices(M, N, K, mode);
  if (!act_f16 || !amax_slots_u32 || !weight || !slab_i32 || !scale_f16 || !slices || (mode == MODE_GRP && (!zeros_i8 || !scales_i8))) return OMNI_EINVAL;
  if ((reinterpret_cast<uintptr_t>(act_f16) | reinterpret_cast<uintptr_t>(weight)) & 15) return OMNI_EINVAL;
  if (slab_bytes < (size_t)slices * M * N * sizeof(int32_t)) return OMNI_ENOMEM;
  GemmArgs a{};
  a.A16 = (const half_t*)act_f16; a.amax = (uint32_t*)amax_slots_u32; a.W = (const uint8_t*)weight;
  a.s2s = (const uint8_t*)scales_i8; a.s2z = (const uint8_t*)zeros_i8;
  a.sum_out = (half_t*)sum_f16; a.scale_out = (half_t*)scale_f16; a.slab = (int32_t*)slab_i32;
  a.M = M; a.N = N; a.K = K;
  const bool nt = !take_prefetched_weight(weight);
  hipStream_t st = (hipStream_t)stream;
  if (mode == MODE_W8) launch<MODE_W8, false>(a, slices, st);
  else if (mode == MODE_CHN) nt ? launch<MODE_CHN, true>(a, slices, st) : launch<MODE_CHN, false>(a, slices, st);
  else nt ? launch<MODE_GRP, true>(a, slices, st) : launch<MODE_GRP, false>(a, slices, st);
  return omni_launch_status();
}
