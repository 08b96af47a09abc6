// residual += the product before, norm, quantisation and the next product as ONE launch, for one or two rows: the decode layer's two edges
// input_layernorm -> qkv_proj and post_attention_layernorm -> gate_up_proj (+ silu_and_mul) (reference: llama_w4a8_unpad.py:410-432).
//
// As two launches (norm_rows.hip, then the GEMV) one compute unit works through the row for 6 us while the others wait, and only then are the product's
// first weights requested.  Handing the row over inside a launch costs what the boundary between two does (norm_gemv_fused.h).  But a row or two
// are little enough for EVERY workgroup of the product to form by itself: 50 - 200 KiB of slabs out of its L2, requested in front of the first
// weights, so that the whole chain -- requests, two reductions, codes -- passes while the weights are on their way, and nothing waits for
// another workgroup.  Each row's codes, scale and sum are the bits that the two launches give (norm_pairs.h: the same additions in the same order).
//
//  * the product is row_product.h's.  gate_up: 32 gate channels and their 32 up channels a workgroup (twice as many, so that a compute unit has one of
//    224 workgroups and the others fetch down_proj's weights: the same 14 us, and down gains what this loses).
//  * qkv: 32 channels a workgroup, so that 6144 channels make 192 workgroups instead of 96.
//  * the new residual goes to a buffer of its own (workgroup 0 stores it): other workgroups still read the old one.
//
// MI355X, 8B model, us a layer, two launches -> one: W4A8 1 row qkv 6.5 + 5.5 -> 6.7, gate_up 6.5 + 12.0 -> 13.7 (down_proj, whose weights the norm
// no longer fetches, 6.8 -> 8.7); the step of 8 layers 472 -> 419 us, 2 rows 511 -> 490; with groups of 128 604 -> 500 and 620 -> 557.  W8A8 1
// row: gate_up 6.5 + 24.5 -> 27.3; four LServe steps of 4 layers 2037 -> 1818.  Two rows
// gain little enough that more are left to the two launches.
#include "row_product.h"

namespace omni {

struct NormProductArgs {
  const half_t* res;
  half_t* res_out;          // with slabs
  const int32_t* slab;      // [sk][M][K]
  int sk;
  const half_t *p_wscales, *p_wsz, *p_ascales, *p_asum;
  const half_t* gamma;
  float eps;
  const uint8_t *W, *s2s, *s2z;
  const half_t *wscales, *wsz;
  half_t* out;
  uint32_t* amax;
  long long out_stride;
  int M, N;
};

// C: K / 1024.  SK: slabs whose requests go out together (those beyond sk read slab 0 again, so there are forms for 2, 4, 8 and 16: qkv of 12288 channels behind one slab of two
// rows in the form for 8, 1048 us a step of 16 layers of 4096 / 11008, 921 in that for 2; the 8B model's step of 16 layers behind 4, 1 and 2 rows, 680 -> 662 and 782 -> 750); 0: the
// residual as it is.  ROWS: M.
template <int MODE, int EPI, int BLOCKS, int C, int SK, int ROWS>
struct NormProduct {
  constexpr static int K = 1024 * C, PITCH = K + 64, PART_BYTES = RowProduct<MODE, EPI ? LAYOUT_GATE : LAYOUT_ROWS32, BLOCKS, K / RP_WAVES, 1, ROWS>::PART_BYTES;
  constexpr static int LDS_BYTES = ROWS * PITCH + PART_BYTES + ROWS * 512;
};

// first: the workgroup's first operand block of all; ng: its place in the grid
template <int MODE, int EPI, int BLOCKS, int C, int SK, int ROWS>
__device__ __forceinline__ void norm_product(const NormProductArgs& p, uint8_t* lds, int first, int ng) {
  constexpr bool ZP = MODE == MODE_CHN, W8 = MODE == MODE_W8;
  constexpr int K = 1024 * C, KPART = K / RP_WAVES;
  // units requested in front of the rows' first wait, and (the slabs' registers are free then) all that fly together
  constexpr bool WIDE = ROWS * SK * C > 16;
  constexpr int FIRST_MAX = W8 ? (EPI ? 1 : 2) : EPI && WIDE ? 3 : 4, RING_MAX = W8 ? 2 : FIRST_MAX;
  typedef RowProduct<MODE, EPI ? LAYOUT_GATE : LAYOUT_ROWS32, BLOCKS, KPART, RING_MAX, ROWS> Product;
  constexpr int FIRST = FIRST_MAX < Product::RING ? FIRST_MAX : Product::RING;
  constexpr int PITCH = K + 64;
  constexpr int LDS_PARTS = ROWS * PITCH, LDS_RED = LDS_PARTS + Product::PART_BYTES;
  uint8_t* const codes = lds;
  uint8_t* const parts = lds + LDS_PARTS;
  float (*red)[128] = reinterpret_cast<float (*)[128]>(lds + LDS_RED);
  asm volatile("" ::"s"(p.res), "s"(p.slab), "s"(p.sk), "s"(p.p_wscales), "s"(p.p_wsz), "s"(p.p_ascales), "s"(p.p_asum), "s"(p.gamma), "s"(p.W),
               "s"(p.wscales), "s"(p.wsz), "s"(p.N));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t at = 4 * tid;

  // ---- requests: the rows ----
  v2h g[C], a[ROWS][C], sw[C], sz[C];
  v2i t[ROWS][SK ? SK : 1][C];
  half_t sa_h[ROWS], as_h[ROWS];
  {
    const RowArray gains(p.gamma), ws(p.p_wscales), wz(p.p_wsz);
#pragma unroll
    for (int m = 0; m < ROWS; ++m) {
      if constexpr (SK > 0) {
        const RowArray slab(p.slab + (size_t)m * K);
        const uint32_t step = ROWS * K * 4;
#pragma unroll
        for (int k = 0; k < SK; ++k)
#pragma unroll
          for (int c = 0; c < C; ++c) t[m][k][c] = slab.two(2 * at, (k < p.sk ? k * step : 0) + 4096 * c);
        sa_h[m] = p.p_ascales[m];
        if constexpr (ZP) as_h[m] = p.p_asum[m];
      }
      const RowArray res(p.res + (size_t)m * K);
#pragma unroll
      for (int c = 0; c < C; ++c) a[m][c] = res.pair(at, 2048 * c);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (SK > 0) {
        sw[c] = ws.pair(at, 2048 * c);
        if constexpr (ZP) sz[c] = wz.pair(at, 2048 * c);
      }
      g[c] = gains.pair(at, 2048 * c);
    }
  }
  // ---- ... the scales of the channel that this lane finishes ----
  int chan;
  const int block = min(lane >> 4, BLOCKS - 1);
  if constexpr (EPI) chan = ((lane >> 3) & 1) * (p.N / 2) + (first + block) * 8 + (lane & 7);
  else chan = ng * 32 + (lane & 31);
  const half_t sw_own = p.wscales[chan];
  half_t sz_own = (half_t)0.0f;
  if constexpr (ZP) sz_own = p.wsz[chan];
  // ---- ... and the weights ----
  Product product;
  product.open(p.W, p.s2s, p.s2z, p.N, K, first, wave * KPART);
  __builtin_amdgcn_sched_barrier(0);      // what the rows need returns first: loads return in order
#pragma unroll
  for (int u = 0; u < FIRST; ++u) product.request(u);
  __builtin_amdgcn_sched_barrier(0);

  // ---- the rows ----
  float x[ROWS][C][2];
  v2h o[ROWS][C];
#pragma unroll
  for (int m = 0; m < ROWS; ++m)
#pragma unroll
    for (int c = 0; c < C; ++c) {
      o[m][c] = a[m][c];
      if constexpr (SK > 0) {
        v2i acc = t[m][0][c];
#pragma unroll
        for (int k = 1; k < SK; ++k) acc += k < p.sk ? t[m][k][c] : (v2i){0, 0};
        const float sa = (float)sa_h[m];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          half_t ep;
          if constexpr (ZP) ep = epilogue<MODE_CHN>(acc[e], (float)sw[c][e], sa, (float)sz[c][e], (float)as_h[m]);
          else ep = epilogue<MODE_W8>(acc[e], (float)sw[c][e], sa, 0.0f, 0.0f);
          o[m][c][e] = (half_t)((float)a[m][c][e] + (float)ep);
        }
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) x[m][c][e] = (float)o[m][c][e];
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = FIRST; u < Product::RING; ++u) product.request(u);
  __builtin_amdgcn_sched_barrier(0);
  const PairPlace place(tid);
#pragma unroll
  for (int m = 0; m < ROWS; ++m) pair_sums<C>(x[m], red[m], place);
  lds_barrier();
#pragma unroll
  for (int m = 0; m < ROWS; ++m) pair_normalise<C, ZP>(x[m], g, p.eps, red[m], place);
  lds_barrier();
  float row_scale[ROWS], row_sum[ROWS];
#pragma unroll
  for (int m = 0; m < ROWS; ++m) {
    const float amax = pair_top(red[m], place);
    row_scale[m] = (float)(half_t)(amax / 127.0f);
    row_sum[m] = 0.0f;
    if constexpr (ZP) row_sum[m] = (float)pair_total(red[m], place);
    const float q = 127.0f / amax;
#pragma unroll
    for (int c = 0; c < C; ++c) *reinterpret_cast<uint16_t*>(codes + m * PITCH + code_place<MODE>(1024 * c + 2 * tid)) = pair_codes(x[m][c], q);
  }
  lds_barrier();

  product.multiply(codes + wave * KPART, PITCH);
  product.leave(parts, wave);
  lds_barrier();
  if (wave < ROWS) {      // (a wave finishes a row, a lane a channel)
    const int m = wave;
    float scale = row_scale[0], sum = row_sum[0];
#pragma unroll
    for (int i = 1; i < ROWS; ++i)
      if (m == i) {
        scale = row_scale[i];
        sum = row_sum[i];
      }
    int total;
    if constexpr (EPI) total = Product::total(parts, block, lane & 15, m);
    else if constexpr (W8) total = Product::total(parts, (lane >> 4) & 1, lane & 15, m);
    else total = Product::total(parts, (lane >> 3) & 3, (lane & 7) + 8 * (lane >> 5), 2 * m + (lane >> 5));
    if constexpr (Product::PAIRED) total += __shfl_xor(total, 32, 64);
    const half_t h = epilogue<MODE == MODE_GRP ? MODE_W8 : MODE>(total, (float)sw_own, scale, (float)sz_own, sum);
    half_t* const out = p.out + (size_t)m * p.out_stride;
    if constexpr (EPI) {
      const int up = __shfl_xor((int)__builtin_bit_cast(uint16_t, h), 8, 64);
      const half_t act = silu_mul_h(h, __builtin_bit_cast(half_t, (uint16_t)up));      // (of lanes with a gate channel)
      const bool gate = !(lane & 8) && (lane >> 4) < BLOCKS;
      if (gate) out[chan] = act;
      const float top = wave_max64(gate ? __builtin_fabsf((float)act) : 0.0f);
      if (lane == 0) amax_raise(p.amax, m, ng >> 3, top);
    } else if (lane < 32) {
      out[chan] = h;
    }
  }
  if constexpr (SK > 0) {
    if (ng == 0) {
#pragma unroll
      for (int m = 0; m < ROWS; ++m)
#pragma unroll
        for (int c = 0; c < C; ++c) RowArray(p.res_out + (size_t)m * K).put(at, 2048 * c, o[m][c]);
    }
  }
}

template <int MODE, int EPI, int BLOCKS, int C, int SK, int ROWS>
__global__ __launch_bounds__(RP_THREADS, EPI ? 4 : 2) void norm_product_kernel(NormProductArgs p) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[NormProduct<MODE, EPI, BLOCKS, C, SK, ROWS>::LDS_BYTES];
  norm_product<MODE, EPI, BLOCKS, C, SK, ROWS>(p, lds, (int)blockIdx.x * BLOCKS, blockIdx.x);
}

// gate_up of int8 weights in two workgroups a compute unit: the first `wide` of them take four blocks of eight gate and eight up channels, the others three.  448
// workgroups of four leave a quarter of the units with one, and a unit takes in its weights at a rate of its own.  (MI355X, 28672 x
// 4096: four LServe steps of 4 layers 1607 -> 1585 us.  Packed weights hold two blocks in a byte and cannot be dealt in threes.  Where: more than three blocks for each of the 512, but not
// so many that few units are left with one.  Workgroups of four / this, us, one slab, weights that no cache holds: 24704 x 4096 26.3 / 23.4, 28672 26.7 / 25.2, 29696 27.3 / 27.2; 24704 x 2048 12.5 / 11.6,
// 28672 12.6 / 12.2, 29696 12.9 / 13.2, 30720 13.0 / 13.3.  Of weights in the last cache rows of 2048 take 10.4 / 11.2 at 26624; a step's come from memory.)
static int even_wide(int N) {      // the first that take four blocks, 0: all take four
  const int wide = N / 16 - 3 * 512;
  return wide > 0 && wide <= 256 ? wide : 0;
}
template <int C, int SK>
__global__ __launch_bounds__(RP_THREADS, 4) void gate_up_even_kernel(NormProductArgs p, int wide) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[NormProduct<MODE_W8, 1, 4, C, SK, 1>::LDS_BYTES];
  const int ng = blockIdx.x;
  if (ng < wide) norm_product<MODE_W8, 1, 4, C, SK, 1>(p, lds, 4 * ng, ng);
  else norm_product<MODE_W8, 1, 3, C, SK, 1>(p, lds, 3 * ng + wide, ng);
}

}  // namespace omni
using namespace omni;

namespace {

template <int MODE, int EPI, int BLOCKS, int C, int SK>
void launch_rows(const NormProductArgs& p, hipStream_t st) {
  const dim3 grid(EPI ? p.N / 64 : p.N / 32), block(RP_THREADS);
  if constexpr (MODE == MODE_W8 && EPI) {
    if (const int wide = even_wide(p.N)) {
      hipLaunchKernelGGL((gate_up_even_kernel<C, SK>), dim3(512), block, 0, st, p, wide);
      return;
    }
  }
  if constexpr (MODE != MODE_W8 && SK <= 8) {      // (two rows with int8 weights, or of 16 slabs, do not fit the registers)
    if (p.M == 2) {
      hipLaunchKernelGGL((norm_product_kernel<MODE, EPI, BLOCKS, C, SK, 2>), grid, block, 0, st, p);
      return;
    }
  }
  hipLaunchKernelGGL((norm_product_kernel<MODE, EPI, BLOCKS, C, SK, 1>), grid, block, 0, st, p);
}
template <int MODE, int C>
void launch_slabs(const NormProductArgs& p, hipStream_t st) {
  constexpr int CHANNELS32 = MODE == MODE_W8 ? 2 : 4;
  if (p.amax) {
    if (p.sk <= 2) launch_rows<MODE, 1, 4, C, 2>(p, st);
    else launch_rows<MODE, 1, 4, C, 4>(p, st);
  } else if (!p.slab) {
    launch_rows<MODE, 0, CHANNELS32, C, 0>(p, st);
  } else if (p.sk <= 2) {
    launch_rows<MODE, 0, CHANNELS32, C, 2>(p, st);
  } else if (p.sk <= 4) {
    launch_rows<MODE, 0, CHANNELS32, C, 4>(p, st);
  } else if (p.sk <= 8) {
    launch_rows<MODE, 0, CHANNELS32, C, 8>(p, st);
  } else {
    launch_rows<MODE, 0, CHANNELS32, C, 16>(p, st);
  }
}
template <int MODE>
int launch(const NormProductArgs& p, int K, hipStream_t st) {
  switch (K >> 10) {
    case 2: launch_slabs<MODE, 2>(p, st); break;
    case 3: launch_slabs<MODE, 3>(p, st); break;
    default: launch_slabs<MODE, 4>(p, st); break;
  }
  return omni_launch_status();
}

}  // namespace

static bool sizes_ok(int M, int N, int K, int mode, bool silu, int sk) {
  if (mode < 0 || mode > 2 || M < 1 || M > (mode == MODE_W8 ? 1 : 2) || K % 1024 || K < 2048 || K > 4096 || N < 64 || N % (silu ? 128 : 64)) return false;
  return silu ? sk >= 1 && sk <= 4 : sk >= 0 && sk <= (M == 1 ? 16 : 8);
}

extern "C" int omni_norm_product_workgroups(int M, int N, int K, int mode, int silu) {
  if (!sizes_ok(M, N, K, mode, silu != 0, 1)) return 0;
  if (mode == MODE_W8 && silu && even_wide(N)) return 512;
  return silu ? N / 64 : N / 32;
}

extern "C" int omni_norm_product_ok(int M, int N, int K, int mode, int silu, int k_before) {
  if (!sizes_ok(M, N, K, mode, silu != 0, 1)) return 0;
  const int kalign = mode == MODE_GRP ? 128 : 64;
  if (k_before == 0) return !silu;
  if (k_before < kalign || k_before % kalign) return 0;
  const int slices = act_product_slices(M, K, k_before, mode);
  return sizes_ok(M, N, K, mode, silu != 0, slices ? slices : plan_gemm(M, K, k_before, kalign, true, mode == MODE_W8).sk);
}

extern "C" int omni_norm_product(int mode, const void* residual_f16, void* residual_out_f16, const void* slab_i32, int sk, const void* p_wscales_f16,
                                 const void* p_ascales_f16, const void* p_wszs_f16, const void* p_asums_f16, const void* gamma_f16, float eps,
                                 const void* weight, const void* zeros_i8, const void* scales_i8, const void* wscales_f16, const void* w_szs_f16,
                                 void* out_f16, int64_t out_row_stride, void* amax_slots_u32, int M, int N, int K, void* stream) {
  if (!residual_f16 || !gamma_f16 || !weight || !wscales_f16 || !out_f16 || !sizes_ok(M, N, K, mode, amax_slots_u32 != nullptr, slab_i32 ? sk : 0))
    return OMNI_EINVAL;
  if (mode == MODE_CHN && !w_szs_f16) return OMNI_EINVAL;
  if (mode == MODE_GRP && (!zeros_i8 || !scales_i8)) return OMNI_EINVAL;
  if (slab_i32 && (sk < 1 || !p_wscales_f16 || !p_ascales_f16 || !residual_out_f16 || residual_out_f16 == residual_f16)) return OMNI_EINVAL;
  if (slab_i32 && mode == MODE_CHN && (!p_wszs_f16 || !p_asums_f16)) return OMNI_EINVAL;
  const NormProductArgs p{(const half_t*)residual_f16, (half_t*)residual_out_f16, (const int32_t*)slab_i32, sk, (const half_t*)p_wscales_f16,
                          (const half_t*)p_wszs_f16, (const half_t*)p_ascales_f16, (const half_t*)p_asums_f16, (const half_t*)gamma_f16, eps,
                          (const uint8_t*)weight, (const uint8_t*)scales_i8, (const uint8_t*)zeros_i8, (const half_t*)wscales_f16,
                          (const half_t*)w_szs_f16, (half_t*)out_f16, (uint32_t*)amax_slots_u32, out_row_stride, M, N};
  hipStream_t st = (hipStream_t)stream;
  if (mode == MODE_CHN) return launch<MODE_CHN>(p, K, st);
  return mode == MODE_GRP ? launch<MODE_GRP>(p, K, st) : launch<MODE_W8>(p, K, st);
}
