// Prompts' gate_up with silu_and_mul in the product's tiles.  A file, and with it a code object, of its own: beside the decode kernels of qgemm_chn.hip a step of 16
// sequences takes 514.3 us for 513.0 (two runs of one side differ by 0.1 %; by what the place of the code makes a difference is not known).
#include "qgemm_kernel.h"
#include "qgemm_group_tiles.h"
using namespace omni;

// out = silu(gate) up fp16 [M, N/2], bit for bit what the product and silu_and_mul leave, in the products' own tiles.
template <int MODE>
static int launch_gemm_silu_rows(GemmArgs a, TileShare share, hipStream_t st) {
  GemmPlan pl;
  PrefillPlan pp;
  if (!silu_rows_plan(a.M, a.N, a.K, MODE, share_fits(&share, a.M, a.N, a.K), &pl, &pp)) return OMNI_EINVAL;
  a.kslice = pl.kslice;
  if (!pp.share) share = TileShare{};
  if (!exact_shape(a, false)) return OMNI_EINVAL;
  if constexpr (MODE == MODE_W8) {
    launch_tiles<MODE, true>(a, share, st);
  } else {
    const bool tiles = pp.w4_tiles;
    if (tiles && MODE == MODE_GRP && ((reinterpret_cast<uintptr_t>(a.s2s) | reinterpret_cast<uintptr_t>(a.s2z)) & 3) != 0) return OMNI_EINVAL;
    if (tiles) launch_w4_tiles_as<MODE, true>(a, share, st);
    else launch_exact_rows<MODE, 1, false, true>(a, pp.mb, 1, st);
  }
  return omni_launch_status();
}

extern "C" int omni_w4a8_per_chn_gemm_silu_rows(const void* in_feats, const void* qweight, const void* wscales, const void* ascales, const void* w_szs,
                                                const void* a_ssums, void* act_f16, int M, int N, int K, void* stream) {
  const TileShare share = take_armed_share();             // (first: an early return must not leave it armed)
  if (!in_feats || !qweight || !wscales || !ascales || !w_szs || !a_ssums || !act_f16) return OMNI_EINVAL;
  GemmArgs a{};
  a.A = (const int8_t*)in_feats; a.W = (const uint8_t*)qweight;
  a.wscales = (const half_t*)wscales; a.ascales = (const half_t*)ascales;
  a.wsz = (const half_t*)w_szs; a.asum = (const half_t*)a_ssums;
  a.out = (half_t*)act_f16; a.M = M; a.N = N; a.K = K; a.out_stride = N / 2;
  return launch_gemm_silu_rows<MODE_CHN>(a, share, (hipStream_t)stream);
}

extern "C" int omni_w4a8_per_group_gemm_silu_rows(const void* in_feats, const void* qweight, const void* zeros, const void* scales_i8, const void* wscales,
                                                  const void* ascales, void* act_f16, int M, int N, int K, void* stream) {
  const TileShare share = take_armed_share();             // (first: an early return must not leave it armed)
  if (!in_feats || !qweight || !zeros || !scales_i8 || !wscales || !ascales || !act_f16) return OMNI_EINVAL;
  GemmArgs a{};
  a.A = (const int8_t*)in_feats; a.W = (const uint8_t*)qweight;
  a.s2s = (const uint8_t*)scales_i8; a.s2z = (const uint8_t*)zeros;
  a.wscales = (const half_t*)wscales; a.ascales = (const half_t*)ascales;
  a.out = (half_t*)act_f16; a.M = M; a.N = N; a.K = K; a.out_stride = N / 2;
  return launch_gemm_silu_rows<MODE_GRP>(a, share, (hipStream_t)stream);
}

extern "C" int omni_w8a8_gemm_silu_rows(const void* in_feats, const void* weight, const void* wscales, const void* ascales, void* act_f16, int M, int N, int K,
                                        void* stream) {
  const TileShare share = take_armed_share();             // (first: an early return must not leave it armed)
  if (!in_feats || !weight || !wscales || !ascales || !act_f16) return OMNI_EINVAL;
  GemmArgs a{};
  a.A = (const int8_t*)in_feats; a.W = (const uint8_t*)weight;
  a.wscales = (const half_t*)wscales; a.ascales = (const half_t*)ascales;
  a.out = (half_t*)act_f16; a.M = M; a.N = N; a.K = K; a.out_stride = N / 2;
  return launch_gemm_silu_rows<MODE_W8>(a, share, (hipStream_t)stream);
}
