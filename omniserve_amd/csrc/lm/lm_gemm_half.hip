// Products of many rows in 256 x 128 tiles: for grids that 256 x 256 tiles (lm_gemm.hip) would leave too small for the chip.  A file, and with it a code
// object, of its own: in lm_gemm.hip's the few-row stream kernels lay differently and took 0.9 % longer (54.15 for 53.7 us of a step's experts).
#include "lm_gemm.h"

namespace lm {

constexpr int HROWB = 64, HK = HROWB / (int)sizeof(elem_t);  // a stage: 64 bytes of k of every row
constexpr int HSTAGE = (TM + HTN) * HROWB, HSTAGES = 3;

// LDS rows of 64 bytes, four 16-byte slots and four rows to a 256-byte line: slot s of row r at s ^ (0, 2, 3, 1)[r / 4 % 4], with
// the property Tile::swizzle has for fragment reads
__device__ __forceinline__ int stage_swizzle(int row) {
  const int q = (row >> 2) & 3;
  return (((q ^ (q >> 1)) & 1) << 1) | (q >> 1);
}

// 4 waves, 128 rows x 64 channels each; three stages: while one multiplies, two are on their way.  Two workgroups share a CU where there are enough.
// half_tiles() says where this one runs.
template <int EPI>
__global__ __launch_bounds__(256, 2) void gemm_half_tiles_kernel(GemmArgs p, int mt_a, int mt_b) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[HSTAGES * HSTAGE];
  __shared__ int y_row[TM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l15 = lane & 15, l4 = lane >> 4;
  // linear order: bands of row tiles, all channel tiles of a band before the next one; of both parts a contiguous range per XCD
  const int nt_a = (p.a.n + HTN - 1) / HTN, nt_b = mt_b ? (p.b.n + HTN - 1) / HTN : 0;
  const int wgs_b = 8 * ((mt_b * nt_b + 7) >> 3);
  const bool is_b = (int)blockIdx.x < wgs_b;
  const Part& pt = is_b ? p.b : p.a;
  const int nt = is_b ? nt_b : nt_a, mts = is_b ? mt_b : mt_a;
  const int id = xcd_contiguous(is_b ? blockIdx.x : blockIdx.x - wgs_b, mts * nt);
  if (id < 0) return;
  constexpr int GM = 4;
  const int band = id / (GM * nt), in = id - band * GM * nt, bm = min(GM, mts - band * GM);
  const int mi = band * GM + in % bm, ni = in / bm;
  const int* perm = is_b ? nullptr : p.perm;
  int first = mi * TM, rows, g = 0;
  if (perm) {
    const i32x4 t = *(const i32x4*)(p.tiles + 4 * mi);       // group, first place, rows
    if (t[2] <= 0) return;
    g = t[0];
    first = t[1];
    rows = t[2];
  } else {
    rows = min(TM, (is_b ? p.rows_b : p.rows_a) - first);
  }
  const int n0 = ni * HTN;
  const elem_t* w = pt.w + (int64_t)g * pt.n * pt.k;
  // pieces of 16 rows: lane -> (row lane / 4, physical slot lane % 4); a wave carries 2 of the weights' and 4 of x's
  const elem_t *wsrc[2], *xsrc[4];
  const int pr = lane >> 2, ps = (lane & 3) ^ stage_swizzle(pr);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = min(16 * (4 * wave + i) + pr, rows - 1);
    const int xr = perm ? perm[first + r] / p.x_div : first + r;
    xsrc[i] = pt.x + (int64_t)xr * pt.ldx + ps * FR;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) wsrc[i] = w + (int64_t)min(n0 + 16 * (2 * wave + i) + pr, pt.n - 1) * pt.k + ps * FR;
  y_row[tid] = tid < rows ? (perm ? perm[first + tid] : first + tid) : -1;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int uw = __builtin_amdgcn_readfirstlane(wave);
  auto stage = [&](int st, int k0) {
    const uint32_t dst = lds0 + st * HSTAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16_uncounted(wsrc[i] + k0, dst + 1024 * (2 * uw + i));
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16_uncounted(xsrc[i] + k0, dst + HTN * HROWB + 1024 * (4 * uw + i));
  };
  const int wn = 64 * (wave & 1), wm = 128 * (wave >> 1);
  f32x4 acc[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = zero4();
  const int nk = pt.k / HK;                                 // (>= 2: k is a multiple of 64)
  const int lane_off = l15 * HROWB + ((l4 ^ stage_swizzle(l15)) << 4);
  wait_pieces<0>();                                         // the compiler's own loads
  stage(0, 0);
  stage(1, HK);
  int st = 0;
  for (int t = 0; t < nk; ++t) {
    if (t + 1 < nk) wait_pieces<6>();                       // stage t is there, the 6 pieces of t + 1 may still fly
    else wait_pieces<0>();
    __builtin_amdgcn_s_barrier();                           // ... for every wave, and everyone has left stage t - 1
    asm volatile("" ::: "memory");
    if (t + 2 < nk) stage(st == 0 ? 2 : st - 1, (t + 2) * HK);
    const uint8_t* wt = lds + st * HSTAGE + wn * HROWB + lane_off;
    const uint8_t* xt = lds + st * HSTAGE + (HTN + wm) * HROWB + lane_off;
    frag_t a[4], b[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = *(const frag_t*)(wt + 16 * HROWB * i);
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = *(const frag_t*)(xt + 16 * HROWB * j);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i][j] = mma(a[i], b[j], acc[i][j]);
    __builtin_amdgcn_s_setprio(0);
    st = st == 2 ? 0 : st + 1;
  }
  __syncthreads();                                          // the stages are free
  if constexpr (EPI == LM_EPI_F32) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int row = y_row[wm + 16 * j + l15];
      if (row < 0) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = n0 + wn + 16 * i + 4 * l4;
        if (c < pt.n) store4<EPI>(pt, row, c, 0, acc[i][j], p.scale);
      }
    }
  } else {
    // through LDS, so that a row leaves in whole 16-byte pieces of neighbouring lanes: 32 rows of the wave's at a time
    constexpr int OC = EPI == LM_EPI_GLU ? 32 : 64, PITCH = OC * (int)sizeof(elem_t) + 16, PPR = OC / FR;
    static_assert(4 * 32 * PITCH <= HSTAGES * HSTAGE, "the waves' buffers");
    uint8_t* buf = lds + wave * 32 * PITCH;
#pragma unroll
    for (int part = 0; part < 4; ++part) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int j = 2 * part + jj;
#pragma unroll
        for (int i = 0; i < 4; i += EPI == LM_EPI_GLU ? 2 : 1) {
          f32x4 v = acc[i][j];
          int c = 16 * i;
          if constexpr (EPI == LM_EPI_GLU) {
            c = 8 * i;
            if (n0 + wn + 16 * i < pt.n) v = glu(pt, p.act, n0 + wn + 16 * i + 4 * l4, v, acc[i + 1][j]);
          }
          *(quad_t*)(buf + (16 * jj + l15) * PITCH + (c + 4 * l4) * (int)sizeof(elem_t)) = to_quad(v);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 32 * PPR / 64; ++i) {
        const int pc = 64 * i + lane, r = pc / PPR, q = pc % PPR;
        const int row = y_row[wm + 32 * part + r], c = (EPI == LM_EPI_GLU ? (n0 + wn) / 2 : n0 + wn) + q * FR;
        if (row >= 0 && c < (EPI == LM_EPI_GLU ? pt.n / 2 : pt.n))
          *(frag_t*)((elem_t*)pt.y + (int64_t)row * pt.ldy + c) = *(const frag_t*)(buf + r * PITCH + q * 16);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

void launch_half_tiles(const GemmArgs& a, int epi, unsigned wgs, int mt_a, int mt_b, hipStream_t s) {
  if (epi == LM_EPI_ELEM) hipLaunchKernelGGL((gemm_half_tiles_kernel<LM_EPI_ELEM>), dim3(wgs), dim3(256), 0, s, a, mt_a, mt_b);
  else if (epi == LM_EPI_F32) hipLaunchKernelGGL((gemm_half_tiles_kernel<LM_EPI_F32>), dim3(wgs), dim3(256), 0, s, a, mt_a, mt_b);
  else hipLaunchKernelGGL((gemm_half_tiles_kernel<LM_EPI_GLU>), dim3(wgs), dim3(256), 0, s, a, mt_a, mt_b);
}

}  // namespace lm
