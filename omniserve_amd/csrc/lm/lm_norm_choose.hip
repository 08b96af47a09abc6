// Few tokens in front of a mixture of experts: residual, norm, router product and expert choice in one launch, a workgroup per token.
//
// Each of the three launches was the latency of a launch, of its loads and of a few barriers, and two of them had one to four of 256 CUs.  Here the router's first
// stages are requested in front of the row's own loads and come in while the row is normed; its 256 KB pass through the workgroup's CU once, 2.9 us
// (every token's does that: they come from the L2; workgroups beside the tokens' that bring them there ahead changed nothing).  The order of the products is left
// to those who need it: a workgroup of lm_gemm_chosen finds its expert's pairs among the choices.
//
// MI355X, bf16, us, norm + router product + choice -> here: 16 tokens, 64 experts, width 2048 4.5 + 4.4 + 6.9 -> 9.8 (in a step of a model 18.6 -> 11.1), 32 tokens 4.5 + 5.2 + 11.5 ->
// 9.8, one 4.3 + 4.4 + 5.5 -> 9.6; 16 tokens, 32 experts, width 4096 5.5 + 6.6 + 4.9 -> 12.6.  A step's empty places choose nothing: 20 steps of
// a model of 6 such layers, 5 sequences in 8 places, 35.6 ms -> 34.6 by the launch and 33.2 by the experts that are not read.
//
// The logits' sums are those of gemm_stream_kernel with 16 channels and four K parts, one product and one addition after the other: a near tie
// between experts falls as it does there.
#include "lm_choose.h"
#include "lm_gemm.h"
#include "lm_residual.h"

namespace lm {

#if LM_ELEM == 0
constexpr int KPARTS = 4, STAGE_B = 128, SLICES = 8;      // K parts of a slice; bytes of k of a stage (of gemm_stream_kernel); slices at most

// NB: blocks of 16 experts.  Stage s belongs to K part s % 4; four stages (one of each part) are a group, a slot of the ring.
template <int TH, int NB>
__global__ __launch_bounds__(TH) void norm_choose_kernel(ResidualArgs p, const int* pos, const elem_t* router, const float* bias, int k, int slices, int experts, int top,
                                                         float* wts, int* ids) {
  constexpr int WAVES = TH / 64, STAGE = NB * 16 * STAGE_B, GROUP = KPARTS * STAGE, R = NB <= 2 ? 8 : 4;
  constexpr int PIECES = GROUP / 1024, P = (PIECES + WAVES - 1) / WAVES;      // of a group, and a wave's (some twice: the same bytes)
  constexpr int TASKS = NB * KPARTS, T = (TASKS + WAVES - 1) / WAVES;         // (block of experts, K part)
  typedef Tile<STAGE_B> Tl;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];               // ring, the row
  __shared__ float red[2 * WAVES], part[SLICES][KPARTS][16 * NB], z[64];
  __shared__ int count[WAVES][64];
  elem_t* const hrow = (elem_t*)(lds + R * GROUP);
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l15 = lane & 15, l4 = lane >> 4;
  if (pos && pos[r] < 0) {      // an empty place of a captured step: it chooses no expert, whose weights would be read for it
    if (tid < top) {
      ids[(int64_t)r * top + tid] = -1;
      wts[(int64_t)r * top + tid] = __builtin_bit_cast(float, LM_NO_EXPERTS_BITS);
    }
    return;
  }
  const uint32_t base = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int groups = k / (KPARTS * STAGE_B / (int)sizeof(elem_t)), own = groups / slices;      // own: of a slice
  // piece i of the wave: eight rows of a stage; lane -> (row lane / 8, slot lane % 8)
  const uint8_t* src[P];
  uint32_t dst[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int pc = (wave + WAVES * i) % PIECES, st = pc / (2 * NB), row = 8 * (pc % (2 * NB)) + (lane >> 3);
    src[i] = (const uint8_t*)(router + (int64_t)row * k) + st * STAGE_B + (((lane & 7) ^ Tl::swizzle(row & 15)) << 4);
    dst[i] = base + 1024 * pc;
  }
  auto request = [&](int g) {
#pragma unroll
    for (int i = 0; i < P; ++i) dma16_uncounted(src[i] + g * (KPARTS * STAGE_B), dst[i] + (g % R) * GROUP);
  };
#pragma unroll
  for (int g = 0; g < R - 1; ++g)
    if (g < groups) request(g);

  f32x4 x[1];
  Row<TH> sums{red};
  residual_row<TH, 1>(p, sums, r, x);
  const int c0 = 4 * tid;
  if (c0 < p.ldh) {
    const quad_t q = to_quad(x[0]);
    *(quad_t*)(p.h + (int64_t)r * p.ldh + c0) = q;
    *(quad_t*)(hrow + c0) = q;
  }

  // sums of 4 stages of a part and the sum of those, slice after slice
  f32x4 acc[T], total[T];
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = total[t] = zero4();
  int slice = 0, in = 0;
  auto multiply = [&](int g) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int task = wave + WAVES * t;
      if (TASKS % WAVES != 0 && task >= TASKS) continue;
      const int b = task / KPARTS, h = task % KPARTS;
      const uint8_t* wt = lds + (g % R) * GROUP + h * STAGE + b * (16 * STAGE_B);
      const elem_t* xt = hrow + (g * KPARTS + h) * (STAGE_B / (int)sizeof(elem_t));
#pragma unroll
      for (int v = 0; v < 2; ++v) acc[t] = mma(Tl::frag(wt, l15, 4 * v + l4), *(const frag_t*)(xt + (4 * v + l4) * FR), acc[t]);
      if ((in & 3) == 3) {
        total[t] += acc[t];
        acc[t] = zero4();
      }
      if (in == own - 1) {
        if (l15 == 0) *(f32x4*)&part[slice][h][16 * b + 4 * l4] = total[t] + acc[t];      // (every column is the token's)
        acc[t] = total[t] = zero4();
      }
    }
    if (++in == own) { in = 0; ++slice; }
  };
  // group g is there for every wave, and everyone has left the one before it, whose slot is filled next
  auto next = [&](auto behind) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(behind)::value * P) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  int g = 0;
  for (; g + R - 1 < groups; ++g) {
    next(Int<R - 2>{});
    request(g + R - 1);
    multiply(g);
  }
  countdown<R - 2>([&](auto behind) {
    constexpr int J = decltype(behind)::value;
    if (groups - 1 - J < 0) return;
    next(behind);
    multiply(groups - 1 - J);
  });
  __syncthreads();

  // The choice, as choose() makes it, by all waves: lane e of a wave counts which of the wave's share of the experts come before expert e.  (One wave over 64
  // experts, readlane after readlane: 2.9 us.)
  float v = -INFINITY;
  if (lane < experts) {
    float sum = 0.f;
    for (int i = 0; i < slices; ++i) {
      float u = part[i][0][lane];
#pragma unroll
      for (int h = 1; h < KPARTS; ++h) u += part[i][h][lane];
      sum += u;
    }
    sum += bias ? bias[lane] : 0.f;
    v = sum == sum ? sum : -INFINITY;        // (NaN: last)
  }
  constexpr int SHARE = 64 / WAVES;
  if (wave == 0) z[lane] = v;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int i = 0; i < SHARE; ++i) {
    const int oe = SHARE * wave + i;
    const float o = z[oe];
    before += (int)(oe < experts) & ((int)(o > v) | ((int)(o == v) & (int)(oe < lane)));
  }
  count[wave][lane] = before;
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 1; w < WAVES; ++w) before += count[w][lane];
  const int first = __builtin_ctzll(__builtin_amdgcn_ballot_w64(before == 0 && lane < experts));
  float best = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), first));
  if (best == -INFINITY) best = 0.f;
  const bool chosen = before < top && lane < experts;
  const float ex = before < top ? __expf(v - best) : 0.f;
  const float sum = wave_sum(ex);
  if (chosen) {
    ids[(int64_t)r * top + before] = lane;
    wts[(int64_t)r * top + before] = ex / sum;
  }
}

template <int TH, int NB>
static int launch_choose(const ResidualArgs& a, const int* pos, const elem_t* router, const float* bias, int k, int slices, int experts, int top, float* wts, int* ids, int tokens,
                         hipStream_t s) {
  const size_t lds = (size_t)(NB <= 2 ? 8 : 4) * KPARTS * NB * 16 * STAGE_B + (size_t)k * sizeof(elem_t);
  if (allow_lds(norm_choose_kernel<TH, NB>, lds)) return LM_EINVAL;
  hipLaunchKernelGGL((norm_choose_kernel<TH, NB>), dim3(tokens), dim3(TH), lds, s, a, pos, router, bias, k, slices, experts, top, wts, ids);
  return launch_status();
}
#endif

}  // namespace lm

using namespace lm;

// Sizes that it has: rows of 2048 - 4096 elements in multiples of 256 (a group of the ring: a stage of 64 of each of four K parts), of which every K slice has equally many
// groups, and up to 64 experts (512 KB and more would take longer through every token's CU than in launches of their own); the router's product as lm_gemm_rows deals it to
// 16 channels and four K parts.  Below 2048 of K that product adds its stages up in shorter chains, which are not built here; a row of 4096 is one piece of 1024 threads.
// K slices of the router's product, or 0: there is no such launch
static int choose_slices(int tokens, int k, int experts, int top) {
#if LM_ELEM == 0
  int slices = 0;
  if (tokens < 1 || tokens > LM_CHOOSE_TOKENS || experts < 1 || experts > 64 || top < 1 || top > MAX_TOP || top > experts || k < 2048 || k > 4096 || k % 256) return 0;
  if (lm_gemm_rows_channels(1, (experts + 15) / 16 * 16, k, tokens, LM_EPI_F32, 1, &slices) != 16 || slices > SLICES || (k / 256) % slices) return 0;
  return slices;
#else
  return 0;
#endif
}
extern "C" int lm_norm_choose_ok(int tokens, int k, int experts, int top) { return choose_slices(tokens, k, experts, top) > 0; }

extern "C" int lm_norm_choose(float* x, int64_t ldx, const void* y, int64_t ldy, const float* post_w, const float* post_b, const float* next_w, const float* next_b, void* h,
                              int64_t ldh, const int* pos, int tokens, int n, int kind, float eps, const void* router, const float* bias, int k, int experts, int top, float* wts, int* ids,
                              void* stream) {
#if LM_ELEM == 0
  const int slices = choose_slices(tokens, k, experts, top);
  if (slices == 0 || !x || !y || !next_w || !h || !router || !wts || !ids || n <= 0 || n > ldx || ldx % 4 || ldh != k || ldx > k || ldh < n || ldy % 4 ||
      ((uintptr_t)router | (uintptr_t)h) % 16)
    return LM_EINVAL;
  const ResidualArgs a{x, ldx, nullptr, nullptr, 1.f, (const elem_t*)y, ldy, nullptr, 0, 0, nullptr, nullptr, 0, 0, 0, post_w, post_b, next_w, next_b, (elem_t*)h, ldh, nullptr, n, kind, 1, eps};
  hipStream_t s = (hipStream_t)stream;
  const elem_t* rt = (const elem_t*)router;
  const int nb = (experts + 15) / 16;
#define LM_CASE(TH, NB) if (nb == NB && k <= 4 * TH) return launch_choose<TH, NB>(a, pos, rt, bias, k, slices, experts, top, wts, ids, tokens, s);
  LM_CASE(512, 1) LM_CASE(512, 2) LM_CASE(512, 3) LM_CASE(512, 4) LM_CASE(1024, 1) LM_CASE(1024, 2) LM_CASE(1024, 3) LM_CASE(1024, 4)
#undef LM_CASE
#endif
  return LM_EINVAL;
}
