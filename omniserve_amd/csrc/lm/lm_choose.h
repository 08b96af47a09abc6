// A token's experts: the `top` largest router logits (ties: the lower expert) and their softmax.
#pragma once
#include "lm_common.h"
#include "omniserve_lm.h"

namespace lm {

constexpr int MAX_EXPERTS = 512, MAX_TOP = LM_MAX_TOP;
// one wave per token; lane l holds its EPL experts l, l + 64, ... and counts for each how many come before it in the order
// (larger logit, then lower number): the first `top` are the choice
template <int EPL>
__device__ __forceinline__ void choose(const float* z, const float* bias, int experts, int top, int lane, int* ids, float* wts) {
  float v[EPL];
  int before[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    const int e = lane + 64 * i;
    const float x = e < experts ? z[e] + (bias ? bias[e] : 0.f) : -INFINITY;
    v[i] = x == x ? x : -INFINITY;        // (NaN: last)
    before[i] = 0;
  }
#pragma unroll
  for (int b = 0; b < EPL; ++b) {
    const int n = min(64, experts - 64 * b);
    for (int l = 0; l < n; ++l) {
      const float o = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[b]), l));
      const int oe = 64 * b + l;
#pragma unroll
      for (int i = 0; i < EPL; ++i) before[i] += (int)(o > v[i]) | ((int)(o == v[i]) & (int)(oe < lane + 64 * i));
    }
  }
  float best = v[0];
#pragma unroll
  for (int i = 1; i < EPL; ++i) best = fmaxf(best, v[i]);
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) best = fmaxf(best, __shfl_xor(best, m, 64));
  if (best == -INFINITY) best = 0.f;
  float ex[EPL], sum = 0.f;
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    ex[i] = before[i] < top ? __expf(v[i] - best) : 0.f;
    sum += ex[i];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int i = 0; i < EPL; ++i)
    if (before[i] < top && lane + 64 * i < experts) {
      ids[before[i]] = lane + 64 * i;
      wts[before[i]] = ex[i] / sum;
    }
}

}  // namespace lm
