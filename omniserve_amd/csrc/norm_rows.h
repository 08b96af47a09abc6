// Row norms of decode-size launches (norm_rows.hip): what elementwise.hip hands over.
#pragma once
#include "common.h"

namespace omni {

struct NormOut {
  int8_t* out;
  const half_t* gamma;
  half_t* sum;      // null: no row sums
  half_t* scale;
  float eps;
};
struct NormSlabs {      // K slabs of a product whose epilogue the norm applies; wsz, asum null: without zero points
  half_t* res;
  const int32_t* slab;      // [sk][tokens][hidden]
  size_t sstride;
  int sk;
  const half_t *wscales, *wsz, *ascales, *asum;
};

void norm_pairs_slabs(const NormOut& o, const NormSlabs& s, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st);
void norm_pairs_add(const NormOut& o, half_t* res, const half_t* delta, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st);
void norm_pairs_plain(const NormOut& o, const half_t* in, int tokens, int hidden, const PrefetchArgs& pf, hipStream_t st);

}  // namespace omni
