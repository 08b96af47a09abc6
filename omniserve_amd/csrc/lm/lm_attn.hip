// Causal attention of prompt portions over the paged cache, with a sliding window, any grouping of query heads and separate
// key / value sizes.  One workgroup per (128 query rows, head): its waves share the K and V tiles (64 keys = one cache
// page) in LDS, brought by LDS-DMA into two buffers; only pages that some row of the workgroup can see are touched.  The output
// is multiplied with sigmoid(gate) before it is stored.
#include "lm_attn.h"
#include "mfma_pinned.h"
#include "omniserve_lm.h"

namespace lm {

struct AttnArgs {
  const elem_t* q; int64_t ldq;                // [tokens][H][dk]
  const elem_t* kc; int64_t k_page; int k_head, k_row;      // key i of head g in page p: kc + p k_page + g k_head + i k_row
  const elem_t* vc; int64_t v_page; int v_head, v_row;
  const int* bt; int bt_stride;                // page numbers, one row per entry
  const int* entry;                            // [entries][4]: first token, tokens, position of the first token, block table row
  const int* tiles; int n_tiles;               // [n_tiles][2]: entry, first row within the entry
  const elem_t* gate; int64_t ldg;             // [tokens][H][dv] or null
  elem_t* o; int64_t ldo;
  float scale;                                 // includes log2(e)
  int window, H, G;
};

// The workgroup's tile and head.  A kv head's work stays on one XCD, late (long) tiles first, so that what runs last is short; an XCD with several
// kv heads takes a tile of all of them in turn.  (MI355X, 128 / 128, list's order / from its end: one prompt of 8000, 32 heads, 822 / 745 us, within a
// window of 4096 614 / 577; 4 of 1500 156 / 136; 16 of 500 90 / 87.  Where a kv head has two XCDs and one prompt's window leaves its tiles equally
// long, neighbours share pages the other way round: 16 heads on 4, window 1024, 115 / 117.)
__device__ __forceinline__ bool attn_work(const AttnArgs& p, int& tile, int& g, int& h) {
  const int gs = p.H / p.G;
  int t;
  if (p.G % 8 == 0) {
    const int hx = p.H / 8, i = blockIdx.x >> 3;
    t = i / hx;
    h = (blockIdx.x & 7) * hx + i - t * hx;
    g = h / gs;
  } else {
    const int id = xcd_contiguous(blockIdx.x, p.n_tiles * p.H);
    if (id < 0) return false;
    t = id / gs % p.n_tiles;
    g = id / (gs * p.n_tiles);
    h = g * gs + id % gs;
  }
  tile = p.n_tiles - 1 - t;
  return true;
}

constexpr int attn_waves_per_simd(int dk, int dv) { return SPLIT && dk + dv <= 256 ? 4 : 2; }      // what the registers allow

template <int DK, int DV, int WAVES>
struct AttnGeom {
  static constexpr int KB = DK * (int)sizeof(elem_t), VB = DV * (int)sizeof(elem_t);
  static constexpr bool DB = 2 * PAGE * (KB + VB) <= 131072 && SPLIT;          // two buffers
};

template <int DK, int DV, int WAVES>
__global__ __launch_bounds__(64 * WAVES, attn_waves_per_simd(DK, DV)) void attn_prefill_kernel(AttnArgs p) {
  typedef AttnGeom<DK, DV, WAVES> Gm;
  typedef Tile<Gm::KB> KT;
  typedef Tile<Gm::VB> VT;
  constexpr int NKF = DK / KSTEP, NVB = DV / 16;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l15 = lane & 15, l4 = lane >> 4;
  int tile, g, h;
  if (!attn_work(p, tile, g, h)) return;
  const int e = p.tiles[2 * tile], row0 = p.tiles[2 * tile + 1];
  const int start = p.entry[4 * e], count = p.entry[4 * e + 1], pos0 = p.entry[4 * e + 2];
  const int* bt = p.bt + (int64_t)p.entry[4 * e + 3] * p.bt_stride;
  const int r_w = row0 + 16 * wave;                      // the wave's first row
  const int row = r_w + l15, rowc = min(row, count - 1);
  const int qpos = pos0 + rowc;
  const int wg_last = pos0 + min(row0 + 16 * WAVES, count) - 1;
  const int w_first = pos0 + min(r_w, count - 1), w_last = pos0 + min(r_w + 15, count - 1);
  const bool idle = r_w >= count;

  frag_t qf[NKF];
  {
    const elem_t* qp = p.q + (int64_t)(start + rowc) * p.ldq + (int64_t)h * DK + FR * l4;
#pragma unroll
    for (int s = 0; s < NKF; ++s) qf[s] = *(const frag_t*)(qp + s * KSTEP);
  }
  f32x4 acc[NVB];
#pragma unroll
  for (int c = 0; c < NVB; ++c) acc[c] = zero4();
  float m_run = NEG, l_run = 0.f;

  const int lo = max(0, pos0 + row0 - p.window + 1);     // first key the workgroup needs
  const int kb0 = lo & ~(PAGE - 1);
  const int k_rowb = p.k_row * (int)sizeof(elem_t), v_rowb = p.v_row * (int)sizeof(elem_t);
  // 1-KiB pieces of a tile, one per wave and turn; physical slot s of row r holds logical slot s ^ swizzle(r)
  auto bring = [&](auto tile, const uint8_t* src, int rowb, uint8_t* dst) {
    typedef decltype(tile) T;
    constexpr int ROWB = T::NS * 16, N = PAGE * ROWB / 1024, STEP = 1024 * WAVES / ROWB;
    constexpr bool EVEN = 1024 * WAVES % ROWB == 0 && STEP % 16 == 0;      // every turn's rows have the first one's swizzles
#pragma unroll
    for (int i = 0; i < (N + WAVES - 1) / WAVES; ++i) {
      const int pc = wave + WAVES * i;
      if (N % WAVES != 0 && pc >= N) continue;
      const int sl = (EVEN ? wave : pc) * 64 + lane, r = sl / T::NS, s = sl % T::NS;
      const uint32_t off = r * rowb + ((s ^ T::swizzle(r)) << 4);
      dma16(src + (EVEN ? i * STEP * rowb : 0) + off, dst + 1024 * pc);
    }
  };
  auto stage = [&](int kb, uint8_t* kt, uint8_t* vt) {
    const int64_t page = bt[kb / PAGE];
    bring(KT{}, (const uint8_t*)(p.kc + page * p.k_page + g * p.k_head), k_rowb, kt);
    bring(VT{}, (const uint8_t*)(p.vc + page * p.v_page + g * p.v_head), v_rowb, vt);
  };
  auto compute = [&](int kb, const uint8_t* kt, const uint8_t* vt, auto prefetch) {
    const bool skip = idle || kb > w_last || kb + PAGE - 1 <= w_first - p.window;      // nothing visible for this wave
    f32x4 x[4];
    if (!skip) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = zero4();
#pragma unroll
        for (int s = 0; s < NKF; ++s) x[u] = mma(KT::frag(kt, 16 * u + l15, 4 * s + l4), qf[s], x[u]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    prefetch();
    if (skip) return;
    if (!(kb + PAGE - 1 <= w_first && kb > w_last - p.window)) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = kb + 16 * u + 4 * l4 + r;
          const int ok = (int)(key <= qpos) & (int)(key > qpos - p.window);
          x[u][r] = ok ? x[u][r] : NEG;
        }
    }
    quad_t pq[4][NOPND];
    const float alpha = softmax_step<4>(x, p.scale, m_run, l_run, pq);
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
      for (int c = 0; c < NVB; ++c) acc[c] *= alpha;
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int c = 0; c < NVB; ++c) {
        const quad_t v0 = VT::column_quad(vt, 32 * kk, c, l15, l4), v1 = VT::column_quad(vt, 32 * kk + 16, c, l15, l4);
#pragma unroll
        for (int o = 0; o < NOPND; ++o) acc[c] = mma_quads(v0, v1, pq[2 * kk][o], pq[2 * kk + 1][o], acc[c]);
      }
    __builtin_amdgcn_s_setprio(0);
  };

  uint8_t *kt0 = lds, *vt0 = lds + PAGE * Gm::KB;
  if constexpr (Gm::DB) {
    uint8_t *kt1 = vt0 + PAGE * Gm::VB, *vt1 = kt1 + PAGE * Gm::KB;
    stage(kb0, kt0, vt0);
    __syncthreads();
    for (int kb = kb0; kb <= wg_last; kb += 2 * PAGE) {
      compute(kb, kt0, vt0, [&] { if (kb + PAGE <= wg_last) stage(kb + PAGE, kt1, vt1); });
      __syncthreads();
      if (kb + PAGE > wg_last) break;
      compute(kb + PAGE, kt1, vt1, [&] { if (kb + 2 * PAGE <= wg_last) stage(kb + 2 * PAGE, kt0, vt0); });
      __syncthreads();
    }
  } else {
    for (int kb = kb0; kb <= wg_last; kb += PAGE) {
      stage(kb, kt0, vt0);
      __syncthreads();
      compute(kb, kt0, vt0, [] {});
      __syncthreads();
    }
  }
  const float inv = 1.0f / column_sum(l_run);
  if (row >= count) return;
  elem_t* op = p.o + (int64_t)(start + row) * p.ldo + (int64_t)h * DV + 4 * l4;
  const elem_t* gp = p.gate ? p.gate + (int64_t)(start + row) * p.ldg + (int64_t)h * DV + 4 * l4 : nullptr;
#pragma unroll
  for (int c = 0; c < NVB; ++c) {
    f32x4 y = acc[c] * inv;
    if (gp) {
      const f32x4 z = from_quad(*(const quad_t*)(gp + 16 * c));
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] *= sigmoid(z[r]);
    }
    *(quad_t*)(op + 16 * c) = to_quad(y);
  }
}

#if LM_ELEM == 0
// The same with 32 query rows per wave (v_mfma_f32_32x32x16_bf16), four waves of 128 rows, two workgroups per CU.
//
// With eight waves of 16 rows there is one workgroup on a CU: its waves form scores, take exponentials and multiply by V in step, and
// every one of them reads all of K and V out of LDS for 16 rows.  Two workgroups run against each other, and an operand read serves 32
// rows.
//
//   S^T = K q^T, 32 keys a block: A = K rows (lane: key lane % 32, 8 dims of 16 s + 8 (lane / 32)), B = q in registers.  A lane then holds
//   ONE query (lane % 32) and 16 keys (r & 3) + 8 (r >> 2) + 4 (lane / 32) of the block: its row maximum is in-lane but for one exchange.
//   O^T = V^T P^T: a k step may take its 16 keys in any order that both operands agree on, so step j of a block takes the lane's own
//   r = 8 j .. 8 j + 7: rows 16 j + 4 (lane / 32) + (0..3) and + 8 of V, two transposed reads.
//
// MI355X, 192 / 128, 16 heads, kernel above -> here: 2 prompts of 8000 1305 -> 920 us (990 TFLOP/s with the second operand of the probabilities
// counted), 48 of 150 57 -> 46; 256 / 64 and 64 / 256 at 2 prompts of 8000, 6 and 8 heads: 579 -> 457 and 766 -> 580.  128 / 128 has four
// waves per SIMD above and stays there (one prompt of 7999 790 us, 841 with 32 rows per wave).  attn_rows32 says where this one runs.
template <int DK, int DV>
struct Attn32 {
  static constexpr int KB = DK * 2, VB = DV * 2, TILE = PAGE * (KB + VB);
};
typedef float f32x16 __attribute__((ext_vector_type(16)));
// V tile: 16-byte slot s of row r at s ^ 4 (r & 3): the four rows that a transposed read touches lie in different bank quarters
__device__ __forceinline__ int v32_swizzle(int row) { return (row & 3) << 2; }

template <int DK, int DV>
__global__ __launch_bounds__(256, 2) void attn_prefill32_kernel(AttnArgs p) {
  typedef Attn32<DK, DV> Gm;
  typedef Tile<Gm::KB> KT;
  constexpr int NQ = DK / 16, NC = DV / 32, VS = Gm::VB / 16;
  static_assert(VS >= 16 ? VS % 16 == 0 : VS == 8, "value rows");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5, l15 = lane & 15;
  int tile, g, h;
  if (!attn_work(p, tile, g, h)) return;
  const int e = p.tiles[2 * tile], row0 = p.tiles[2 * tile + 1];
  const int start = p.entry[4 * e], count = p.entry[4 * e + 1], pos0 = p.entry[4 * e + 2];
  const int* bt = p.bt + (int64_t)p.entry[4 * e + 3] * p.bt_stride;
  const int r_w = row0 + 32 * wave;
  const int row = r_w + l32, rowc = min(row, count - 1);
  const int qpos = pos0 + rowc;
  const int wg_last = pos0 + min(row0 + 128, count) - 1;
  const int w_first = pos0 + min(r_w, count - 1), w_last = pos0 + min(r_w + 31, count - 1);
  const bool idle = r_w >= count;

  bf16x8 qf[NQ];
  {
    const elem_t* qp = p.q + (int64_t)(start + rowc) * p.ldq + (int64_t)h * DK + 8 * hi;
#pragma unroll
    for (int s = 0; s < NQ; ++s) qf[s] = *(const bf16x8*)(qp + 16 * s);
  }
  f32x16 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[c][r] = 0.f;
  float m_run = NEG, l_run = 0.f;

  const int lo = max(0, pos0 + row0 - p.window + 1);
  const int kb0 = lo & ~(PAGE - 1);
  const int k_rowb = p.k_row * 2, v_rowb = p.v_row * 2;
  // pieces of 1 KiB, lane-linear in LDS; physical slot s of row r holds logical slot s ^ swizzle(r)
  auto stage = [&](int kb, uint32_t kt, uint32_t vt) {
    const int64_t page = bt[kb / PAGE];
    const uint8_t* ks = (const uint8_t*)(p.kc + page * p.k_page + g * p.k_head);
    const uint8_t* vs = (const uint8_t*)(p.vc + page * p.v_page + g * p.v_head);
    const int ol = opaque(lane);
    constexpr int NK = PAGE * Gm::KB / 4096, NV = PAGE * Gm::VB / 4096;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int pc = NK * wave + i, sl = pc * 64 + ol, r = sl / KT::NS, s = sl % KT::NS;
      dma16_uncounted(ks + r * k_rowb + ((s ^ KT::swizzle(r)) << 4), kt + 1024 * pc);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int pc = NV * wave + i, sl = pc * 64 + ol, r = sl / VS, s = sl % VS;
      dma16_uncounted(vs + r * v_rowb + ((s ^ (v32_swizzle(r) & (VS - 1))) << 4), vt + 1024 * pc);
    }
  };
  // V^T operand: row 4 hi + l15 / 4 (+ 16 j + 32 u, + 8), dims 32 c + 16 ((lane / 16) & 1) + 4 (l15 & 3)
  const int vrow = 4 * hi + (l15 >> 2);
  int vaddr[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
    vaddr[c] = vrow * Gm::VB + (((4 * c + 2 * ((lane >> 4) & 1) + ((l15 & 3) >> 1)) ^ (v32_swizzle(vrow) & (VS - 1))) << 4) + 8 * (l15 & 1);

  auto compute = [&](int kb, const uint8_t* kt, const uint8_t* vt, auto prefetch) {
    const bool skip = idle || kb > w_last || kb + PAGE - 1 <= w_first - p.window;
    f32x16 x[2];
    if (!skip) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int r = 0; r < 16; ++r) x[u][r] = 0.f;
#pragma unroll
        for (int s = 0; s < NQ; ++s)
          x[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(kt + KT::slot(32 * u + l32, 2 * s + hi)), qf[s], x[u], 0, 0, 0);
      }
      // operand reads four products ahead
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 2 * NQ - 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
    }
    prefetch();
    if (skip) return;
    if (!(kb + PAGE - 1 <= w_first && kb > w_last - p.window)) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kb + 32 * u + (r & 3) + 8 * (r >> 2) + 4 * hi;
          const int ok = (int)(key <= qpos) & (int)(key > qpos - p.window);
          x[u][r] = ok ? x[u][r] : NEG;
        }
    }
    float t = NEG;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) t = fmaxf(t, x[u][r]);
    t = fmaxf(t, __shfl_xor(t, 32, 64));
    const float m_new = t <= NEG ? m_run : fmaxf(m_run, t * p.scale);
    const float m_sub = m_new <= NEG ? 0.f : m_new;          // no key seen yet: every probability underflows to 0
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    float sum = 0.f;
    bf16x8 ph[2][2], pl[2][2];                               // f32 probabilities as the sum of two operands
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float v = __builtin_amdgcn_exp2f(__builtin_fmaf(x[u][r], p.scale, -m_sub));
        sum += v;
        const __bf16 hb = (__bf16)v;
        ph[u][r >> 3][r & 7] = hb;
        pl[u][r >> 3][r & 7] = (__bf16)(v - (float)hb);
      }
    l_run = l_run * alpha + sum;
    m_run = m_new;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[c][r] *= alpha;
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int uj = 0; uj < 4; ++uj)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint8_t* src = vt + 16 * uj * Gm::VB + vaddr[c];
        const quad_t v0 = KT::transposed(src), v1 = KT::transposed(src + 8 * Gm::VB);
        const bf16x8 a = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, ph[uj >> 1][uj & 1], acc[c], 0, 0, 0);
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pl[uj >> 1][uj & 1], acc[c], 0, 0, 0);
      }
    // ... two operands (four products) ahead
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int i = 0; i < 4 * NC - 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  uint8_t *kt0 = lds, *vt0 = lds + PAGE * Gm::KB, *kt1 = lds + Gm::TILE, *vt1 = kt1 + PAGE * Gm::KB;
  auto at = [](const uint8_t* t) { return (uint32_t)(size_t)(const __attribute__((address_space(3))) uint8_t*)t; };
  // the wave's pieces have landed, then everybody's; everybody has left the tile before
  auto next = [&] {
    wait_pieces<0>();
    __syncthreads();
  };
  stage(kb0, at(kt0), at(vt0));
  next();
  for (int kb = kb0; kb <= wg_last; kb += 2 * PAGE) {
    compute(kb, kt0, vt0, [&] { if (kb + PAGE <= wg_last) stage(kb + PAGE, at(kt1), at(vt1)); });
    next();
    if (kb + PAGE > wg_last) break;
    compute(kb + PAGE, kt1, vt1, [&] { if (kb + 2 * PAGE <= wg_last) stage(kb + 2 * PAGE, at(kt0), at(vt0)); });
    next();
  }
  const float inv = 1.0f / (l_run + __shfl_xor(l_run, 32, 64));
  if (row >= count) return;
  elem_t* op = p.o + (int64_t)(start + row) * p.ldo + (int64_t)h * DV + 4 * hi;
  const elem_t* gp = p.gate ? p.gate + (int64_t)(start + row) * p.ldg + (int64_t)h * DV + 4 * hi : nullptr;
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 y = {acc[c][4 * q] * inv, acc[c][4 * q + 1] * inv, acc[c][4 * q + 2] * inv, acc[c][4 * q + 3] * inv};
      if (gp) {
        const f32x4 z = from_quad(*(const quad_t*)(gp + 32 * c + 8 * q));
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] *= sigmoid(z[r]);
      }
      *(quad_t*)(op + 32 * c + 8 * q) = to_quad(y);
    }
}
#endif

// Which sizes have the 32-row form: sums up to 256 have four waves per SIMD in the 16-row form, sums above 320 leave LDS for one workgroup of
// the 32-row form on a CU.  And it pays where workgroups share CUs: alone on one, its four waves have the SIMDs to themselves and wait for what eight
// of the other form overlap.  (MI355X, 16 rows / 32 rows per wave: 256 workgroups -- 16 prompts of 100 behind 400, 1 of 2000, 16 heads of 192 / 128 --
// 26.7 / 28.4 and 74.2 / 75.8 us, 128 rows behind 7000 241 / 246, 8 heads of 64 / 256 257 / 282; 288 workgroups, 3 prompts of 333 with 32
// heads, 27.4 / 22.0.)
constexpr bool has_rows32(int dk, int dv) { return !LM_ELEM && dk + dv == 320; }
static bool attn_rows32(int dk, int dv, int64_t workgroups) { return has_rows32(dk, dv) && workgroups > 256; }

template <int DK, int DV>
static int launch(const AttnArgs& a, hipStream_t s) {
  const int64_t total = (int64_t)a.n_tiles * a.H;
#if LM_ELEM == 0
  static_assert(LM_ATTN_ROWS == 128, "four waves of 32 rows");
  if constexpr (has_rows32(DK, DV)) if (attn_rows32(DK, DV, total)) {
    auto k = attn_prefill32_kernel<DK, DV>;
    constexpr size_t lds = 2 * Attn32<DK, DV>::TILE;
    if (allow_lds(k, lds)) return LM_EINVAL;
    hipLaunchKernelGGL(k, dim3((unsigned)(8 * ((total + 7) / 8))), dim3(256), lds, s, a);
    return launch_status();
  }
#endif
  constexpr int WAVES = LM_ATTN_ROWS / 16;
  typedef AttnGeom<DK, DV, WAVES> Gm;
  constexpr size_t lds = (size_t)PAGE * (Gm::KB + Gm::VB) * (Gm::DB ? 2 : 1);
  auto k = attn_prefill_kernel<DK, DV, WAVES>;
  if (allow_lds(k, lds)) return LM_EINVAL;
  hipLaunchKernelGGL(k, dim3((unsigned)(8 * ((total + 7) / 8))), dim3(64 * WAVES), lds, s, a);
  return launch_status();
}

}  // namespace lm

using namespace lm;

extern "C" int lm_attn_prefill_rows(int dk, int dv, int n_tiles, int H) { return attn_rows32(dk, dv, (int64_t)n_tiles * H) ? 32 : 16; }

extern "C" int lm_attn_prefill(const void* q, int64_t ldq, const void* kc, int64_t k_page, int k_head, int k_row,
                               const void* vc, int64_t v_page, int v_head, int v_row, const int* bt, int bt_stride, const int* entry, const int* tiles, int n_tiles, const void* gate, int64_t ldg, void* o, int64_t ldo,
                               float scale, int window, int H, int G, int dk, int dv, void* stream) {
  if (n_tiles <= 0 || G <= 0 || H % G || !(scale > 0.f) || window <= 0 || ldq % FR || ldo % 4 || ldg % 4 ||
      k_page % FR || k_head % FR || k_row % FR || v_page % FR || v_head % FR || v_row % FR ||
      k_row <= 0 || v_row <= 0 || k_row > (1 << 22) || v_row > (1 << 22) ||
      (int64_t)n_tiles * H > (1 << 28))
    return LM_EINVAL;
  AttnArgs a{(const elem_t*)q, ldq, (const elem_t*)kc, k_page, k_head, k_row, (const elem_t*)vc, v_page, v_head, v_row, bt, bt_stride, entry, tiles, n_tiles, (const elem_t*)gate,
             ldg, (elem_t*)o, ldo, scale * 1.4426950408889634f, window, H, G};
  hipStream_t s = (hipStream_t)stream;
#define LM_CASE(K, V) if (dk == K && dv == V) return launch<K, V>(a, s);
  LM_CASE(64, 64) LM_CASE(64, 128) LM_CASE(64, 256) LM_CASE(128, 64) LM_CASE(128, 128) LM_CASE(128, 256)
  LM_CASE(192, 64) LM_CASE(192, 128) LM_CASE(192, 256) LM_CASE(256, 64) LM_CASE(256, 128) LM_CASE(256, 256)
#undef LM_CASE
  return LM_EINVAL;
}
