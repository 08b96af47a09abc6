// Matrix products y = x W^T, one launch for a set of weight matrices ("groups"): a dense projection is one group, a mixture of
// experts is one group per expert over the tokens routed to it, plus one for the shared expert over all tokens.
//
//   lm_gemm_rows   few rows (decode): HBM bound.  A workgroup streams the weights of 16 - 80 channels of a group once, through an LDS
//                  ring filled by DMA; the rows of x come the same way, shared by its waves.  Small ones: operands straight to registers.
//   lm_gemm_tiles  many rows (prefill): MFMA bound.  256 x 256 tiles, both operands by LDS-DMA, a workgroup per CU that takes tile after tile;
//                  256 x 128 where those are too few for the chip, or their last round too empty.
//
// Epilogues: element type, f32 times a factor, the gated unit act(gate + bias) * (up + bias) of a matrix whose rows alternate in
// blocks of 16 between gate and up channels (both halves of a pair then sit in the same lane), or the product with sigmoid(gate).
#include "lm_gemm.h"
#include "mfma_pinned.h"

namespace lm {

// A workgroup owns NR 16-channel blocks; its KW waves split K and meet in LDS.  16 MB rows at a time; blockIdx.z takes every
// gridDim.z-th such part.
template <int NR, int MB, int KW, int EPI>
__global__ __launch_bounds__(64 * KW) void gemm_rows_kernel(GemmArgs p) {
  constexpr int U = NR > 1 ? 4 : 8;             // k-steps of weights requested together (a multiple of 4: see xf)
  __shared__ __attribute__((aligned(16))) float red[KW][16 * MB][16 * NR + 4];
  const int g = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l15 = lane & 15, l4 = lane >> 4;
  const bool is_b = g >= p.groups;
  const Part& pt = is_b ? p.b : p.a;
  const int n0 = blockIdx.x * 16 * NR;
  if (n0 >= pt.n) return;
  int first = 0, rows = is_b ? p.rows_b : p.rows_a;
  const int* perm = is_b ? nullptr : p.perm;
  if (perm) { first = p.off[g]; rows = p.off[g + 1] - first; }
  if (rows <= 0) return;
  const elem_t* w = pt.w + (is_b ? 0 : (int64_t)g * pt.n * pt.k);
  const int64_t x0 = is_b || perm ? 0 : g * pt.gx, y0 = is_b || perm ? 0 : g * pt.gy;
  const int steps = pt.k / KSTEP, s0 = steps * wave / KW, s1 = steps * (wave + 1) / KW;
  const elem_t* wp[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int c = n0 + 16 * r + l15;
    wp[r] = w + (int64_t)(c < pt.n ? c : pt.n - 1) * pt.k + FR * l4;
  }
  const int div = is_b ? 1 : p.x_div;
  for (int m0 = 16 * MB * blockIdx.z; m0 < rows; m0 += 16 * MB * gridDim.z) {
    const elem_t* xp[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int i = m0 + 16 * m + l15, ic = i < rows ? i : rows - 1;
      const int pair = perm ? perm[first + ic] : ic;
      xp[m] = pt.x + (int64_t)(pair / div) * pt.ldx + x0 + FR * l4;
    }
    const int mb = min(MB, (rows - m0 + 15) >> 4);     // row blocks with work (uniform)
    f32x4 acc[NR][MB];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[r][m] = zero4();
    // two sets of U steps of weights in turn (HBM), two sets of two steps of x in turn (L1 / L2), each requested one set ahead
    frag_t wf[2][NR][U], xf[2][MB][2];
    auto request_w = [&](frag_t (&f)[NR][U], int s) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < NR; ++r) f[r][u] = __builtin_nontemporal_load((const frag_t*)(wp[r] + (int64_t)(s + u) * KSTEP));
    };
    auto request_x = [&](frag_t (&f)[MB][2], int s) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        if (m < mb) {
          f[m][0] = *(const frag_t*)(xp[m] + (int64_t)s * KSTEP);
          f[m][1] = *(const frag_t*)(xp[m] + (int64_t)(s + 1) * KSTEP);
        }
      }
    };
    auto multiply = [&](frag_t (&f)[NR][U], int s) {
#pragma unroll
      for (int u = 0; u < U; u += 2) {
        if (s + u + 4 <= s1) request_x(xf[(u / 2 + 1) & 1], s + u + 2);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          if (m < mb) {
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
              for (int r = 0; r < NR; ++r) acc[r][m] = mma(f[r][u + v], xf[(u / 2) & 1][m][v], acc[r][m]);
          }
        }
      }
    };
    int s = s0;
    if (s + U <= s1) {
      request_w(wf[0], s);
      request_x(xf[0], s);
      while (true) {
        if (s + 2 * U <= s1) request_w(wf[1], s + U);
        multiply(wf[0], s);
        s += U;
        if (s + U > s1) break;
        if (s + 2 * U <= s1) request_w(wf[0], s + U);
        multiply(wf[1], s);
        s += U;
        if (s + U > s1) break;
      }
    }
    for (; s < s1; ++s) {
      frag_t w1[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) w1[r] = *(const frag_t*)(wp[r] + (int64_t)s * KSTEP);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        if (m < mb) {
          const frag_t x1 = *(const frag_t*)(xp[m] + (int64_t)s * KSTEP);
#pragma unroll
          for (int r = 0; r < NR; ++r) acc[r][m] = mma(w1[r], x1, acc[r][m]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int m = 0; m < MB; ++m) *(f32x4*)&red[wave][16 * m + l15][16 * r + 4 * l4] = acc[r][m];
    __syncthreads();
    constexpr int OB = EPI == LM_EPI_GLU ? NR / 2 : NR;      // 16-channel blocks of the result
    for (int i = tid; i < 16 * MB * OB * 4; i += 64 * KW) {
      const int m = i / (OB * 4), q = i - m * (OB * 4), blk = q >> 2, c4 = 4 * (q & 3);
      const int sb = EPI == LM_EPI_GLU ? 2 * blk : blk;
      if (m0 + m >= rows) continue;
      f32x4 v = zero4(), up = zero4();
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        v += *(const f32x4*)&red[k][m][16 * sb + c4];
        if constexpr (EPI == LM_EPI_GLU) up += *(const f32x4*)&red[k][m][16 * sb + 16 + c4];
      }
      const int pair = perm ? perm[first + m0 + m] : m0 + m;
      const int c = (EPI == LM_EPI_GLU ? n0 / 2 : n0) + 16 * blk + c4;
      if (c < (EPI == LM_EPI_GLU ? pt.n / 2 : pt.n)) {
        if constexpr (EPI == LM_EPI_GLU) v = glu(pt, p.act, n0 + 16 * sb + c4, v, up);
        store4<EPI>(pt, pair, c, y0, v, p.scale);
      }
    }
    __syncthreads();
  }
}

// ---- few rows: the weights' stream --------------------------------------------------------------------------------------------
// Both operands arrive by LDS-DMA in pieces of 8 rows x 128 bytes: 8 neighbouring lanes read 128 consecutive bytes.  An operand fragment
// loaded straight into registers reads 64 bytes of each of 16 rows, which the address path takes at 15 B per clock and CU; with x read that way
// once per 16 channels (4 bytes of x per byte of weights at 64 rows) that path and not HBM bounded the products: 4096 x 14336 at 48 rows 59 us
// -> 26 (117 MB: 4.5 TB/s), 28672 x 4096 75 -> 49, 32 experts at 60 tokens (998 MB) 278 -> 172 us (5.8 TB/s).  A stage is consumed behind one
// barrier; R - 1 more are on their way.
constexpr int RB = 128;                // bytes of k of a stage's rows
template <int NW, int KW> constexpr int ring_bytes = KW > 1 ? (144 << 10) / KW : NW <= 4 ? 64 << 10 : NW == 5 ? 80 << 10 : 144 << 10;      // of one K part

// at most N pieces of this wave still fly, and its LDS reads have been answered
template <int N>
__device__ __forceinline__ void wait_stage() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// rows (at most 16 MB) of x times 16 NW channels of w, stages s0 .. s1 - 1 of k, into red [KW][16 MB][16 NW + 4]: part h of the
// workgroup's waves takes every KW-th stage through a ring of its own
// SHORT: k may be below CHAIN_K.
// TURN: rows lie whole KiBs apart, and workgroups in step ask the same channels of the memory.  So the workgroups of an XCD begin with different numbers (`early`) of
// K's last chains of stages, whose sums wait in registers for those in front of them: the additions keep their order, and a channel's sum does not hang
// on its place.  (MI355X, without | with: 28672 x 4096 at 48 rows 48.9 | 39.9 us, 32000 x 4096 59.7 | 43.4, 32000 x 2048 at 16 rows 25.4 | 22.9; each workgroup
// 256 bytes further than the one before it and an order of its own, 38.5, 42.1, 21.5; at most 8 and 4 chains 40.1, 45.1, 22.4.)
constexpr int CHAIN_K = 64 * KSTEP;
template <int MB, int NW, int KW, bool SHORT, bool TURN>
__device__ __forceinline__ void stream_stages(uint8_t* lds, const elem_t* w, int n, int64_t k, int n0, const elem_t* x, int64_t ldx,
                                              const int* perm, int div, int rows, int s0, int s1) {
  constexpr int WST = 16 * NW * RB, XST = 16 * MB * RB, ST = WST + XST, R0 = ring_bytes<NW, KW> / ST;
  constexpr int XP = (2 * MB + NW - 1) / NW;                   // pieces (8 rows) of x a wave carries (some twice: the same bytes)
  constexpr int P = 2 + XP, RMAX = 63 / P + 2 < 10 ? 63 / P + 2 : 10, R = R0 < RMAX ? R0 : RMAX;      // (vmcnt counts to 63)
  typedef Tile<RB> T;
  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, l4 = lane >> 4;
  const int all = __builtin_amdgcn_readfirstlane(tid >> 6), h = KW == 1 ? 0 : all / NW, wave = all - h * NW;
  lds += h * ring_bytes<NW, KW>;
  const int pr = lane >> 3, ps = lane & 7;                 // a piece: lane -> (row, physical slot)
  const uint8_t *wsrc[2], *xsrc[XP];
  int xp[XP];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * i + pr, c = min(n0 + 16 * wave + r, n - 1);
    wsrc[i] = (const uint8_t*)(w + c * k) + (int64_t)(s0 + h) * RB + ((ps ^ T::swizzle(r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    xp[i] = (NW * i + wave) % (2 * MB);
    const int r = 8 * xp[i] + pr, rc = min(r, rows - 1);
    const int64_t row = perm ? perm[rc] / div : rc;
    xsrc[i] = (const uint8_t*)(x + row * ldx) + (int64_t)(s0 + h) * RB + ((ps ^ T::swizzle(r)) << 4);
  }
  const uint32_t base = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int nst = (s1 - s0 - h + KW - 1) / KW;
  constexpr int EARLY = !TURN || SHORT ? 0 : NW == 5 ? (MB <= 2 ? 7 : 4) : MB <= 2 ? 15 : 7;      // (as the registers have room; of 80 channels 3 waves share a SIMD's)
  const int early = EARLY ? max(0, min((int)(blockIdx.x >> 3) % (EARLY + 1), (nst + 3) / 4 - 3)) : 0;      // (12 stages or more stay behind them, R - 1 <= 9)
  const int turn = early ? 4 * ((nst + 3) / 4 - early) : 0, first = early ? nst - turn : 0;      // first: stages of those chains
  auto stage = [&](int t) {                                // the t-th stage that this part takes
    const uint32_t dst = base + (uint32_t)(t % R) * ST;
    const int at = (EARLY == 0 || t + turn < nst ? t + turn : t + turn - nst) * (KW * RB);
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16_stream(wsrc[i] + at, dst + 2048 * wave + 1024 * i);
#pragma unroll
    for (int i = 0; i < XP; ++i) dma16_uncounted(xsrc[i] + at, dst + WST + 1024 * xp[i]);
  };
  // sums of 4 stages (2, 1, half a one) and the sum of those: chains of f32 additions no longer than an eighth of K.  (A form of its own for long K: with
  // the choice in it that one took 3 - 7 % more, 16 tokens of 8 of 64 x 1280 x 2048 52.8 -> 55.5 us.)
  const int chain = !SHORT || k >= CHAIN_K ? 3 : k >= CHAIN_K / 2 ? 1 : 0;
  const bool halves = SHORT && k < CHAIN_K / 4;
  f32x4 acc[MB], total[MB], later[EARLY + 1][MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) acc[m] = total[m] = zero4();
  auto end_chain = [&] {
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      total[m] += acc[m];
      acc[m] = zero4();
    }
  };
  auto multiply = [&](int t) {
    const uint8_t* wt = lds + (t % R) * ST + wave * (16 * RB);
    const uint8_t* xt = lds + (t % R) * ST + WST;
    frag_t a[2], b[2][MB];
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      a[v] = T::frag(wt, l15, 4 * v + l4);
#pragma unroll
      for (int m = 0; m < MB; ++m) b[v][m] = *(const frag_t*)(xt + 16 * m * RB + T::slot(l15, 4 * v + l4));
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[m] = mma(a[v], b[v][m], acc[m]);
      if (v == 0 && halves) end_chain();
    }
  };
  auto multiply_on = [&](int t) {                          // ... of the chains that are added up at once
    multiply(t);
    if (((t - first) & chain) == chain) end_chain();
  };
  wait_pieces<0>();                                        // the compiler's own loads
#pragma unroll
  for (int t = 0; t < R - 1; ++t)
    if (t < nst) stage(t);
  int t = 0;
  auto next = [&] {                                        // R - 2 stages fly behind stage t
    wait_stage<(R - 2) * P>();
    __builtin_amdgcn_s_barrier();                          // stage t is there for every wave, everyone has left stage t - 1
    asm volatile("" ::: "memory");
    stage(t + R - 1);
  };
#pragma unroll
  for (int c = 0; c < EARLY; ++c) {
    for (const int end = c < early ? min(t + 4, first) : t; t < end; ++t) {
      next();
      multiply(t);
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      later[c][m] = acc[m];
      acc[m] = zero4();
    }
  }
  for (; t + R - 1 < nst; ++t) {
    next();
    multiply_on(t);
  }
  // the last R - 1 stages: j fly behind this one
  auto last = [&](auto jt) {
    constexpr int J = decltype(jt)::value;
    if (nst - 1 - J < 0) return;
    wait_stage<J * P>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply_on(nst - 1 - J);
  };
  countdown<R - 2>(last);
  if (KW > 1 && nst < (s1 - s0 + KW - 1) / KW) __builtin_amdgcn_s_barrier();      // (other parts have a stage more)
#pragma unroll
  for (int c = 0; c < EARLY; ++c)
#pragma unroll
    for (int m = 0; m < MB; ++m)
      if (c < early) total[m] += later[c][m];
  __syncthreads();                                         // the rings are free
  float* red = (float*)(lds - h * ring_bytes<NW, KW>) + h * (16 * MB * (16 * NW + 4));
#pragma unroll
  for (int m = 0; m < MB; ++m) *(f32x4*)&red[(16 * m + l15) * (16 * NW + 4) + 16 * wave + 4 * l4] = total[m] + acc[m];
  __syncthreads();
}

// A workgroup: 16 NW channels of a group, rows 0 .. 16 MB - 1 of it, K slice blockIdx.z.  With several slices (one group) the f32 sums of a
// slice go to part [slice][rows][n] and gemm_reduce_kernel finishes them.
// IDS: the rows of a group are the pairs whose expert it is: every wave looks through the choices (a load per 64 pairs, all at once), one of them notes
// the places.  Their order does not matter: a row's sums are its own.
// ROWS16: blocks of 16 rows that there are (0: up to four).
template <int EPI, int NW, int KW, bool SHORT, bool TURN, bool IDS, int ROWS16>
__global__ __launch_bounds__(64 * NW * KW) void gemm_stream_kernel(GemmArgs p, float* part) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[KW * ring_bytes<NW, KW>];
  __shared__ int own[IDS ? LM_CHOOSE_TOKENS : 1];
  constexpr int RC = 16 * NW, NT = 64 * NW * KW;
  const int g = blockIdx.y, tid = threadIdx.x;
  const bool is_b = g >= p.groups;
  const Part& pt = is_b ? p.b : p.a;
  const int n0 = blockIdx.x * RC;
  if (n0 >= pt.n) return;
  int first = 0, rows = is_b ? p.rows_b : p.rows_a;
  const int* perm = is_b ? nullptr : p.perm;
  if (IDS && !is_b) {
    const int lane = tid & 63;
    rows = 0;
    auto look = [&](auto chunks) {
      constexpr int CHUNKS = decltype(chunks)::value;
      int e[CHUNKS];
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i) e[i] = p.off[min(64 * i + lane, p.rows_a - 1)];
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i) {
        const bool it = e[i] == g && 64 * i + lane < p.rows_a;
        const uint64_t mine = __builtin_amdgcn_ballot_w64(it);
        const int at = rows + __builtin_amdgcn_mbcnt_hi((uint32_t)(mine >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mine, 0));
        if (tid < 64 && it && at < LM_CHOOSE_TOKENS) own[at] = 64 * i + lane;
        rows += __builtin_popcountll(mine);
      }
    };
    if (p.rows_a <= 128) look(Int<2>{});
    else look(Int<LM_CHOOSE_TOKENS * LM_MAX_TOP / 64>{});
    rows = min(rows, LM_CHOOSE_TOKENS);      // (a token chooses an expert once)
    perm = own;
    if (rows > 0) __syncthreads();
  } else if (perm) {
    first = p.off[g]; rows = p.off[g + 1] - first; perm += first;
  }
  if (rows <= 0) return;
  const elem_t* w = pt.w + (is_b ? 0 : (int64_t)g * pt.n * pt.k);
  const int64_t x0 = is_b || perm ? 0 : g * pt.gx, y0 = is_b || perm ? 0 : g * pt.gy;
  const int stages = pt.k * (int)sizeof(elem_t) / RB, slice = blockIdx.z, slices = gridDim.z;
  const int s0 = stages * slice / slices, s1 = stages * (slice + 1) / slices;
  const int div = is_b ? 1 : p.x_div;
  static_assert(!IDS || LM_CHOOSE_TOKENS <= 32, "rows of a chosen group");
  for (int m0 = 0; m0 < (IDS ? 1 : rows); m0 += 64) {
    const int here = min(64, rows - m0), mb = ROWS16 ? ROWS16 : (here + 15) >> 4;
    const elem_t* x = pt.x + x0 + (perm ? 0 : m0 * pt.ldx);
    const int* pm = perm ? perm + m0 : nullptr;
    if constexpr (ROWS16 > 0) stream_stages<ROWS16, NW, KW, SHORT, TURN>(lds, w, pt.n, pt.k, n0, x, pt.ldx, pm, div, here, s0, s1);
    else if (mb == 1) stream_stages<1, NW, KW, SHORT, TURN>(lds, w, pt.n, pt.k, n0, x, pt.ldx, pm, div, here, s0, s1);
    else if (IDS || mb == 2) stream_stages<2, NW, KW, SHORT, TURN>(lds, w, pt.n, pt.k, n0, x, pt.ldx, pm, div, here, s0, s1);
    else if (mb == 3) stream_stages<3, NW, KW, SHORT, TURN>(lds, w, pt.n, pt.k, n0, x, pt.ldx, pm, div, here, s0, s1);
    else stream_stages<4, NW, KW, SHORT, TURN>(lds, w, pt.n, pt.k, n0, x, pt.ldx, pm, div, here, s0, s1);
    const float* red = (const float*)lds;
    auto sum = [&](int m, int c) {
      f32x4 v = *(const f32x4*)&red[m * (RC + 4) + c];
#pragma unroll
      for (int h = 1; h < KW; ++h) v += *(const f32x4*)&red[(16 * mb * h + m) * (RC + 4) + c];
      return v;
    };
    if (slices > 1) {
      for (int i = tid; i < here * (RC / 4); i += NT) {
        const int m = i / (RC / 4), c = 4 * (i % (RC / 4));
        if (n0 + c < pt.n) *(f32x4*)(part + ((int64_t)slice * rows + m0 + m) * pt.n + n0 + c) = sum(m, c);
      }
    } else {
      constexpr int OC = EPI == LM_EPI_GLU ? RC / 2 : RC;
      for (int i = tid; i < here * (OC / 4); i += NT) {
        const int m = i / (OC / 4), c = 4 * (i % (OC / 4));
        const int sc = EPI == LM_EPI_GLU ? 32 * (c >> 4) + (c & 15) : c;      // the gate's (or the only) channel inside the tile
        if (n0 + sc >= pt.n) continue;
        f32x4 v = sum(m, sc);
        if constexpr (EPI == LM_EPI_GLU) v = glu(pt, p.act, n0 + sc, v, sum(m, sc + 16));
        store4<EPI>(pt, pm ? pm[m] : m0 + m, (EPI == LM_EPI_GLU ? n0 / 2 : n0) + c, y0, v, p.scale);
      }
    }
    __syncthreads();
  }
}

// sums of the K slices in their order, then the epilogue
template <int EPI>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs p, const float* part, int slices) {
  const Part& pt = p.a;
  const int oq = (EPI == LM_EPI_GLU ? pt.n / 2 : pt.n) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)p.rows_a * oq) return;
  const int m = (int)(i / oq), c = 4 * (int)(i % oq);
  const int sc = EPI == LM_EPI_GLU ? 32 * (c >> 4) + (c & 15) : c;
  f32x4 v = zero4(), up = zero4();
  for (int k = 0; k < slices; ++k) {
    const float* r = part + ((int64_t)k * p.rows_a + m) * pt.n + sc;
    v += *(const f32x4*)r;
    if constexpr (EPI == LM_EPI_GLU) up += *(const f32x4*)(r + 16);
  }
  if constexpr (EPI == LM_EPI_GLU) v = glu(pt, p.act, sc, v, up);
  store4<EPI>(pt, m, c, 0, v, p.scale);
}

// ---- many rows: 256 x 256 tiles -----------------------------------------------------------------------------------------------
constexpr int TN = 256;                                     // channels of a tile
constexpr int SROWB = 128, SK = SROWB / (int)sizeof(elem_t); // a stage: 128 bytes of k of every row (whole lines of the L2)
constexpr int STAGE = (TM + TN) * SROWB;

// c += a b, c pinned (mfma_pinned.h)
__device__ __forceinline__ void mma_in_place(f32x4& c, frag_t a, frag_t b) {
#if LM_ELEM == 0
  OMNI_MFMA_PINNED("v_mfma_f32_16x16x32_bf16", c, a, b);
#else
#pragma unroll
  for (int i = 0; i < 4; ++i) OMNI_MFMA_PINNED("v_mfma_f32_16x16x4_f32", c, a[i], b[i]);
#endif
}
// three of them and an LDS-DMA request.  SADDR: src is a 32-bit offset from base.
template <bool SADDR, typename S>
__device__ __forceinline__ void mma3_dma16(f32x4& c0, f32x4& c1, f32x4& c2, frag_t a0, frag_t a1, frag_t a2, frag_t b, S src, const void* base,
                                           uint32_t lds_dst) {
#if LM_ELEM == 0
  if constexpr (SADDR) OMNI_MFMA3_DMA16("v_mfma_f32_16x16x32_bf16", "%10", c0, c1, c2, a0, a1, a2, b, src, base, lds_dst);
  else OMNI_MFMA3_DMA16("v_mfma_f32_16x16x32_bf16", "off", c0, c1, c2, a0, a1, a2, b, src, 0, lds_dst);
#else
  mma_in_place(c0, a0, b);
  mma_in_place(c1, a1, b);
  if constexpr (SADDR) dma16_uncounted((const uint8_t*)base + src, lds_dst);
  else dma16_uncounted(src, lds_dst);
  mma_in_place(c2, a2, b);
#endif
}

// 4 waves, 128 rows x 128 channels each.  A wave's operands are 16 fragments for 64 MFMAs (256 accumulator registers, one wave per SIMD):
// with 64 x 128 per wave and two workgroups per CU the LDS had 72 KB to move per 512 MFMA cycles and SIMD, more than its 128 B per clock.
// Nothing overlaps with a lone wave but what it issues itself: the fragments of a half stage are read while the half before it
// multiplies, a stage ahead of it is requested.
//
// A workgroup takes tile after tile: the first two stages of the next one are on their way while it stores this one (16 us passed between
// the products of a tile and those of the next where every tile had a workgroup; a stage takes 1 us and K = 640 has 10 of them).
//
// MI355X, bf16, before: 256 x 128 tiles of 64-byte stages, a workgroup per tile, two of them on a CU.  7999
// tokens, 6 of 32 experts of 1792, width 4096: 2407 -> 1883 us up (998 TFLOP/s with the rows of the half empty tiles not counted), 1084 ->
// 938 down; 6733 tokens, 8 of 64 experts of 640, width 2048: 410 -> 382 up, 256 -> 259 down; 8192 x 7168 x 4096 to f32: 569 -> 469.
// Ahead of the requests a wave touches 32 lines of the stage behind them (touch_lines32): 64 rows of each operand a workgroup, the others by the workgroups
// of the band and of the neighbouring columns; where a band's tiles are several experts', their weights' other rows come untouched.  7999 tokens as
// above: 1687 -> 1644 up, 947 -> 920 down.  To f32, 30 sizes of 300 - 4100 rows: 0.94x on average, 2000 rows of 16384 x 4096 236 -> 198, but 1000 of 32000 x 4096 229 -> 239, 2000 of
// 8192 x 4096 99 -> 102 (of the two steps, no zeroing alone 0.998x).
template <int EPI>
__global__ __launch_bounds__(256, 1) void gemm_tiles_kernel(GemmArgs p, int mt_a, int mt_b) {
  constexpr bool DIRECT = EPI == LM_EPI_F32 || sizeof(elem_t) == 4;      // accumulators straight to memory
  constexpr bool TOUCH = sizeof(elem_t) == 2;                            // (f32's products take too long for memory and ends of tiles to matter)
  constexpr int OC = EPI == LM_EPI_GLU ? 64 : 128, PITCH = OC * (int)sizeof(elem_t) + 16, OUT = DIRECT ? 0 : 4 * 16 * PITCH;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * STAGE + OUT + 128];
  __shared__ int y_rows[2][TM];
  typedef Tile<SROWB> T;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // linear order of a part: bands of row tiles, all channel tiles of a band before the next one; an XCD has a contiguous range of both
  // parts, its workgroups take the tiles of it in turn
  if (p.perm) mt_a = row_tiles(p.tiles, mt_a);
  const int nt_a = (p.a.n + TN - 1) / TN, nt_b = mt_b ? (p.b.n + TN - 1) / TN : 0;
  const int per_a = (mt_a * nt_a + 7) >> 3, per_b = (mt_b * nt_b + 7) >> 3, xcd = blockIdx.x & 7;
  const int own_b = max(0, min(per_b, mt_b * nt_b - xcd * per_b)), own = own_b + max(0, min(per_a, mt_a * nt_a - xcd * per_a));
  // in the XCD's range: a place further among its workgroups with every turn, so that a row of short tiles in every band is not always the same ones'
  const int turn = (int)gridDim.x >> 3;
  int place = blockIdx.x >> 3, turns = 0;

  // pieces of 8 rows: lane -> (row lane / 8, physical slot lane % 8); a wave carries 8 of the weights' and 8 of x's.  (A row of the tile past
  // the matrix: its last one again; none of it is stored.)
  const uint8_t* xsrc[8];
  uint32_t woff[8];                                         // from the tile's first channel
  const uint8_t* wbase = nullptr;
  const uint8_t* soon = nullptr;                            // the lane's line of the stage behind the one requested last: of the weights (lanes 0 - 15) or of x
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const uint32_t dst0 = __builtin_amdgcn_readfirstlane(lds0 + 64 * SROWB * wave);
  auto dst = [&](int t, int i) { return dst0 + (t & 1) * STAGE + 1024 * (i & 7) + (i < 8 ? 0 : TN * SROWB); };      // of piece i
  auto stage = [&](int t) {                                 // requests the next stage of k
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i < 8) dma16_uncounted(wbase + woff[i], dst(t, i));
      else {
        dma16_uncounted(xsrc[i & 7], dst(t, i));
        xsrc[i & 7] += SROWB;
      }
    }
    wbase += SROWB;
  };
  bool is_b = false, few_next = false;
  int n0 = 0, ns = 0;
  // the next tile with rows from place `at` on: its rows of y, its first two stages requested; false: there is none
  auto open_tile = [&](int (&y_row)[TM]) {
    while (turns + place < own) {
      const int at = turns + place;
      turns += turn;
      place = place + 1 == turn ? 0 : place + 1;
      is_b = at < own_b;
      const Part& pt = is_b ? p.b : p.a;
      const int nt = is_b ? nt_b : nt_a, mts = is_b ? mt_b : mt_a;
      const int id = is_b ? xcd * per_b + at : xcd * per_a + at - own_b;
      constexpr int GM = 4;
      const int band = id / (GM * nt), in = id - band * GM * nt, bm = min(GM, mts - band * GM);
      const int mi = band * GM + in % bm;
      const int* perm = is_b ? nullptr : p.perm;
      int first = mi * TM, rows, g = 0;
      if (perm) {
        const i32x4 t = *(const i32x4*)(p.tiles + 4 * mi);     // group, first place, rows
        if (t[2] <= 0) continue;
        g = t[0];
        first = t[1];
        rows = t[2];
      } else {
        rows = min(TM, (is_b ? p.rows_b : p.rows_a) - first);
      }
      const int ol = lane_here(), pr = ol >> 3, ps = ol & 7, otid = 64 * wave + ol, x_div = opaque(p.x_div);
      n0 = in / bm * TN;
      ns = pt.k / SK;
      wbase = (const uint8_t*)(pt.w + ((int64_t)g * pt.n + n0) * pt.k);
      int xr[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int rc = first + min(64 * wave + 8 * i + pr, rows - 1);
        xr[i] = perm ? perm[rc] : rc;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = 64 * wave + 8 * i + pr;
        woff[i] = (uint32_t)min(r, pt.n - 1 - n0) * (uint32_t)(pt.k * (int)sizeof(elem_t)) + ((ps ^ T::swizzle(r)) << 4);
        xsrc[i] = (const uint8_t*)(pt.x + (int64_t)(perm ? xr[i] / x_div : xr[i]) * pt.ldx) + ((ps ^ T::swizzle(r)) << 4);
        __builtin_amdgcn_sched_barrier(0);                  // (not eight divisions at once beside the results of the tile before)
      }
      {
        const int r = 64 * ((ol & 16 ? in / bm : mi) & 3) + 16 * wave + (ol & 15), rc = first + min(r, rows - 1);
        const int xr = perm ? perm[rc] / x_div : rc;
        soon = (ol & 16 ? (const uint8_t*)(pt.x + (int64_t)xr * pt.ldx) : wbase + (uint32_t)min(r, pt.n - 1 - n0) * (uint32_t)(pt.k * (int)sizeof(elem_t))) +
               SROWB * min(2, ns - 1);
      }
      y_row[otid] = otid < rows ? (perm ? perm[first + otid] : first + otid) : -1;
      wait_pieces<0>();                                     // the compiler's own loads
      stage(0);
      if (ns > 1) stage(1);
      if constexpr (TOUCH) touch_lines32(soon, lds0 + 2 * STAGE + OUT);
      few_next = rows <= TM / 2;
      return true;
    }
    return false;
  };

  const int wn = 128 * (wave & 1);
  int wm = 0;                                               // the wave's first row
  int off[2];                                               // of a fragment of half u inside 16 rows
  frag_t a[2][8], b[2][8];
  auto fetch_b = [&](int t, auto half, int i) {
    constexpr int U = decltype(half)::value;
    b[U][i] = *(const frag_t*)(lds + (t & 1) * STAGE + 16 * SROWB * i + off[U] + (TN + wm) * SROWB);
  };
  auto fetch_a = [&](int t, auto half, int i) {
    constexpr int U = decltype(half)::value;
    a[U][i] = *(const frag_t*)(lds + (t & 1) * STAGE + 16 * SROWB * i + off[U] + wn * SROWB);
  };
  f32x4 acc[8][8];
  // Stage t: FRESH: the tile's first (its accumulators were not zeroed: 256 instructions of a lone wave), MORE: there is a stage t + 1, DMA: and a stage t + 2.  Requests and reads go out one by one between the products: a burst of
  // them fills the queues of the address path and the LDS, and the lone wave, which issues in order, waits there with its matrix
  // unit idle.  No condition inside: reads and products have to share a basic block.
  auto step = [&](int t, auto blocks, auto fresh, auto more, auto dma) {
    constexpr int NJ = decltype(blocks)::value;            // blocks of 16 rows of the wave: 8, or 4 of a tile of up to 128 rows
    constexpr bool FRESH = decltype(fresh)::value, MORE = decltype(more)::value, DMA = decltype(dma)::value;
    auto four = [&](auto half, int i0, int j) {
      constexpr int U = decltype(half)::value;
#pragma unroll
      for (int i = i0; i < i0 + 4; ++i) {
        if constexpr (FRESH && U == 0) OMNI_MFMA_FRESH("v_mfma_f32_16x16x32_bf16", acc[i][j], a[U][i], b[U][j]);
        else mma_in_place(acc[i][j], a[U][i], b[U][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      fetch_b(t, Int<1>{}, j);
      if constexpr (NJ == 4) fetch_a(t, Int<1>{}, 2 * j);
      __builtin_amdgcn_sched_barrier(0);
      four(Int<0>{}, 0, j);
      fetch_a(t, Int<1>{}, NJ == 4 ? 2 * j + 1 : j);
      __builtin_amdgcn_sched_barrier(0);
      four(Int<0>{}, 4, j);
    }
    // stage t + 1 is there for every wave, and everyone has stage t in registers
    if constexpr (DMA && TOUCH) asm volatile("s_waitcnt vmcnt(1) lgkmcnt(0)" ::: "memory");      // (behind its requests only lines are touched)
    else if constexpr (MORE) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      constexpr int PER = 8 / NJ;                           // pieces of each operand with a block of rows
      if constexpr (MORE) {
        fetch_b(t + 1, Int<0>{}, j);
        if constexpr (PER == 2) fetch_a(t + 1, Int<0>{}, 2 * j);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (DMA) {
        mma3_dma16<true>(acc[0][j], acc[1][j], acc[2][j], a[1][0], a[1][1], a[1][2], b[1][j], woff[PER * j], wbase, dst(t, PER * j));
        mma_in_place(acc[3][j], a[1][3], b[1][j]);
        if constexpr (PER == 2) dma16_uncounted(wbase + woff[2 * j + 1 & 7], dst(t, 2 * j + 1));
        __builtin_amdgcn_sched_barrier(0);
      } else {
        four(Int<1>{}, 0, j);
      }
      if constexpr (MORE) fetch_a(t + 1, Int<0>{}, PER * j + PER - 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (DMA) {
        mma3_dma16<false>(acc[4][j], acc[5][j], acc[6][j], a[1][4], a[1][5], a[1][6], b[1][j], xsrc[PER * j], nullptr, dst(t, 8 + PER * j));
        xsrc[PER * j] += SROWB;
        mma_in_place(acc[7][j], a[1][7], b[1][j]);
        if constexpr (PER == 2) {
          dma16_uncounted(xsrc[2 * j + 1 & 7], dst(t, 8 + 2 * j + 1));
          xsrc[2 * j + 1 & 7] += SROWB;
        }
        __builtin_amdgcn_sched_barrier(0);
      } else {
        four(Int<1>{}, 4, j);
      }
    }
    if constexpr (DMA) {
      wbase += SROWB;
      soon += SROWB & (t + 3 < ns ? -1 : 0);
      if constexpr (TOUCH) touch_lines32(soon, lds0 + 2 * STAGE + OUT);
    }
  };

  int parity = 0;
  bool open = open_tile(y_rows[0]);
  while (open) {
    // stage 0 is there: of what was requested last -- stage 1 and lines, or stores of the tile before -- 16 (17) may still fly
    if (ns > 1) wait_pieces<16 + TOUCH>();
    else wait_pieces<0>();
    __syncthreads();
    const bool few = few_next;
    wm = (few ? 64 : 128) * (wave >> 1);
    const int fl = lane_here();
#pragma unroll
    for (int u = 0; u < 2; ++u) off[u] = T::slot(fl & 15, 4 * u + (fl >> 4));
    auto products = [&](auto blocks) __attribute__((always_inline)) {
      constexpr int NJ = decltype(blocks)::value;
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = NJ; j < 8; ++j) asm volatile("" : "=a"(acc[i][j]));      // (nothing: no value of the tile before is carried along)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i < NJ) fetch_b(0, Int<0>{}, i);
        fetch_a(0, Int<0>{}, i);
      }
      int t = 0;
      if (TOUCH && ns > 2) {
        step(0, blocks, Int<TOUCH>{}, Int<1>{}, Int<1>{});
        t = 1;
      } else {
        const float z = __builtin_bit_cast(float, opaque(0));
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{z, z, z, z};
      }
      for (; t + 2 < ns; ++t) step(t, blocks, Int<0>{}, Int<1>{}, Int<1>{});
      if (t + 1 < ns) {
        step(t, blocks, Int<0>{}, Int<1>{}, Int<0>{});
        ++t;
      }
      step(t, blocks, Int<0>{}, Int<0>{}, Int<0>{});        // (behind its barrier both stages are free)
    };
    if (few) products(Int<4>{});
    else products(Int<8>{});
    accumulators_settle(acc);

    const Part& pt = is_b ? p.b : p.a;
    const int el = lane_here(), e15 = el & 15, e4 = el >> 4;
    const int c0 = n0 + wn;                                 // the wave's first channel
    const int* y_row = y_rows[parity];
    const int span = few ? 64 : 128;                        // the wave's rows (behind them is what other tiles left)
    // the next tile's requests, then the results: they stay in the accumulation registers until they are stored
    open = open_tile(y_rows[parity ^ 1]);
    accumulators_stay(acc);
    if constexpr (DIRECT) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int row = 16 * j < span ? y_row[wm + 16 * j + e15] : -1;
        if (row >= 0) {
#pragma unroll
          for (int i = 0; i < 8; i += EPI == LM_EPI_GLU ? 2 : 1) {
            const int c = c0 + 16 * i + 4 * e4;
            if (c >= pt.n) continue;
            if constexpr (EPI == LM_EPI_GLU) store4<EPI>(pt, row, (c0 + 16 * i) / 2 + 4 * e4, 0, glu(pt, p.act, c, acc[i][j], acc[i + 1][j]), p.scale);
            else store4<EPI>(pt, row, c, 0, acc[i][j], p.scale);
          }
        }
        accumulators_stay(acc);                             // (no addresses of later rows kept beside them either)
      }
    } else {
      // through LDS, so that a row leaves in whole 16-byte pieces of neighbouring lanes: 16 rows of the wave's at a time
      constexpr int PPR = OC / FR, NI = EPI == LM_EPI_GLU ? 4 : 8;
      uint8_t* buf = lds + 2 * STAGE + wave * 16 * PITCH;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          quad_t v;
          if constexpr (EPI == LM_EPI_GLU) v = to_quad(glu(pt, p.act, min(c0 + 32 * i, pt.n - 32) + 4 * e4, acc[2 * i][j], acc[2 * i + 1][j]));
          else v = to_quad(acc[i][j]);
          *(quad_t*)(buf + e15 * PITCH + (16 * i + 4 * e4) * (int)sizeof(elem_t)) = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 16 * PPR / 64; ++i) {
          const int pc = 64 * i + el, r = pc / PPR, q = pc % PPR;
          const int row = 16 * j < span ? y_row[wm + 16 * j + r] : -1, c = (EPI == LM_EPI_GLU ? c0 / 2 : c0) + q * FR;
          if (row >= 0 && c < (EPI == LM_EPI_GLU ? pt.n / 2 : pt.n))
            *(frag_t*)((elem_t*)pt.y + (int64_t)row * pt.ldy + c) = *(const frag_t*)(buf + r * PITCH + q * 16);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        accumulators_stay(acc);
      }
    }
    parity ^= 1;
  }
}

// 256 x 128 tiles instead of 256 x 256?  Whichever has the smaller time in rounds of the latter (one workgroup per CU) by a model of both: on
// the XCD with the most tiles, pairs of half tiles share a CU and take 0.97 - 1.26 rounds, the more the longer their K and the fewer rows of them are empty
// (1.05 with fewer than 48 rows in a tile, where they wait for weights), a rest that is alone on its CUs 0.8.  What it is about: grids that leave CUs idle, and last rounds.
// (MI355X, bf16, 256 x 256 / 256 x 128, us: to f32, 65 rows of 32000 x 4096 103 / 84, 300 rows 110 / 133, 1000 rows of 8192 x 4096 79 / 72, 2000
// rows 103 / 138.  Experts: 12 rows each of 32 x 4096 x 1792 145 / 131, 131 rows 158 / 176, 750 rows 415 / 498; 64 x 2048 x 640, 8, 87 and 500 rows, 62 / 49, 62 / 58, 152 / 156.
// With the rows' tiles shared out evenly (row_tiles): 300 tokens, 6 of 32 experts of 1792, width 4096, up, 229 / 303 (before: whole 311), 1200 331 / 542 and, down, 205 / 292, 2000 509 / 715 and 294 / 351; 8 of
// 64 experts of 640, width 2048, 2000 tokens 129 / 212 and 83 / 117, 5800 276 / 388 and 201 / 234.  Over those 44 sizes the choice costs 0.1 % on average, 3.9 % before.
// f32, 65 rows of 4096 x 1024 234 / 129.  Over 113 bf16 sizes the choice costs 0.4 % on average and 9 % at most, 700 tokens' two of 16 experts of 4096 x 4096, 209 us for 192, against the
// better one.)
// max_tiles > 0: rows sorted by group, of which there is a tile for every 256 and one per group.  Part b over rows_b rows: its tiles are the first that
// workgroups of the whole form take, and where its K is longer those end later, by a third of it.
static bool half_tiles(int n, int k, int groups, int max_tiles, int rows_a, int n_b, int k_b, int rows_b) {
  const int row_tiles = max_tiles > 0 ? max_tiles : (rows_a + TM - 1) / TM;
  const int64_t rows = max_tiles > 0 ? (int64_t)TM * max(0, max_tiles - groups) : rows_a;
  auto per_xcd = [&](int tn, int tiles_a) {
    auto part = [&](int tiles, int c) { return ((int64_t)tiles * ((c + tn - 1) / tn) + 7) / 8; };
    return part(tiles_a, n) + part((rows_b + TM - 1) / TM, n_b);
  };
  // (the whole tiles' XCDs share out those that have rows, of experts that differ as many as their mean has and 0.45 more; the half tiles' those that may have.  Of fewer than 144 rows of each
  // expert, 48 of 8 KB of K, which wait for weights, the difference is not made)
  const int filled = max_tiles > 0 && rows >= (k * (int)sizeof(elem_t) >= 8192 ? 48 : 144) * (int64_t)groups ? min(max_tiles, (int)((float)groups * fmaxf(1.f, (float)rows / (float)(TM * groups) + 0.45f))) : row_tiles;
  const int64_t per_h = per_xcd(HTN, row_tiles), per_f = per_xcd(TN, filled);
  const int64_t places = max_tiles > 0 ? groups : row_tiles;
  const float pair = rows < 48 * places ? 1.05f
                                        : (rows < 1000 * places ? 0.97f : 1.01f) + 0.25f * (float)min((int64_t)k * (int)sizeof(elem_t), (int64_t)8192) / 8192.f;
  const int64_t rest = per_h % 64;
  const float half = (float)(per_h / 64) * pair + (rest == 0 ? 0.f : rest <= 32 ? 0.8f : pair);
  const float late = rows_b > 0 && k_b > k ? ((float)k_b / (float)k - 1.f) / 3.f : 0.f;
  return half <= (float)((per_f + 31) / 32) + late;
}

template <int EPI>
static void launch_tiles(const GemmArgs& a, bool half, int64_t wgs, int mt_a, int mt_b, hipStream_t s) {
  if (half) launch_half_tiles(a, EPI, (unsigned)wgs, mt_a, mt_b, s);
  else hipLaunchKernelGGL((gemm_tiles_kernel<EPI>), dim3((unsigned)min((int64_t)256, wgs)), dim3(256), 0, s, a, mt_a, mt_b);      // a workgroup per CU
}

static int check_part(const Part& p, int epi, int act) {
  if (!p.w || !p.x || !p.y || p.n <= 0 || p.k <= 0 || p.k % 64 || p.n % 16 || p.ldx < p.k || p.ldx % FR || p.ldy % FR) return LM_EINVAL;
  if (epi == LM_EPI_GLU && (p.n % 32 || (act != LM_ACT_SILU && act != LM_ACT_GELU_TANH))) return LM_EINVAL;
  if (epi == LM_EPI_GATE && (!p.gate || p.ldg % 4)) return LM_EINVAL;
  if (p.gx % FR || p.gy % 4) return LM_EINVAL;
  return LM_OK;
}

static int fill(GemmArgs& a, const LmGemmPart* pa, const LmGemmPart* pb, int groups, const int* perm, const int* off, int rows_a,
                int rows_b, int x_div, float scale, int epi, int act) {
  auto conv = [](const LmGemmPart* s) {
    return Part{(const elem_t*)s->w, (const elem_t*)s->x, s->ldx, s->y, s->ldy, s->n, s->k, s->gx, s->gy, s->bias,
                (const elem_t*)s->gate, s->ldg};
  };
  if (!pa || groups <= 0 || x_div <= 0 || (perm && !off) || epi < 0 || epi > LM_EPI_GATE) return LM_EINVAL;
  a.a = conv(pa);
  a.b = pb ? conv(pb) : Part{};
  if (check_part(a.a, epi, act) || (pb && check_part(a.b, epi, act))) return LM_EINVAL;
  a.groups = groups; a.perm = perm; a.off = off; a.rows_a = rows_a; a.rows_b = pb ? rows_b : 0; a.x_div = perm ? x_div : 1;
  a.tiles = nullptr; a.scale = scale; a.act = act;
  return LM_OK;
}

template <int NR, int MB, int EPI, int KW = 8>
static int launch_rows(const GemmArgs& a, int max_rows, int has_b, hipStream_t s) {
  const int n = has_b && a.b.n > a.a.n ? a.b.n : a.a.n;
  const dim3 grid((n + 16 * NR - 1) / (16 * NR), a.groups + has_b, a.perm ? 1 : (max_rows + 16 * MB - 1) / (16 * MB));
  hipLaunchKernelGGL((gemm_rows_kernel<NR, MB, KW, EPI>), grid, dim3(64 * KW), 0, s, a);
  return launch_status();
}

// How the products of few rows are dealt: workgroups of 16 nw channels, K slices over the grid (of one matrix, `sliced`).
//
// The least time of a model fitted to the kernel (MI355X, bf16, 1 - 64 rows, 8 - 260 MB of weights): a workgroup takes 0.07 nw + 0.02 per
// 16 rows + 0.02 us per stage, workgroups beyond one per CU add up (a CU takes in about 22 GB/s times 1000, so a 257th tile costs as much as
// 256 more: 16448 channels at 48 rows take 42 us as 257 tiles of 64, 30 as 206 of 80), and slices cost the launch that adds them.  By what
// was measured the channels per workgroup matter most where n / 64 is far from a multiple of 256 (10816 x 4096, 48 rows: 26.5 us at 64,
// 20.8 at 48; 4096 x 4096, 16 rows: 11.8 us at 64 and 4 slices, 9.8 at 16), slices where K is long (4096 x 14336, 48 rows: 40 us, 26
// with 4).  128 channels, bf16: 2 us a round for a ring of 144 KiB that nothing runs beside, but x comes in half as often, and 224 or 250 workgroups are one round where 448
// or 500 are two (heads and gated units; 28672 x 4096, 64 / 128 channels: 16 rows 42.3 / 37.1 us, 48 rows 48.3 / 39.9, 64 rows 51.8 / 41.5; 32000 x 4096, 80 / 128: 48 rows
// 52.0 / 43.4; 32000 x 2048, 16 rows 25.4 / 22.9; two and four rounds of few rows and short K lose: 64000 x 2048 at 1 row 45.9 / 48.5, 128256 x 1024 43.1 / 46.7; 96 and
// 112 channels nowhere the fastest).
// Gated units (64 or 128 channels) of one round of 128: slices of several rounds cost 3.5 us a round more than that, two rounds of 64 channels have none, and 128 channels take 0.39 - 0.58 us a stage as they fill the chip.  (us, one | 64
// rows, what the model without these two chose / now: 28672 x 4096, 4 slices, 48.8 / 36.0 at one row; 24576 x 4096, 2 slices, 43.6 / 31.1 | 51.0 / 37.4; 22016 x 4096, 8 slices, 43.3 / 29.3 | 47.5 /
// 36.5; 10240 x 4096, 8 slices, 23.2 / 18.5; 5120 x 2048, 8 slices, 11.8 / 8.5.)
struct RowsPlan {
  int nw, slices;      // nw 0: gemm_rows_kernel
};
static RowsPlan plan_stream(int groups, int n, int k, int rows, bool glu, bool sliced) {
  RowsPlan best{4, 1};
  float time = 1e30f;
  const int stages = (int)((int64_t)k * (int)sizeof(elem_t) / RB), mb = min(4, (rows + 15) / 16);
  const bool one_round = LM_ELEM == 0 && glu && (int64_t)groups * ((n + 127) / 128) <= 256;
  for (int nw = 5; nw >= 1; --nw) {
    if (glu && nw != 4) continue;                          // (a gate block and its up block share a workgroup)
    const int64_t tiles = (int64_t)groups * ((n + 16 * nw - 1) / (16 * nw));
    for (int s = 1; s <= (sliced ? 8 : 1) && (s == 1 || stages >= 4 * s); s *= 2) {
      float t = (float)((tiles * s + 255) / 256) * (float)((stages + s - 1) / s) * (0.07f * nw + 0.02f * mb + 0.02f);
      if (s > 1) t += 4.5f + (float)s * rows * n * 8.f / 5e6f;
      if (one_round && s > 1) t += tiles > 256 ? 1e30f : 3.5f * (float)((tiles * s - 1) / 256);
      if (t < time) { time = t; best = RowsPlan{nw, s}; }
    }
  }
  auto tiles = [&](int nw) { return (int64_t)groups * ((n + 16 * nw - 1) / (16 * nw)); };
  // 128 channels only in place of workgroups that take K in one chain of stages, as they do: the same order of sums
  if (one_round) {
    if (best.slices == 1 && tiles(best.nw) > 256 && (float)stages * (0.19f + 0.39f * (float)tiles(8) / 256.f + 0.03f * (mb - 1)) + 2.5f < time) best.nw = 8;
    return best;
  }
  if (LM_ELEM == 0 && best.slices == 1 && tiles(best.nw) > 256 &&
      (float)((tiles(8) + 255) / 256) * ((float)stages * (0.07f * 8 + 0.02f * mb + 0.02f) + 2.f) + 0.5f < time)
    best.nw = 8;
  return best;
}

// K parts inside a workgroup where there is no second one to run beside it on its CU
template <int EPI, int NW, bool SHORT, bool TURN, bool IDS, int ROWS16>
static void launch_stream_rows(const GemmArgs& a, int n, int has_b, int slices, float* part, hipStream_t s) {
  const dim3 grid((n + 16 * NW - 1) / (16 * NW), a.groups + has_b, slices);
  constexpr int KW = NW <= 2 ? 4 : NW <= 5 ? 2 : 1;
  if (KW > 1 && (int64_t)grid.x * grid.y * grid.z <= 256)
    hipLaunchKernelGGL((gemm_stream_kernel<EPI, NW, KW, SHORT, TURN, IDS, ROWS16>), grid, dim3(64 * NW * KW), 0, s, a, part);
  else
    hipLaunchKernelGGL((gemm_stream_kernel<EPI, NW, 1, SHORT, TURN, IDS, ROWS16>), grid, dim3(64 * NW), 0, s, a, part);
}
// One matrix, or one per head: a kernel for the very number of row blocks.  A kernel with all four in it keeps more in registers than it has scalar ones.
// (MI355X, bf16, 64 rows, all in one | this: 28672 x 4096 gated 41.9 | 40.8 us, 12352 x 4096 28.0 | 26.1, 10816 x 4096 24.6 | 23.5, 32000 x 4096 45.9 | 44.4; 16 rows of 32000 x 2048
// 23.7 | 23.2, of 2048 x 2048 6.1 | 5.9.)  Experts' rows are known on the device only.
template <int EPI, int NW, bool SHORT, bool TURN = false, bool IDS = false>
static void launch_stream_form(const GemmArgs& a, int n, int has_b, int slices, float* part, hipStream_t s) {
  if constexpr (!IDS && LM_ELEM == 0) {
    if (!a.perm && !has_b && a.rows_a > 64) {      // (in one slice; more rows than a caller's max_rows said, or gated units of more)
      for (int m = 0; m < a.rows_a; m += 64) {
        GemmArgs c = a;
        c.rows_a = min(64, a.rows_a - m);
        c.a.x += m * a.a.ldx;
        c.a.y = (uint8_t*)a.a.y + m * a.a.ldy * (EPI == LM_EPI_F32 ? (int64_t)sizeof(float) : (int64_t)sizeof(elem_t));
        if (EPI == LM_EPI_GATE) c.a.gate += m * a.a.ldg;
        launch_stream_form<EPI, NW, SHORT, TURN, IDS>(c, n, has_b, slices, part, s);
      }
      return;
    }
    const int blocks = a.perm || has_b ? 0 : (a.rows_a + 15) / 16;
    if (blocks == 1) return launch_stream_rows<EPI, NW, SHORT, TURN, IDS, 1>(a, n, has_b, slices, part, s);
    if (blocks == 2) return launch_stream_rows<EPI, NW, SHORT, TURN, IDS, 2>(a, n, has_b, slices, part, s);
    if (blocks == 3) return launch_stream_rows<EPI, NW, SHORT, TURN, IDS, 3>(a, n, has_b, slices, part, s);
    if (blocks == 4) return launch_stream_rows<EPI, NW, SHORT, TURN, IDS, 4>(a, n, has_b, slices, part, s);
  }
  if constexpr (NW == 4 || LM_ELEM != 0) launch_stream_rows<EPI, NW, SHORT, TURN, IDS, 0>(a, n, has_b, slices, part, s);      // (experts: 64 channels a workgroup)
}

// bf16: heads, and gated units of 128 channels, in one slice: workgroups that begin at different k where rows lie whole 4 KiBs apart and are enough to be bound by the memory's
// channels.  (MI355X, in step | so, 16 rows, f32 results, us: 16448 x 4096 27.9 | 24.6, 40960 x 4096 63.0 | 55.3, 8192 x 8192 33.5 | 28.1, 8192 x 4096 16.6 | 16.0; other rows 2 - 5 % the
// other way: 24576 x 2560 23.2 | 24.4, 36864 x 3072 37.6 | 39.0; small products, the router's among them, by 0.6 us: 512 x 2048 5.4 | 6.0, 4096 x 4096 9.5 | 10.1.)
[[maybe_unused]] static bool turns(int n, int64_t k, int slices) { return slices == 1 && k % 2048 == 0 && n * k >= 24 << 20; }

template <int EPI, int NW>
static void launch_stream_tiles(const GemmArgs& a, int n, int has_b, int slices, float* part, hipStream_t s) {
  if (a.a.k < CHAIN_K || (has_b && a.b.k < CHAIN_K)) return launch_stream_form<EPI, NW, true>(a, n, has_b, slices, part, s);
  if constexpr (LM_ELEM == 0 && (EPI == LM_EPI_F32 || (EPI == LM_EPI_GLU && NW == 8))) {
    if (turns(n, a.a.k, slices)) return launch_stream_form<EPI, NW, false, true>(a, n, has_b, slices, part, s);
  }
  launch_stream_form<EPI, NW, false>(a, n, has_b, slices, part, s);
}

template <int EPI>
static int launch_stream(const GemmArgs& a, int has_b, RowsPlan pl, float* part, hipStream_t s, bool leave = false) {      // leave: the K slices' sums stay as they are
  const int n = has_b && a.b.n > a.a.n ? a.b.n : a.a.n;
  if (LM_ELEM == 0 && (a.perm || has_b) && pl.nw != 4) return LM_EINVAL;      // (no such kernels: launch_stream_form)
  if constexpr (EPI == LM_EPI_GLU) {
    if (LM_ELEM == 0 && pl.nw == 8) launch_stream_tiles<EPI, LM_ELEM == 0 ? 8 : 4>(a, n, has_b, pl.slices, part, s);
    else launch_stream_tiles<EPI, 4>(a, n, has_b, pl.slices, part, s);
  } else {
    switch (pl.nw) {
#if LM_ELEM == 0
      case 8: launch_stream_tiles<EPI, 8>(a, n, has_b, pl.slices, part, s); break;
#endif
      case 1: launch_stream_tiles<EPI, 1>(a, n, has_b, pl.slices, part, s); break;
      case 2: launch_stream_tiles<EPI, 2>(a, n, has_b, pl.slices, part, s); break;
      case 3: launch_stream_tiles<EPI, 3>(a, n, has_b, pl.slices, part, s); break;
      case 4: launch_stream_tiles<EPI, 4>(a, n, has_b, pl.slices, part, s); break;
      default: launch_stream_tiles<EPI, 5>(a, n, has_b, pl.slices, part, s); break;
    }
  }
  if (pl.slices > 1 && !leave) {
    const int64_t q = (int64_t)a.rows_a * ((EPI == LM_EPI_GLU ? n / 2 : n) / 4);
    hipLaunchKernelGGL((gemm_reduce_kernel<EPI>), dim3((unsigned)((q + 255) / 256)), dim3(256), 0, s, a, part, pl.slices);
  }
  return launch_status();
}

// Which kernel, and how dealt.  experts: groups by perm or two parts; how many of them have rows is not known here, and 64 channels measured best from
// 60 to 1000 MB.  gemm_rows_kernel takes (figures: MI355X, us, stream / gemm_rows_kernel, bf16 where nothing else is said)
//   * more than 64 rows of few channels (the router of a prompt) or of one matrix per head: workgroups along the rows;
//   * 33 - 64 rows where channels and K slices make too few workgroups: there too (64 rows: 64 x 2048 7.7 in 8 slices / 6.1; 8 heads of
//     128 x 512 4.2 / 3.8; but 16 heads of 128 x 256 3.7 / 4.7, and 128 x 4096 is better in slices);
//   * up to 16 rows where a ring is only filled once: up to 4096 channels (16 heads of 256 x 128 3.5 / 3.2, 4096 x 128 3.2 / 2.8; 4096 x 256 3.2 / 3.3; f32
//     4096 x 192 4.0 / 3.6, 16 heads of 128 x 256 3.7 / 3.3, and at 32 rows 4.0 / 3.5), 9600 to 16384 of K up to 128 with 32 channels per
//     workgroup (32 heads of 512 x 128 3.8 / 3.8, weights in the caches 3.5 / 3.0; of 512 x 64 3.3 / 2.9; 512 x 256 4.4 / 4.8; 32000 x 128 4.5 / 5.8);
//   * up to 16 tokens of few small experts, which leave the stream too few workgroups (1 and 16 tokens, 2 of 8 x 1024 x 1024 5.5 / 3.9 and 6.7 / 6.4, of
//     512 x 512 4.4 / 3.2 and 4.7 / 3.5; but 4 of 16 x 1024 x 512 5.2 / 8.6 at 16);
//   * the gated unit of up to 16 rows over few weights, whose stream of 64 channels per workgroup has too few workgroups (16 rows: 2048 x 512
//     4.7 / 3.9, 4096 x 256 4.2 / 3.7, 2048 x 1024 6.4 / 6.1, 4096 x 1024 6.5 / 6.2; 1024 x 2048 9.1 / 9.2; f32 2048 x 1024 9.3 / 10.2), with short K also of more rows (17 and 32 rows: 2048 x 512 4.8 /
//     4.4 and 4.9 / 4.6, 4096 x 512 4.9 / 4.5 and 5.0 / 4.6; 1024 x 512 4.2 / 4.4; 64 rows 5.7 / 5.8; f32 13.3 / 11.4).
static RowsPlan plan_rows(int groups, int n, int k, int rows, int epi, bool experts, bool sliced) {
  const int64_t bytes_k = (int64_t)k * (int)sizeof(elem_t), channels = (int64_t)groups * n;
  if (experts && epi != LM_EPI_GLU && rows <= 16 && channels <= 8192) return RowsPlan{0, 1};
  if (experts && (epi == LM_EPI_GLU || rows <= 64)) return RowsPlan{4, 1};
  if (epi == LM_EPI_GLU) {
    if (rows <= 16 && channels * bytes_k <= (bytes_k <= 2048 ? 8 << 20 : 4 << 20)) return RowsPlan{0, 1};
    if (rows <= (LM_ELEM ? 64 : 32) && k <= 512 && channels >= 2048 && channels <= 4096) return RowsPlan{0, 1};
    return plan_stream(groups, n, k, rows, true, sliced);
  }
  if (rows > 64) return RowsPlan{0, 1};
  const RowsPlan pl = plan_stream(groups, n, k, rows, false, sliced);
  if (rows > 32 && n <= 256 && channels <= 1024 && (pl.slices == 1 || bytes_k <= 4096)) return RowsPlan{0, 1};
  if (k <= 256 && n <= 256 && channels <= 2048 && rows <= 32) return RowsPlan{0, 1};
  if (rows <= 16 && channels <= 4096 && k <= 256 && bytes_k <= 768) return RowsPlan{0, 1};
  if (rows <= 16 && channels >= 9600 && channels <= 16384 && k <= 128) return RowsPlan{0, 1};
  return pl;
}

// ... of a product whose slices the norm behind it adds up (lm_gemm_sums): as lm_gemm_rows has them where those are slices; else slices too where whole K leaves a workgroup few channels, each of
// which brings x in again, and they pay for what the norm reads: 1.5 us by the model, in one round of workgroups.  (MI355X, bf16, product and norm, whole K | slices, us: 4096 x 4096, 64 rows 18.1 | 15.4,
// 48 16.8 | 14.9, 24 14.6 | 13.1; 2048 x 2048, 64 rows 11.8 | 10.2, 24 9.6 | 8.6, 16 8.6 | 8.1; 3072 x 3072, 48 rows 14.2 | 12.4; without the launch that adds up, 2048 x 4096, 48 rows 14.7 | 11.7.)
static RowsPlan plan_sums(int n, int k, int rows) {
  RowsPlan best = plan_rows(1, n, k, rows, LM_EPI_ELEM, false, true);
#if LM_ELEM == 0
  if (best.nw == 0 || best.slices > 1 || n < 2048) return best;
  const int stages = (int)((int64_t)k * (int)sizeof(elem_t) / RB), mb = min(4, (rows + 15) / 16);
  auto stage = [&](int nw) { return 0.07f * nw + 0.02f * mb + 0.02f; };
  float time = (float)((((n + 16 * best.nw - 1) / (16 * best.nw)) + 255) / 256) * (float)stages * stage(best.nw) - 1.5f;
  for (int nw = 4; nw >= 1; nw /= 2)
    for (int s = 2; s <= 4 && stages >= 8 * s && (n + 16 * nw - 1) / (16 * nw) * s <= 256; s *= 2) {
      const float t = (float)((stages + s - 1) / s) * stage(nw) + (float)s * rows * n * 8.f / 5e6f;
      if (t < time) { time = t; best = RowsPlan{nw, s}; }
    }
#endif
  return best;
}

template <int EPI>
static int launch_few(const GemmArgs& a, int max_rows, int has_b, float* part, hipStream_t s) {
  const bool one = a.groups == 1 && !a.perm && !has_b && max_rows <= 64 && max_rows == a.rows_a;
  RowsPlan pl = plan_rows(a.groups, has_b && a.b.n > a.a.n ? a.b.n : a.a.n, a.a.k, max_rows, EPI, a.perm || has_b, one && part != nullptr);
  // the stream's DMA takes whole 16-byte pieces; loads into registers may start anywhere
  uintptr_t at = (uintptr_t)a.a.w | (uintptr_t)a.a.x;
  if (has_b) at |= (uintptr_t)a.b.w | (uintptr_t)a.b.x;
  if (at & 15) pl = RowsPlan{0, 1};
  if (pl.nw > 0) return launch_stream<EPI>(a, has_b, pl, part, s);
  if constexpr (EPI == LM_EPI_GLU) {
    if (max_rows <= 16) return launch_rows<2, 1, EPI>(a, max_rows, has_b, s);
    else if (max_rows <= 32) return launch_rows<2, 2, EPI>(a, max_rows, has_b, s);
    else return launch_rows<2, 4, EPI>(a, max_rows, has_b, s);
  } else {
    if (max_rows > 64) return launch_rows<2, 4, EPI>(a, max_rows, has_b, s);
    else if (max_rows <= 16 && (int64_t)a.groups * a.a.n > 4096 && !a.perm) return launch_rows<2, 1, EPI, 4>(a, max_rows, has_b, s);
    else return launch_rows<1, 1, EPI>(a, max_rows, has_b, s);
  }
}

}  // namespace lm

using namespace lm;

extern "C" int lm_gemm_rows(const LmGemmPart* pa, const LmGemmPart* pb, int groups, const int* perm, const int* off, int rows_a,
                            int rows_b, int x_div, int max_rows, float scale, int epi, int act, float* part, void* stream) {
  GemmArgs a;
  if (fill(a, pa, pb, groups, perm, off, rows_a, rows_b, x_div, scale, epi, act) || max_rows <= 0) return LM_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const int has_b = pb && rows_b > 0;
  if (epi == LM_EPI_GLU) return launch_few<LM_EPI_GLU>(a, max_rows, has_b, part, s);
  if (epi == LM_EPI_GATE) return launch_few<LM_EPI_GATE>(a, max_rows, has_b, part, s);
  return epi == LM_EPI_F32 ? launch_few<LM_EPI_F32>(a, max_rows, has_b, part, s) : launch_few<LM_EPI_ELEM>(a, max_rows, has_b, part, s);
}

// are the products of a mixture of experts those of gemm_stream_kernel with 64 channels?
static bool chosen_streams(int groups, int n, int k, int tokens, int epi) { return plan_rows(groups, n, k, tokens, epi, true, false).nw == 4; }

extern "C" int lm_gemm_chosen_ok(int groups, int n, int k, int tokens, int top, int epi) {
  return LM_ELEM == 0 && groups > 0 && n > 0 && k > 0 && tokens > 0 && tokens <= LM_CHOOSE_TOKENS && top > 0 && top <= LM_MAX_TOP && (epi == LM_EPI_GLU || epi == LM_EPI_ELEM) &&
         chosen_streams(groups, n, k, tokens, epi);
}

extern "C" int lm_gemm_chosen(const LmGemmPart* pa, const LmGemmPart* pb, int groups, const int* ids, int tokens, int top, int x_is_pairs, float scale, int epi, int act,
                              void* stream) {
#if LM_ELEM == 0
  GemmArgs a;
  if (!ids || tokens <= 0 || top <= 0 || fill(a, pa, pb, groups, nullptr, nullptr, 0, tokens, x_is_pairs ? 1 : top, scale, epi, act)) return LM_EINVAL;
  const int has_b = pb != nullptr, n = has_b && a.b.n > a.a.n ? a.b.n : a.a.n;
  if (!lm_gemm_chosen_ok(groups, n, a.a.k, tokens, top, epi)) return LM_EINVAL;
  uintptr_t at = (uintptr_t)a.a.w | (uintptr_t)a.a.x;
  if (has_b) at |= (uintptr_t)a.b.w | (uintptr_t)a.b.x;
  if (at & 15) return LM_EINVAL;
  a.off = ids; a.rows_a = tokens * top; a.x_div = x_is_pairs ? 1 : top;
  hipStream_t s = (hipStream_t)stream;
  const bool is_short = a.a.k < CHAIN_K || (has_b && a.b.k < CHAIN_K);
  if (epi == LM_EPI_GLU) {
    if (is_short) launch_stream_form<LM_EPI_GLU, 4, true, false, true>(a, n, has_b, 1, nullptr, s);
    else launch_stream_form<LM_EPI_GLU, 4, false, false, true>(a, n, has_b, 1, nullptr, s);
  } else {
    if (is_short) launch_stream_form<LM_EPI_ELEM, 4, true, false, true>(a, n, has_b, 1, nullptr, s);
    else launch_stream_form<LM_EPI_ELEM, 4, false, false, true>(a, n, has_b, 1, nullptr, s);
  }
  return launch_status();
#else
  return LM_EINVAL;
#endif
}

extern "C" int lm_gemm_sums(const LmGemmPart* pa, int rows, float* sums, void* stream) {
  GemmArgs a;
  if (fill(a, pa, nullptr, 1, nullptr, nullptr, rows, 0, 1, 1.f, LM_EPI_ELEM, 0) || rows <= 0 || rows > 64 || !sums || ((uintptr_t)a.a.w | (uintptr_t)a.a.x) % 16) return LM_EINVAL;
  const RowsPlan pl = plan_sums(a.a.n, a.a.k, rows);
  if (pl.nw == 0 || pl.slices < 2) return LM_EINVAL;
  return launch_stream<LM_EPI_ELEM>(a, 0, pl, sums, (hipStream_t)stream, true);
}

extern "C" int64_t lm_gemm_rows_scratch(int n, int k, int rows, int epi) {
  if (n <= 0 || k <= 0 || rows <= 0 || rows > 64) return 0;
  const int s = plan_rows(1, n, k, rows, epi, false, true).slices;
  return s > 1 ? (int64_t)s * rows * n : 0;
}

extern "C" int64_t lm_gemm_sums_room(int n, int k, int rows) {
  if (n <= 0 || k <= 0 || rows <= 0 || rows > 64) return 0;
  const RowsPlan pl = plan_sums(n, k, rows);
  return pl.nw > 0 && pl.slices > 1 ? (int64_t)pl.slices * rows * n : 0;
}

extern "C" int lm_gemm_rows_channels(int groups, int n, int k, int rows, int epi, int sliced, int* slices) {
  const RowsPlan pl = plan_rows(groups, n, k, rows, epi, false, sliced != 0);
  if (slices) *slices = pl.slices;
  return 16 * pl.nw;
}

extern "C" int lm_gemm_tile_channels(int n, int k, int groups, int max_tiles, int rows_a, int n_b, int k_b, int rows_b) {
  return half_tiles(n, k, groups, max_tiles, rows_a, n_b, k_b, rows_b) ? HTN : TN;
}

extern "C" int lm_gemm_tiles(const LmGemmPart* pa, const LmGemmPart* pb, int groups, const int* perm, const int* off,
                             const int* tiles, int max_tiles, int rows_a, int rows_b, int x_div,
                             float scale, int epi, int act, void* stream) {
  GemmArgs a;
  if (fill(a, pa, pb, groups, perm, off, rows_a, rows_b, x_div, scale, epi, act)) return LM_EINVAL;
  if (epi == LM_EPI_GATE || (groups > 1 && !perm)) return LM_EINVAL;      // few rows only
  if (perm && (!tiles || max_tiles <= 0)) return LM_EINVAL;
  a.tiles = perm ? tiles : nullptr;
  const int mt_a = perm ? max_tiles : (rows_a + TM - 1) / TM, mt_b = pb && rows_b > 0 ? (rows_b + TM - 1) / TM : 0;
  const bool half = half_tiles(a.a.n, a.a.k, groups, perm ? max_tiles : 0, rows_a, a.b.n, a.b.k, mt_b ? rows_b : 0);
  const int tn = half ? HTN : TN;
  const int64_t tiles_a = (int64_t)mt_a * ((a.a.n + tn - 1) / tn), tiles_b = mt_b ? (int64_t)mt_b * ((a.b.n + tn - 1) / tn) : 0;
  if (tiles_a <= 0 || tiles_a + tiles_b > (1 << 30)) return LM_EINVAL;
  const int64_t wgs = 8 * ((tiles_a + 7) / 8 + (tiles_b + 7) / 8);
  hipStream_t s = (hipStream_t)stream;
  if (epi == LM_EPI_ELEM) launch_tiles<LM_EPI_ELEM>(a, half, wgs, mt_a, mt_b, s);
  else if (epi == LM_EPI_F32) launch_tiles<LM_EPI_F32>(a, half, wgs, mt_a, mt_b, s);
  else launch_tiles<LM_EPI_GLU>(a, half, wgs, mt_a, mt_b, s);
  return launch_status();
}
