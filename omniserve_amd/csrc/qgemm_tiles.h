// W8A8 prefill GEMM in 256-row x 256-channel tiles: M >= 256, N % 256 == 0, K % 256 == 0.  (included by qgemm_kernel.h)
//
// What bounds w4a8_gemm_exact_kernel at W8A8 is neither HBM nor the matrix units but what a CU takes in: a 128 x 256 tile asks for 96 bytes
// per 16.8 KOP (11 TB/s of L2 reads at 1950 TOPS, and its weights cross the LDS twice to be transposed).  A 256 x 256 tile asks for 64, and
// both operands lie in LDS as the matrix instruction wants them.  The price is a whole CU per workgroup: four waves of 128 rows x 128
// channels with 256 accumulation registers each, one per SIMD, so that nothing overlaps but what a wave issues itself (mfma_pinned.h):
//
//  * stages of 128 bytes of k (64 KB), two of them: the fragments of a half stage are read while the half before it multiplies, the stage
//    after next is requested as soon as every wave has the current one in registers.
//  * ahead of the requests a wave touches 32 lines of the stage behind them (touch_lines32): 64 rows of each operand a workgroup, the other rows by
//    those of the 32 workgroups of an XCD that have the same rows (four neighbouring columns) or channels: as many as a band has row tiles.  Four of them touch all
//    channels; bands of three, which 5, 6 and 9 row tiles make, leave a quarter to the requests.
//  * a workgroup takes tile after tile of its XCD; the first two stages of the next one are on their way while it stores this one.
//
// Integer sums and the general kernel's epilogue: the same bits.
//
//  * the stores stream: 256 workgroups write 33 MB at the ends of their tiles, as much as all L2s hold, which keep the operands.
// MI355X, us, 12001 rows of 28672 x 4096 | 4096 x 14336, what is compared in turn on one box (boxes differ by a tenth, by the card's power):
//  * w4a8_gemm_exact_kernel's best tiles -> here 1406 -> 1057 (2670 TOPS) | 681 -> 499 (2820 TOPS); of 6144 x 4096 304 -> 245;
//  * without -> with lines touched ahead 1206 -> 1118 | 512 -> 487 (two stages ahead 1134 | 489; every workgroup its whole tile 1168 | 535; the operands of all tiles the first
//    one's, so that the L2 has everything, 983 | 445; no requests at all 934 | 398; no LDS reads 1182 | 498); a line of the tile that is there anyway -> the lines ahead 1067 -> 1056 |
//    516 -> 500, and of 28672 x 4096 in bands of four 1024 rows 113 -> 105, 2048 213 -> 200, in bands of three 1501 163 -> 157, 2100 217 -> 216; of 4096 x 14336 2100 166 -> 150, 2331 166 -> 131;
//  * results stored -> streamed 1038 -> 1013 | 470 -> 461, accumulators zeroed -> not 1013 -> 996 | 460 -> 459.
//  * the next tile requested behind -> before the scaling of the results: 0.99 of the time over 31 sizes without the unit (12001 rows of 6144 x 4096 246 -> 242, 4000 of 4096 x 4096 54.1 -> 52.3, 12001 of 4096 x 14336 482 -> 480;
//    3700 of 6144 x 4096 92.1 -> 94.4, 7900 of 4096 x 4096 105.6 -> 107.0 are the slower ones); with the unit: launch_tiles.
// What is left of the 5 POPS nominal is the clock under this load, the ends of a tile, which 4096 of K show, and the L2.
#pragma once
#include "lm/mfma_pinned.h"

namespace omni {

constexpr int TILES_M = 256, TILES_N = 256, TILES_K = 128;
constexpr int TILES_STAGE = (TILES_M + TILES_N) * TILES_K;

// LDS row of 128 bytes: 16-byte piece s of row r at slot s ^ tiles_swizzle(r).  ds_read_b128 serves rows 0 - 3 and 12 - 15 at one piece with
// rows 4 - 11 at its neighbour: sixteen different places of two rows' 256 bytes answer.
__device__ __forceinline__ int tiles_swizzle(int row) {
  const int q = (row >> 1) & 7;
  return (((q ^ ((q >> 1) & 2)) & 3) << 1) | (q >> 2);
}
__device__ __forceinline__ void tiles_dma16(uint32_t src, const void* base, uint32_t lds_dst) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(src), "s"(lds_dst), "s"(base)
               : "memory");
}

// SILU: out = silu(gate) up of a [gate | up] weight, [M][N / 2]: rows 0 - 63 and 128 - 191 of a tile are 128 gate channels, the others the up channels of the same place, so that
// a wave has both.  Half the stores pay for the exponentials; what it saves is the other half's way
// through memory: 12001 rows of 28672 x 4096, the quantiser behind the product 156 -> 90 us, both 1.03x of a whole prompt.
// SHARE: tile_share.h.  LATE: the next tile is requested behind the scaling of this one's results, not in front of it (launch_tiles).
template <int MODE, bool SILU = false, bool SHARE = false, bool LATE = false>
__global__ __launch_bounds__(256, 1) void w8a8_tiles_kernel(GemmArgs p, TileShare share) {
  static_assert(MODE == MODE_W8, "rows of int8 weights");
  static_assert(!(LATE && SHARE), "parts of a tile are left with the next part requested");
  constexpr int PITCH = 128 * 2 + 16;                       // a row of the write-back buffers: a wave's 128 channels
  // one object: the stages, four write-back buffers of 16 rows, the scales of two tiles
  constexpr int LDS_OUT = 2 * TILES_STAGE, LDS_SC = LDS_OUT + 4 * 16 * PITCH, LDS_SINK = LDS_SC + 2 * 1024;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_SINK + 128 + (SHARE ? 16 : 0)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = 128 * (wave & 1), wm = 128 * (wave >> 1);
  // XCD x takes the x-th contiguous eighth of the tiles, counted down the columns of bands of row tiles (as w4a8_gemm_exact_kernel)
  const int tiles = p.tiles_m * p.tiles_n, xcd = blockIdx.x & 7;
  const int own = (tiles >> 3) + (xcd < (tiles & 7)), first = xcd * (tiles >> 3) + min(xcd, tiles & 7);
  int at = blockIdx.x >> 3;
  TileParts parts(at, own, p.K / TILES_K);                  // (SHARE)

  // a wave's part of a stage: 64 rows of the weights and 64 of the activations, 8 a piece (lane: row lane / 8, slot lane % 8)
  uint32_t src[8];
  {
    const int l = lane_here();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 64 * wave + 8 * i + (l >> 3);
      src[i] = (uint32_t)r * (uint32_t)p.K + (((l & 7) ^ tiles_swizzle(r)) << 4);
    }
  }
  const uint8_t *wbase = nullptr, *abase = nullptr;         // of the next stage
  const uint32_t dst0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds + 64 * TILES_K * wave);
  auto dst = [&](int t, int i) { return dst0 + (t & 1) * TILES_STAGE + 1024 * (i & 7) + (i < 8 ? 0 : TILES_N * TILES_K); };
  auto stage = [&](int t) {
#pragma unroll
    for (int i = 0; i < 16; ++i) tiles_dma16(src[i & 7], i < 8 ? wbase : abase, dst(t, i));
    wbase += TILES_K;
    abase += TILES_K;
  };
  int ns = p.K / TILES_K;                                   // stages of the part opened last: four or more
  // first channel of a quarter of the tile's rows, from the tile's
  auto quarter = [&](int q) { return SILU ? 64 * (q >> 1) + (q & 1) * (p.N >> 1) : 64 * q; };
  const uint8_t* soon = nullptr;                            // the lane's line of the stage behind the one requested last: of the weights (lanes 0 - 15) or the activations
  const uint32_t sink = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds + LDS_SINK);
  int m0 = 0, n0 = 0;
  uint16_t sw_next = 0, sa_next = 0;                        // the thread's channel's and row's scales of the tile opened last
  // requests the next tile's first two stages; false: there is none.  The last row tile starts at M - 256: the rows that it shares with the
  // one before are computed twice, to the same bits.
  auto open_tile = [&]() {
    int k0 = 0;
    if constexpr (SHARE) {
      if (!parts.next(at)) return false;
      k0 = parts.k0 * TILES_K;
      ns = parts.stages;
    } else {
      if (at >= own) return false;
    }
    const int id = first + (SHARE ? parts.tile : at), band = id / (p.tile_linear * p.tiles_n), in = id - band * p.tile_linear * p.tiles_n;
    const int rows = min(p.tile_linear, p.tiles_m - band * p.tile_linear), tn = in / rows;
    at += (int)gridDim.x >> 3;
    n0 = tn * (SILU ? TILES_N / 2 : TILES_N);
    m0 = min((band * p.tile_linear + in - tn * rows) * TILES_M, p.M - TILES_M);
    {
      const int l = lane_here();                            // (in & 3: in % rows where rows is four)
      const uint8_t *aq = (const uint8_t*)p.A + (size_t)(m0 + 64 * (tn & 3)) * p.K, *wq = p.W + (size_t)(n0 + quarter(in & 3)) * p.K;
      soon = (l & 16 ? aq : wq) + ((uint32_t)(16 * wave + (l & 15)) * (uint32_t)p.K + k0 + 2 * TILES_K);
    }
    wbase = p.W + (int64_t)__builtin_amdgcn_readfirstlane(n0 + (quarter(wave) - 64 * wave)) * p.K + k0;      // (its rows' offsets hold 64 * wave)
    abase = (const uint8_t*)p.A + (size_t)m0 * p.K + k0;
    if constexpr (SHARE) {
      wbase = wave_uniform(wbase);
      abase = wave_uniform(abase);
    }
    const int tid = 64 * wave + lane_here();
    sw_next = ((const uint16_t*)p.wscales)[n0 + quarter(wave) + lane_here()];
    sa_next = ((const uint16_t*)p.ascales)[m0 + tid];
    stage(0);
    stage(1);
    touch_lines32(soon, sink);                              // (there are four stages)
    return true;
  };
  // ... its scales in LDS: 256 channels', 256 rows'
  auto park = [&](int parity) {
    uint16_t* s = (uint16_t*)(lds + LDS_SC + 1024 * parity) + 64 * wave + lane_here();
    s[0] = sw_next;
    s[256] = sa_next;
  };

  int off[2];                                               // of a fragment of half u inside 16 rows
  v4i a[2][8], b[2][8], acc[8][8];
  auto fetch_a = [&](int t, auto half, int i) {
    constexpr int U = decltype(half)::value;
    a[U][i] = *(const v4i*)(lds + (t & 1) * TILES_STAGE + 16 * TILES_K * i + off[U] + wn * TILES_K);
  };
  auto fetch_b = [&](int t, auto half, int i) {
    constexpr int U = decltype(half)::value;
    b[U][i] = *(const v4i*)(lds + (t & 1) * TILES_STAGE + 16 * TILES_K * i + off[U] + (TILES_N + wm) * TILES_K);
  };
#define OMNI_TILES_OP "v_mfma_i32_16x16x64_i8"
  // Stage t: FRESH: the tile's first (no accumulators are zeroed: 256 instructions of a lone wave), MORE: there is a stage t + 1, DMA: and a stage t + 2.  Requests and reads go out one by one between the products (a burst of them
  // fills the queues, where the lone wave, which issues in order, waits).  No condition inside: one basic block.
  auto step = [&](int t, auto fresh, auto more, auto dma) {
    constexpr bool FRESH = decltype(fresh)::value, MORE = decltype(more)::value, DMA = decltype(dma)::value;
    auto four = [&](auto half, int i0, int j) {
      constexpr int U = decltype(half)::value;
#pragma unroll
      for (int i = i0; i < i0 + 4; ++i) {
        if constexpr (FRESH && U == 0) OMNI_MFMA_FRESH(OMNI_TILES_OP, acc[i][j], a[U][i], b[U][j]);
        else OMNI_MFMA_PINNED(OMNI_TILES_OP, acc[i][j], a[U][i], b[U][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      fetch_b(t, IntTag<1>{}, j);
      __builtin_amdgcn_sched_barrier(0);
      four(IntTag<0>{}, 0, j);
      fetch_a(t, IntTag<1>{}, j);
      __builtin_amdgcn_sched_barrier(0);
      four(IntTag<0>{}, 4, j);
    }
    // stage t + 1 is there for every wave, and everyone has stage t in registers
    if constexpr (MORE && DMA) asm volatile("s_waitcnt vmcnt(1) lgkmcnt(0)" ::: "memory");      // (behind its requests only lines are touched)
    else if constexpr (MORE) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (MORE) {
          if (h) fetch_a(t + 1, IntTag<0>{}, j);
          else fetch_b(t + 1, IntTag<0>{}, j);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (DMA) {
          OMNI_MFMA3_DMA16(OMNI_TILES_OP, "%10", acc[4 * h][j], acc[4 * h + 1][j], acc[4 * h + 2][j], a[1][4 * h], a[1][4 * h + 1], a[1][4 * h + 2],
                           b[1][j], src[j], h ? abase : wbase, dst(t, 8 * h + j));
          OMNI_MFMA_PINNED(OMNI_TILES_OP, acc[4 * h + 3][j], a[1][4 * h + 3], b[1][j]);
          __builtin_amdgcn_sched_barrier(0);
        } else {
          four(IntTag<1>{}, 4 * h, j);
        }
      }
    }
    if constexpr (DMA) {
      wbase += TILES_K;
      abase += TILES_K;
      soon += TILES_K & (t + 3 < ns ? -1 : 0);
      touch_lines32(soon, sink);
    }
  };

  int parity = 0;
  bool open = open_tile();
  if (open) park(0);
  while (open) {
    // stage 0 is there: of what was requested last -- stage 1 and lines, or stores of the tile before -- 17 may still fly
    asm volatile("s_waitcnt vmcnt(17)" ::: "memory");
    __syncthreads();
    if constexpr (SHARE) {
      wbase = wave_uniform(wbase);
      abase = wave_uniform(abase);
    }
    const int fl = lane_here();
#pragma unroll
    for (int u = 0; u < 2; ++u) off[u] = (fl & 15) * TILES_K + (((4 * u + (fl >> 4)) ^ tiles_swizzle(fl & 15)) << 4);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      fetch_b(0, IntTag<0>{}, i);
      fetch_a(0, IntTag<0>{}, i);
    }
    int t = 1;
    step(0, BoolTag<true>{}, BoolTag<true>{}, BoolTag<true>{});
    for (; t + 2 < ns; ++t) step(t, BoolTag<false>{}, BoolTag<true>{}, BoolTag<true>{});
    if (t + 1 < ns) {                                       // (always: it keeps the two steps in blocks of their own)
      step(t, BoolTag<false>{}, BoolTag<true>{}, BoolTag<false>{});
      ++t;
    }
    step(t, BoolTag<false>{}, BoolTag<false>{}, BoolTag<false>{});      // (behind its barrier both stages are free)
    accumulators_settle(acc);

    // The next tile's requests, then the results, which stay in the accumulation registers until they are stored (LATE: the results packed, then the requests, then the stores).  The arithmetic of the general kernel: both scales' product, the sum times it, each
    // rounded to f32, then to fp16 -- opaque in between, or hipcc folds the last two into one rounding.
    const int el = lane_here(), e15 = el & 15, e4 = el >> 4;
    const uint8_t* sc = lds + LDS_SC + 1024 * parity;
    half_t* const out = p.out + (size_t)(m0 + wm) * p.out_stride + n0 + (SILU ? wn / 2 : wn);
    const TileParts mine = parts;
    bool opened = false;
    if constexpr (SHARE) {
      if (mine.shared()) {
        const bool last = mine.finishes(share, lds + LDS_SINK + 128, acc, [&] {
          opened = true;
          open = open_tile();
        });
        if (!last) {
          parity ^= 1;
          if (open) park(parity);
          continue;
        }
      }
    }
    if (!LATE && !opened) open = open_tile();
    uint8_t* buf = lds + LDS_OUT + wave * 16 * PITCH;
    // through LDS, so that a row leaves in whole 16-byte pieces of neighbouring lanes: 16 rows of the wave's at a time
    auto put = [&](int j, const uint2 (&h)[8]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < (SILU ? 4 : 8); ++i) *(uint2*)(buf + e15 * PITCH + (16 * i + 4 * e4) * 2) = SILU ? silu_mul_h4(h[i], h[i + 4 & 7]) : h[i];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < (SILU ? 2 : 4); ++i) {
        const int r = SILU ? 8 * i + (el >> 3) : 4 * i + e4, q = SILU ? el & 7 : e15;
        __builtin_nontemporal_store(*(const v4i*)(buf + r * PITCH + q * 16), (v4i*)(out + (size_t)(16 * j + r) * p.out_stride + q * 8));
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    auto store = [&](auto add) __attribute__((always_inline)) {
      constexpr bool ADD = decltype(add)::value;
      accumulators_stay(acc);
      float sw[8][4];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint2 w = *(const uint2*)(sc + 2 * (wn + 16 * i + 4 * e4));
        const uint32_t wv[2] = {w.x, w.y};
#pragma unroll
        for (int e = 0; e < 4; ++e) sw[i][e] = (float)__builtin_bit_cast(half_t, (uint16_t)(wv[e >> 1] >> (16 * (e & 1))));
      }
      v4i x[16];                                            // ADD: of two blocks of rows
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (ADD) if (j % 2 == 0) {
          mine.others(share, [&](int q) { return 8 * (q & 7) + j + (q >> 3); }, x);
          accumulators_stay(acc);
        }
        const float sa = (float)*(const half_t*)(sc + 512 + 2 * (wm + 16 * j + e15));
        uint2 h[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          uint32_t hw[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const v4i& y = x[8 * (j & 1) + i];
            const int c0 = acc[i][j][2 * e] + (ADD ? y[2 * e] : 0), c1 = acc[i][j][2 * e + 1] + (ADD ? y[2 * e + 1] : 0);
            v2f r = (v2f){(float)c0 * (sw[i][2 * e] * sa), (float)c1 * (sw[i][2 * e + 1] * sa)};
            asm volatile("" : "+v"(r));
            hw[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, v2h));
          }
          h[i] = make_uint2(hw[0], hw[1]);
        }
        put(j, h);
      }
    };
    if constexpr (LATE) {
      uint2 packed[8][8];                                   // [row block][channel block]
      float sa[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sa[j] = (float)*(const half_t*)(sc + 512 + 2 * (wm + 16 * j + e15));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint2 w = *(const uint2*)(sc + 2 * (wn + 16 * i + 4 * e4));
        const uint32_t wv[2] = {w.x, w.y};
        float sw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) sw[e] = (float)__builtin_bit_cast(half_t, (uint16_t)(wv[e >> 1] >> (16 * (e & 1))));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          uint32_t hw[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            v2f r = (v2f){(float)acc[i][j][2 * e] * (sw[2 * e] * sa[j]), (float)acc[i][j][2 * e + 1] * (sw[2 * e + 1] * sa[j])};
            asm volatile("" : "+v"(r));
            hw[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, v2h));
            asm volatile("" : "+v"(hw[e]));                 // (converted here, not where it is stored: half the registers)
          }
          packed[j][i] = make_uint2(hw[0], hw[1]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      open = open_tile();
#pragma unroll
      for (int j = 0; j < 8; ++j) put(j, packed[j]);
    } else if (SHARE && mine.shared()) {
      store(BoolTag<SHARE>{});
    } else {
      store(BoolTag<false>{});
    }
    parity ^= 1;
    if (open) park(parity);
  }
#undef OMNI_TILES_OP
}

}  // namespace omni
