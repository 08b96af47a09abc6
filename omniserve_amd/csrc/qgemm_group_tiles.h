// W4A8 prefill GEMM in 256-row x 256-channel tiles: M >= 256, N % 256 == 0, K % 256 == 0, K >= 512.  (included by qgemm_grp.hip, qgemm_chn_tiles.hip and qgemm_silu_rows.hip)
//
// What bounds w4a8_gemm_exact_kernel per-group is the second level: 5.5 operations (9.5 where a scale is above 17) for each word of four weights, done again for
// every 64 - 128 rows, beside products that leave three issue slots each.  Here a wave has 64 channels and all 256 rows of the tile, so that a word is
// unpacked once for 16 row blocks: 16 words and 64 products for 64 k, one word between four products.  The frame is qgemm_tiles.h's: a workgroup of four waves
// to a compute unit, 256 accumulation registers each, stages of 128 k (a group of the second level), tile after tile of an XCD.
//
//  * activations (32 KB a stage) lie in LDS as the matrix instruction wants them; the packed weights (16 KB) as they come: a wave reads its own back in 16-byte
//    pieces and turns them by permlane swaps (w4a8_gemm_exact_kernel).  The group's scales and zero points (a dword of each a lane) come the same way.
//  * half 0 of a stage multiplies while half 1 is unpacked and fetched, and the other way round with the next stage's half 0.
//  * three stages: packed weights are half as long as W8A8's.
//
// Measured (MI355X): 512 rows of 28672 x 4096, one tile a CU, 62 us where the other kernel takes 76 (W8A8 61); 4096 rows 430 / 494 (404); 6000 rows of 4096 x 14336
// 336 / 396; 2331 rows of 28672 x 4096 318 / 342.  The matrix units are busy half of the time, as in the W8A8 tiles; unpacking in 8.5 operations a word took
// 2 - 3 % more, letting the stores of a tile fly into the next one nothing less.
//
// The next tile's requests go out before the results are scaled, which wait in the accumulation registers (accumulators_stay): 2331 rows of 28672 x 4096 with the unit 291 -> 279 us, of 6144 x 4096
// 59.5 -> 56.8, 6000 rows of 28672 x 4096 620 -> 600.
//
// Per-channel (MODE_CHN) there is no second level: a word is a shift and a mask, a stage has no parameters, and 64 products wait for nothing but their operands: 1.24 us a stage with all CUs at
// work, 0.98 with few, where the package's power lets the clock be higher.  What it gains on w4a8_gemm_exact_kernel is operands brought in half as often, where its tiles fill whole rounds: us, 4000
// rows of 4096 x 14336 162 -> 148 (3190 TOPS), of 28672 x 4096 with the unit 340 -> 331, of 8192 x 8192 188 -> 175, of 8192 x 28672 664 -> 572.
//
// SHARE: K of the last round's tiles shared out (tile_share.h).
//
// Integer sums and the general kernel's epilogue: the same bits.
#pragma once
#include "tile_share.h"

namespace omni {

constexpr int GT_ACT = TILES_M * TILES_K, GT_W = TILES_N * TILES_K / 2, GT_PAR = 4 * 256, GT_BUFS = 3;

// A word of four weights, u * scale + zero per byte, as the general form has it: the whole word's product, in which a byte's overflow goes into the next,
// then four byte additions.  In full-rate operations, 6.5 a word where a quarter-rate multiplication and the additions one by one are 9.5, and without a
// condition, around which the accumulators would move.  In pieces, which stand between products.
// Written out, as hipcc would join them to the quarter-rate multiplication again and undo (y ^ w) + z7.
#define OMNI_GT_BYTE3(h, x, sc) "v_mul_u32_u24_sdwa " h ", " x ", " sc " dst_sel:BYTE_3 dst_unused:UNUSED_PAD src0_sel:BYTE_3 src1_sel:DWORD\n\t"
#define OMNI_GT_MULTIPLY(y, x, sc, h) "v_mad_u32_u24 " y ", " x ", " sc ", " h "\n\t"
#define OMNI_GT_ADD(w, t, y, z7) "v_and_b32 " w ", 0x80808080, " y "\n\tv_xad_u32 " t ", " y ", " w ", " z7 "\n\t"
#define OMNI_GT_RESULT(r, t, w, z80) "v_bitop3_b32 " r ", " t ", " w ", " z80 " bitop3:0x96\n\t"

// SILU: out = silu(gate) up of a [gate | up] weight, [M][N / 2]: of a wave's 64 channels the first 32 are gate channels, the others the up channels of the same place.  (2331 rows of
// 28672 x 4096: the product takes 307 us either way, the quantiser behind it 31 -> 18.)
template <int MODE, bool SILU, bool SHARE>
__global__ __launch_bounds__(256, 1) void w4a8_tiles_kernel(GemmArgs p, TileShare share) {
  static_assert(MODE == MODE_CHN || MODE == MODE_GRP, "packed weights");
  constexpr bool GRP = MODE == MODE_GRP;
  constexpr int GT_STAGE = GT_ACT + GT_W + (GRP ? GT_PAR : 0), PIECES = GRP ? 13 : 12;
  constexpr int PITCH = 64 * 2 + 16;                        // a row of the write-back buffers: a wave's 64 channels
  constexpr int LDS_OUT = GT_BUFS * GT_STAGE, LDS_SC = LDS_OUT + 4 * 16 * PITCH, SC = GRP ? 1024 : 2048;      // (SC: scales of 256 channels and 256 rows, CHN: zero points and sums too)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_SC + 2 * SC + (SHARE ? 16 : 0)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (tile order: w8a8_tiles_kernel's)
  const int tiles = p.tiles_m * p.tiles_n, xcd = blockIdx.x & 7;
  const int own = (tiles >> 3) + (xcd < (tiles & 7)), first = xcd * (tiles >> 3) + min(xcd, tiles & 7);
  int at = blockIdx.x >> 3;
  const int all_stages = p.K / TILES_K;
  TileParts parts(at, own, all_stages);                     // (SHARE)

  // a wave's part of a stage: 64 rows of the activations, 8 a piece (lane: row lane / 8, slot lane % 8), and its two tile rows of weights, 2 KB each
  uint32_t src[8], wsrc[4];
  {
    const int l = lane_here();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 64 * wave + 8 * i + (l >> 3);
      src[i] = (uint32_t)r * (uint32_t)p.K + (((l & 7) ^ tiles_swizzle(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      wsrc[i] = (uint32_t)(SILU ? wave + (i >> 1) * (p.N >> 6) : 2 * wave + (i >> 1)) * (uint32_t)p.K * 16u + (i & 1) * 1024 + l * 16;
  }
  const uint8_t *wbase = nullptr, *abase = nullptr;         // of the next stage
  const uint8_t* par = nullptr;                             // ... the lane's dword of its parameters: scales in the first 16 lanes, zero points in the next
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds);
  // buf: byte of a stage's buffer
  auto dst = [&](int buf, int i) __attribute__((always_inline)) {
    return lds0 + buf + (i < 8 ? 8192 * wave + 1024 * i : GT_ACT + 4096 * wave + 1024 * (i - 8));
  };
  auto after = [&](int buf) __attribute__((always_inline)) { return buf == (GT_BUFS - 1) * GT_STAGE ? 0 : buf + GT_STAGE; };
  auto dma_params = [&](int buf) __attribute__((always_inline)) {
    const uint32_t to = lds0 + buf + GT_ACT + GT_W + 256 * wave;
    const uint8_t* const from = par;
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(from), "s"(to) : "memory");
  };
  auto advance = [&]() __attribute__((always_inline)) {
    wbase += 4 * 512;
    abase += TILES_K;
    if constexpr (GRP) par += p.N;
  };
  auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 12; ++i) tiles_dma16(i < 8 ? src[i & 7] : wsrc[i & 3], i < 8 ? abase : wbase, dst(buf, i));
    if constexpr (GRP) dma_params(buf);
    advance();
  };
  int m0 = 0, n0 = 0, ns = all_stages;                      // ns: stages of the tile opened last
  uint16_t sw_next = 0, sa_next = 0, sz_next = 0, as_next = 0;      // the thread's channel's and row's scales of the tile opened last; CHN: zero point and sum
  // (the last row tile starts at M - 256: the rows that it shares with the one before are computed twice, to the same bits)
  auto open_tile = [&]() __attribute__((always_inline)) {
    int k0 = 0;
    if constexpr (SHARE) {
      if (!parts.next(at)) return false;
      k0 = parts.k0;
      ns = parts.stages;
    } else {
      if (at >= own) return false;
    }
    const int id = first + (SHARE ? parts.tile : at), band = id / (p.tile_linear * p.tiles_n), in = id - band * p.tile_linear * p.tiles_n;
    const int rows = min(p.tile_linear, p.tiles_m - band * p.tile_linear), tn = in / rows;
    at += (int)gridDim.x >> 3;
    n0 = tn * (SILU ? TILES_N / 2 : TILES_N);
    m0 = min((band * p.tile_linear + in - tn * rows) * TILES_M, p.M - TILES_M);
    wbase = p.W + (size_t)n0 * (p.K / 2) + k0 * (4 * 512);
    abase = (const uint8_t*)p.A + (size_t)m0 * p.K + k0 * TILES_K;
    const int tid = 64 * wave + lane_here();
    // (lane l of 64 channels: the first of the wave's and, SILU, the other half's)
    auto channel = [&](int l) __attribute__((always_inline)) { return SILU ? n0 + 32 * wave + (l & 31) + (l >> 5) * (p.N >> 1) : n0 + 64 * wave + l; };
    if constexpr (GRP) par = ((tid & 16) ? p.s2z : p.s2s) + (size_t)k0 * p.N + channel(4 * (tid & 15));
    sw_next = ((const uint16_t*)p.wscales)[channel(lane_here())];
    sa_next = ((const uint16_t*)p.ascales)[m0 + tid];
    if constexpr (!GRP) {
      sz_next = ((const uint16_t*)p.wsz)[channel(lane_here())];
      as_next = ((const uint16_t*)p.asum)[m0 + tid];
    }
    if constexpr (SHARE) {
      wbase = wave_uniform(wbase);
      abase = wave_uniform(abase);
    }
#pragma unroll
    for (int i = 0; i < GT_BUFS; ++i) stage(i * GT_STAGE);
    return true;
  };
  // ... its scales in LDS: 256 channels', 256 rows'
  auto park = [&](int parity) __attribute__((always_inline)) {
    uint16_t* s = (uint16_t*)(lds + LDS_SC + SC * parity) + 64 * wave + lane_here();
    s[0] = sw_next;
    s[256] = sa_next;
    if constexpr (!GRP) {
      s[512] = sz_next;
      s[768] = as_next;
    }
  };

  int off[2], woff = 0, poff = 0;                           // of a fragment of half u inside 16 rows; of a piece of the wave's weights; of its parameters
  v4i a[2][4], b[2][16], acc[4][16];
  auto fetch_b = [&](int buf, auto half, int j) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    b[U][j] = *(const v4i*)(lds + 16 * TILES_K * j + (buf + off[U]));
  };
  uint4 raw[2];                                             // the packed weights of the half that is unpacked next
  auto fetch_raw = [&](int buf, auto half, int j) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    raw[j] = *(const uint4*)(lds + GT_ACT + 1024 * U + 512 * j + (buf + woff));
  };
  uint32_t ps = 0, pz = 0, ps_next = 0, pz_next = 0;        // the parameters of the stage that is being unpacked, and of the next
  auto fetch_params = [&](int buf) __attribute__((always_inline)) {
    const uint32_t* const q = (const uint32_t*)(lds + GT_ACT + GT_W + (buf + poff));
    ps_next = q[0];
    pz_next = q[16];
  };
  // dwords of a 16-B piece: x = (k5 = 0, n2 = 0) y = (0, 1) z = (1, 0) w = (1, 1); behind it d[n2][q] = k6 = q of (tile parity, k5) = lane >> 4
  uint32_t d[2][4];
  auto turn = [&](int n2) __attribute__((always_inline)) {
    const uint32_t e0 = n2 ? raw[0].y : raw[0].x, e1 = n2 ? raw[0].w : raw[0].z;
    const uint32_t e2 = n2 ? raw[1].y : raw[1].x, e3 = n2 ? raw[1].w : raw[1].z;
    const auto s02 = __builtin_amdgcn_permlane32_swap(e0, e2, false, false);
    const auto s13 = __builtin_amdgcn_permlane32_swap(e1, e3, false, false);
    const auto s01 = __builtin_amdgcn_permlane16_swap((uint32_t)s02[0], (uint32_t)s13[0], false, false);
    const auto s23 = __builtin_amdgcn_permlane16_swap((uint32_t)s02[1], (uint32_t)s13[1], false, false);
    d[n2][0] = (uint32_t)s01[0]; d[n2][1] = (uint32_t)s01[1]; d[n2][2] = (uint32_t)s23[0]; d[n2][3] = (uint32_t)s23[1];
  };
  // word w of a half: dword w % 4 of nibbles w / 4 % 2 of n2 = w / 8 (so that a half's d[0] is free for the next one's); its block of channels
  auto block_of = [](int w) { return 2 * ((w >> 2) & 1) + (w >> 3); };
  uint32_t sc = 0, z7 = 0, z80 = 0;           // the block's scale; its zero point in every byte: seven bits, the eighth
  auto scale = [&](int w) __attribute__((always_inline)) { sc = (ps >> (8 * block_of(w))) & 0xFFu; };
  auto zero_point = [&](int w) __attribute__((always_inline)) {
    const uint32_t zero = __builtin_amdgcn_perm(0u, pz, 0x01010101u * (uint32_t)block_of(w));
    z7 = zero & 0x7F7F7F7Fu;
    z80 = zero & 0x80808080u;
  };
#define OMNI_GT_OP "v_mfma_i32_16x16x64_i8"
#define OMNI_GT_FENCE() __builtin_amdgcn_sched_barrier(0)
  auto product = [&](auto half, int i, int j) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    v4i& c = acc[i][j];
    const v4i &x = a[U][i], &y = b[U][j];
    OMNI_MFMA_PINNED(OMNI_GT_OP, c, x, y);
  };
  // ... with pieces of a word around it (gx, gh, gy, gw, gt): the fourth product may not be read by the instruction behind it
  uint32_t gx, gy, gw, gt;
  auto nibbles = [&](int w) __attribute__((always_inline)) { gx = (d[w >> 3][w & 3] >> (4 * ((w >> 2) & 1))) & 0x0F0F0F0Fu; };
  auto product_multiply = [&](auto half, int i, int j) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    v4i& c = acc[i][j];
    const v4i &x = a[U][i], &y = b[U][j];
    uint32_t gh;
    uint32_t& to = gy;
    const uint32_t word = gx, by = sc;
    asm volatile(OMNI_GT_BYTE3("%0", "%3", "%4") OMNI_GT_OP " %2, %5, %6, %2\n\t" OMNI_GT_MULTIPLY("%1", "%3", "%4", "%0")
                 : "=&v"(gh), "=&v"(to), "+a"(c) : "v"(word), "v"(by), "v"(x), "v"(y));
  };
  auto product_add = [&](auto half, int i, int j) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    v4i& c = acc[i][j];
    const v4i &x = a[U][i], &y = b[U][j];
    uint32_t &top = gw, &sum = gt;
    const uint32_t word = gy, by = z7;
    asm volatile(OMNI_GT_OP " %2, %5, %6, %2\n\t" OMNI_GT_ADD("%0", "%1", "%3", "%4") : "=&v"(top), "=&v"(sum), "+a"(c) : "v"(word), "v"(by), "v"(x), "v"(y));
  };
  auto product_result = [&](auto half, int i, int j, int w) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    v4i& c = acc[i][j];
    const v4i &x = a[U][i], &y = b[U][j];
    const uint32_t top = gw, sum = gt, by = z80;
    int to;
    asm volatile(OMNI_GT_OP " %1, %5, %6, %1\n\t" OMNI_GT_RESULT("%0", "%2", "%3", "%4") : "=&v"(to), "+a"(c) : "v"(sum), "v"(top), "v"(by), "v"(x), "v"(y));
    a[U ^ 1][block_of(w)][w & 3] = to;
  };
  // ... with piece i of a stage requested around it
  auto product_dma = [&](auto half, int i, int j, int piece, int buf) __attribute__((always_inline)) {
    constexpr int U = decltype(half)::value;
    v4i& c = acc[i][j];
    const v4i &x = a[U][i], &y = b[U][j];
    if (piece < 12) {
      const uint32_t from = piece < 8 ? src[piece & 7] : wsrc[piece & 3], to = dst(buf, piece);
      const uint8_t* const base = piece < 8 ? abase : wbase;
      asm volatile("s_mov_b32 m0, %4\n\t" OMNI_GT_OP " %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, %5"
                   : "+a"(c) : "v"(x), "v"(y), "v"(from), "s"(to), "s"(base) : "memory", "m0");
    } else {
      const uint32_t to = lds0 + buf + GT_ACT + GT_W + 256 * wave;
      const uint8_t* const from = par;
      asm volatile("s_mov_b32 m0, %4\n\t" OMNI_GT_OP " %0, %1, %2, %0\n\tglobal_load_lds_dword %3, off"
                   : "+a"(c) : "v"(x), "v"(y), "v"(from), "s"(to) : "memory", "m0");
    }
  };
  // The 64 products of half U of a stage.  Between them: the other half's activations (NEXT: there is one), for U = 0 of the same stage (buffer `same`),
  // else of the next (`next`); that half's 16 words are unpacked, d[0] and its first block's parameters being there; the packed weights of the half
  // behind it, of the next stage; U = 1: the stage three further on (DMA) into this one's buffer.
  // At most three instructions fit behind a product: a group of four has 12 - 14 others.
  auto half = [&](auto hu, int same, int next, auto has_next, auto has_raw, auto dma) __attribute__((always_inline)) {
    constexpr int U = decltype(hu)::value;
    constexpr bool NEXT = decltype(has_next)::value, RAW = decltype(has_raw)::value, DMA = decltype(dma)::value;
    if constexpr (!GRP) {      // (a group of four has five others)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        OMNI_GT_FENCE();
        product(hu, 0, j);
        if constexpr (NEXT) nibbles(j);
        OMNI_GT_FENCE();
        if (DMA && j < PIECES) product_dma(hu, 1, j, j, same);
        else product(hu, 1, j);
        if constexpr (NEXT) {
          a[U ^ 1][block_of(j)][j & 3] = (int)gx;
          if (j < 12 && j % 3 == 0) fetch_b(U ? next : same, IntTag<U ^ 1>{}, 12 + j / 3);
        }
        OMNI_GT_FENCE();
        product(hu, 2, j);
        if constexpr (NEXT) {
          if (j < 12) fetch_b(U ? next : same, IntTag<U ^ 1>{}, j);
          if (j == 6) turn(1);
        }
        OMNI_GT_FENCE();
        product(hu, 3, j);
        if constexpr (RAW) {
          if (j == 8 || j == 9) fetch_raw(next, IntTag<U>{}, j - 8);
          if (j == 14) turn(0);
        }
      }
      OMNI_GT_FENCE();
      if constexpr (DMA) advance();
      return;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      OMNI_GT_FENCE();
      if (NEXT && j > 0) product_result(hu, 0, j, j - 1);
      else product(hu, 0, j);
      if constexpr (NEXT) {
        if (j == 0) nibbles(0);
        if (j > 0 && (j & 3) == 0) scale(j);
      }
      OMNI_GT_FENCE();
      if (DMA && j < 13) product_dma(hu, 1, j, j, same);
      else product(hu, 1, j);
      if constexpr (NEXT) {
        if (j > 0 && (j & 3) == 0) zero_point(j);
        if (j < 12 && j % 3 == 0) fetch_b(U ? next : same, IntTag<U ^ 1>{}, 12 + j / 3);     // activations: four in three groups
      }
      OMNI_GT_FENCE();
      if constexpr (NEXT) {
        product_multiply(hu, 2, j);
        if (j < 12) fetch_b(U ? next : same, IntTag<U ^ 1>{}, j);
      } else {
        product(hu, 2, j);
      }
      OMNI_GT_FENCE();
      if constexpr (NEXT) {
        product_add(hu, 3, j);
        if (j < 15) nibbles(j + 1);
        if (j == 6) turn(1);
      } else {
        product(hu, 3, j);
      }
      if constexpr (RAW) {
        if (j == 8 || j == 9) fetch_raw(next, IntTag<U>{}, j - 8);
        if (U == 0 && j == 10) fetch_params(next);
        if (j == 14) turn(0);
      }
    }
    OMNI_GT_FENCE();
    if constexpr (NEXT) a[U ^ 1][3][3] = (int)(gt ^ gw ^ z80);
    if constexpr (RAW) {
      if constexpr (U == 0) {
        ps = ps_next;
        pz = pz_next;
      }
      scale(0);
      zero_point(0);
    }
    if constexpr (DMA) advance();
  };
  // MORE: there is a next stage; DMA: and two behind it
  auto step = [&](int buf, int next, auto more, auto dma) __attribute__((always_inline)) {
    half(IntTag<0>{}, buf, next, BoolTag<true>{}, more, BoolTag<false>{});
    // the stage after the next is there for every wave, and everyone has this one in registers
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    half(IntTag<1>{}, buf, next, more, more, dma);
  };

  int parity = 0;
  bool open = open_tile();
  if (open) park(0);
  while (open) {
    const int zero = opaque(0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        v4i& c = acc[i][j];
        c = (v4i){zero, zero, zero, zero};
        asm volatile("" : "+a"(c));                         // (here, not between the first products, behind whose writes hipcc would not wait)
      }
    // stages 0 and 1 are there: of what was requested last -- a stage, or stores of the tile before -- 13 (CHN 12) may still fly (let fly all 32 stores,
    // a tile takes the same time)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PIECES) : "memory");
    __syncthreads();
    if constexpr (SHARE) {
      wbase = wave_uniform(wbase);
      abase = wave_uniform(abase);
    }
    const int fl = lane_here();
#pragma unroll
    for (int u = 0; u < 2; ++u) off[u] = (fl & 15) * TILES_K + (((4 * u + (fl >> 4)) ^ tiles_swizzle(fl & 15)) << 4);
    woff = 4096 * wave + ((fl >> 3) & 1) * 2048 + ((fl & 7) * 4 + (fl >> 4)) * 16;
    poff = 256 * wave + 4 * (fl & 15);
    if constexpr (GRP) fetch_params(0);
#pragma unroll
    for (int j = 0; j < 2; ++j) fetch_raw(0, IntTag<0>{}, j);
#pragma unroll
    for (int j = 0; j < 16; ++j) fetch_b(0, IntTag<0>{}, j);
    ps = ps_next;
    pz = pz_next;
    turn(0);
    turn(1);
#pragma unroll
    for (int j = 0; j < 2; ++j) fetch_raw(0, IntTag<1>{}, j);
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      if constexpr (!GRP) {
        nibbles(w);
        a[0][block_of(w)][w & 3] = (int)gx;
        continue;
      }
      if ((w & 3) == 0) {
        scale(w);
        zero_point(w);
      }
      nibbles(w);
      const uint32_t word = gx, by = sc, add = z7, top = z80;
      uint32_t h, y, w7, t7;
      int to;
      asm(OMNI_GT_BYTE3("%0", "%5", "%6") "s_nop 1\n\t" OMNI_GT_MULTIPLY("%1", "%5", "%6", "%0") OMNI_GT_ADD("%2", "%3", "%1", "%7") OMNI_GT_RESULT("%4", "%3", "%2", "%8")
          : "=&v"(h), "=&v"(y), "=&v"(w7), "=&v"(t7), "=&v"(to) : "v"(word), "v"(by), "v"(add), "v"(top));
      a[0][block_of(w)][w & 3] = to;
    }
    turn(0);
    if constexpr (GRP) {
      scale(0);
      zero_point(0);
    }
    int t = 0, buf = 0;
    do {                                                    // (at least once: zeros on a way around it would be kept beside the accumulators)
      step(buf, after(buf), BoolTag<true>{}, BoolTag<true>{});
      buf = after(buf);
    } while (++t + 3 < ns);
    step(buf, after(buf), BoolTag<true>{}, BoolTag<false>{});
    buf = after(buf);
    step(buf, after(buf), BoolTag<true>{}, BoolTag<false>{});
    buf = after(buf);
    step(buf, 0, BoolTag<false>{}, BoolTag<false>{});       // (behind its barrier all buffers are free)
    accumulators_settle(acc);

    // the next tile's requests, then the results, which stay in the accumulation registers until they are stored (w8a8_tiles_kernel's arithmetic)
    const int el = lane_here(), e15 = el & 15, i0 = (el >> 4) * 4;
    const int chan = (i0 >> 3) * 32 + (i0 & 7);             // of block 0
    const uint8_t* scales = lds + LDS_SC + SC * parity;
    half_t* const out = p.out + (size_t)m0 * p.out_stride + n0 + (SILU ? 32 : 64) * wave;
    const TileParts mine = parts;
    bool opened = false;
    if constexpr (SHARE) {
      if (mine.shared()) {
        const bool last = mine.finishes(share, lds + LDS_SC + 2 * SC, acc, [&] {
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
    if (!opened) open = open_tile();
    uint8_t* rows = lds + LDS_OUT + wave * 16 * PITCH;
    auto store = [&](auto add) __attribute__((always_inline)) {
      constexpr bool ADD = decltype(add)::value;
      accumulators_stay(acc);
      float sw[4][4], sz[4][4];
      auto channels = [&](int at, float (&to)[4][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint2 w = *(const uint2*)(scales + at + 2 * (64 * wave + chan + 8 * i));
          const uint32_t wv[2] = {w.x, w.y};
#pragma unroll
          for (int e = 0; e < 4; ++e) to[i][e] = (float)__builtin_bit_cast(half_t, (uint16_t)(wv[e >> 1] >> (16 * (e & 1))));
        }
      };
      channels(0, sw);
      if constexpr (!GRP) channels(1024, sz);
      v4i x[16];                                            // ADD: of four blocks of rows
      uint2 h[2][4];                                        // [row block][channel block]
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        if constexpr (ADD) if (j % 4 == 0) {
          mine.others(share, [&](int q) { return 16 * (q & 3) + j + (q >> 2); }, x);
          accumulators_stay(acc);
        }
        const float sa = (float)*(const half_t*)(scales + 512 + 2 * (16 * j + e15));
        const float as = GRP ? 0.f : (float)*(const half_t*)(scales + (GRP ? 0 : 1536) + 2 * (16 * j + e15));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t hw[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const v4i& y = x[4 * (j & 3) + i];
            const int c0 = acc[i][j][2 * e] + (ADD ? y[2 * e] : 0), c1 = acc[i][j][2 * e + 1] + (ADD ? y[2 * e + 1] : 0);
            v2f r;
            if constexpr (GRP) r = (v2f){(float)c0 * (sw[i][2 * e] * sa), (float)c1 * (sw[i][2 * e + 1] * sa)};
            else r = (v2f){(float)c0 * sw[i][2 * e] * sa - sz[i][2 * e] * as, (float)c1 * sw[i][2 * e + 1] * sa - sz[i][2 * e + 1] * as};
            asm volatile("" : "+v"(r));
            hw[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, v2h));
          }
          h[j & 1][i] = make_uint2(hw[0], hw[1]);
        }
        if constexpr (SILU) {      // two row blocks at a time; lanes l and l ^ 16 have a block's eight channels
          if (j & 1) {
            const int odd = (el >> 4) & 1;
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const uint2 v = silu_mul_blocks(h[0][i], h[1][i]), y = silu_mul_blocks(h[0][i + 1], h[1][i + 1]);
              const auto lo = __builtin_amdgcn_permlane16_swap(v.x, y.x, false, false), hi = __builtin_amdgcn_permlane16_swap(v.y, y.y, false, false);
              *(uint4*)(out + (size_t)(16 * (j - 1) + 16 * (el >> 5) + e15) * p.out_stride + 8 * (i + odd)) =
                  make_uint4((uint32_t)lo[0], (uint32_t)hi[0], (uint32_t)lo[1], (uint32_t)hi[1]);
            }
          }
        } else {      // through LDS, so that a row leaves in whole 16-byte pieces of neighbouring lanes: 16 rows of the wave's 64 channels at a time
#pragma unroll
          for (int i = 0; i < 4; ++i) *(uint2*)(rows + e15 * PITCH + (chan + 8 * i) * 2) = h[j & 1][i];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int r = 8 * i + (el >> 3);
            *(uint4*)(out + (size_t)(16 * j + r) * p.out_stride + (el & 7) * 8) = *(const uint4*)(rows + r * PITCH + (el & 7) * 16);
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (SHARE && mine.shared()) store(BoolTag<SHARE>{});
    else store(BoolTag<false>{});
    parity ^= 1;
    if (open) park(parity);
  }
#undef OMNI_GT_OP
#undef OMNI_GT_FENCE
}

// a workgroup per CU
template <int MODE, bool SILU>
static void launch_w4_tiles_as(GemmArgs b, const TileShare& share, hipStream_t st) {
  b.tiles_n = b.N / TILES_N;
  b.tiles_m = (b.M + TILES_M - 1) / TILES_M;
  const int bands = (b.tiles_m + 3) / 4, tiles = b.tiles_m * b.tiles_n;
  b.tile_linear = (b.tiles_m + bands - 1) / bands;
  if (share.sums) hipLaunchKernelGGL((w4a8_tiles_kernel<MODE, SILU, true>), dim3(256), dim3(256), 0, st, b, share);
  else hipLaunchKernelGGL((w4a8_tiles_kernel<MODE, SILU, false>), dim3(std::min(256, (tiles + 7) / 8 * 8)), dim3(256), 0, st, b, share);
}

}  // namespace omni
