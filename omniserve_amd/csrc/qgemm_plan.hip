// Host-side tiling / split-K planning for the W4A8 / W8A8 GEMMs (shared by the three GEMM TUs).
#include "qgemm_kernel.h"
#include <atomic>
#include <chrono>

namespace omni {

// (plan overrides: test / sweep hooks, per enqueueing thread like everything else here)
static thread_local int g_override_waves = 0;
static thread_local int g_override_sk = 0;
static thread_local int g_midm_mode = -1;     // omni_gemm_set_midm_override
static thread_local int g_midm_sk = 0;
static thread_local PrefetchArgs g_armed_prefetch = {};   // per enqueueing thread: armed and consumed by the same caller
// weight tensors named by omni_prefetch_arm_gemm whose GEMV has not been enqueued yet (one-shot, per thread): that GEMV
// reads its weights with plain loads (they sit in L2), every other one streams non-temporally.  A decode layer has at
// most two such entries alive at a time (down_proj armed while gate_up runs); 4 slots, oldest replaced.
static thread_local const void* g_prefetched_w[4] = {nullptr, nullptr, nullptr, nullptr};
static thread_local unsigned g_prefetched_next = 0;

bool take_prefetched_weight(const void* weight) {
  if (!weight) return false;
  for (auto& w : g_prefetched_w)
    if (w == weight) { w = nullptr; return true; }
  return false;
}
static void note_prefetched_weight(const void* weight) {
  for (auto& w : g_prefetched_w)
    if (w == weight) return;
  g_prefetched_w[g_prefetched_next++ & 3] = weight;
}

PrefetchArgs take_armed_prefetch() {
  PrefetchArgs pf = g_armed_prefetch;
  g_armed_prefetch = PrefetchArgs{};
  return pf;
}

static thread_local TileShare g_armed_share = {};
TileShare take_armed_share() {
  const TileShare s = g_armed_share;
  g_armed_share = TileShare{};
  return s;
}
// of the XCDs with a tile more and of those without
static int share_places_of(int M, int N, int K) {
  const long long tiles = (long long)((M + TILES_M - 1) / TILES_M) * (N / TILES_N);
  int places = 0;
  for (const long long own : {tiles / 8, (tiles + 7) / 8}) {
    const int left = (int)(own % SHARE_PER);
    const ShareSplit sp = share_split(left, K / TILES_K);
    if (left > 0 && sp.head < K / TILES_K) places = std::max(places, share_places(left, sp.used));
  }
  return places;
}
bool share_fits(TileShare* s, int M, int N, int K) {
  if (!s->sums || N < TILES_N || K < TILES_K) return false;
  const int places = share_places_of(M, N, K);
  if (places == 0 || s->places < places) return false;
  s->places = places;
  return true;
}

GemmPlan plan_gemm(int M, int N, int K, int kalign, bool deferred, bool w8) {
  GemmPlan pl;
  pl.kw = 1;
  pl.mz = 1;
  pl.narrow = 0;
  pl.midm = 0;
  // Mid-M kernel (qgemm_midm.h): M = 33 .. 128 rows (one row tile), N in whole 128-channel tiles, K slices of whole 256-k
  // chunks.  A launch of it carries ~7 us that do not depend on K (first requests, the K-phase exchange, stores) and streams
  // at about twice the single-wave tiles' rate beyond them, so it takes the BIG matrices (measured, tools/midm_sweep.py,
  // profiles/r05_a: Llama-3-8B gate_up at M = 128 35.4 -> 23.1 us, Llama-2-70B gate_up 138 -> 71, down 106 -> 41 -- and
  // Llama-3-8B qkv 11.7 -> 19.6, which stays where it was): N x K >= 80 M weights, or >= 50 M where the caller wants the
  // slabs anyway (the deferred forms: no slab epilogue launch to pay for; Llama-3-8B down at M = 64: 11.4 -> 10.7 us, g128
  // 13.6 -> 12.6; g128 gate_up at M = 64 21.2 -> 19.5).
  // K split: one workgroup per CU and launch (its LDS rings fill the CU) -- the largest split that keeps the grid inside one
  // round of 256 and >= 4 chunks per slice (Llama-2-70B qkv, 80 tiles: 2 slices 28.5 us, 4 slices 34.7).
  // (the kernel addresses weights and activations with 32-bit lane offsets: matrices of 4 GiB and more keep the other tiles)
  const bool midm_fits = (unsigned long long)N * K * (w8 ? 2 : 1) < (2ull << 32) && (unsigned long long)M * K < (1ull << 32);
  if (g_midm_mode != 0 && g_override_waves == 0 && g_override_sk == 0 && M > 32 && M <= 128 && N % 128 == 0 && K % KCHUNK == 0 &&
      midm_fits) {
    const long long weights = (long long)N * K;
    bool take = g_midm_mode > 0;
    if (g_midm_mode < 0) take = weights >= 80000000LL || (deferred && weights >= 50000000LL);
    if (take) {
      const int tiles = N / 128;
      int best = 1;
      for (int s2 = 2; s2 <= 16; ++s2) {
        if (K % (s2 * KCHUNK) != 0 || (K / s2) % kalign != 0 || K / s2 < 4 * KCHUNK || tiles * s2 > 256) continue;
        best = s2;
      }
      if (g_midm_sk > 0 && K % (g_midm_sk * KCHUNK) == 0) best = g_midm_sk;
      pl.midm = 1; pl.mb = M <= 64 ? 4 : 8; pl.mz = 1; pl.waves = 2; pl.kw = 1;
      pl.sk = best; pl.kslice = K / best;
      return pl;
    }
  }
  if (M > 128) {  // MFMA-bound regime: 128 x 256 tile per workgroup
    pl.mb = 8; pl.waves = 4; pl.sk = 1; pl.kslice = K;
    // Few tiles (decode at batch 129..512: the published A100 figure is quoted at bs = 256): Llama-3-8B's down_proj is
    // 2 x 16 = 32 tiles of 56 K chunks on 256 CUs (80 us per layer at bs = 256, profiles/r04_b), o_proj 32, qkv 48.  Split K over
    // grid.y into int32 slabs (+ the slab epilogue launch) until about one workgroup per CU streams: the smallest split with
    // >= 256 workgroups, whole 256-k chunks and >= 1024 k per workgroup.  A grid that already covers half the chip stays whole.
    const long long tiles = (long long)((M + 127) / 128) * ((N + 255) / 256);
    if (M <= 512 && tiles <= 128 && g_override_waves == 0) {
      int best = 1;
      for (int s2 = 2; s2 <= 8; s2 *= 2) {
        if (K % (s2 * KCHUNK) != 0 || K / s2 < 1024 || tiles * s2 > 512) break;
        best = s2;
        if (tiles * s2 >= 256) break;
      }
      if (g_override_sk > 0 && K % (g_override_sk * KCHUNK) == 0) best = g_override_sk;
      pl.sk = best;
      pl.kslice = K / best;
    }
    return pl;
  }
  // bandwidth-bound regime (decode): every CU must stream weights.  One wave owns 64 channels
  // and a K-slice; activations are staged per round of RING steps, so the slice length is free.
  pl.mb = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  pl.mz = M <= 64 ? 1 : 2;         // M = 65..128: two 64-row tiles per channel group
  pl.waves = 1;                    // fixed per tile height (GemvCfg)
  const int ngroups = N / 64;
  auto ok = [&](int s) { return s >= 1 && (K % s) == 0 && ((K / s) % kalign) == 0; };
  int sk = 1;
  // M = 33..128, int4 modes: 32-row tiles (ceil(M / 32) row tiles per channel group, the re-reads of a weight byte are
  // served by L1 / L2) beat the 64-row tile whenever their grid still fits the chip in one round -- smaller serial
  // chains per wave at the same two waves per SIMD (measured, profiles/r03_c_*: Llama-2-70B TP=8 shard at M = 128
  // gate_up 24.8 -> 21.6 us, down 18.4 -> 12.9, qkv 12.5 -> 10.0, o 7.6 -> 5.6; Llama-3-8B g128 at M = 64 down 20.4 ->
  // 18.6, qkv 12.8 -> 10.1, o 10.9 -> 9.9, but gate_up 23.0 -> 31.5: 896 workgroups, two rounds -- stays on 64 rows).
  static const int narrow_mode = omni_knob("OMNI_GEMV_NARROW", 1);   // 0: never (A/B, tuning builds)
  // (g128 at M <= 64: faster launch by launch, but the Llama-3-8B bs = 64 decode step measured 1.2 % slower with it -- off)
  if (!w8 && M > 32 && !(kalign == 128 && M <= 64) && narrow_mode != 0 && g_override_waves == 0 && g_override_sk == 0) {
    const int mz = (M + 31) / 32;
    if (ngroups * mz <= 640 && (K % (4 * kalign)) == 0) {
      pl.mb = 2; pl.mz = mz; pl.waves = 1; pl.narrow = 1; pl.kw = 4;
      // smallest split with <= 2048 k per wave and >= 128 workgroups; parts of at least 256 k
      int best = 1;
      for (int s = 1; s <= 64; ++s) {
        if (!ok(s) || ((K / s) % (4 * kalign)) != 0 || K / (s * 4) < 256) continue;
        best = s;
        if (K / (s * 4) <= 2048 && ngroups * mz * s >= 128) break;
      }
      pl.sk = best;
      pl.kslice = K / best;
      return pl;
    }
  }
  if (pl.mb == 1) {
    // M <= 16: single-wave tiles, K split first inside the workgroup (kw waves, no slab traffic) and only
    // then across workgroups.  Measured on MI355X (tools/kw_sweep*.py): a wave should stream <= 1024 k
    // (two ring rounds) when the split is free (one kernel), <= 512 k when the int32 slabs are consumed
    // by a fused kernel anyway (deferred) or a split cannot be avoided.
    int kw = 4;
    while (kw > 1 && (K % (kw * kalign)) != 0) kw >>= 1;
    auto part = [&](int s) { return K / (s * kw); };
    auto fits = [&](int s) { return ok(s) && ((K / s) % (kw * kalign)) == 0; };
    // W8A8 rows are twice the bytes per k: the deferred (slab-only) plan halves the k per wave (same bytes per wave)
    static const int part_w4_deferred = omni_knob("OMNI_DEFERRED_PART", 512);   // (A/B knob, tuning builds)
    const int part_target = (deferred && w8) ? 256 : (deferred ? part_w4_deferred : 512);
    // W8A8 rows are twice the bytes per k: with few channel groups (qkv at batch 1: 96 workgroups streaming 256 KiB each)
    // a split to 512 k per wave + the slab epilogue launch beats the single kernel (OMNI_W8_SMALL_SPLIT=0: off, A/B)
    static const int w8_small_split = omni_knob("OMNI_W8_SMALL_SPLIT", 1);
    const bool w8_small = w8 && !deferred && w8_small_split && ngroups <= 128 && part(1) > 512;
    if (!deferred && part(1) <= 1024 && !w8_small) {
      sk = 1;
    } else {
      int best = 0;
      for (int s = 1; s <= 64; ++s) {
        if (!fits(s) || part(s) < 256) continue;
        if (part(s) <= part_target) { best = s; break; }
        best = s;   // largest usable split so far
      }
      sk = best > 0 ? best : 1;
    }
    if (g_override_sk > 0 && ok(g_override_sk)) sk = g_override_sk;
    if (g_override_waves == 1 || g_override_waves == 2 || g_override_waves == 4) kw = g_override_waves;
    while (kw > 1 && ((K / sk) % (kw * kalign)) != 0) kw >>= 1;
    pl.kw = kw;
  } else {
    // 16 < M <= 128: single-wave tiles of MB*16 rows, two K parts per workgroup; split across workgroups until a
    // wave streams <= 2048 k (a wave keeps only RING x 2 KiB in flight, so short parts = more bytes in flight).
    // M > 32 (64-row tiles: 20-us kernels, the 5-us slab epilogue is cheap next to them) keeps splitting, down to
    // 512 k per wave, until ~1.5 workgroups per CU are in flight: at bs = 64 the Llama-3-8B qkv / o projections ran
    // on 96 / 64 workgroups at 0.6 TB/s (profiles/r02_*).
    int kw = (pl.mb == 4 && !w8 && OMNI_GEMV_AR_MB4 == 2) ? 4 : 2;
    while (kw > 1 && (K % (kw * kalign)) != 0) kw >>= 1;
    auto fits = [&](int s) { return ok(s) && ((K / s) % (kw * kalign)) == 0; };
    // a part should be whole ring rounds (the remainder runs one unpipelined step at a time)
    const int ring_k = 64 * (w8 ? 4 : (pl.mb == 4 ? OMNI_GEMV_RING_MB4 : 8));
    int best = 0;
    for (int strict = 1; strict >= 0 && best == 0; --strict) {
      for (int s = 1; s <= 64; ++s) {
        const int part = K / (s * kw);
        if (!fits(s) || part < (kw == 4 ? 256 : 512) || (strict && (part % ring_k) != 0)) continue;
        best = s;
        if (kw == 4) {   // 64-row tile, four K parts per workgroup: <= 1024 k per wave and >= 768 waves (measured, r02_e)
          if (part <= 1024 && ngroups * s * pl.mz * kw >= 768) break;
        } else if (part <= 2048 && (pl.mb < 4 || ngroups * s * pl.mz >= 384)) {
          break;
        }
      }
    }
    if (best == 0) best = 1;
    sk = best;
    if (g_override_sk > 0 && ok(g_override_sk)) sk = g_override_sk;
    if (g_override_waves == 1 || g_override_waves == 2 || (g_override_waves == 4 && kw == 4)) kw = g_override_waves;
    while (kw > 1 && ((K / sk) % (kw * kalign)) != 0) kw >>= 1;
    pl.kw = kw;
  }
  pl.sk = sk;
  pl.kslice = K / sk;
  return pl;
}

// Tile height, K parts inside a workgroup and use of the slab form for w4a8_gemm_exact_kernel: the smallest modelled time.
//
// The model's numbers are measured times of the kernel on an MI355X (us; 150 - 4096 rows at N x K = 6144 x 4096, 4096 x 4096, 28672 x 4096
// and 4096 x 14336): one four-wave workgroup on a CU, two of them, and one eight-wave workgroup (KW = 2), each as fixed + per 256-k chunk
// and 16-row blocks.  A grid of n workgroups per CU is whole pairs and a rest that runs alone or in pairs.  What the choice is about is
// the last round: 1501 rows of the 4096 x 14336 projection were 192 tiles of 128 rows on 256 CUs (86.6 us per-channel, 171 per-group,
// 129 W8A8); 256 tiles of 96 rows with two K parts each take 70.5 / 116 / 95.  2331 rows: 304 tiles, i.e. two rounds (141 / 226 / 197 us);
// 480 tiles of 80 rows 111 / 184 / 160.  Few rows: 333 rows of 4096 x 4096 24.6 us with K slices over the grid, slabs and their epilogue
// launch, 18.6 with 64-row tiles and KW = 2.
struct TileCost {
  float fix[3], chunk[3][5];      // [alone, pair, KW = 2][mb - 4]
};
static const TileCost kTileCost[3] = {
    {{3.8f, 7.5f, 5.5f}, {{1.12f, 1.20f, 1.36f, 1.21f, 1.44f}, {1.50f, 1.80f, 2.10f, 2.14f, 2.40f}, {0.82f, 0.92f, 1.06f, 1.08f, 1.16f}}},
    {{1.5f, 5.0f, 5.0f}, {{2.18f, 2.52f, 2.74f, 2.65f, 3.00f}, {2.92f, 3.18f, 3.46f, 3.54f, 3.94f}, {1.52f, 1.72f, 1.95f, 2.00f, 2.20f}}},
    {{3.5f, 6.5f, 4.7f}, {{1.63f, 1.80f, 1.88f, 2.12f, 2.24f}, {2.18f, 2.65f, 3.00f, 3.08f, 3.36f}, {1.22f, 1.36f, 1.48f, 1.62f, 1.78f}}},
};

static float grid_time(const TileCost& c, int mb, int kw, long long workgroups, float chunks) {
  auto t = [&](int kind) { return c.fix[kind] + c.chunk[kind][mb - 4] * chunks; };
  if (kw == 2) {      // (nothing runs beside the next one's start: 4 us more per further round)
    const long long rounds = (workgroups + 255) / 256;
    return (float)rounds * (t(2) + 4.f) - 4.f;
  }
  const long long pairs = workgroups / 512, rest = workgroups - pairs * 512;
  return (float)pairs * t(1) + (rest == 0 ? 0.f : rest <= 256 ? t(0) : t(1));
}

// w8a8_tiles_kernel: rounds of a tile per CU.  A stage takes 0.95 us where few CUs have a tile and 1.4 where all have one; 8 us a tile for its
// ends, which is what short K loses here.  (MI355X, this kernel against the best tiles of the other: 12001 rows of 28672 x 4096 1057 us / 1406, of 4096 x 14336 499 / 681, of
// 16640 x 1024 213 / 252, of 16384 x 512 152 / 158; 2331 rows of 6144 x 4096 52 / 66; 1501 rows of 4096 x 14336, 96 tiles, 149 / 112.  The stages' times are those of the kernel
// before its lines were touched ahead; with them it is up to a tenth faster, and sizes at the line go to the slower one: over 142 sizes of 300 - 12001 rows the rule takes 1.4 % more
// time than the better of the two, 8000 rows of 2048 x 2048 41 us for 32, 1501 of 16640 x 1024 43 for 35, 1024 of 8192 x 28672 255 for 229.  From 512 of K: the kernel's first
// stage and its last two are not the same.)
static float tiles_time(long long tiles, int stages) {
  const long long rounds = tiles / 256;
  const float rest = (float)(tiles - rounds * 256) / 256.f;
  return 3.f + (float)rounds * (8.f + 1.4f * (float)stages) + (rest > 0.f ? 8.f + (0.95f + 0.45f * rest * rest) * (float)stages : 0.f);
}

// w4a8_tiles_kernel, per-group: the same, a stage of 1.3 us where few CUs have a tile and 1.65 where all have one.  (MI355X, this kernel against the other's best: 8000 rows
// of 8192 x 28672 1560 us / 1914, of 28672 x 4096 845 / 971, of 16384 x 1024 185 / 187, of 2048 x 512 21 / 20; 2331 rows of 4096 x 14336, 160 tiles, 178 / 192; 1800
// rows of it, 128 tiles, 158 / 128; 1024 rows of 6144 x 4096, 96 tiles, 53 / 36.  Over 150 sizes of 257 - 8000 rows the rule takes 10 % less time than without
// this kernel, the better of the two 10.2 %.)
static float w4_tiles_time(int mode, long long tiles, int stages) {
  const long long rounds = tiles / 256;
  const float rest = (float)(tiles - rounds * 256) / 256.f;
  // per-channel: 0.98 and 1.24.  (MI355X, us, the best of w4a8_gemm_exact_kernel / here: 4096 rows of 4096 x 14336 162 / 149, of 28672 x 4096 346 / 328, 4000 of 8192 x 28672 664 / 572, of 8192 x 8192
  // 188 / 175; 1280 of 28672 x 4096 118 / 133, 3000 of 6144 x 4096 65 / 86, 1500 of 4096 x 4096 26 / 42.)
  if (mode == MODE_CHN) return (float)rounds * (9.f + 1.24f * (float)stages) + (rest > 0.f ? 9.f + (0.98f + 0.27f * rest * rest) * (float)stages : 0.f);
  return (float)rounds * (8.f + 1.65f * (float)stages) + (rest > 0.f ? 8.f + (1.3f + 0.35f * rest) * (float)stages : 0.f);
}

// The same with K of the last round's tiles shared out (the rounds in front of it as above): every CU at work for the stages of a head, and 17 us (per-channel 21) for a second part's sums and two more ends, 4 for each
// part more.  1e30f: it has nothing
// to share.  (MI355X, whole tiles / shared, us: per-group 2331 rows of 4096 x 14336, 20 tiles of an XCD, 181 / 152; 3000, 24 tiles, 181 / 164; 6000, 32 + 16, 342 / 300; 2331 of 28672 x 4096, 4 x 32 + 12, 284 / 278;
// 1500, 2 x 32 + 20, 167 / 172, 3000 of 4096 x 4096, 24 tiles, 54 / 61; per-channel 3000 of
// 4096 x 14336 137 / 128, 6000 265 / 237, 5000 264 / 209, 1000 of 8192 x 28672, 16 tiles, 241 / 165; 1501 of 28672 x 4096 with the unit, 2 x 32 + 20, 140 / 145.)
static float shared_time(int mode, long long tiles, int stages) {
  const float stage = mode == MODE_GRP ? 1.65f : mode == MODE_W8 ? 1.4f : 1.24f, ends = mode == MODE_CHN ? 9.f : 8.f, more = mode == MODE_CHN ? 21.f : 17.f;
  const int left = (int)((tiles + 7) / 8 % SHARE_PER);
  const ShareSplit sp = share_split(left, stages);
  if (left == 0 || sp.head == stages) return 1e30f;
  return (float)((tiles + 7) / 8 / SHARE_PER) * (ends + stage * (float)stages) + more + 4.f * (float)(sp.used - left - 1) / (float)left + stage * (float)sp.head;
}

PrefillPlan plan_prefill(int M, int N, int K, int mode, int sk, bool slab_only, bool scratch) {
  const TileCost& c = kTileCost[mode];
  PrefillPlan best{8, 1, slab_only ? sk : 1};
  // rows far apart are slower to read, but not where K slices read them at several places (512 rows of 8192 x 28672 per-channel: 1.08 us per chunk of
  // two K parts, 0.83 at 14336; 256 rows of 7168 x 8192 W8A8 1.68, 1.25 at 4096: 126 and 58 us where slices take 105 and 47)
  const float far = mode == MODE_W8 && K >= 8192 ? 1.2f : mode == MODE_CHN && K >= 16384 ? 1.17f : 1.f;
  // whole bands of 8 full row tiles go in an order of their own (w4a8_gemm_exact_kernel): 4096 rows of 8192 x 28672 per-channel 607 us, 632 with K in two
  // parts; 4096 of 10240 x 8192 per-group 336, 346 in tiles of 112 rows; 8192 of 5120 x 13824 546, 563
  const float whole_bands = mode != MODE_W8 && M % 1024 == 0 ? 0.96f : 1.f;
  float time = 1e30f;
  auto offer = [&](int mb, int kw, int split) {
    const long long tiles = (long long)((M + 16 * mb - 1) / (16 * mb)) * (N / 256) * split;
    float t = grid_time(c, mb, kw, tiles, (split == 1 ? far : 1.f) * (float)(K / (split * KCHUNK)));
    // the slabs written, read and reduced by a launch of their own
    if (split > 1 && !slab_only) t += 4.5f + (float)split * M * N * 8.f / 4.5e6f;
    if (mb == 8 && kw == 1 && split == 1) t *= whole_bands;
    if (t < time) { time = t; best = PrefillPlan{mb, kw, split}; }
  };
  for (int mb = 8; mb >= 4; --mb) {
    if (slab_only || g_override_sk > 0) {
      offer(mb, 1, sk);
      continue;
    }
    offer(mb, 1, 1);
    if (K % (2 * KCHUNK) == 0) offer(mb, 2, 1);
    if (sk > 1) offer(mb, 1, sk);
  }
  if (!slab_only && g_override_sk <= 0 && M >= TILES_M && K >= 4 * TILES_K) {
    const long long tiles = (long long)((M + TILES_M - 1) / TILES_M) * (N / TILES_N);
    const int stages = K / TILES_K;
    const float whole = mode == MODE_W8 ? tiles_time(tiles, stages) : w4_tiles_time(mode, tiles, stages);
    // (the models' errors: per-channel the other kernel takes 1.05 - 1.15 of the time above where all CUs are at work, in whole bands of 8 row tiles too: 4096 rows of 4096 x 14336 136 us, in truth 162)
    if (mode == MODE_CHN) {
      const long long places = best.kw == 1 && best.sk == 1 ? 512 : 0, grid = (long long)((M + 16 * best.mb - 1) / (16 * best.mb)) * (N / 256);
      const float busy = places ? (float)grid / (float)((grid + places - 1) / places * places) : 1.f;
      if (best.mb == 8 && best.kw == 1 && best.sk == 1) time /= whole_bands;
      time *= 1.f + 0.08f * std::max(0.f, (busy - 0.8f) / 0.2f);
    }
    const bool take = mode == MODE_W8 ? whole < time : g_override_waves == 16 || whole < (mode == MODE_GRP ? 0.98f : 0.985f) * time;      // (per-channel 1501 rows of 28672 x 4096, 0.994 here, 147 / 145 us in a prompt, whose step is no faster for it)
    // (in place of whole W8A8 tiles: by 18 us, which are faster than reckoned in a last round of two thirds and more of the CUs.  us, whole / shared, rounds of tiles in brackets.  Shared by this rule: 4096 x 14336, 1501 rows (0.38)
    // 109 / 92, 2100 (0.56) 153 / 125, 4200 (1.06) 275 / 209, 6000 (1.50) 282 / 258; 10240 x 8192, 2000 (1.25) 167 / 147; 8192 x 28672, 1501 (0.75) 310 / 280.  Left whole: 4096 x 14336, 3000 (0.75) 142 / 143, a whole prompt
    // 3342 / 3402, 3500 (0.88) 153 / 165, 7000 (1.75) 300 / 304; 6144 x 4096, 4800 (1.78) 98 / 112; 28672 x 4096 with the unit, 3000 (5.25) 291 / 297.  Where the last round has few tiles and K is short the line leaves
    // some: 6144 x 4096, 2700 - 3400 (1.03 - 1.31) 88 - 105 / 80 - 94; 4096 x 4096, 4800 (1.19) 94 / 84; 4096 x 14336, 2331 (0.62) 131 - 140 / 130; 8192 x 8192, 1000 (0.50) 78 / 66, 2600 (1.38) 175 / 163)
    const bool share = scratch && shared_time(mode, tiles, stages) < (take ? whole - (mode == MODE_W8 ? 18.f : 4.f) : (mode == MODE_CHN ? 1.f : 0.93f) * time - 4.f);
    if ((take || share) && mode == MODE_W8) best = PrefillPlan{16, 1, 1};
    best.w4_tiles = (take || share) && mode != MODE_W8;
    best.share = share;
  }
  return best;
}

// One pass over K by the kernels that have the unit: the tiles, and w4a8_gemm_exact_kernel of one K part.
bool silu_rows_plan(int M, int N, int K, int mode, bool scratch, GemmPlan* pl, PrefillPlan* pp) {
  if (M <= 128 || N < 256 || K < 64 || mode < MODE_CHN || mode > MODE_W8) return false;
  if (N % 256 != 0 || K % KCHUNK != 0) return false;
  *pl = plan_gemm(M, N, K, mode == MODE_GRP ? 128 : 64, false, mode == MODE_W8);
  if (pl->midm || !exact_sizes(M, N, K, pl->kslice)) return false;
  *pp = plan_prefill(M, N, K, mode, pl->sk, false);
  if (mode == MODE_W8 ? pp->mb != 16 : !pp->w4_tiles && (pp->sk != 1 || pp->kw != 1)) return false;
  if (scratch) *pp = plan_prefill(M, N, K, mode, pl->sk, false, true);
  return true;
}

}  // namespace omni

extern "C" int omni_gemm_silu_rows_ok(int M, int N, int K, int mode) {
  omni::GemmPlan pl;
  omni::PrefillPlan pp;
  return omni::silu_rows_plan(M, N, K, mode, false, &pl, &pp) ? 1 : 0;
}

extern "C" void omni_gemm_set_plan_override(int waves, int sk) {
  omni::g_override_waves = waves;
  omni::g_override_sk = sk;
}

extern "C" void omni_gemm_set_midm_override(int mode, int sk) {
  omni::g_midm_mode = mode;
  omni::g_midm_sk = sk;
}

extern "C" void omni_gemm_get_plan(int M, int N, int K, int kalign, int* mb, int* waves, int* sk) {
  omni::GemmPlan pl = omni::plan_gemm(M, N, K, kalign, false, false);
  if (mb) *mb = pl.mb;
  if (waves) *waves = pl.waves;
  if (sk) *sk = pl.sk;
}

extern "C" int omni_gemm_get_prefill_plan(int M, int N, int K, int mode, int slabs_only, int* mb, int* kw, int* sk) {
  using namespace omni;
  if (M <= 128 || N < 64 || N % 64 || K < 64 || K % 64 || mode < 0 || mode > 2 || (slabs_only && M > 512)) return 0;
  const GemmPlan pl = plan_gemm(M, N, K, mode == MODE_GRP ? 128 : 64, slabs_only != 0, mode == MODE_W8);
  const bool exact = exact_sizes(M, N, K, pl.kslice);
  const PrefillPlan pp = exact ? plan_prefill(M, N, K, mode, pl.sk, slabs_only != 0) : PrefillPlan{8, 1, pl.sk};
  if (mb) *mb = pp.mb;
  if (kw) *kw = pp.kw;
  if (sk) *sk = pp.sk;
  return exact ? 1 : 2;
}

static int prefill_w4_tiles(int M, int N, int K, int mode) {
  using namespace omni;
  if (M <= 128 || N < 64 || N % 64 || K < 64 || K % 64) return 0;
  const GemmPlan pl = plan_gemm(M, N, K, mode == MODE_GRP ? 128 : 64, false, false);
  return exact_sizes(M, N, K, pl.kslice) && plan_prefill(M, N, K, mode, pl.sk, false).w4_tiles;
}
extern "C" int omni_gemm_prefill_group_tiles(int M, int N, int K) { return prefill_w4_tiles(M, N, K, omni::MODE_GRP); }
extern "C" int omni_gemm_prefill_channel_tiles(int M, int N, int K) { return prefill_w4_tiles(M, N, K, omni::MODE_CHN); }

extern "C" size_t omni_gemm_share_bytes(int M, int N, int K, int mode) {
  using namespace omni;
  if (M < TILES_M || N < TILES_N || K < 4 * TILES_K || mode < MODE_CHN || mode > MODE_W8) return 0;
  const GemmPlan pl = plan_gemm(M, N, K, mode == MODE_GRP ? 128 : 64, false, mode == MODE_W8);
  return !pl.midm && exact_sizes(M, N, K, pl.kslice) && plan_prefill(M, N, K, mode, pl.sk, false, true).share ? SHARE_MARKS + (size_t)8 * share_places_of(M, N, K) * SHARE_PART : 0;
}

extern "C" int omni_gemm_arm_share(void* scratch, size_t bytes) {
  using namespace omni;
  g_armed_share = TileShare{};
  if (!scratch) return OMNI_OK;
  // (two parts of a tile on every XCD are the least)
  if (bytes < SHARE_MARKS + (size_t)8 * 2 * SHARE_PART || (reinterpret_cast<uintptr_t>(scratch) & 15) != 0) return OMNI_EINVAL;
  static std::atomic<unsigned long long> launches{(unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count()};
  const size_t places = std::min<size_t>((bytes - SHARE_MARKS) / ((size_t)8 * SHARE_PART), 2 * SHARE_PER);
  g_armed_share = TileShare{static_cast<v4i*>(scratch), reinterpret_cast<unsigned long long*>(static_cast<char*>(scratch) + 8 * places * SHARE_PART), launches.fetch_add(1, std::memory_order_relaxed) << 8,
                            (int)places};
  return OMNI_OK;
}

extern "C" int omni_gemm_share_parts(int own, int stages, int* parts, int room) {
  using namespace omni;
  if (own < 0 || stages < SHARE_MIN || stages > 1 << 16 || !parts) return OMNI_EINVAL;
  int n = 0;
  for (int wg = 0; wg < SHARE_PER; ++wg) {
    TileParts p(wg, own, stages);
    for (int at = wg; p.next(at); at += SHARE_PER, ++n) {
      if (n == room) return OMNI_EINVAL;
      const int part[7] = {wg, p.tile, p.k0, p.stages, p.shared() ? p.slot(p.me()) : -1, p.lo, p.hi};
      std::copy(part, part + 7, parts + 7 * n);
    }
  }
  return n;
}

extern "C" int omni_gemm_share_armed(void) { return omni::g_armed_share.sums != nullptr; }

// Would the row-kernel-free decode forms (omni_*_gemm_silu for gate_up, omni_*_gemm_partial_f16 for o / down) accept a layer
// with these dimensions?  The same plan conditions launch_gemm_silu / launch_gemm_partial_f16 check at launch (one place to
// keep in step: qgemm_kernel.h), so that a driver can choose its fusion level BEFORE its first step instead of running into
// EINVAL there (hidden > 4096: the gate_up plan splits K across workgroups; rows > N / 64: no rider per row).
// mode: 0 per-channel W4A8 (row sums needed), 1 per-group W4A8, 2 W8A8.
extern "C" int omni_gemm_rowfree_ok(int M, int hidden, int attn_dim, int inter, int mode) {
  using namespace omni;
  if (mode < 0 || mode > 2 || M < 1 || M > 16 || hidden < 64 || attn_dim < 64 || inter < 64) return 0;
  const int kalign = mode == MODE_GRP ? 128 : 64;
  const bool w8 = mode == MODE_W8;
  if (hidden % 64 || attn_dim % kalign || inter % kalign || (2 * inter) % 128 || hidden % kalign) return 0;
  const GemmPlan gu = plan_gemm(M, 2 * inter, hidden, kalign, false, w8);
  if (gu.sk != 1 || gu.mb != 1) return 0;
  const int ar = w8 ? GemvCfg<1, MODE_W8>::AR : GemvCfg<1, MODE_CHN>::AR;
  for (const int K : {attn_dim, inter}) {
    if (hidden / 64 < M) return 0;
    const GemmPlan pl = plan_gemm(M, hidden, K, kalign, true, w8);
    if (pl.mb != 1 || pl.kw < 2) return 0;
    if (mode == MODE_CHN && (size_t)K * sizeof(float) > (size_t)pl.kw * 2 * 16 * ar * KSTEP) return 0;   // rider's LDS row
  }
  return 1;
}

// Largest K split any plan of an (M, N, K) problem can take: the maximum over the K alignments of the three GEMM flavours (64;
// 128 for per-group), over W4 / W8 rows and over the mid-M kernel off / forced on WITH every legal forced split (so that a
// buffer sized once stays large enough under omni_gemm_set_midm_override(1, sk), whatever the mode was when it was sized;
// the loop used to skip forced mode 1 and the forced sk).  `deferred`: the slab-only forms' plans.
static int max_plan_sk(int M, int N, int K, bool deferred) {
  using namespace omni;
  int sk = 1;
  const int keep_mode = g_midm_mode, keep_sk = g_midm_sk;
  for (int midm = 0; midm < 2; ++midm) {
    g_midm_mode = midm;
    for (int force = midm ? 16 : 0; force >= 0; force = (force > 2 ? force - 1 : (force == 2 ? 0 : -1))) {
      g_midm_sk = force;      // 0: the heuristic split; 2 .. 16: omni_gemm_set_midm_override(1, force)
      for (int kalign = 64; kalign <= 128; kalign *= 2) {
        if (K % kalign != 0) continue;
        for (int w8 = 0; w8 < 2; ++w8) {
          const GemmPlan pl = plan_gemm(M, N, K, kalign, deferred, w8 != 0);
          if (pl.sk > sk) sk = pl.sk;
        }
      }
    }
  }
  g_midm_mode = keep_mode;
  g_midm_sk = keep_sk;
  return sk;
}

// plain entry points (omni_*_gemm): scratch only where a plan splits K (0 otherwise: M = 129 .. 512 used to pin one
// M x N slab here for the sake of the slab-only forms, which now have their own query)
extern "C" size_t omni_gemm_workspace_bytes(int M, int N, int K) {
  if (M < 1 || N < 64 || K < 64) return 0;
  const int sk = max_plan_sk(M, N, K, false);
  return sk > 1 ? (size_t)sk * M * N * sizeof(int32_t) : 0;
}

// slab-only forms (omni_*_gemm_partial[_f16], M <= 512): they write their int32 accumulators even when the plan keeps K whole
extern "C" size_t omni_gemm_partial_workspace_bytes(int M, int N, int K) {
  if (M < 1 || M > 512 || N < 64 || K < 64) return 0;
  const int a = max_plan_sk(M, N, K, true), b = max_plan_sk(M, N, K, false);
  return (size_t)(a > b ? a : b) * M * N * sizeof(int32_t);
}

// ---- fused extension: L2 weight prefetch riding on the next row kernel (common.h: PrefetchArgs) -------------------
extern "C" int omni_prefetch_arm_gemm(const void* weight, int M, int N, int K, int mode, int deferred,
                                      int64_t budget_bytes, int blocks) {
  using namespace omni;
  g_armed_prefetch = PrefetchArgs{};
  if (!weight || blocks <= 0 || budget_bytes <= 0) {                        // disarm (and forget every pending load-policy entry)
    if (!weight)
      for (auto& w : g_prefetched_w) w = nullptr;
    return OMNI_OK;
  }
  // mode | 0x10: the gate_up form with the fused SiLU epilogue (omni_w4a8_per_*_gemm_silu): workgroup x streams tile row x
  // of the gate half and tile row N/64 + x of the up half
  const bool silu = (mode & 0x10) != 0;
  // mode | 0x20: the consuming GEMV keeps its non-temporal weight loads (the prefetch then only warms the memory-side
  // cache); default: that GEMV -- the next decode-shape GEMM enqueued by this thread on this weight tensor -- loads plain
  const bool keep_nt = (mode & 0x20) != 0;
  mode &= 0xF;
  if (silu && (mode == MODE_W8 || deferred || (N / 64) % 8 != 0)) return mode == MODE_W8 ? OMNI_EINVAL : OMNI_OK;
  if (mode < 0 || mode > 2 || M < 1 || M > 128 || N % 64 != 0 || K % 64 != 0 || K < 64) return OMNI_EINVAL;
  const GemmPlan pl = plan_gemm(M, N, K, mode == MODE_GRP ? 128 : 64, deferred != 0, mode == MODE_W8);
  PrefetchArgs pf{};
  pf.base = static_cast<const uint8_t*>(weight);
  const int groups_per_wg = pl.waves;                                       // 64-channel groups per workgroup
  pf.gx = (N / 64 + groups_per_wg - 1) / groups_per_wg;
  pf.gy = pl.sk;
  pf.kw = pl.kw;
  if ((N / 64) % groups_per_wg != 0) return OMNI_OK;                         // ragged last workgroup: skip the hint
  if (mode == MODE_W8) {
    // [N][K] int8 rows of K bytes: a wave walks its 64 rows together along k, so a budget below the matrix size
    // fetches whole rows of the first rows of every workgroup (K-parts of a row can be shorter than a 1-KiB piece)
    if (pf.gy > 1 && (pf.gx & 7) != 0) return OMNI_OK;                       // K-slices of a row group on different XCDs
    pf.row_bytes = K; pf.rows_per_wg = 64 * groups_per_wg;
    pf.gy = 1; pf.kw = 1;
    const long long total = (long long)N * K;
    double f = total > budget_bytes ? (double)budget_bytes / (double)total : 1.0;
    pf.rows_pf = (int)(pf.rows_per_wg * f);
    pf.pf_bytes = (K / 1024) * 1024;
    if (pf.rows_pf < 1 || pf.pf_bytes < 1024) return OMNI_OK;
  } else {
    pf.row_bytes = (long long)K * 16; pf.rows_per_wg = 2 * groups_per_wg;
    if (silu) {
      // as 2 * (N/64) single-row workgroups: item v = tile row v is fetched on XCD v % 8, and (N/64) % 8 == 0 makes that
      // the XCD of the real workgroup v % (N/64) for both of its rows
      pf.rows_per_wg = 1;
      pf.gx = N / 32;
    }
    pf.rows_pf = pf.rows_per_wg;
    const long long part_bytes = pf.row_bytes / ((long long)pf.gy * pf.kw);
    const long long total = pf.row_bytes * pf.rows_per_wg * pf.gx;
    long long want = part_bytes;
    if (total > budget_bytes) want = (long long)((double)part_bytes * (double)budget_bytes / (double)total);
    want = (want / 1024) * 1024;
    if (want < 1024 || part_bytes < 1024) return OMNI_OK;                    // parts too small for 1-KiB pieces: skip
    pf.pf_bytes = (int)want;
  }
  pf.blocks = (blocks + 7) & ~7;
  static const int delay = omni_knob("OMNI_PREFETCH_DELAY", 0);
  pf.delay = delay;
  g_armed_prefetch = pf;
  if (!keep_nt) note_prefetched_weight(weight);     // the GEMV on this weight tensor reads L2-resident lines: plain loads
  return OMNI_OK;
}

// 3: omni_gemm_set_weight_policy removed (the load policy is per call: omni_prefetch_arm_gemm mode bit 0x20);
//    omni_gemm_workspace_bytes covers the slab-only forms (>= one slab up to 512 rows); omni_gemm_set_midm_override added.
// 4: the slab-only forms have their own query (omni_gemm_partial_workspace_bytes) and omni_gemm_workspace_bytes is the plain
//    entry points' again (0 without a K split); both cover every legal omni_gemm_set_midm_override; the (norm -> GEMV) pair
//    entry points (omni_w4a8_per_*_norm_gemm_fused, omni_norm_gemm_fused_ok) added.
extern "C" int omni_abi_version(void) { return 4; }
