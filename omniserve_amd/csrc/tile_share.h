// The K of the last round's tiles shared out among an XCD's workgroups (int8 tiles of 256 x 256: qgemm_tiles.h, qgemm_group_tiles.h).
//
// A grid of one workgroup per CU that takes whole tiles leaves much of the chip idle in its last round: 160 tiles on 256 CUs take as long as 256.  Here a workgroup that has a tile of that round
// takes its first stages only; the workgroups that have none divide the others' stages, in equal shares: the end of one tile's, perhaps whole ones, the beginning of another's.  The first
// stages are as many as make both kinds of workgroups end together, a part beginning and leaving its sums counted as three and a half stages.  (Equal shares of everything from one end to the other, which
// splits as many tiles: workgroups that work at different k find less of each other's operands in the L2, a stage of the per-group tiles takes 1.9 us instead of 1.65.)
//
// Whoever comes to a tile's mark last finishes it: the others leave their int32 sums (256 KB a part, 16 bytes a lane and piece) in a scratch buffer of up to 62 parts an XCD (share_places: 10 - 124 MB in all).  Nobody waits for anybody.
//  * sums and marks are written and read at agent scope (sc1), past the XCDs' L2s and the CUs' L1s: a part's stores are through before its arrival.
//  * a mark holds the launch's token and the number of arrivals.  Whatever else it holds counts as none, so that nobody clears it; a tile's last arrival leaves 0 in it, for a captured launch
//    that runs again.
// Sums of integers in another order: the same bits.
//
// MI355X, us, whole tiles (or the other kernel's, where those were faster) / shared: per-group 2331 rows of 4096 x 14336, 160 tiles, 181 / 150; 6000 rows, 384 tiles, 342 / 300; 4940, 320 tiles, 359 / 270; 2774 rows of
// 8192 x 28672 666 / 528; 2331 of 28672 x 4096 with the unit, 1120 tiles, 284 / 279; W8A8 1937 rows of 4096 x 14336, 128 tiles, 114 / 99, 4225 272 / 206.  Short of the rounds saved (1.5 instead of 2
// would be 256) by what a whole chip at work costs: the card's power lets 160 CUs run faster than 256.  Of the 150 us of the first, 12 are the sums written and 5 the sums read.
#pragma once
#include "common.h"
#include "lm/mfma_pinned.h"

namespace omni {

struct TileShare {
  v4i* sums;                       // [8 XCDs][places][64][256]; null: every tile whole
  unsigned long long* marks;       // [8 XCDs][32]
  unsigned long long token;        // << 8
  int places;                      // of an XCD's parts
};
constexpr int SHARE_PER = 32;                               // workgroups of an XCD
constexpr int SHARE_COST2 = 7;                               // twice the stages that a part's ends are worth
constexpr int SHARE_MIN = 4;                                // stages that a part has at least: the kernels' loops want them
constexpr int SHARE_PART = 64 * 256 * 16, SHARE_MARKS = 8 * SHARE_PER * 8;      // bytes of a part's sums and of all marks

// How an XCD's last `left` tiles (1 .. 31) of ns stages are dealt: `used` workgroups, the first `left` of which take `head` stages of a tile each; head = ns: not shared.
struct ShareSplit {
  int used, head;
};
__host__ __device__ inline ShareSplit share_split(int left, int ns) {
  ShareSplit r{SHARE_PER, ns};
  if (r.used > left * ns / 8) r.used = left * ns / 8;
  if (r.used > left * 5) r.used = left * 5;
  if (r.used <= left) return r;
  const int head = (left * (2 * ns + SHARE_COST2) + 2 * r.used - 1) / (2 * r.used);
  if (ns - head >= SHARE_MIN && left * (ns - head) >= 7 * (r.used - left)) r.head = head;      // (7: no two borders move to one place)
  return r;
}
// Places that the parts of an XCD's last `left` tiles lie in: share and tile number together are below used - 1 (a share and the next have one tile in common at most, so that the sum is another for
// each part), the first stages' parts behind them.
__host__ __device__ inline int share_places(int left, int used) { return used - 1 + left; }

__device__ __forceinline__ const uint8_t* wave_uniform(const uint8_t* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));      // (of type int: no sign into the upper half)
  return (const uint8_t*)((uint64_t)hi << 32 | lo);
}

// (of a value that all lanes have)
__host__ __device__ inline int wave_uniform(int v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}

// The parts of an XCD's wg-th workgroup (of SHARE_PER), one after the other.  How they are dealt is host code, too: omni_gemm_share_parts.
struct TileParts {
  int wg, own, ns, left, whole, head, used, from, to;       // whole: tiles taken one by one; from, to: this workgroup's share of the last round's stages behind the first ones, tile after tile
  int tile = 0, k0 = 0, stages = 0, rest = 0, lo = 0, hi = 0;      // the part opened last; rest: its tile among the last round's; lo .. hi: the workgroups behind the first `left` that have parts of it

  __host__ __device__ __forceinline__ int border(int s) const {      // where the share of the s-th of them begins
    const int n = ns - head, x = s * left * n / (used - left), in = x % n;
    return in < SHARE_MIN ? x - in : n - in < SHARE_MIN ? x - in + n : x;
  }
  __host__ __device__ __forceinline__ TileParts(int wg_, int own_, int ns_) : wg(wg_), own(own_), ns(ns_), left(own_ % SHARE_PER), whole(own_), head(ns_), used(0), from(0), to(0) {
    if (left == 0) return;
    const ShareSplit sp = share_split(left, ns);
    if (sp.head == ns) return;
    whole = own - left;
    used = sp.used;
    head = sp.head;
    const int s = wg - left;
    if (s >= 0 && s < used - left) {
      from = border(s);
      to = border(s + 1);
    }
  }
  __host__ __device__ __forceinline__ bool next(int at) {
    tile = at;
    k0 = 0;
    stages = ns;
    lo = hi = -1;
    if (at < whole) return true;
    if (at < own) {
      rest = at - whole;
      stages = head;
    } else {
      if (from >= to) return false;
      const int n = ns - head;
      rest = from / n;
      tile = whole + rest;
      k0 = from - rest * n;
      stages = n - k0 < to - from ? n - k0 : to - from;
      k0 += head;
      from += stages;
    }
    // the share that has the tile's first stage behind the head, and the one that has the last
    const int n = ns - head;
    lo = rest * (used - left) / left;
    while (lo > 0 && border(lo) > rest * n) --lo;
    while (border(lo + 1) <= rest * n) ++lo;
    hi = lo;
    while (border(hi + 1) < (rest + 1) * n) ++hi;
    lo = wave_uniform(lo), hi = wave_uniform(hi), from = wave_uniform(from);
    return true;
  }
  __host__ __device__ __forceinline__ bool shared() const { return lo >= 0; }
  // where the part of the s-th of them lies in the scratch buffer, -1 the first stages'
  __host__ __device__ __forceinline__ int slot(int s) const { return rest + (s < 0 ? used - 1 : s); }
  __device__ __forceinline__ uint32_t place(const TileShare& p, int s) const {
    return __builtin_amdgcn_readfirstlane(((int)(blockIdx.x & 7) * p.places + slot(s)) * SHARE_PART);
  }
  static __device__ __forceinline__ auto buffer(const TileShare& p) { return __builtin_amdgcn_make_buffer_rsrc(p.sums, 0, 8 * p.places * SHARE_PART, 0x00020000); }
  __host__ __device__ __forceinline__ int me() const { return k0 == 0 ? -1 : wg - left; }

  // A part's sums are in c: does this workgroup finish the tile, with what others() adds to them?  If not, or if that was not certain at first, other() has been called, which may request what the
  // next part needs.
  template <int N, int M, class Other>
  __device__ __forceinline__ bool finishes(const TileShare& p, uint8_t* lds_word, v4i (&c)[N][M], Other other) const {
    static_assert(N * M == 64, "64 pieces a lane");
    const int tid = threadIdx.x;
    const unsigned rivals = hi - lo + 1;
    unsigned long long* const mark = p.marks + SHARE_PER * (blockIdx.x & 7) + rest;
    volatile uint32_t* const word = (volatile uint32_t*)lds_word;
    if (tid == 0) *word = __hip_atomic_load(mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (p.token | rivals);
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(*word)) {
      const auto rsrc = buffer(p);
      const uint32_t mine = place(p, me());
      accumulators_stay(c);
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) __builtin_amdgcn_raw_buffer_store_b128(c[i][j], rsrc, tid * 16, mine + (i * M + j) * 4096, 16);
      other();
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        unsigned long long was = __hip_atomic_load(mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), is;
        do is = (was & ~255ull) == p.token ? was + 1 : p.token | 1;
        while (!__hip_atomic_compare_exchange_strong(mark, &was, is, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        *word = (unsigned)(is & 255) == rivals + 1;
      }
      __syncthreads();
      if (!__builtin_amdgcn_readfirstlane(*word)) return false;
    }
    if (tid == 0) __hip_atomic_store(mark, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  // x[q]: the other parts' sums of piece number(q)
  template <int M, class Number>
  __device__ __forceinline__ void others(const TileShare& p, Number number, v4i (&x)[M]) const {
    const int tid = threadIdx.x;
    const auto rsrc = buffer(p);
    auto piece = [&](uint32_t at, int q) { return __builtin_amdgcn_raw_buffer_load_b128(rsrc, tid * 16, at + number(q) * 4096, 16); };
    // (the first of them is this one or another)
    int s = me() < 0 ? lo : -1;
    uint32_t at = place(p, s);
#pragma unroll
    for (int q = 0; q < M; ++q) x[q] = piece(at, q);
    for (s = max(s + 1, lo); s <= hi; ++s) {
      if (s == me()) continue;
      at = place(p, s);
      v4i y[M];
#pragma unroll
      for (int q = 0; q < M; ++q) y[q] = piece(at, q);
#pragma unroll
      for (int q = 0; q < M; ++q) x[q] += y[q];
    }
  }
};

}  // namespace omni
