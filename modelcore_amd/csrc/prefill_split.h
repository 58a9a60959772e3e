// Key ranges of a chunked prefill with few query blocks (a short chunk against a long prefix, a
// single row): each block's tiles of keys are cut into ranges, a workgroup per range, whose
// unnormalised (o, m, l) go to scratch in fp32 and are merged by a second launch.
//
// How far a block is cut depends on the row's position, which only the device knows, so both
// launches work it out from cache_seqlens. S ranges take a block's n tiles from n * tile time to
// n / S of it and cost S times the writing and reading of the call's partials, so the best S is
// sqrt(n * tile time / partial time). The host gives that ratio and the most ranges for which the
// chip has room. No range is much shorter than kMinRangeKeys keys, so blocks of fewer than twice as many
// are never cut. Ranges are as long as is best for the block of the row with the most tiles (the one with
// its last queries), blocks with fewer tiles get fewer of them, and one that is not cut writes its output
// itself. A cut call's sums run in another order than an uncut one's: the same outputs within the
// dtype's rounding, not the same bits.
//
// A partial is laid out as the accumulators hold it, which is also how the merge reads it: 32 pairs
// by 32 dims in 4 x 64 lanes of four dims (lane (h, col) of step j: pair col, dims 8j + 4h ..), so
// that every access of a wave is 1 KiB in one piece.
//
// Where nothing is cut (a first prompt in a long cache: the host sees the same sizes), the second
// launch is not to cost more than it saves elsewhere: on the bf16 / 128 path it appends the chunk, whose
// keys the ranges read from k and v, and so takes the place of the append's launch; the first ranges of
// all blocks are launched first; and rows too short for a cut are known by one comparison
// (uncut_keys). 100 tokens from position 0 of a 16384-key cache, 32 / 8 heads of 128: 13.0 us with the
// append (15.7 with an append of its own and every workgroup working out its ranges; 12.6 without
// scratch); 500 tokens 24.9 (31.8; 23.9).
//
// Measured (100 tokens of 32 query / 8 KV heads of 128 in bf16 after 8000 keys; 16 blocks of 126
// tiles): uncut 182 us; cut 36.3, of which the merge, with the append, 9.3. With
// partials as rows of D floats (16 bytes of each of 32 rows per store) 6 us more, with the merge's loads
// one range at a time 4. The partials' rate was swept: 2e6 44 us, 4e6 40, 6e6 38, 9e6 36.7; from
// 9e6 on, calls of many rows and few keys lose to the uncut ones (8 x 20 tokens after 500 keys: 28.7
// against 21.0 us).
#pragma once

#include "kernels.h"

#include <algorithm>
#include <cmath>

namespace mcamd {

constexpr int kMaxPrefillSplits = 32;
#ifndef MCAMD_SPLIT_MIN_KEYS
#define MCAMD_SPLIT_MIN_KEYS 256
#endif
constexpr int kMinRangeKeys = MCAMD_SPLIT_MIN_KEYS;

struct SplitGeo {
  int pairs;       // (position, head) pairs per block
  int kt;          // keys per tile
  int n_split;     // ranges per block, at most
  int n_qt, n_bh;  // blocks per (row, KV head), (row, KV head)s
  int groups;      // 32-pair groups per block
  int md;          // 32-dim pieces of the head
  int G, window;
  int uncut_keys;  // rows of at most that many keys are not cut, whatever the block
  float ratio;     // tile time / time of one range's partials of the whole call
  float *part_o;   // [n_split][n_qt * n_bh * groups][md][4][64][4]
  float *part_ml;  // [n_split][n_qt * n_bh * groups][32][2]
  // Index of 32-pair group w of block (qt, bh) within range `part`.
  __device__ __forceinline__ int64_t group(int part, int qt, int bh, int w) const {
    return ((int64_t(part) * n_qt + qt) * n_bh + bh) * groups + w;
  }
  // Four dims 32 d + 8 j + 4 (lane / 32) .. of pair lane % 32 of a group.
  __device__ __forceinline__ float *o(int64_t group, int d, int j, int lane) const {
    return part_o + ((group * md + d) * 4 + j) * 256 + lane * 4;
  }
  __device__ __forceinline__ float *ml(int64_t group, int pair) const {
    return part_ml + (group * 32 + pair) * 2;
  }
};

// First and last key of block qt of a row at position s0 with T_b new tokens.
__device__ __forceinline__ void block_keys(const SplitGeo &g, int s0, int T_b, int qt, int &lo,
                                           int &hi) {
  const int64_t p0 = int64_t(qt) * g.pairs;
  const int64_t pend = min(p0 + g.pairs, int64_t(T_b) * g.G);
  hi = s0 + int((pend - 1) / g.G);
  lo = g.window >= 0 ? max(0, s0 + int(p0 / g.G) - g.window) : 0;
}

// Ranges for `tiles` tiles by the cost rule above.
__host__ __device__ inline int best_splits(float ratio, int tiles, int kt, int most) {
  most = most < tiles / (kMinRangeKeys / kt) ? most : tiles / (kMinRangeKeys / kt);
  const int s = int(sqrtf(float(tiles) * ratio));
  return s < 1 || most < 1 ? 1 : s > most ? most : s;
}

// Ranges of a block of n_tiles tiles.
__device__ __forceinline__ int block_splits(const SplitGeo &g, int s0, int T_b, int n_tiles) {
  if (s0 + T_b <= g.uncut_keys) return 1;
  int lo, hi;
  block_keys(g, s0, T_b, int((int64_t(T_b) * g.G - 1) / g.pairs), lo, hi);
  const int longest = max((hi - lo) / g.kt + 1, n_tiles);
  const int s = best_splits(g.ratio, longest, g.kt, g.n_split);
  const int range = (longest + s - 1) / s;
  return max(1, (n_tiles + range / 2) / range);  // at most s: n_tiles <= longest <= s * range
}

// What a call's kernel makes of it: pairs per block and keys per tile, its blocks, and by
// plan_splits() the most ranges of one and the ratio of the cost rule.
struct SplitPlan {
  int pairs, kt;
  int64_t blocks;
  int n_split;
  float ratio;
};

#ifndef MCAMD_SPLIT_BYTES_PER_US
#define MCAMD_SPLIT_BYTES_PER_US 6.0e6f
#endif

// Partials of one range, in floats.
inline int64_t split_floats(const AttnArgs &a, const SplitPlan &p) {
  return p.blocks * (p.pairs + 31) / 32 * 32 * ((a.head_dim + 31) / 32 * 32 + 2);
}

// room: how many workgroups of the call the chip holds; tile_us: the time of a tile; keys: the most a
// block can have.
inline void plan_splits(const AttnArgs &a, int64_t room, float tile_us, int64_t keys,
                        SplitPlan &p) {
  p.n_split = 1;
  p.ratio = 0.f;
  // Varlen calls have no scratch; two ranges at least must find room.
  if (a.rows || a.cu || p.blocks <= 0 || 2 * p.blocks > room) return;
  p.ratio = tile_us * MCAMD_SPLIT_BYTES_PER_US / (float(split_floats(a, p)) * 8.f);
  const int64_t most = std::min<int64_t>(room / p.blocks, kMaxPrefillSplits);
  p.n_split = best_splits(p.ratio, int((keys + p.kt - 1) / p.kt), p.kt, int(most));
}

inline size_t split_bytes(const AttnArgs &a, const SplitPlan &p) {
  return p.n_split <= 1 ? 0 : size_t(p.n_split) * size_t(split_floats(a, p)) * 4;
}

// Whether the call has the scratch to cut its keys; without it they stay whole.
inline bool cuts_keys(const AttnArgs &a, const SplitPlan &p) {
  return p.n_split > 1 && a.workspace && a.workspace_bytes >= split_bytes(a, p);
}

// The geometry for the kernels.
inline SplitGeo split_geo(const AttnArgs &a, const SplitPlan &p) {
  SplitGeo g;
  g.pairs = p.pairs;
  g.kt = p.kt;
  g.n_split = cuts_keys(a, p) ? p.n_split : 1;
  g.n_bh = int(a.batch * a.n_kv_head);
  g.n_qt = int(p.blocks / g.n_bh);
  g.groups = (p.pairs + 31) / 32;
  g.md = int((a.head_dim + 31) / 32);
  g.G = int(a.n_head / a.n_kv_head);
  g.window = int(a.window < 0 ? -1 : a.window);
  g.ratio = p.ratio;
  g.uncut_keys = 0;
  if (g.n_split > 1) {  // one tile less than would be cut: the device's roots need not be the host's
    int tiles = std::max(1, int(4.f / p.ratio) - 1);  // two ranges from sqrt(tiles * ratio) = 2 on
    while (best_splits(p.ratio, tiles, p.kt, g.n_split) < 2) ++tiles;
    g.uncut_keys = (tiles - 2) * p.kt;
  }
  g.part_o = static_cast<float *>(a.workspace);
  g.part_ml = g.part_o + size_t(g.n_split) * p.blocks * g.groups * g.md * 1024;
  return g;
}

}  // namespace mcamd
