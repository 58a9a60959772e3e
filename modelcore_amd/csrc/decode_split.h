// Keys per split of the general single-token decode (decode_splitk.hip). A pure function of the sizes,
// so that every entry point gives the same sums. Host code of the standard library alone.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mcamd {

constexpr int64_t kDecodeSplitLen = 256;
// Workgroups that remain where splits are made longer than that, and how long they get.
constexpr int64_t kLongSplitBlocks = 8192;
constexpr int64_t kLongestSplit = 2048;
// Workgroups from which rows of up to 512 keys are not cut: there is no merge then (300 rows of 200
// keys in a cache of 512, 8 heads of 64 in bf16: 27 us against 42 with splits of 256).
constexpr int64_t kWholeRowBlocks = 2048;
constexpr int64_t kMostSplits = 65535;  // a grid's blocks along y

// Keys a row can attend, and its splits of `len` keys.
inline int64_t span_of(int64_t t_max, int64_t window) {
  return window >= 0 ? std::min<int64_t>(t_max, window + 1) : t_max;
}
inline int64_t splits_of(int64_t t_max, int64_t window, int64_t len) {
  return (span_of(t_max, window) + len - 1) / len;
}

// kDecodeSplitLen, or less where even a full cache gives few workgroups, down to 32 KB of keys (two
// rows' chunks in flight are 16 KB each) and as far as `fits(splits)` allows their partials. Measured,
// shorter against 256 keys, with the merge: 16 query / 2 KV heads of 128 in fp32, one row of 4000 keys
// 26.4 against 35.8 us; 8 heads of 256 in fp32, one row of 300 keys 10.2 against 16.6; but 12 heads of 64
// in bf16 (32 KB are 256 keys), one row of 2000 keys, 11.0 at 64 keys against 8.5.
//
// Longer only where the grid is so large that its empty workgroups, about 1 ns each, cost more than
// the longer walk: how much of the cache the rows fill is known on the device only, and a row shorter
// than a split is walked by one workgroup per KV head. 8 heads of 64 in bf16, 8 rows of 2000 keys in a
// cache of 65536: 256 keys 16.6 us, 512 13.8 (this rule), 1024 17.6, 2048 33.3. Full caches gain less
// from longer ones than short rows lose: 16 / 4 heads of 64 in bf16, 32 rows of 512-8192 keys in a cache
// of 8218, 256 keys (this rule) 44.7 us, 512 41.0, but 32 rows of 1000 in it 24.3 and 31.3; 8 heads of 256
// in fp32, 8 rows of 2000 in a cache of 16384, 63 and 97.
template <class Fits>
int64_t split_len(int64_t batch, int64_t n_kv_head, int64_t head_dim, int64_t t_max, int64_t window,
                  int64_t elem, const Fits &fits) {
  int64_t len = 64;
  while (len < kDecodeSplitLen && len * head_dim * elem < 32768) len *= 2;
  for (; len < kDecodeSplitLen; len *= 2) {
    const int64_t ns = splits_of(t_max, window, len);
    if (ns <= 64 && batch * n_kv_head * ns <= 1024 && fits(ns)) return len;
  }
  len = kDecodeSplitLen;
  if (span_of(t_max, window) > len && span_of(t_max, window) <= 2 * len &&
      batch * n_kv_head >= kWholeRowBlocks)
    return 2 * len;
  while (len < kLongestSplit &&
         batch * n_kv_head * splits_of(t_max, window, 2 * len) >= kLongSplitBlocks)
    len *= 2;
  while (splits_of(t_max, window, len) > kMostSplits) len *= 2;
  return len;
}

}  // namespace mcamd
