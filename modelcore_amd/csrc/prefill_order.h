// The order in which a chunked prefill's blocks of queries are launched.
//
// Workgroup ids are dealt round-robin over the chip's 8 XCDs and to compute units as they fall free,
// so a launch ends evenly when its longest blocks come first and every XCD gets its share of them.
#pragma once

#include "kernels.h"

namespace mcamd {

// Which of `n` blocks, longest first, workgroup id takes where all of them run at once. Ids go to
// the compute units (`cus` of them) round after round, so in plain order a compute unit with one
// of the longest blocks of a round gets one of the longest of the next too; every other round is
// dealt the other way round instead, in steps of 8 ids, which keeps a (row, KV head) on its XCD where
// n_bh is a multiple of 8. Two prompts of 1000 tokens, 32 / 8 heads of 128 in fp32 (two workgroups a compute
// unit) 232 -> 187 us with the append, four of 2048, 12 heads of 64 in fp32 309 -> 278, in bf16 (three) 75.7 -> 74.
__device__ __forceinline__ int dealt_block(int id, int n, int cus) {
  const int round = id / cus;
  if ((round & 1) == 0) return id;
  const int j = id - round * cus;
  const int eights = min(cus, n - round * cus) / 8;
  return (j >> 3) < eights ? round * cus + (eights - 1 - (j >> 3)) * 8 + (j & 7) : id;
}

// Block i of a varlen launch of up to 64 sequences, lane b of the wave holding in `mine` how many
// blocks sequence b has, at most n_qt: the blocks that exist, by their number qt within their
// sequence, last first (the most keys before the window's edge), a sequence per id within a
// number. Returns false past the last. Sequences of very different lengths so keep every XCD
// busy: with an id per (sequence, qt), existing or not, an XCD's share was that of a few sequences
// (eight prompts of 37 to 4001 tokens, window 1024: 222 us; this way 135, of which the append
// is 14).
__device__ __forceinline__ bool varlen_block(int i, int mine, int n_qt, int &b, int &qt) {
  // Blocks numbered k or more: the largest k with more than i of them is block i's number.
  int lo = -1, hi = n_qt;  // more than i blocks from `lo` on (if lo >= 0), at most i from `hi` on
  while (hi - lo > 1) {
    const int k = (lo + hi) >> 1;
    if (wave_total(max(mine - k, 0)) > i)
      lo = k;
    else
      hi = k;
  }
  if (lo < 0) return false;
  qt = lo;
  int nth = i - wave_total(max(mine - lo - 1, 0));  // among the sequences that have a block lo
  uint64_t has = __builtin_amdgcn_ballot_w64(mine > lo);
  for (; nth > 0; --nth) has &= has - 1;
  b = __builtin_ctzll(has);
  return true;
}

// Sequences of a varlen launch for which varlen_block() is used.
constexpr int kOrderedSeqs = 64;

// A block of a varlen launch: sequence b's block qt, its tokens [tok0, tok0 + T_b), its cache row and
// that row's position.
struct VarlenBlock {
  int b, qt, row, T_b, s0;
  int64_t tok0;
};

// Block i of a launch of n_seqs sequences of up to n_qt blocks of `pairs` (position, head) pairs
// (G heads). Returns false past the last. Each lane reads one sequence's lengths, row and position
// up front, in two rounds of loads that the search runs beside.
__device__ __forceinline__ bool find_varlen_block(const int32_t *cu, const int32_t *rows,
                                                  const int32_t *seqlens, int n_seqs, int n_qt,
                                                  int pairs, int G, int i, int lane,
                                                  VarlenBlock &v) {
  const int l = min(lane, n_seqs - 1);
  const int c0 = cu[l], c1 = cu[l + 1];
  const int row = rows ? rows[l] : l;
  const int pos = seqlens[row];
  const int64_t n = lane < n_seqs ? int64_t(c1 - c0) * G : 0;
  const int mine = int(min((n + pairs - 1) / pairs, int64_t(n_qt)));
  if (!varlen_block(i, mine, n_qt, v.b, v.qt)) return false;
  v.row = __builtin_amdgcn_readlane(row, v.b);
  v.T_b = __builtin_amdgcn_readlane(c1 - c0, v.b);
  v.s0 = __builtin_amdgcn_readlane(pos, v.b);
  v.tok0 = __builtin_amdgcn_readlane(c0, v.b);
  return true;
}

}  // namespace mcamd
