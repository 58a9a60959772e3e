// Next-token sampling on the device with a counter-based RNG per row.
//
// Row b draws token argmax_i (logits[b, i] / T + g_i), where g_i = -log(-log(u_i)) is standard
// Gumbel noise and u_i is uniform in (0, 1): the Gumbel-max form of sampling from
// softmax(logits[b] / T), the distribution modelcore/generate.py:18-34 draws from with
// torch.multinomial. T == 0 takes the plain argmax (greedy), as the reference does. Ties go to
// the lowest index, as torch.argmax does.
//
// The uniforms come from Philox4x32-10 (Salmon, Moraes, Dror and Shaw, "Parallel random numbers:
// as easy as 1, 2, 3", SC 2011): key = the row's 64-bit seed, counter = (i / 4, row offset,
// 0, 0), word i % 4; u = ((x >> 9) + 1/2) / 2^23, an exact float32 in (0, 1). Each call
// consumes one offset per row and advances offsets[b] by one on the device, so a row's draws
// depend only on its seed and on how many tokens it has drawn -- never on the batch it sits in
// -- and no host sync is needed.
//
// One workgroup per row; each lane scans a strided part of the vocabulary, then a wave64
// reduction and an LDS reduction over the waves pick the (score, index) maximum. The result does
// not depend on the workgroup size: a token's noise is keyed by its own index.
//
// top_k (0 < k < vocab) restricts the draw to the k largest logits, ties at the k-th value going
// to the lowest indices -- the set torch.topk returns for distinct values -- and the Gumbel-max
// over that set is a draw from softmax(top-k logits / T), the distribution of the reference's
// top_k branch. The k-th largest value is found without sorting: logits map to 32-bit keys in
// the same order (NaN lowest). The keys are dealt to 1024 parts (4096 for k > 256) and each part's
// maximum taken: about the k-th largest of the maxima has k keys at or above it, so the k largest are
// among the keys that reach it, about k of them while k is small against the parts (k = 50: ~60 of
// 32768; k = 1000: ~1200). Those go to LDS; up to 384 of them are ranked against each other,
// more are counted by one wave in a binary search over the key bits, without barriers. Noise is
// made for the kept ones only. A row whose candidates do not fit (larger k, many equal logits) is
// searched as a whole. Bound by latency (a row is one workgroup's 128 KiB): 64 rows of 32768 at
// k = 50 take 10.7 us, at k = 1000 33; counting the whole row for every bit, with a
// barrier each, and noise for every token took 76 and 86 (2366 where 131072 logits had to be read
// again for every count).
#include "kernels.h"

#include <cmath>
#include <type_traits>

namespace mcamd {
namespace {

// The plain draw: sixteen waves per row, so that the Philox rounds and logarithms of a row (its
// cost; one row per CU) run on every SIMD with four waves each to interleave (measured on the
// 64-row, 32768-token sampling step: 31.5 -> 18.1 us per draw against four waves).
constexpr int kDrawThreads = 1024;

struct Philox {
  uint32_t c0, c1, c2, c3;
};

// Philox4x32 with 10 rounds on counter (c0..c3) and key (k0, k1).
__device__ __forceinline__ Philox philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                uint32_t k0, uint32_t k1) {
  constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;  // round multipliers
  constexpr uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;  // key schedule increments
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t hi0 = __umulhi(M0, c0), lo0 = M0 * c0;
    const uint32_t hi1 = __umulhi(M1, c2), lo1 = M1 * c2;
    const uint32_t n0 = hi1 ^ c1 ^ k0, n1 = lo1, n2 = hi0 ^ c3 ^ k1, n3 = lo0;
    c0 = n0;
    c1 = n1;
    c2 = n2;
    c3 = n3;
    k0 += W0;
    k1 += W1;
  }
  return {c0, c1, c2, c3};
}

// (k + 1/2) / 2^23 for the top 23 bits k of x: exactly representable, strictly inside (0, 1).
__device__ __forceinline__ float uniform23(uint32_t x) {
  return (float(x >> 9) + 0.5f) * (1.0f / 8388608.0f);
}

__device__ __forceinline__ bool better(float s, int i, float bs, int bi) {
  return s > bs || (s == bs && i < bi);
}

// A 32-bit key in the order of the float (NaN below everything, -inf next; -0 equal to +0).
__device__ __forceinline__ uint32_t order_key(float f) {
  if (f != f) return 0u;
  uint32_t u = __float_as_uint(f);
  if (u == 0x80000000u) u = 0u;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The float of an order key above that of -inf.
__device__ __forceinline__ float order_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

// Sum of one int per thread over the workgroup; `slot` alternates between calls so that one
// barrier per call suffices.
__device__ __forceinline__ int block_sum(int v, int (*s_cnt)[kDrawThreads / 64], int &slot) {
  v = wave_total(v);
  if ((threadIdx.x & 63) == 0) s_cnt[slot][threadIdx.x >> 6] = v;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int w = 0; w < kDrawThreads / 64; ++w) t += s_cnt[slot][w];
  slot ^= 1;
  return t;
}

// Four logits at any float's address.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Groups of four logits a thread loads at once; a row of that many per thread (vocab <= 32768)
// stays in registers.
constexpr int kRegGroups = 8;
// Candidates of a top_k draw held in LDS, and those ranked against each other.
constexpr int kCandidates = 4096;
constexpr int kRanked = 384;
constexpr int kManyParts = 256;  // top_k past which the keys are dealt to four parts per thread

// (score, index) maximum over the workgroup's threads, in thread 0.
__device__ __forceinline__ void block_best(float &best, int &best_i, float *s_score, int *s_index) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float os = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(best_i, o, 64);
    if (better(os, oi, best, best_i)) {
      best = os;
      best_i = oi;
    }
  }
  if ((tid & 63) == 0) {
    s_score[tid >> 6] = best;
    s_index[tid >> 6] = best_i;
  }
  __syncthreads();
  if (tid == 0)
    for (int w = 1; w < kDrawThreads / 64; ++w)
      if (better(s_score[w], s_index[w], best, best_i)) {
        best = s_score[w];
        best_i = s_index[w];
      }
}

__global__ __launch_bounds__(kDrawThreads) void sample_kernel(const float *__restrict__ logits,
                                                          int64_t row_stride, int vocab,
                                                          float inv_temp, int greedy,
                                                          const uint64_t *__restrict__ seeds,
                                                          int64_t *__restrict__ offsets,
                                                          int64_t *__restrict__ out) {
  __shared__ float s_score[kDrawThreads / 64];
  __shared__ int s_index[kDrawThreads / 64];
  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  const float *row = logits + int64_t(b) * row_stride;
  const uint64_t seed = seeds[b];
  const uint64_t off = uint64_t(offsets[b]);
  const uint32_t k0 = uint32_t(seed), k1 = uint32_t(seed >> 32);
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  // Thread tid handles groups of four consecutive tokens 4 g .. 4 g + 3, g = tid, tid + 1024, ...
  for (int g = tid; 4 * g < vocab; g += kDrawThreads) {
    Philox r{0, 0, 0, 0};
    if (!greedy) r = philox4x32_10(uint32_t(g), uint32_t(off), uint32_t(off >> 32), 0u, k0, k1);
    const uint32_t w[4] = {r.c0, r.c1, r.c2, r.c3};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = 4 * g + j;
      if (i >= vocab) break;
      float s = row[i];
      if (!greedy) s = s * inv_temp - logf(-logf(uniform23(w[j])));
      if (s != s) s = -INFINITY;  // a NaN logit never wins
      if (better(s, i, best, best_i)) {
        best = s;
        best_i = i;
      }
    }
  }
  block_best(best, best_i, s_score, s_index);
  if (tid == 0) {
    out[b] = best_i == 0x7fffffff ? 0 : best_i;
    offsets[b] = int64_t(off + 1);
  }
}

// The k-th largest of a set of keys and the kept ones among its equals: a key is kept when it is
// above K, or K at an index up to last_tie.
struct TopK {
  uint32_t K;
  int last_tie;
};

// `ge(c)` counts the set's keys >= c, `eq_below(c, i)` those equal to c at an index below i, each
// the same in every thread that calls; at least top_k of the set's keys are >= lo.
template <class Ge, class EqBelow>
__device__ __forceinline__ TopK find_top_k(int top_k, uint32_t lo, uint32_t hi, const Ge &ge,
                                           const EqBelow &eq_below) {
  // K is the largest key with top_k of the set's keys >= it: lo has them, hi + 1 has not.
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2 + 1;
    if (ge(mid) >= top_k)
      lo = mid;
    else
      hi = mid - 1;
  }
  TopK r{lo, 0x7fffffff};
  const int above = lo == 0xffffffffu ? 0 : ge(lo + 1);
  const int ties = eq_below(lo, 0x7fffffff);
  const int need = top_k - above;  // 1 <= need <= ties
  if (need < ties) {  // the largest index with fewer than `need` ties below it is the last kept
    int last = 0;
    for (int bit = 30; bit >= 0; --bit) {
      const int cand = last | (1 << bit);
      if (eq_below(lo, cand) < need) last = cand;
    }
    r.last_tie = last;
  }
  return r;
}

// The draw restricted to the top_k largest logits of the row (see the top of the file). REG: the
// row is held in registers (vocab <= 4 * kDrawThreads * kRegGroups), else read again for every use.
template <bool REG>
__global__ __launch_bounds__(kDrawThreads) void sample_topk_kernel(
    const float *__restrict__ logits, int64_t row_stride, int vocab, int top_k, float inv_temp,
    const uint64_t *__restrict__ seeds, int64_t *__restrict__ offsets, int64_t *__restrict__ out) {
  // The parts' maxima (keys), then the candidates: key, and the complement of the token below it, so
  // that the larger of two is the one kept first.
  __shared__ uint64_t s_cand[kCandidates];
  uint32_t *const s_max = reinterpret_cast<uint32_t *>(s_cand);
  __shared__ int s_cnt[2][kDrawThreads / 64];
  __shared__ float s_score[kDrawThreads / 64];
  __shared__ int s_index[kDrawThreads / 64];
  __shared__ int s_n;
  __shared__ TopK s_top;
  __shared__ uint32_t s_bound;
  const int b = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float *row = logits + int64_t(b) * row_stride;
  const int n_groups = (vocab + 3) / 4;
  // kRegGroups groups from g0 + tid on, kDrawThreads apart: group g holds tokens 4 g .. 4 g + 3
  // (NaN past the vocabulary).
  auto load_groups = [&](int g0, f32x4u (&v)[kRegGroups]) __attribute__((always_inline)) {
    const int last = vocab - 4;
    if (vocab < 4) {  // no whole group: thread 0 has them all
#pragma unroll
      for (int m = 0; m < kRegGroups; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[m][j] = m == 0 && tid == 0 && j < vocab ? row[j] : NAN;
      return;
    }
    // The loads first and without a branch between them, so that they are in flight together:
    // groups past the last whole one read the row's last four logits and pick theirs below.
#pragma unroll
    for (int m = 0; m < kRegGroups; ++m)
      v[m] = *reinterpret_cast<const f32x4u *>(row + min(4 * (g0 + tid + m * kDrawThreads), last));
#pragma unroll
    for (int m = 0; m < kRegGroups; ++m) {
      const int past = 4 * (g0 + tid + m * kDrawThreads) - last;  // of the first token loaded
      if (past > 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[m][j] = past + j == 1 ? v[m][1] : past + j == 2 ? v[m][2] : past + j == 3 ? v[m][3] : NAN;
      }
    }
  };
  f32x4u val[kRegGroups];
  if constexpr (REG) load_groups(0, val);
  // f(logit, token, part) for every logit of this thread; they fall into four parts. NaN stands in
  // for tokens past the vocabulary.
  auto each = [&](auto f) __attribute__((always_inline)) {
    for (int g0 = 0; g0 < n_groups; g0 += kRegGroups * kDrawThreads) {
      if constexpr (!REG) load_groups(g0, val);
#pragma unroll
      for (int m = 0; m < kRegGroups; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) f(val[m][j], 4 * (g0 + tid + m * kDrawThreads) + j, m & 3);
      if constexpr (REG) break;
    }
  };

  // The same for the rare whole-row searches: small code where the row is not in registers.
  auto each_again = [&](auto f) __attribute__((always_inline)) {
    if constexpr (REG) {
      each(f);
    } else {
#pragma unroll 4
      for (int i = tid; i < vocab; i += kDrawThreads) f(row[i], i, 0);
    }
  };

  // The bound: a key that at least k parts' maxima reach, not many more; and the largest key. The
  // maxima are taken as floats (a part of NaNs alone has -inf).
  float most[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  each([&](float v, int, int part) { most[part] = fmaxf(most[part], v); });
  const bool many = top_k > kManyParts;
  if (many) {
#pragma unroll
    for (int u = 0; u < 4; ++u) s_max[u * kDrawThreads + tid] = order_key(most[u]);
  } else {
    s_max[tid] = order_key(fmaxf(fmaxf(most[0], most[1]), fmaxf(most[2], most[3])));
  }
  if (tid == 0) s_n = 0;
  __syncthreads();
  if (wave == 0) {
    auto search = [&](auto n_c) {
      constexpr int N = decltype(n_c)::value;
      uint32_t mx[N];
      uint32_t top = 0;
#pragma unroll
      for (int u = 0; u < N; ++u) {
        mx[u] = s_max[64 * u + lane];
        top = max(top, mx[u]);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) top = max(top, uint32_t(__shfl_xor(int(top), o, 64)));
      uint32_t lo = 0, hi = top_k <= 64 * N ? top : 0;
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2 + 1;
        int n = 0;
#pragma unroll
        for (int u = 0; u < N; ++u) n += mx[u] >= mid ? 1 : 0;
        n = wave_total(n);
        if (n >= top_k)
          lo = mid;
        else
          hi = mid - 1;
        if (n >= top_k && n <= top_k + (top_k >> 3) + 8) break;  // close enough
      }
      if (lane == 0) {
        s_bound = lo > order_key(-INFINITY) ? lo : 0u;  // -inf may stand for no logit at all
        s_top.K = top;
      }
    };
    if (many)
      search(std::integral_constant<int, kCandidates / 64>{});
    else
      search(std::integral_constant<int, kDrawThreads / 64>{});
  }
  __syncthreads();
  const uint32_t bound = s_bound, top = s_top.K;

  // The candidates, in LDS while they fit (their order does not matter).
  auto take = [&](uint32_t k, int i) __attribute__((always_inline)) {
    const int at = atomicAdd(&s_n, 1);
    if (at < kCandidates) s_cand[at] = uint64_t(k) << 32 | uint32_t(~i);
  };
  if (bound == 0) {
    each_again([&](float v, int i, int) {
      if (i < vocab) take(order_key(v), i);
    });
  } else {
    const float least = order_value(bound);
    each([&](float v, int i, int) {
      if (v >= least) take(order_key(v), i);
    });
  }
  __syncthreads();
  const int n_cand = s_n;
  const bool listed = n_cand <= kCandidates;
  TopK r{0u, 0x7fffffff};
  bool mine = true;  // of candidate tid, where they are ranked
  if (n_cand <= kRanked) {
    if (tid < n_cand) {
      const uint64_t own = s_cand[tid];
      int rank = 0;
#pragma unroll 16
      for (int c = 0; c < n_cand; ++c) rank += s_cand[c] > own ? 1 : 0;
      mine = rank < top_k;
    }
  } else if (listed) {
    if (wave == 0) {
      constexpr int N = kCandidates / 64;
      uint32_t k[N];
#pragma unroll
      for (int u = 0; u < N; ++u)
        k[u] = 64 * u + lane < n_cand ? uint32_t(s_cand[64 * u + lane] >> 32) : 0u;
      const TopK t = find_top_k(
          top_k, bound, top,
          [&](uint32_t c) {  // c > bound >= 0: the places without a candidate do not count
            int n = 0;
#pragma unroll
            for (int u = 0; u < N; ++u) n += k[u] >= c ? 1 : 0;
            return wave_total(n);
          },
          [&](uint32_t c, int below) {
            int n = 0;
            for (int u = lane; u < n_cand; u += 64) {
              const uint64_t x = s_cand[u];
              n += uint32_t(x >> 32) == c && int(~uint32_t(x)) < below ? 1 : 0;
            }
            return wave_total(n);
          });
      if (lane == 0) s_top = t;
    }
    __syncthreads();
    r = s_top;
  } else {
    int slot = 0;
    auto count = [&](auto which) {
      int n = 0;
      each_again([&](float v, int i, int) { n += i < vocab && which(order_key(v), i) ? 1 : 0; });
      return block_sum(n, s_cnt, slot);
    };
    r = find_top_k(
        top_k, bound, top,
        [&](uint32_t c) { return count([&](uint32_t k, int) { return k >= c; }); },
        [&](uint32_t c, int below) {
          return count([&](uint32_t k, int i) { return k == c && i < below; });
        });
  }

  const uint64_t seed = seeds[b];
  const uint64_t off = uint64_t(offsets[b]);
  const uint32_t k0 = uint32_t(seed), k1 = uint32_t(seed >> 32);
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  // Gumbel-max over the kept logits: token i takes word i % 4 of group i / 4's Philox counter.
  auto draw = [&](uint32_t k, int i) __attribute__((always_inline)) {
    if (!(k > r.K || (k == r.K && i <= r.last_tie))) return;
    const Philox p = philox4x32_10(uint32_t(i >> 2), uint32_t(off), uint32_t(off >> 32), 0u, k0, k1);
    const uint32_t w = (i & 3) == 0 ? p.c0 : (i & 3) == 1 ? p.c1 : (i & 3) == 2 ? p.c2 : p.c3;
    float sc = row[i] * inv_temp - logf(-logf(uniform23(w)));
    if (sc != sc) sc = -INFINITY;
    if (better(sc, i, best, best_i)) {
      best = sc;
      best_i = i;
    }
  };
  if (listed) {
    for (int c = tid; c < n_cand; c += kDrawThreads)
      if (mine) draw(uint32_t(s_cand[c] >> 32), int(~uint32_t(s_cand[c])));
  } else {
    each_again([&](float v, int i, int) {
      if (i < vocab) draw(order_key(v), i);
    });
  }
  block_best(best, best_i, s_score, s_index);
  if (tid == 0) {
    out[b] = best_i == 0x7fffffff ? 0 : best_i;
    offsets[b] = int64_t(off + 1);
  }
}

}  // namespace
}  // namespace mcamd

using namespace mcamd;

extern "C" int mcamd_sample_tokens(const float *logits, int64_t batch, int64_t vocab,
                                   int64_t row_stride, float temperature, int64_t top_k,
                                   const uint64_t *seeds, int64_t *offsets, int64_t *out,
                                   void *stream) {
  if (batch < 0 || vocab <= 0 || vocab > (int64_t(1) << 30) || (row_stride != 0 && row_stride < vocab))
    return fail(MCAMD_EINVAL,
                "sample_tokens: need batch >= 0, 0 < vocab <= 2^30, row_stride 0 or >= vocab");
  if (!(temperature >= 0.f) || std::isinf(temperature))
    return fail(MCAMD_EINVAL, "sample_tokens: temperature must be finite and non-negative");
  if (batch > 0 && (!logits || !seeds || !offsets || !out))
    return fail(MCAMD_EINVAL, "sample_tokens: null pointer");
  if (batch > 0x7fffffff) return fail(MCAMD_EUNSUPPORTED, "sample_tokens: batch too large");
  if (batch == 0) {
    clear_error();
    return MCAMD_OK;
  }
  const int greedy = temperature == 0.f ? 1 : 0;
  const float inv_temp = greedy ? 1.f : 1.f / temperature;
  if (!greedy && top_k > 0 && top_k < vocab) {
    if (vocab <= int64_t(4) * kDrawThreads * kRegGroups)
      hipLaunchKernelGGL(sample_topk_kernel<true>, dim3(unsigned(batch)), dim3(kDrawThreads), 0,
                         as_stream(stream), logits, row_stride, int(vocab), int(top_k), inv_temp,
                         seeds, offsets, out);
    else
      hipLaunchKernelGGL(sample_topk_kernel<false>, dim3(unsigned(batch)), dim3(kDrawThreads), 0,
                         as_stream(stream), logits, row_stride, int(vocab), int(top_k), inv_temp,
                         seeds, offsets, out);
    return launch_status("sample_tokens (top_k)");
  }
  hipLaunchKernelGGL(sample_kernel, dim3(unsigned(batch)), dim3(kDrawThreads), 0, as_stream(stream),
                     logits, row_stride, int(vocab), inv_temp, greedy, seeds, offsets, out);
  return launch_status("sample_tokens");
}
