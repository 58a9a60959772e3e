// Single-token decode attention over the KV cache, as split-K flash-decoding.
//
// Semantics: modelcore/kernels/flash_attn.py:348-366 with T_new == 1. The query of row b sits at
// p = cache_seqlens[b] and attends keys [lo, p], lo = max(0, p - window) (window < 0: lo = 0),
// which is both the sliced uniform path (:217-224) and the ragged mask (:246-264). Query head h
// reads KV head h / G, G = H / H_kv (SDPA enable_gqa). Scale 1/sqrt(D).
//
// Work split. The key range of a row is cut into splits, aligned to lo. One workgroup owns (row b,
// KV head, split) and serves every query head of that KV head's GQA group (up to GM at a time), so
// each K/V byte of the split is read from HBM once. The grid is sized from T_max (no host sync on
// cache_seqlens); splits past a row's length exit at once. The length of a split: decode_split.h.
//
// Inside a workgroup (256 threads): LPT = DP / VEC lanes cover one key's D elements with one
// 16-byte load each, so a wave reads 64/LPT whole head rows per instruction, and each group of LPT
// lanes keeps a softmax of its own (running maximum, sum and weighted sum over its keys, exp2
// domain) in registers: a score is complete in every lane of the group after log2(LPT) DPP adds, and
// its weight goes straight to the value row. Keys go by in chunks of U per group, K and V of the next
// chunk in flight while one is used. The groups merge once, at the end of the split: over the wave in
// registers, over the four waves through LDS. A row of one split writes its output there; otherwise
// the split's (m, l, o[D]) go to the workspace and the combine kernel merges the splits of a
// (row, head) by log-sum-exp.
//
// Append: the split that ends at the row's position takes the new token from k/v instead of the
// cache and writes it there (bit-exact), the workgroup of the KV head's first query heads.
//
// Measured (one call with its append): 16 rows of 128-2047 keys, 12 heads of 64 in bf16 (53.6 MB)
// 16.7 us (3.2 TB/s; 24.4 before); two rows of 80 keys, 12 heads of 64 in fp32 4.3 (10.5); 32 rows of
// 256-4096 keys, 16 / 4 heads of 128 in fp32 (286 MB) 62 (92). Before, each split read K, stored its
// scores in LDS, took the softmax there and read V after it, with the append and the merge as
// launches of their own.
#include "decode_split.h"
#include "kernels.h"

#include <cmath>

namespace mcamd {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

struct DecodeParams {
  const void *q, *k_new, *v_new;
  void *k_cache, *v_cache;
  const int32_t *seqlens;
  void *out;
  float *part_o;   // [B][H][n_splits][D]
  float *part_ml;  // [B][H][n_splits][2]
  int H, H_kv, G, n_hchunks, T_max, window, n_splits, D, SL;
  int64_t cache_b;
  float scale_log2;
};

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
// x of the lane 16 (32) away added to, or compared with, this lane's.
template <class Op>
__device__ __forceinline__ float across16(float x, const Op &op) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <class Op>
__device__ __forceinline__ float across32(float x, const Op &op) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Sum over a group of LPT neighbouring lanes, in each of them: within quads, then mirrored halves
// of a row of 16 lanes, then rows.
template <int LPT>
__device__ __forceinline__ float group_sum(float x) {
  const auto add = [](float a, float b) { return a + b; };
  if constexpr (LPT >= 2) x += dpp<0xB1>(x);   // quad_perm [1,0,3,2]
  if constexpr (LPT >= 4) x += dpp<0x4E>(x);   // quad_perm [2,3,0,1]
  if constexpr (LPT >= 8) x += dpp<0x141>(x);  // row_half_mirror
  if constexpr (LPT >= 16) x += dpp<0x140>(x); // row_mirror
  if constexpr (LPT >= 32) x = across16(x, add);
  if constexpr (LPT >= 64) x = across32(x, add);
  return x;
}
// op over the lanes LPT apart (the same dims of the wave's 64 / LPT key groups), in each of them.
template <int LPT, class Op>
__device__ __forceinline__ float over_groups(float x, const Op &op) {
  if constexpr (LPT <= 2) x = op(x, dpp<0x122>(x));  // row_ror:2
  if constexpr (LPT <= 4) x = op(x, dpp<0x124>(x));  // row_ror:4
  if constexpr (LPT <= 8) x = op(x, dpp<0x128>(x));  // row_ror:8
  if constexpr (LPT <= 16) x = across16(x, op);
  if constexpr (LPT <= 32) x = across32(x, op);
  return x;
}

// DP is head_dim rounded up to a power of two (at least 16): LPT = DP / VEC lanes cover one key
// row, and lanes past the real head_dim D hold nothing (they load no data and add zeros).
// PAIRED: the order of the splits and heads in the grid (run_decode()).
template <class E, int DP, int GM, bool PAIRED>
__global__ __launch_bounds__(kThreads) void decode_split_kernel(DecodeParams P) {
  constexpr int VEC = Vec<E>::N;
  constexpr int LPT = DP / VEC;        // lanes per key row
  constexpr int TPI = kThreads / LPT;  // keys per pass of the workgroup
  constexpr int U = GM <= 4 ? 4 : 2;   // keys per group and chunk
  static_assert(LPT >= 2 && LPT <= 64 && (64 % LPT) == 0, "head_dim too large for one wave");
  const int D = P.D;

  __shared__ float s_ml[kWaves][GM][2];
  __shared__ float s_o[kWaves][GM][DP];

  const int b = blockIdx.z;
  const int head = PAIRED ? blockIdx.x >> 1 : blockIdx.x;
  // Paired: a split past the last one starts past the row's end.
  const int split = PAIRED ? 2 * blockIdx.y + ((blockIdx.x + head + b) & 1) : blockIdx.y;
  const int kvh = head / P.n_hchunks;
  const int hc = head - kvh * P.n_hchunks;
  const int h0 = kvh * P.G + hc * GM;
  const int gcount = min(GM, P.G - hc * GM);
  const int tid = threadIdx.x;
  E *out = static_cast<E *>(P.out) + (int64_t(b) * P.H + h0) * D;

  const int pos = P.seqlens[b];
  if (pos < 0 || pos >= P.T_max) {
    if (split == 0)
      for (int i = tid; i < gcount * D; i += kThreads) out[i] = from_f32<E>(NAN);
    return;
  }
  const int lo = key_lo(pos, P.window);
  const int t0 = lo + split * P.SL;
  if (t0 > pos) return;
  const int n = min(P.SL, pos - t0 + 1);

  const int li = tid % LPT;
  const int tg = tid / LPT;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const bool live = li * VEC < D;  // this lane holds dims of the head

  const E *q = static_cast<const E *>(P.q);
  E *kc = static_cast<E *>(P.k_cache);
  E *vc = static_cast<E *>(P.v_cache);
  const int64_t row_base = int64_t(b) * P.cache_b + int64_t(kvh) * D + li * VEC;
  const int64_t tok_stride = int64_t(P.H_kv) * D;
  const int64_t new_off = (int64_t(b) * P.H_kv + kvh) * D + li * VEC;
  const E *kn = P.k_new ? static_cast<const E *>(P.k_new) + new_off : nullptr;
  const E *vn = P.k_new ? static_cast<const E *>(P.v_new) + new_off : nullptr;

  // Keys r0 + u TPI (u < U) of the split, r0 = chunk * U * TPI + tg; those past its end re-read its
  // last one (their weight is zero, and their values are zeroed before use).
  struct Chunk {
    uint4 k[U], v[U];
  };
  auto load_chunk = [&](Chunk &c, int r0) {
#pragma unroll
    for (int u = 0; u < U; ++u) c.k[u] = c.v[u] = make_uint4(0, 0, 0, 0);
    if (live) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = t0 + min(r0 + u * TPI, n - 1);
        const bool is_new = t == pos && kn != nullptr;
        const int64_t at = row_base + int64_t(t) * tok_stride;
        c.k[u] = load_stream(is_new ? kn : kc + at);  // K/V are read once per pass
        c.v[u] = load_stream(is_new ? vn : vc + at);
      }
    }
  };

  Chunk cur;
  load_chunk(cur, tg);

  float qv[GM][VEC];
#pragma unroll
  for (int g = 0; g < GM; ++g) {
    if (g < gcount && live) {
      float x[VEC];
      Vec<E>::load(q + (int64_t(b) * P.H + h0 + g) * D + li * VEC, x);
#pragma unroll
      for (int e = 0; e < VEC; ++e) qv[g][e] = x[e] * P.scale_log2;
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) qv[g][e] = 0.f;
    }
  }

  float m[GM], l[GM], o[GM][VEC];
#pragma unroll
  for (int g = 0; g < GM; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < VEC; ++e) o[g][e] = 0.f;
  }

  for (int c0 = 0; c0 < n; c0 += U * TPI) {
    Chunk next;
    if (c0 + U * TPI < n) load_chunk(next, c0 + U * TPI + tg);
    float s[U][GM];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float kx[VEC];
      Vec<E>::unpack(cur.k[u], kx);
#pragma unroll
      for (int g = 0; g < GM; ++g) {
        float a = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) a = fmaf(qv[g][e], kx[e], a);
        s[u][g] = group_sum<LPT>(a);
      }
    }
    if (c0 + U * TPI > n) {  // the split's end: some keys are not there
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c0 + tg + u * TPI >= n) {
          cur.v[u] = make_uint4(0, 0, 0, 0);
#pragma unroll
          for (int g = 0; g < GM; ++g) s[u][g] = -INFINITY;
        }
    }
#pragma unroll
    for (int g = 0; g < GM; ++g) {
      float mx = m[g];
#pragma unroll
      for (int u = 0; u < U; ++u) mx = fmaxf(mx, s[u][g]);
      const float ref = mx == -INFINITY ? 0.f : mx;  // no key yet: weights of zero
      const float alpha = fast_exp2(m[g] - ref);
      m[g] = mx;
      l[g] *= alpha;
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[g][e] *= alpha;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        s[u][g] = fast_exp2(s[u][g] - ref);
        l[g] += s[u][g];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float vx[VEC];
      Vec<E>::unpack(cur.v[u], vx);
#pragma unroll
      for (int g = 0; g < GM; ++g)
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[g][e] = fmaf(s[u][g], vx[e], o[g][e]);
    }
    cur = next;
  }

  // The new token into the cache, from the split that ends with it.
  if (kn != nullptr && hc == 0 && t0 + n - 1 == pos && tg == 0 && live) {
    const int64_t at = row_base + int64_t(pos) * tok_stride;
    *reinterpret_cast<uint4 *>(kc + at) = *reinterpret_cast<const uint4 *>(kn);
    *reinterpret_cast<uint4 *>(vc + at) = *reinterpret_cast<const uint4 *>(vn);
  }

  // Merge the wave's key groups, then the waves.
  const auto add = [](float a, float b) { return a + b; };
#pragma unroll
  for (int g = 0; g < GM; ++g) {
    const float M = over_groups<LPT>(m[g], [](float a, float b) { return fmaxf(a, b); });
    // A group with no key has l = 0; a NaN l (a NaN score) must stay.
    const float a = m[g] == -INFINITY ? 0.f : fast_exp2(m[g] - M);
    const float L = over_groups<LPT>(m[g] == -INFINITY ? l[g] : l[g] * a, add);
#pragma unroll
    for (int e = 0; e < VEC; ++e) o[g][e] = over_groups<LPT>(o[g][e] * a, add);
    if (lane < LPT) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) s_o[wave][g][li * VEC + e] = o[g][e];
      if (lane == 0) {
        s_ml[wave][g][0] = M;
        s_ml[wave][g][1] = L;
      }
    }
  }
  __syncthreads();

  const bool whole = pos - lo < P.SL;  // the row's only split
  const int64_t base = (int64_t(b) * P.H + h0) * P.n_splits + split;
  for (int i = tid; i < gcount * D; i += kThreads) {
    const int g = i / D;
    const int d = i - g * D;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, s_ml[w][g][0]);
    float L = 0.f, x = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float mw = s_ml[w][g][0];
      const float a = mw == -INFINITY ? 0.f : fast_exp2(mw - M);
      L += s_ml[w][g][1] * (mw == -INFINITY ? 1.f : a);
      x = fmaf(s_o[w][g][d], a, x);
    }
    if (whole) {
      out[i] = from_f32<E>(x / L);
    } else {
      P.part_o[(base + int64_t(g) * P.n_splits) * D + d] = x;
      if (d == 0) {
        P.part_ml[(base + int64_t(g) * P.n_splits) * 2 + 0] = M;
        P.part_ml[(base + int64_t(g) * P.n_splits) * 2 + 1] = L;
      }
    }
  }
}

// Merge of the splits of one (row, head): out = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M). Four
// waves take every fourth split each; rows of one split are written already.
template <class E>
__global__ __launch_bounds__(kThreads) void decode_combine_kernel(DecodeParams P) {
  __shared__ float s_x[kWaves][256 + 1];
  const int h = blockIdx.x;
  const int b = blockIdx.y;
  const int D = P.D;
  const int pos = P.seqlens[b];
  if (pos < 0 || pos >= P.T_max) return;  // NaN, written already
  const int lo = key_lo(pos, P.window);
  const int ns = (pos - lo) / P.SL + 1;
  if (ns == 1) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t base = (int64_t(b) * P.H + h) * P.n_splits;
  const float *ml = P.part_ml + base * 2;
  const float *po = P.part_o + base * D;
  // Every wave takes the maximum over all splits, a split per lane.
  float M = -INFINITY;
  for (int s = lane; s < ns; s += 64) M = fmaxf(M, ml[2 * s]);
  M = wave_max<64>(M);
  float L = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = wave; s < ns; s += kWaves) {
    const float a = fast_exp2(ml[2 * s] - M);
    L = fmaf(ml[2 * s + 1], a, L);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (lane + 64 * i < D) acc[i] = fmaf(po[int64_t(s) * D + lane + 64 * i], a, acc[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) s_x[wave][lane + 64 * i] = acc[i];
  if (lane == 0) s_x[wave][256] = L;
  __syncthreads();
  const int d = threadIdx.x;
  if (d >= D) return;
  float x = 0.f;
  L = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    x += s_x[w][d];
    L += s_x[w][256];
  }
  static_cast<E *>(P.out)[(int64_t(b) * P.H + h) * D + d] = from_f32<E>(x / L);
}

template <class E, int DP, int GM>
int run_decode(const DecodeParams &P, int B, hipStream_t stream) {
  // The KV heads of a split are neighbours: together they read whole token rows (16 rows of 12
  // heads of 64 in bf16: 18.8 us with the splits of a head side by side, 16.7 so). Paired: two splits
  // of a head side by side, then the next head's, the first of the two in turn.
  //
  // Rows of 512 bytes or 1 KB of a head, where the workgroups fill the chip several times over, are
  // paired: with a head beside a head, 16 rows of 8000 keys, 8 heads of 256, run at 5.6 TB/s in fp32 (375
  // us; paired 330) and 5.7 in bf16 (183; 174). Smaller calls don't gain (3 rows of 11000 keys of it in
  // bf16 58.2 us, paired 61.0), nor other rows (16 rows of 8000 keys, 8 heads of 192 in fp32, 240 and 251).
  const unsigned heads = P.H_kv * P.n_hchunks, splits = P.n_splits;
  constexpr bool kWide = DP * sizeof(E) >= 512;
  if (kWide && P.D * sizeof(E) % 512 == 0 && int64_t(B) * P.H_kv * P.n_splits >= 2048)
    hipLaunchKernelGGL((decode_split_kernel<E, DP, GM, kWide>), dim3(2 * heads, (splits + 1) / 2, B),
                       dim3(kThreads), 0, stream, P);
  else
    hipLaunchKernelGGL((decode_split_kernel<E, DP, GM, false>), dim3(heads, splits, B),
                       dim3(kThreads), 0, stream, P);
  int st = launch_status("decode_split");
  if (st != MCAMD_OK || P.n_splits == 1) return st;
  hipLaunchKernelGGL(decode_combine_kernel<E>, dim3(P.H, B), dim3(kThreads), 0, stream, P);
  return launch_status("decode_combine");
}

template <class E, int DP>
int dispatch_gm(DecodeParams &P, int B, hipStream_t s) {
  if (P.G == 1) { P.n_hchunks = 1; return run_decode<E, DP, 1>(P, B, s); }
  if (P.G == 2) { P.n_hchunks = 1; return run_decode<E, DP, 2>(P, B, s); }
  if (P.G <= 4) { P.n_hchunks = 1; return run_decode<E, DP, 4>(P, B, s); }
  P.n_hchunks = (P.G + 7) / 8;
  return run_decode<E, DP, 8>(P, B, s);
}

// Any head_dim up to 256 whose rows are whole 16-byte vectors (checked before; wider heads take
// the general prefill kernel, see launch_decode), run in the
// instantiation of the next power of two.
template <class E>
int dispatch_d(DecodeParams &P, int B, hipStream_t s) {
  switch (head_dim_bucket(P.D)) {
    case 16: return dispatch_gm<E, 16>(P, B, s);
    case 32: return dispatch_gm<E, 32>(P, B, s);
    case 64: return dispatch_gm<E, 64>(P, B, s);
    case 128: return dispatch_gm<E, 128>(P, B, s);
    case 256: return dispatch_gm<E, 256>(P, B, s);
    default:
      return fail(MCAMD_EUNSUPPORTED, "decode: head_dim must be at most 256");
  }
}

}  // namespace

namespace {

size_t general_bytes(int64_t batch, int64_t n_head, int64_t head_dim, int64_t splits) {
  return size_t(batch * n_head * splits * (head_dim + 2) * 4);
}
// What the other decode path of a head dim needs, or 4 MB: shorter splits stay within it.
size_t short_split_room(int64_t batch, int64_t n_head, int64_t n_kv_head, int64_t head_dim,
                        int64_t t_max, int64_t window) {
  return head_dim == 128 ? decode_fused_partial_bytes(batch, n_head, n_kv_head, t_max, window)
                         : size_t(4) << 20;
}

int64_t decode_split_len(int64_t batch, int64_t n_head, int64_t n_kv_head, int64_t head_dim,
                         int64_t t_max, int64_t window, int64_t elem) {
  return split_len(batch, n_kv_head, head_dim, t_max, window, elem, [&](int64_t splits) {
    return general_bytes(batch, n_head, head_dim, splits) <=
           short_split_room(batch, n_head, n_kv_head, head_dim, t_max, window);
  });
}

}  // namespace

size_t decode_workspace_bytes(int64_t batch, int64_t n_head, int64_t n_kv_head, int64_t head_dim,
                              int64_t t_max, int64_t window) {
  // Head dims above 256 take the general prefill kernel, which needs no workspace.
  size_t generic = 0;
  if (head_dim <= 256) {
    for (int64_t elem : {2, 4}) {  // the sizes do not tell the type
      const int64_t len = decode_split_len(batch, n_head, n_kv_head, head_dim, t_max, window, elem);
      generic = std::max(generic, general_bytes(batch, n_head, head_dim,
                                                splits_of(t_max, window, len)));
    }
    generic = std::max(generic, general_bytes(batch, n_head, head_dim,
                                              splits_of(t_max, window, kDecodeSplitLen)));
  }
  // The fused path serves head_dim 128 (bf16); other head dims only ever take the general one.
  const size_t fused =
      head_dim == 128 ? decode_fused_partial_bytes(batch, n_head, n_kv_head, t_max, window) : 0;
  const size_t part = generic > fused ? generic : fused;
  return (part + 255) / 256 * 256;
}

int launch_decode(const AttnArgs &a) {
  int st = check_attn_shapes(a, true);
  if (st != MCAMD_OK) return st;
  if (a.t_new != 1) return fail(MCAMD_EINVAL, "decode: t_new must be 1");
  if (a.batch == 0) {
    clear_error();
    return MCAMD_OK;
  }
  if (decode_fused_supported(a)) return launch_decode_fused(a);
  if (a.k_new && a.head_dim > 256) {
    // The kernel of these head dims reads the cache only: append first.
    AppendArgs ap{a.k_new, a.v_new, const_cast<void *>(a.k_cache), const_cast<void *>(a.v_cache),
                  a.seqlens, a.batch, 1, a.n_kv_head, a.head_dim, a.t_max, a.cache_batch_stride,
                  a.dtype, a.stream};
    st = launch_append(ap);
    if (st != MCAMD_OK) return st;
  }
  if (a.head_dim > 256) {
    // Past 256 an fp32 key row needs more than a wave's 64 lanes of 16 bytes, and the cross-wave
    // sum buffer (4 x GM x D floats) outgrows the LDS budget: the general prefill kernel (one
    // query per row here) walks the keys instead, with no split and no workspace.
    AttnArgs pa = a;
    pa.k_new = pa.v_new = nullptr;  // appended above
    st = launch_prefill_generic(pa);
    if (st != MCAMD_OK || !a.advance_seqlens) return st;
    return launch_advance(a.advance_seqlens, a.batch, a.advance, a.stream);
  }
  DecodeParams P;
  P.q = a.q;
  P.k_new = a.k_new;
  P.v_new = a.v_new;
  P.k_cache = const_cast<void *>(a.k_cache);
  P.v_cache = const_cast<void *>(a.v_cache);
  P.seqlens = a.seqlens;
  P.out = a.out;
  P.H = int(a.n_head);
  P.H_kv = int(a.n_kv_head);
  P.G = int(a.n_head / a.n_kv_head);
  P.n_hchunks = 1;
  P.T_max = int(a.t_max);
  P.window = int(a.window < 0 ? -1 : a.window);
  const int64_t elem = a.dtype == MCAMD_F32 ? 4 : 2;
  P.SL = int(decode_split_len(a.batch, a.n_head, a.n_kv_head, a.head_dim, a.t_max, a.window, elem));
  P.n_splits = int(splits_of(a.t_max, a.window, P.SL));
  P.D = int(a.head_dim);
  P.cache_b = a.cache_batch_stride;
  P.scale_log2 = float(kLog2e / std::sqrt(double(a.head_dim)));
  const int64_t floats_o = a.batch * a.n_head * P.n_splits * a.head_dim;
  P.part_o = static_cast<float *>(a.workspace);
  P.part_ml = P.part_o + floats_o;
  st = a.dtype == MCAMD_BF16 ? dispatch_d<bf16>(P, int(a.batch), a.stream)
                             : dispatch_d<float>(P, int(a.batch), a.stream);
  if (st != MCAMD_OK || !a.advance_seqlens) return st;
  return launch_advance(a.advance_seqlens, a.batch, a.advance, a.stream);
}

}  // namespace mcamd
