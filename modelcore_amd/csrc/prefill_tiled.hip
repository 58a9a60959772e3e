// Multi-token attention against the cache prefix on the matrix cores, for the shapes the bf16 /
// head_dim 128 kernel (prefill_mfma.hip) does not take: fp32 caches, and head dims up to 256 made
// of whole 16-byte vectors.
//
// Semantics: modelcore/kernels/flash_attn.py:226-244 (uniform, explicit mask with row offset
// Tk - Tq) and :362-364 (ragged mask). Query t of row b sits at p = cache_seqlens[b] + t and
// attends keys col <= p with p - col <= window when window >= 0. The cache already holds the new
// tokens (the append runs first), so the prefix includes the chunk itself.
//
// Work split. The (position, query head) pairs of one (row, KV head), head fastest, are laid end
// to end and cut into blocks of 32 per wave, so that every K/V tile serves the whole GQA group.
// KS = 1: the four waves of a workgroup take 128 pairs and share each staged tile of keys. KS = 4:
// they take the same 32 pairs and a quarter of each staged tile each, and merge at the end; four
// times the workgroups and a quarter of the serial chain, for calls with too few pairs to fill the
// chip (each K/V byte is then staged for a quarter of the pairs). Blocks with the most keys (the
// last positions) are launched first; a compute unit holds two or three at once, so they are dealt to
// the compute units there and back (dealt_block()).
//
// Products, per wave and 32 keys, with both 32 x 32 results transposed so that a lane owns one
// pair (lane l: pair l % 32, keys 8j + 4(l / 32) + i):
//   S^T (keys x pairs) = K . Q^T     A = K from LDS, B = Q in registers
//   O^T (D x pairs)   += V^T . P^T   A = V^T from LDS, B = the weights, where they are
//  * bf16: v_mfma_f32_32x32x16_bf16. K and V are bf16 as they are and the scores leave in fp32;
//    the weights are fp32 and go in as two bf16 terms, p = hi + lo with lo = bf16(p - hi), which
//    keeps them to 2^-17: half again the matrix work for the accuracy of fp32 weights.
//  * fp32: v_mfma_f32_32x32x2_f32, fp32 throughout. A step of the second product takes the keys
//    8j + i and 8j + 4 + i, the two that one accumulator of the scores holds in the two halves of
//    the wave, so the weights are its B operand in place; the first takes dims 8c + i and
//    8c + 4 + i, so that a lane reads its K row as 16-byte vectors.
//
// Measured against the VALU kernel this replaced (four lanes a row, an LDS float per FMA), the call
// with its append: four 2048-token prompts of 12 heads of 64 in bf16 1868 -> 73 us (355 TFLOP/s of the
// attended pairs), two of 512 tokens in fp32 194 -> 32.
//
// Online softmax per pair in fp32 (exp2 domain): weights are made against the running maximum, and
// the tile's own maximum is taken (and O rescaled) only when a lane's weights of the tile sum past
// 2^15 or are not finite, or the pair has no maximum yet.
//
// LDS holds one tile; the next is loaded while it is consumed, into arrays of which the compiler keeps
// one in scratch memory in most instantiations (48 to 272 bytes a lane: half a tile's loads are waited
// for, and stored there, before the products start). K rows are padded by
// 16 bytes (a 16-lane group reads 16 rows at once: their 16-byte pieces then fall on all banks);
// bf16 V rows to 16 or 48 banks modulo 64 for the transpose reads (four rows of 64 bytes), fp32 V
// rows by 32 bytes (the two wave halves read rows four apart).
//
// Not finite. The products multiply masked keys' values by a weight of zero, so an infinity or
// NaN in V would reach pairs that may not see it, and an infinite value meets a zero lo term. A
// pair whose result is not finite is therefore redone over the keys it sees alone (careful_pair()).
#include "prefill_order.h"
#include "prefill_split.h"

#include <cmath>
#include <type_traits>

namespace mcamd {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = 4;
constexpr float kTileSumLimit = 32768.f;  // 2^15: a lane's weights of one tile sum to at most this

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 lds_bf16x4 __attribute__((__vector_size__(4 * sizeof(__bf16))));

struct TiledParams {
  const void *q, *k_cache, *v_cache;
  const int32_t *seqlens;
  const int32_t *rows, *cu;  // varlen (optional): cache row and token range per sequence
  void *out;
  int T_new, H, H_kv, G, T_max, window, D, n_bh, n_qt;
  int deal;  // workgroups per round of dealt_block()
  int64_t cache_b;
  float scale_log2;
  SplitGeo split;
};

// Tile geometry of an instantiation (elements of E; DP is head_dim rounded up).
template <class E, int DP, int KS>
struct Geo {
  static constexpr bool kBf16 = sizeof(E) == 2;
  static constexpr int VEC = Vec<E>::N;
  static constexpr int KW = kBf16 && DP <= 128 && KS == 1 ? 64 : 32;  // keys per wave and tile
  static constexpr int MK = KW / 32;
  static constexpr int KT = KW * KS;                  // keys per tile
  static constexpr int PAIRS = 32 * kWaves / KS;      // pairs per workgroup
  static constexpr int MD = DP / 32;                  // 32-row blocks of O^T
  static constexpr int KSTR = DP + VEC;               // K row stride
  // V row stride: bf16 16 or 48 dwords modulo 64 (DP / 2 is 16, 48 or a multiple of 32), fp32
  // DP + 8.
  static constexpr int VSTR = kBf16 ? (DP % 64 == 0 ? DP + 32 : DP) : DP + 8;
  static constexpr int CH = KT * DP / VEC / kThreads;  // 16-byte pieces of K (or V) per thread
  static constexpr int TILE_BYTES = (KSTR + VSTR) * KT * int(sizeof(E));
  static constexpr int OSTR = DP + 4;                 // row stride of the KS = 4 merge, floats
  static constexpr int MERGE_BYTES = KS == 1 ? 0 : (32 * OSTR + 64) * 4 * kWaves + 32 * 4;
  static constexpr int LDS_BYTES = TILE_BYTES > MERGE_BYTES ? TILE_BYTES : MERGE_BYTES;
  static_assert(KT * DP % (VEC * kThreads) == 0, "whole pieces per thread");
  static_assert(!kBf16 || VSTR / 2 % 32 == 16, "V rows on 16 or 48 banks modulo 64");
};

__device__ __forceinline__ float max_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }

// Four consecutive LDS rows of one column, transposed into a lane: lane L of each 16-lane group
// passes the address of row L / 4, columns 4 (L % 4) .. + 3 of a 4 x 16 block and receives
// column L of it.
__device__ __forceinline__ bf16x4 lds_read_tr(const uint16_t *p) {
  auto lp = (__attribute__((address_space(3))) lds_bf16x4 *)(p);
  return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4bf16(lp));
}

// Dims [d0, d1) of one pair redone by a wave over the keys it sees alone, for pairs whose result is not
// finite: 64 keys a step, a key per lane for its score, then a dim per lane (l, l + 64, ..) for the sums.
// Four prompts of 2048 tokens, 12 heads of 64, with an infinity in one head's first value: 4.7 ms in bf16
// (a key at a time 28; without the infinity 0.07), in every head's 8.1 in fp32 (38; 0.26). 64 values in
// flight instead of 32 gave 6% and cost the kernel's other waves their registers.
template <class E, int DP, int LOADS = 32>  // LOADS: values (and 16-byte pieces of keys) in flight
__device__ void careful_pair(const TiledParams &P, int row, int kvh, int64_t at, int p, int lane,
                             int d0, int d1) {
  constexpr int N = (DP + 63) / 64, VEC = Vec<E>::N, U = N == 3 ? LOADS / 4 : LOADS / N;
  static_assert(64 % U == 0, "whole batches per step");
  const int D = P.D;
  const E *q = static_cast<const E *>(P.q) + at;
  E *out = static_cast<E *>(P.out) + at;
  const int64_t tok = int64_t(P.H_kv) * D;
  const E *kc = static_cast<const E *>(P.k_cache) + int64_t(row) * P.cache_b + int64_t(kvh) * D;
  const E *vc = static_cast<const E *>(P.v_cache) + int64_t(row) * P.cache_b + int64_t(kvh) * D;
  float o[N];
#pragma unroll
  for (int i = 0; i < N; ++i) o[i] = 0.f;
  float m = -INFINITY, l = 0.f;  // l: of this lane's keys
  for (int t0 = key_lo(p, P.window); t0 <= p; t0 += 64) {
    const int t = min(t0 + lane, p);
    float s = 0.f;
    constexpr int KU = DP / VEC < LOADS / 4 ? DP / VEC : LOADS / 4;
    for (int c0 = 0; c0 < D; c0 += KU * VEC) {
      uint4 y[KU];
#pragma unroll
      for (int c = 0; c < KU; ++c)
        y[c] = *reinterpret_cast<const uint4 *>(kc + int64_t(t) * tok + min(c0 + c * VEC, D - VEC));
#pragma unroll
      for (int c = 0; c < KU; ++c) {
        float x[VEC], z[VEC], dot = s;
        Vec<E>::load(q + min(c0 + c * VEC, D - VEC), x);
        Vec<E>::unpack(y[c], z);
#pragma unroll
        for (int e = 0; e < VEC; ++e) dot = fmaf(x[e] * P.scale_log2, z[e], dot);
        s = c0 + c * VEC < D ? dot : s;
      }
    }
    if (t0 + lane > p) s = -INFINITY;
    if (__builtin_amdgcn_ballot_w64(s != s) != 0) {  // a NaN key makes the output NaN, as in the softmax
      l = NAN;
      break;
    }
    const float m_new = fmaxf(m, wave_max<64>(s));
    if (m_new == -INFINITY) continue;
    const float corr = fast_exp2(m - m_new), w = fast_exp2(s - m_new);
    m = m_new;
    l = fmaf(l, corr, s == -INFINITY ? 0.f : w);
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] *= corr;
    const uint64_t seen = __builtin_amdgcn_ballot_w64(s != -INFINITY);
    for (int k0 = 0; k0 < min(64, p - t0 + 1); k0 += U) {
      E v[U][N];  // without a branch between the loads: lanes without a dim take a neighbour's
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < N; ++i)
          v[u][i] = vc[int64_t(min(t0 + k0 + u, p)) * tok + max(d0, min(lane + 64 * i, d1 - 1))];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float wk = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), k0 + u));
        const bool there = (seen >> (k0 + u)) & 1;  // a weight of zero must not meet an infinity
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = there ? fmaf(wk, to_f32<E>(v[u][i]), o[i]) : o[i];
      }
    }
  }
  const float inv = 1.f / wave_sum<64>(l);
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (lane + 64 * i >= d0 && lane + 64 * i < d1) out[lane + 64 * i] = from_f32<E>(o[i] * inv);
}

// Four consecutive output dims.
__device__ __forceinline__ void store4(float *p, const f32x4 &x) {
  *reinterpret_cast<f32x4 *>(p) = x;
}
__device__ __forceinline__ void store4(bf16 *p, const f32x4 &x) {
  *reinterpret_cast<uint2 *>(p) =
      __builtin_bit_cast(uint2, __builtin_convertvector(x, bf16x4));
}

template <class E, int DP, int KS>
__global__ __launch_bounds__(kThreads) void prefill_tiled_kernel(TiledParams P) {
  using G_ = Geo<E, DP, KS>;
  constexpr bool kBf16 = G_::kBf16;
  constexpr int VEC = G_::VEC, KW = G_::KW, MK = G_::MK, KT = G_::KT, MD = G_::MD, CH = G_::CH;
  constexpr int KSTR = G_::KSTR, VSTR = G_::VSTR, OSTR = G_::OSTR;
  __shared__ __attribute__((aligned(16))) unsigned char s_raw[G_::LDS_BYTES];
  E *const sK = reinterpret_cast<E *>(s_raw);
  E *const sV = sK + KT * KSTR;

  const int id = P.cu ? int(blockIdx.x) : dealt_block(int(blockIdx.x), int(gridDim.x), P.deal);
  int bh = id % P.n_bh;
  const int part = int(id / P.n_bh) % P.split.n_split;  // key range
  int qt = P.n_qt - 1 - int(id / P.n_bh) / P.split.n_split;
  int b = bh / P.H_kv;
  int kvh = bh - b * P.H_kv;
  int row = b, T_b = P.T_new, s0;
  int64_t tok0 = int64_t(b) * P.T_new;
  if (P.cu && P.n_bh <= kOrderedSeqs * P.H_kv) {
    VarlenBlock v;
    if (!find_varlen_block(P.cu, P.rows, P.seqlens, P.n_bh / P.H_kv, P.n_qt, G_::PAIRS, P.G,
                           int(blockIdx.x) / P.H_kv, threadIdx.x & 63, v))
      return;
    kvh = int(blockIdx.x) % P.H_kv;
    bh = v.b * P.H_kv + kvh;
    b = v.b, qt = v.qt, row = v.row, tok0 = v.tok0, T_b = v.T_b, s0 = v.s0;
  } else {
    if (P.cu) {
      row = P.rows ? P.rows[b] : b;
      tok0 = P.cu[b];
      T_b = P.cu[b + 1] - P.cu[b];
    }
    s0 = P.seqlens[row];
  }
  // This workgroup's pairs: n of them from pair p0 on, which is head r0 of position q0.
  const int64_t n_pairs = int64_t(T_b) * P.G;
  const int64_t p0 = int64_t(qt) * G_::PAIRS;
  if (p0 >= n_pairs) return;  // a block past a shorter sequence's end (a whole workgroup)
  const int n = int(min(int64_t(G_::PAIRS), n_pairs - p0));
  const int q0 = int(p0 / P.G), r0 = int(p0 - int64_t(q0) * P.G);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5;    // lane half
  const int col = lane & 31;  // this lane's pair within the wave's 32
  const int D = P.D;

  const bool row_ok = s0 >= 0 && int64_t(s0) + T_b <= P.T_max;
  const int w0 = KS == 1 ? 32 * wave : 0;  // the wave's first pair
  const bool live = w0 + col < n;
  // Position of pair i of the workgroup, and where its query and output lie.
  auto pair_pos = [&](int i) { return q0 + (r0 + i) / P.G; };
  auto pair_at = [&](int i) {
    const int pos = (r0 + i) / P.G;
    return ((tok0 + q0 + pos) * P.H + int64_t(kvh) * P.G + (r0 + i - pos * P.G)) * D;
  };
  const int pr = live ? w0 + col : 0;  // dead pairs compute on a live one
  const int tq = pair_pos(pr);
  const int64_t at = pair_at(pr);
  E *out = static_cast<E *>(P.out) + at;
  if (!row_ok) {
    if (live && part == 0 && (KS == 1 || wave == 0))
      for (int d = h; d < D; d += 2) out[d] = from_f32<E>(NAN);
    return;
  }

  const int p_abs = s0 + tq;
  const int p_first = s0 + q0;
  const int last = s0 + pair_pos(n - 1);  // the last key any pair of the workgroup sees
  const int n_part = P.split.n_split;
  int lo = P.window >= 0 ? max(0, p_first - P.window) : 0, hi = last;
  int n_tiles = (hi - lo) / KT + 1;
  bool whole = true;
  if (n_part > 1) {  // this workgroup's range of the block's tiles
    const int ranges = block_splits(P.split, s0, T_b, n_tiles);
    if (part >= ranges) return;
    whole = ranges == 1;
    const int t0 = part * n_tiles / ranges, t1 = (part + 1) * n_tiles / ranges;
    hi = min(hi, lo + t1 * KT - 1);
    lo += t0 * KT;
    n_tiles = t1 - t0;
  }

  // Q^T fragments, B[k = dim][n = pair]. bf16: dims 16 kd + 8h .. + 7 of step kd; fp32: dims
  // 8c + 4h .. + 3, one for each of four steps. Dims past the head_dim are zero.
  constexpr int NQ = kBf16 ? DP / 16 : DP / 8;
  using QF = typename std::conditional<kBf16, bf16x8, f32x4>::type;
  QF qf[NQ];
  {
    const E *qp = static_cast<const E *>(P.q) + at;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int d = (kBf16 ? 16 : 8) * i + VEC * h;
      uint4 u = make_uint4(0, 0, 0, 0);
      if (d < D) u = *reinterpret_cast<const uint4 *>(qp + d);
      qf[i] = __builtin_bit_cast(QF, u);
    }
  }
  const int64_t tok = int64_t(P.H_kv) * D;
  const E *kbase = static_cast<const E *>(P.k_cache) + int64_t(row) * P.cache_b + int64_t(kvh) * D;
  const E *vbase = static_cast<const E *>(P.v_cache) + int64_t(row) * P.cache_b + int64_t(kvh) * D;

  // The next tile, on its way to LDS (see above where it waits): piece c = tid + 256 i is 16 bytes of key c / (DP / VEC).
  // Keys past `hi` re-read key `hi` (they are masked); K's dims past the head_dim are zero, V's
  // re-read the last ones (they reach no output).
  uint4 kr[CH], vr[CH];
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = tid + kThreads * i;
      const int key = min(k0 + c / (DP / VEC), hi);
      const int d = (c % (DP / VEC)) * VEC;
      const int64_t off = int64_t(key) * tok + min(d, D - VEC);
      kr[i] = *reinterpret_cast<const uint4 *>(kbase + off);
      vr[i] = *reinterpret_cast<const uint4 *>(vbase + off);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = tid + kThreads * i;
      const int key = c / (DP / VEC), d = (c % (DP / VEC)) * VEC;
      // The zeroes go in here and not at the load, all of which would then be waited for at once.
      *reinterpret_cast<uint4 *>(&sK[key * KSTR + d]) = d < D ? kr[i] : make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4 *>(&sV[key * VSTR + d]) = vr[i];
    }
  };

  f32x16 o[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[md][e] = 0.f;
  float m = -INFINITY, l = 0.f;

  const int wk = KS == 1 ? 0 : wave * KW;  // the wave's first key within a tile
  const int tr_row = (lane & 15) >> 2;     // bf16: this lane's part of a transpose read
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  load_tile(lo);
  for (int t = 0; t < n_tiles; ++t) {
    const int k0 = lo + t * KT + wk;
    if (t > 0) __syncthreads();  // every wave has read the tile before
    store_tile();
    __syncthreads();
    if (t + 1 < n_tiles) load_tile(lo + (t + 1) * KT);
    if (KS > 1 && k0 > hi) continue;  // no key of this wave's quarter (barriers stay paired)

    f32x16 s[MK];
#pragma unroll
    for (int mk = 0; mk < MK; ++mk) {
      const E *kp = &sK[(wk + 32 * mk + col) * KSTR + VEC * h];
      // fp32: four interleaved chains of sums, added at the end: a quarter of one chain's rounding.
      constexpr int NC = kBf16 ? 1 : 4;
      f32x16 sc[NC];
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[j][e] = 0.f;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const QF a = __builtin_bit_cast(
            QF, *reinterpret_cast<const uint4 *>(kp + (kBf16 ? 16 : 8) * i));
        if constexpr (kBf16) {
          sc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[i], sc[0], 0, 0, 0);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            sc[j % NC] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], qf[i][j], sc[j % NC], 0, 0, 0);
        }
      }
      s[mk] = sc[0];
      if constexpr (!kBf16) s[mk] = (sc[0] + sc[1]) + (sc[2] + sc[3]);
    }
    // Keys the pair may not see, in tiles that straddle the diagonal or the window's edge.
    if (k0 + KW - 1 > p_first || (P.window >= 0 && k0 < last - P.window)) {
#pragma unroll
      for (int mk = 0; mk < MK; ++mk)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int dpos = p_abs - (k0 + 32 * mk + 8 * (e >> 2) + 4 * h + (e & 3));
          if (!(dpos >= 0 && (P.window < 0 || dpos <= P.window))) s[mk][e] = -INFINITY;
        }
    }

    float w[MK][16];
    auto weigh = [&]() {
      const float mu = m == -INFINITY ? 0.f : m;
      float ts[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mk = 0; mk < MK; ++mk)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          w[mk][e] = fast_exp2(fmaf(s[mk][e], P.scale_log2, -mu));
          ts[e & 3] += w[mk][e];
        }
      return (ts[0] + ts[1]) + (ts[2] + ts[3]);
    };
    float tl = weigh();
    if (__builtin_amdgcn_ballot_w64(!(tl <= kTileSumLimit) || m == -INFINITY) != 0) {
      float m4[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
      for (int mk = 0; mk < MK; ++mk)
#pragma unroll
        for (int e = 0; e < 16; ++e) m4[e & 3] = fmaxf(m4[e & 3], s[mk][e]);
      const float mx =
          max_halves(fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]))) * P.scale_log2;
      const float m_new = fmaxf(m, mx);
      const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - m_new);
      l *= alpha;
#pragma unroll
      for (int md = 0; md < MD; ++md)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[md][e] *= alpha;
      m = m_new;
      tl = weigh();
    }
    l += tl;

    if constexpr (kBf16) {
#pragma unroll
      for (int ks = 0; ks < 2 * MK; ++ks) {  // 16 keys: the eight accumulators 8 (ks % 2) ..
        f32x8 pv;
#pragma unroll
        for (int e = 0; e < 8; ++e) pv[e] = w[ks >> 1][8 * (ks & 1) + e];
        const bf16x8 hi8 = __builtin_convertvector(pv, bf16x8);
        const bf16x8 lo8 =
            __builtin_convertvector(pv - __builtin_convertvector(hi8, f32x8), bf16x8);
        const uint16_t *vp = reinterpret_cast<const uint16_t *>(sV) +
                             (wk + 16 * ks + 4 * h + tr_row) * VSTR + tr_col;
        bf16x8 a[MD];  // the lo terms after all hi terms: no product waits for the one before it
#pragma unroll
        for (int md = 0; md < MD; ++md) {
          const bf16x4 a0 = lds_read_tr(vp + 32 * md);
          const bf16x4 a1 = lds_read_tr(vp + 8 * VSTR + 32 * md);
          a[md] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
          o[md] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[md], hi8, o[md], 0, 0, 0);
        }
#pragma unroll
        for (int md = 0; md < MD; ++md)
          o[md] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[md], lo8, o[md], 0, 0, 0);
      }
    } else {
      const float *vp = reinterpret_cast<const float *>(sV) + (wk + 4 * h) * VSTR + col;
#pragma unroll
      for (int mk = 0; mk < MK; ++mk)
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int md = 0; md < MD; ++md)
            o[md] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                vp[(32 * mk + 8 * (e >> 2) + (e & 3)) * VSTR + 32 * md], w[mk][e], o[md], 0, 0, 0);
    }
  }

  l = sum_halves(l);
  if constexpr (KS == 1) {
    if (!whole) {
      if (!live) return;
      const int64_t g = P.split.group(part, qt, bh, wave);
#pragma unroll
      for (int md = 0; md < MD; ++md)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (32 * md < D)
            store4(P.split.o(g, md, j, lane), f32x4{o[md][4 * j], o[md][4 * j + 1],
                                                    o[md][4 * j + 2], o[md][4 * j + 3]});
      if (h == 0) *reinterpret_cast<float2 *>(P.split.ml(g, col)) = make_float2(m, l);
      return;
    }
    const float inv = 1.f / l;
    bool ok = true;
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        o[md][e] *= inv;
        ok = ok && (finite(o[md][e]) || 32 * md + 8 * (e >> 2) >= D);
      }
    const uint64_t bad64 = __builtin_amdgcn_ballot_w64(live && !ok);
    const uint32_t bad = uint32_t(bad64) | uint32_t(bad64 >> 32);
    if (live && !((bad >> col) & 1u)) {
#pragma unroll
      for (int md = 0; md < MD; ++md)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int d = 32 * md + 8 * j + 4 * h;
          if (d < D)
            store4(out + d, f32x4{o[md][4 * j], o[md][4 * j + 1], o[md][4 * j + 2],
                                  o[md][4 * j + 3]});
        }
    }
    for (uint32_t left = bad; __builtin_expect(left != 0, 0); left &= left - 1) {
      const int c = w0 + __builtin_ctz(left);
      careful_pair<E, DP>(P, row, kvh, pair_at(c), s0 + pair_pos(c), lane, 0, D);
    }
  } else {
    // Merge the four waves' (o, m, l) of the same 32 pairs; thread t then owns an eighth of the
    // dims of pair t / 8.
    float *const so = reinterpret_cast<float *>(s_raw);
    float *const sm = so + kWaves * 32 * OSTR;  // m[4][32], then l[4][32]
    int *const s_bad = reinterpret_cast<int *>(sm + 64 * kWaves);
    __syncthreads();  // the last tile has been read
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4 *>(&so[(wave * 32 + col) * OSTR + 32 * md + 8 * j + 4 * h]) =
            f32x4{o[md][4 * j], o[md][4 * j + 1], o[md][4 * j + 2], o[md][4 * j + 3]};
    if (h == 0) {
      sm[wave * 32 + col] = m;
      sm[kWaves * 32 + wave * 32 + col] = l;
    }
    if (tid < 32) s_bad[tid] = 0;
    __syncthreads();
    const int c = tid >> 3;
    float M = -INFINITY, L = 0.f, a[kWaves];
#pragma unroll
    for (int u = 0; u < kWaves; ++u) M = fmaxf(M, sm[u * 32 + c]);
#pragma unroll
    for (int u = 0; u < kWaves; ++u) {
      const float mu = sm[u * 32 + c];
      a[u] = mu == -INFINITY ? 0.f : fast_exp2(mu - M);
      // A wave that saw no key has l = 0; a NaN l (a NaN score) must stay.
      L += sm[kWaves * 32 + u * 32 + c] * (mu == -INFINITY ? 1.f : a[u]);
    }
    const float inv = whole ? 1.f / L : 1.f;
    constexpr int DT = DP / 8;
    f32x4 y[DT / 4];
    bool ok = true;
#pragma unroll
    for (int i = 0; i < DT / 4; ++i) {
      const int d = 32 * i + 4 * (tid & 7);
      y[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < kWaves; ++u) {
        const f32x4 x = *reinterpret_cast<const f32x4 *>(&so[(u * 32 + c) * OSTR + d]);
        y[i] += x * a[u];
      }
      y[i] *= inv;
#pragma unroll
      for (int e = 0; e < 4; ++e) ok = ok && (finite(y[i][e]) || d >= D);
    }
    const bool c_live = c < n;
    if (!whole) {
      if (!c_live) return;
      const int64_t g = P.split.group(part, qt, bh, 0);
      const int x = tid & 7;
#pragma unroll
      for (int i = 0; i < DT / 4; ++i)
        if (32 * i < D) store4(P.split.o(g, i, x >> 1, 32 * (x & 1) + c), y[i]);
      if (x == 0) *reinterpret_cast<float2 *>(P.split.ml(g, c)) = make_float2(M, L);
      return;
    }
    if (c_live && !ok) s_bad[c] = 1;
    __syncthreads();
    if (c_live && s_bad[c] == 0) {
      E *co = static_cast<E *>(P.out) + pair_at(c);
#pragma unroll
      for (int i = 0; i < DT / 4; ++i) {
        const int d = 32 * i + 4 * (tid & 7);
        if (d < D) store4(co + d, y[i]);
      }
    }
    for (int x = wave; x < 32; x += kWaves) {
      if (__builtin_expect(s_bad[x] == 0, 1)) continue;
      careful_pair<E, DP>(P, row, kvh, pair_at(x), s0 + pair_pos(x), lane, 0, D);
    }
  }
}

// Merges the partials of key ranges, in the partials' own layout: a workgroup per 32 pairs and 32
// dims, a wave per step j of them, eight ranges' loads in flight. Bound by the latency of those
// loads at these sizes. (A workgroup per 32 pairs, of 1024 threads, is slower: 10.8 us against 8.6 for 100
// tokens after 8000 keys, and 7.3 against 5.8 where 2048 workgroups find nothing to merge.)
//
// Where the ranges have read the chunk from k and v (prefill_appends()), the first workgroups of
// each row append it.
constexpr int kMergeThreads = 256;
constexpr int kAppendUnits = 2 * kMergeThreads;  // of 16 bytes, of a workgroup

struct NewTokens {
  const void *k, *v;
  int64_t units;  // of 16 bytes, per row of k (or v)
  int tok;        // and per token of it
  int blocks;     // appending workgroups per row of k (or v)
};

// Part `i` of row b's append: its new tokens are one run in the cache, clipped to its positions.
template <class E>
__device__ __forceinline__ void append_part(const TiledParams &P, const NewTokens &N, int b, int i) {
  const bool is_v = i >= N.blocks;
  const int64_t s0 = P.seqlens[b];
  const int64_t from = max(int64_t(0), -s0) * N.tok;
  const int64_t to = min(int64_t(P.T_new), P.T_max - s0) * N.tok;
  const uint4 *src = static_cast<const uint4 *>(is_v ? N.v : N.k) + b * N.units;
  uint4 *dst = static_cast<uint4 *>(const_cast<void *>(is_v ? P.v_cache : P.k_cache)) +
               (b * P.cache_b / Vec<E>::N + s0 * N.tok);
  const int64_t at = int64_t(is_v ? i - N.blocks : i) * kAppendUnits + threadIdx.x;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t c = at + u * kMergeThreads;
    if (c >= from && c < to) dst[c] = src[c];
  }
}

template <class E>
__global__ __launch_bounds__(kMergeThreads) void prefill_combine_kernel(TiledParams P, SplitGeo g,
                                                                        int careful, NewTokens N) {
  const int b = blockIdx.y;
  int at = int(blockIdx.x) - 2 * N.blocks;
  if (at < 0) {
    append_part<E>(P, N, b, blockIdx.x);
    return;
  }
  const int s0 = P.seqlens[b];
  if (s0 < 0 || int64_t(s0) + P.T_new > P.T_max) return;  // NaN, written already
  if (s0 + P.T_new <= g.uncut_keys) return;               // written by the blocks themselves
  const int lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int md = at % g.md;
  at /= g.md;
  const int w = at % g.groups;
  at /= g.groups;
  const int kvh = at % P.H_kv, qt = at / P.H_kv;
  const int bh = b * P.H_kv + kvh;
  const int d = 32 * md + 8 * j;  // this wave's dims d .. d + 7, lane half h d + 4h ..
  if (d >= P.D) return;
  int lo, hi;
  block_keys(g, s0, P.T_new, qt, lo, hi);
  const int ranges = block_splits(g, s0, P.T_new, (hi - lo) / g.kt + 1);
  if (ranges == 1) return;  // written by the block itself
  const int64_t p0 = int64_t(qt) * g.pairs;
  const int in_block = 32 * w + col;
  const bool live = in_block < g.pairs && p0 + in_block < int64_t(P.T_new) * P.G;

  constexpr int U = 8;
  const int64_t group = g.group(0, qt, bh, w), step = g.group(1, qt, bh, w) - group;
  const float *ml = g.ml(group, col);
  const float *po = g.o(group, md, j, lane);
  const int64_t ml_step = step * 64, o_step = step * g.md * 1024;
  float M = -INFINITY, L = 0.f;
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
  for (int r0 = 0; r0 < ranges; r0 += U) {
    float2 x[U];
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = min(r0 + u, ranges - 1);
      x[u] = *reinterpret_cast<const float2 *>(ml + r * ml_step);
      v[u] = *reinterpret_cast<const f32x4 *>(po + r * o_step);
    }
    float m_new = M;
#pragma unroll
    for (int u = 0; u < U; ++u) m_new = fmaxf(m_new, x[u].x);
    const float keep = M == -INFINITY ? 0.f : fast_exp2(M - m_new);
    L *= M == -INFINITY ? 1.f : keep;  // 0 then, or a NaN that must stay
    y *= keep;
    M = m_new;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (r0 + u >= ranges) break;
      const float a = x[u].x == -INFINITY ? 0.f : fast_exp2(x[u].x - M);
      L += x[u].y * (x[u].x == -INFINITY ? 1.f : a);
      y += a * v[u];
    }
  }
  y *= 1.f / L;
  const bool ok = finite(y[0]) && finite(y[1]) && finite(y[2]) && finite(y[3]);
  const int pos = live ? int((p0 + in_block) / P.G) : 0;
  const int64_t row = (int64_t(b) * P.T_new + pos) * P.H + int64_t(kvh) * P.G +
                      (live ? int(p0 + in_block - int64_t(pos) * P.G) : 0);
  const uint64_t bad64 =
      careful ? __builtin_amdgcn_ballot_w64(live && !ok && d + 4 * h < P.D) : 0;
  const uint32_t bad = uint32_t(bad64) | uint32_t(bad64 >> 32);
  if (live && !((bad >> col) & 1u) && d + 4 * h < P.D)
    store4(static_cast<E *>(P.out) + row * P.D + d + 4 * h, y);
  for (uint32_t left = bad; left != 0; left &= left - 1) {
    const int c = __builtin_ctz(left);
    const int rlo = __shfl(int(uint64_t(row)), c, 64), rhi = __shfl(int(uint64_t(row) >> 32), c, 64);
    const int64_t r = int64_t((uint64_t(uint32_t(rhi)) << 32) | uint32_t(rlo));
    careful_pair<E, 256, 4>(P, b, kvh, r * P.D, s0 + __shfl(pos, c, 64), lane, d, min(d + 8, P.D));
  }
}

TiledParams tiled_params(const AttnArgs &a) {
  TiledParams P;
  P.q = a.q;
  P.k_cache = a.k_cache;
  P.v_cache = a.v_cache;
  P.seqlens = a.seqlens;
  P.rows = a.rows;
  P.cu = a.cu;
  P.out = a.out;
  P.T_new = int(a.t_new);
  P.H = int(a.n_head);
  P.H_kv = int(a.n_kv_head);
  P.G = int(a.n_head / a.n_kv_head);
  P.T_max = int(a.t_max);
  P.window = int(a.window < 0 ? -1 : a.window);
  P.D = int(a.head_dim);
  P.n_bh = int(a.batch * a.n_kv_head);
  P.n_qt = 0;
  P.deal = device_cus();
  P.cache_b = a.cache_batch_stride;
  P.scale_log2 = float(kLog2e / std::sqrt(double(a.head_dim)));
  P.split = SplitGeo{};
  P.split.n_split = 1;
  return P;
}


// What a call runs: the waves over pairs (KS = 1) or keys (KS = 4), and the key ranges.
struct TiledPlan {
  int ks;
  SplitPlan split;
};
TiledPlan tiled_plan(const AttnArgs &a) {
  const int64_t G = a.n_head / a.n_kv_head;
  const int64_t n_bh = a.batch * a.n_kv_head;
  const bool bf = a.dtype == MCAMD_BF16;
  TiledPlan t;
  SplitPlan &p = t.split;
  // Fewer workgroups of 128 pairs than compute units: 32 pairs and a quarter of the keys per wave
  // instead (12 heads of 64: 2 x 512 tokens fp32 33 against 50 us, bf16 15.0 against 18.6; 8 x 512,
  // 384 workgroups: 78 against 67 and 31.6 against 21.8). Head dims above 128 keep KS = 1 (a tile of four waves' keys outgrows the LDS).
  t.ks = a.head_dim <= 128 && (a.t_new * G + 127) / 128 * n_bh < device_cus() ? 4 : 1;
  p.pairs = 128 / t.ks;
  p.kt = t.ks == 4 ? 128 : bf && a.head_dim <= 128 ? 64 : 32;
  p.blocks = (a.t_new * G + p.pairs - 1) / p.pairs * n_bh;
  // Measured time of a tile on a compute unit of its own, per head dim. The chip counts as full at
  // one workgroup per compute unit: cutting 192 blocks in two gains on long prefixes (512 tokens of
  // 12 heads of 64 after 4096 keys, bf16: 52 against 63 us) what it loses on short ones (from
  // empty: 17 against 11.6).
  const float tile_us = float(a.head_dim) * (t.ks == 4 ? (bf ? 0.027f : 0.085f)
                                                       : (bf ? 0.012f : 0.035f));
  plan_splits(a, device_cus(), tile_us,
              a.window >= 0 ? std::min<int64_t>(a.t_max, a.window + 1 + (p.pairs + G - 1) / G)
                            : a.t_max, p);
  return t;
}

template <class E, int DP, int KS>
int run(TiledParams &P, const AttnArgs &a, const TiledPlan &plan) {
  using G_ = Geo<E, DP, KS>;
  if (plan.split.pairs != G_::PAIRS || plan.split.kt != G_::KT)
    return fail(MCAMD_EINVAL, "prefill: plan and kernel disagree");
  P.split = split_geo(a, plan.split);
  P.n_qt = P.split.n_qt;
  const int64_t blocks = plan.split.blocks * P.split.n_split;
  if (blocks > 0x7fffffff) return fail(MCAMD_EUNSUPPORTED, "prefill: grid too large");
  hipLaunchKernelGGL((prefill_tiled_kernel<E, DP, KS>), dim3(unsigned(blocks)), dim3(kThreads), 0,
                     a.stream, P);
  const int st = launch_status("prefill_tiled");
  if (st != MCAMD_OK || P.split.n_split == 1) return st;
  return launch_prefill_combine(a, P.split, true);
}

template <class E, int DP>
int run_ks(TiledParams &P, const AttnArgs &a, const TiledPlan &plan) {
  if constexpr (DP <= 128) {
    if (plan.ks == 4) return run<E, DP, 4>(P, a, plan);
  }
  return run<E, DP, 1>(P, a, plan);
}

template <class E>
int dispatch(TiledParams &P, const AttnArgs &a, const TiledPlan &plan) {
  if (P.D <= 32) return run_ks<E, 32>(P, a, plan);
  if (P.D <= 64) return run_ks<E, 64>(P, a, plan);
  if (P.D <= 96) return run_ks<E, 96>(P, a, plan);
  if (P.D <= 128) return run_ks<E, 128>(P, a, plan);
  if (P.D <= 192) return run_ks<E, 192>(P, a, plan);
  return run_ks<E, 256>(P, a, plan);
}

}  // namespace

int launch_prefill_combine(const AttnArgs &a, const SplitGeo &g, bool careful) {
  const TiledParams P = tiled_params(a);
  NewTokens N{a.k_new, a.v_new, 0, 0, 0};
  if (a.k_new) {
    N.tok = int(a.n_kv_head * a.head_dim * (a.dtype == MCAMD_BF16 ? 2 : 4) / 16);
    N.units = a.t_new * N.tok;
    N.blocks = int((N.units + kAppendUnits - 1) / kAppendUnits);
  }
  // A row's workgroups; calls are cut only while their blocks leave half the chip idle, so few.
  const int64_t blocks = 2 * int64_t(N.blocks) + int64_t(g.n_qt) * P.H_kv * g.groups * g.md;
  if (blocks >= (int64_t(1) << 32) / kMergeThreads)  // a grid's threads along x
    return fail(MCAMD_EUNSUPPORTED, "prefill: grid too large");
  const dim3 grid{unsigned(blocks), unsigned(a.batch)}, threads{kMergeThreads};
  if (a.dtype == MCAMD_BF16)
    hipLaunchKernelGGL(prefill_combine_kernel<bf16>, grid, threads, 0, a.stream, P, g, int(careful),
                       N);
  else
    hipLaunchKernelGGL(prefill_combine_kernel<float>, grid, threads, 0, a.stream, P, g, int(careful),
                       N);
  return launch_status("prefill_combine");
}

SplitPlan prefill_tiled_splits(const AttnArgs &a) { return tiled_plan(a).split; }

int launch_prefill_tiled(const AttnArgs &a) {
  TiledParams P = tiled_params(a);
  if (P.G > 64) return fail(MCAMD_EUNSUPPORTED, "prefill: more than 64 query heads per KV head");
  const TiledPlan plan = tiled_plan(a);
  if (plan.split.blocks > 0x7fffffff) return fail(MCAMD_EUNSUPPORTED, "prefill: grid too large");
  if (a.dtype == MCAMD_BF16) return dispatch<bf16>(P, a, plan);
  return dispatch<float>(P, a, plan);
}

}  // namespace mcamd
