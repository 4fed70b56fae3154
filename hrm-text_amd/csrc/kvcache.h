// KV-cache attention: the inference path of the reference's attention layer
// (flash_attn_with_kvcache at models/layers.py:147-151, driven by
// simple_inference_engine.py:105-112, :131, :179-180).
//
// Semantics (FlashAttention's documented kv-cache call, as the reference uses it):
// the new rows k, v [B, S, H, D] are written into the caches [B, Smax, H, D] at
// rows len_b .. len_b + S - 1 (len_b = cache_seqlens[b]); query i of batch row b
// then attends the lk = len_b + S cache keys (lk = len_b when no new rows are
// given), and with `causal` only keys j <= lk - S + i (bottom-right alignment). No
// segment structure: a cache row is one sequence.
//
// Kernels:
//   append  : copies the new k, v rows into the caches (rows past Smax are dropped), where the
//             kernels below do not (see P.fused);
//   decode  : one query per row, split-K over the keys. A workgroup = (b, h, split); each
//             16-lane group owns one key at a time (16 x 16-byte chunks of a 256-byte row),
//             four keys per step, with an online softmax in fp32; the 16 groups are merged
//             and the split writes (max, sum, o[D]) unnormalised to the workspace, or out
//             when it is the only one. HBM-bound: 2 * D * 2 bytes per key.
//   extend  : several queries per row (S >= 2): the same split-K on the matrix cores, every
//             staged key serving 32 QW queries (see the kernel);
//   combine : merges the splits of each (b, i, h) and writes bf16 out.
#pragma once
#include "common.h"

namespace prefixlm {
namespace kvc {

constexpr int D = 128;
constexpr int NT = 256;
constexpr int GROUPS = NT / 16;      // keys in flight per workgroup step (x kUnroll)
constexpr int kUnroll = 4;
constexpr int kStep = GROUPS * kUnroll;   // keys per step of a workgroup of NT threads
constexpr int kPart = D + 4;         // floats per partial: max (log2 units), sum, 2 unused, o[D]
static_assert(kPart % 4 == 0, "partials keep o 16-byte aligned");

struct Params {
  const bf16* q;
  const bf16* k;          // new rows (may be null)
  const bf16* v;
  bf16* kc;
  bf16* vc;
  bf16* out;
  float* part;            // [B, S, H, nsplit, kPart]
  const int32_t* seqlens; // device [B]; null: every row has seqlen_const
  int64_t q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, v_sb, v_ss, v_sh;
  int64_t kc_sb, kc_ss, kc_sh, vc_sb, vc_ss, vc_sh, o_sb, o_ss, o_sh;
  int B, S, H, Smax, nsplit, causal, seqlen_const;
  int s_new;              // rows appended by this call: S, or 0 without new k, v
  int fused;              // new rows are read from k, v and written to the caches by the same kernel
  int nqb;                // extend: query blocks of 32 QW rows
  float scale_log2;
};

__device__ __forceinline__ int cache_len(const Params& P, int b) {
  return P.seqlens ? P.seqlens[b] : P.seqlen_const;
}

// The keys that query i sees of a cache row of length len: [0, n)
__device__ __forceinline__ int keys_seen(const Params& P, int len, int i) {
  const int lk = min(P.Smax, len + P.s_new);
  return P.causal ? min(lk, len + P.s_new - P.S + i + 1) : lk;
}
// 1 / (sum of the weights) of a query that sees n keys. Without keys its row is 0; with keys whose
// scores are all -inf the sum is 0 and the row NaN, as softmax gives it.
__device__ __forceinline__ float row_inv(int n, float sum) { return n > 0 ? 1.f / sum : 0.f; }
// What exponents are taken against: a running max of -inf (no key yet, or only keys whose score is
// -inf) would turn exp2(-inf - max) into NaN where the weight is 0.
__device__ __forceinline__ float max_ref(float m) { return m == -INFINITY ? 0.f : m; }

// thread = 16-byte chunk of one (b, i, h) row of k and of v
__global__ __launch_bounds__(256) void append_kernel(Params P) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int c = (int)(gid & 15);
  const int64_t r = gid >> 4;
  if (r >= (int64_t)P.B * P.S * P.H) return;
  const int h = (int)(r % P.H);
  const int i = (int)((r / P.H) % P.S);
  const int b = (int)(r / ((int64_t)P.H * P.S));
  const int row = cache_len(P, b) + i;
  if (row < 0 || row >= P.Smax) return;
  const u32x4 kv = *reinterpret_cast<const u32x4*>(P.k + b * P.k_sb + i * P.k_ss + h * P.k_sh + 8 * c);
  const u32x4 vv = *reinterpret_cast<const u32x4*>(P.v + b * P.v_sb + i * P.v_ss + h * P.v_sh + 8 * c);
  *reinterpret_cast<u32x4*>(P.kc + b * P.kc_sb + row * P.kc_ss + h * P.kc_sh + 8 * c) = kv;
  *reinterpret_cast<u32x4*>(P.vc + b * P.vc_sb + row * P.vc_ss + h * P.vc_sh + 8 * c) = vv;
}

// 16 bytes of a cached row: read once per call, by one workgroup
__device__ __forceinline__ u32x4 load_once(const bf16* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

// One query per row (S = 1): blockIdx.x = ((b * H + h) * nsplit + split). The splits share
// each sequence's own length, in whole steps of 64 keys: all but the last with keys hold the
// same number, and those past the length none (4200 keys in 64 splits: 128 each in 33 of them). A
// ragged batch so has no sequence whose splits are all full beside one whose splits are mostly
// empty, as splits of fixed 512 keys had. Bound by HBM. The cache loads are non-temporal:
// a row is read once, and kept out of the caches it costs no write-back of what it would
// evict. 64 x 16 heads, 2100-4000 of 4096 rows (1.6 GB): 262 us with the combine, 6.1 TB/s,
// against 285 with plain loads and 322 for fixed 512-key splits, plain loads and an append
// launch. Loading the next 64 keys at the end of a step instead of at its start is worth 2%;
// doing it before the step's P V, or the heads as the fastest grid index, changes nothing.
// NTH = 512 for calls of one split and few workgroups, where a CU would hold four waves only and
// the walk is a chain of memory round trips: twice the keys per step (16 pairs x 256 keys 5.5 ->
// 4.9 us, 256 pairs x 512 13.6 -> 10.9).
template <int NTH>
__global__ __launch_bounds__(NTH) void decode_kernel(Params P) {
  constexpr int NWAVE = NTH / 64, GROUPS = NTH / 16, kStep = GROUPS * kUnroll;   // keys per workgroup step
  __shared__ float s_m[NWAVE], s_l[NWAVE];
  __shared__ f32x4 s_o[NWAVE][D / 4];
  const int split = blockIdx.x % P.nsplit;
  const int bh = blockIdx.x / P.nsplit;
  const int h = bh % P.H, b = bh / P.H;
  const int tid = threadIdx.x, grp = tid >> 4, g16 = tid & 15;
  const int len = cache_len(P, b);
  // keys read from the cache; with P.fused the new row is not one of them
  const int lk = min(P.Smax, len + (P.fused ? 0 : P.s_new));
  const int per = ((lk + P.nsplit - 1) / P.nsplit + kStep - 1) / kStep * kStep;
  const int k0 = split * per, k1 = min(lk, k0 + per);
  const bf16* kbase = P.kc + b * P.kc_sb + h * P.kc_sh + 8 * g16;
  const bf16* vbase = P.vc + b * P.vc_sb + h * P.vc_sh + 8 * g16;
  u32x4 kw[kUnroll], vw[kUnroll];
  auto load = [&](int j0) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int j = min(j0 + u * GROUPS, k1 - 1);   // clamped rows are masked below
      kw[u] = load_once(kbase + j * P.kc_ss);
      vw[u] = load_once(vbase + j * P.vc_ss);
    }
  };
  if (k0 + grp < k1) load(k0 + grp);
  float q[8];
  {
    const u32x4 w = *reinterpret_cast<const u32x4*>(P.q + b * P.q_sb + h * P.q_sh + 8 * g16);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      q[2 * e] = bf16lo(w[e]) * P.scale_log2;
      q[2 * e + 1] = bf16hi(w[e]) * P.scale_log2;
    }
  }
  auto dot = [&](const u32x4& k) {
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) d += q[2 * e] * bf16lo(k[e]) + q[2 * e + 1] * bf16hi(k[e]);
    return row16_sum(d);
  };
  float m = -INFINITY, l = 0.f, o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  if (P.fused && split == 0 && grp == 0 && len >= 0 && len < P.Smax) {
    // the new row, key len: into the caches, and the first key of this group
    const u32x4 kn = *reinterpret_cast<const u32x4*>(P.k + b * P.k_sb + h * P.k_sh + 8 * g16);
    const u32x4 vn = *reinterpret_cast<const u32x4*>(P.v + b * P.v_sb + h * P.v_sh + 8 * g16);
    *reinterpret_cast<u32x4*>(P.kc + b * P.kc_sb + h * P.kc_sh + len * P.kc_ss + 8 * g16) = kn;
    *reinterpret_cast<u32x4*>(P.vc + b * P.vc_sb + h * P.vc_sh + len * P.vc_ss + 8 * g16) = vn;
    m = dot(kn);
    l = __builtin_amdgcn_exp2f(m - max_ref(m));   // 1, or 0 for a score of -inf
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[2 * e] = l * bf16lo(vn[e]);
      o[2 * e + 1] = l * bf16hi(vn[e]);
    }
  }
  for (int j0 = k0 + grp; j0 < k1; j0 += kStep) {
    float s[kUnroll], mx = m;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      s[u] = (j0 + u * GROUPS < k1) ? dot(kw[u]) : -INFINITY;
      mx = fmaxf(mx, s[u]);
    }
    const float ref = max_ref(mx), alpha = __builtin_amdgcn_exp2f(m - ref);   // m = -inf at first: 0
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= alpha;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const float p = __builtin_amdgcn_exp2f(s[u] - ref);
      l += p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] += p * bf16lo(vw[u][e]);
        o[2 * e + 1] += p * bf16hi(vw[u][e]);
      }
    }
    m = mx;
    if (j0 + kStep < k1) load(j0 + kStep);
  }
  // merge the wave's four groups, then the four waves
  float M = fmaxf(m, __shfl_xor(m, 16));
  M = fmaxf(M, __shfl_xor(M, 32));
  const float a = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
  l *= a;
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    o[e] *= a;
    o[e] += __shfl_xor(o[e], 16);
    o[e] += __shfl_xor(o[e], 32);
  }
  const int w = tid >> 6;
  if ((tid & 63) < 16) {
    if (g16 == 0) {
      s_m[w] = M;
      s_l[w] = l;
    }
    s_o[w][2 * g16] = f32x4{o[0], o[1], o[2], o[3]};
    s_o[w][2 * g16 + 1] = f32x4{o[4], o[5], o[6], o[7]};
  }
  __syncthreads();
  if (tid < D / 4) {
    M = s_m[0];
#pragma unroll
    for (int g = 1; g < NWAVE; ++g) M = fmaxf(M, s_m[g]);
    float L = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < NWAVE; ++g) {
      const float wgt = s_m[g] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[g] - M);
      L += wgt * s_l[g];
      acc += wgt * s_o[g][tid];
    }
    if (P.nsplit == 1) {
      const float inv = row_inv(keys_seen(P, len, 0), L);
      *reinterpret_cast<bf16x4*>(P.out + b * P.o_sb + h * P.o_sh + 4 * tid) =
          cvt4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
      return;
    }
    float* dst = P.part + (((int64_t)b * P.H + h) * P.nsplit + split) * kPart;
    if (tid == 0) {
      dst[0] = M;
      dst[1] = L;
    }
    *reinterpret_cast<f32x4*>(dst + 4 + 4 * tid) = acc;   // kPart keeps o 16-byte aligned
  }
}

// ---- several queries per row ---------------------------------------------------------
// Workgroup = (b, h, 32 QW queries, split of the keys); 4 waves, QW along the queries and
// KW = 4 / QW along the keys: a staged tile holds 32 KW keys, wave (qw, kw) multiplies its
// 32 queries with 32 of them, and the KW partial results meet in LDS at the end. QW = 1, 2,
// 4 for S <= 32, <= 64 and above, so that a short turn still keeps four waves busy and each
// cached row is read once per 32 QW queries.
//
// Same data flow as the varlen forward (fwd.h): S^T = K Q^T with the query as the lane
// column, Q in registers, K and V staged row-major (304-byte rows, V's permuted), V^T from
// transposing reads, O^T in four 32x32 tiles. The probabilities go into P V as three bf16
// terms, the upper 8 bits of what the terms before leave, which add up to the 24 bits of the
// fp32 value: the product keeps the bits of a walk in fp32. Two terms (16 bits) are 2% faster
// on the whole and up to 14% where several hundred queries meet long caches (16 x 16 heads x 200
// queries on 3700 rows 266 us, 300 with three), but leave 2e-6 of cancelling sums.
//
// Bound by HBM (512 bytes per key and query block) up to about 64 queries, by the MFMA ->
// softmax -> MFMA chain above. Measured against the walk of the queries one after another that
// this replaces (each query read all keys again): 4 x 16 heads x 45 queries on 4096-row half
// full caches 658 -> 28 us with the combine; 16 x 16 x 512 queries on 7000 of 8192 rows 1.11 ms (437
// TFLOP/s useful). Two workgroups per CU: at three (168 VGPRs) the 128-query form spills, a fifth
// slower.
//
// New rows (keys len .. len + S - 1) are read from k, v, and every workgroup copies its
// share of them into the caches: nothing in the launch reads those cache rows, so no
// launch has to come before it (P.fused = 0: they are in the caches already).
constexpr int kMaxSplits = 64;

template <int QW>
struct ExtGeo {
  static constexpr int KW = 4 / QW;
  static constexpr int TK = 32 * KW;             // keys per staged tile
  static constexpr int NBUF = QW == 1 ? 1 : 2;
  static constexpr int TILE = TK * RS;
  static constexpr int BUF = 2 * TILE;           // K tile, V tile
  static constexpr int LDS_BYTES = NBUF * BUF;   // 76, 76 and 38 KB: two workgroups per CU, or more
  static constexpr int MERGE = 64 * 64 * 4 + 2 * 64 * 4;   // one wave's O, max and sum
  static_assert((4 - QW) * MERGE <= LDS_BYTES && QW * OUT_WAVE_BYTES <= LDS_BYTES, "epilogue areas fit");
};

// the larger of m and the magnitudes of 8 bf16 (as 4 words), as 16-bit integers per half
__device__ __forceinline__ u16x2 max_mag(u16x2 m, const u32x4& w) {
#pragma unroll
  for (int e = 0; e < 4; ++e) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w[e] & 0x7fff7fffu));
  return m;
}

// Queries [q0, q1) over keys [k0, k1) without the matrix cores: a 16-lane group per query,
// key by key. For blocks whose values hold an infinity or NaN: in P V on the matrix cores
// 0 * inf would reach queries that must not see the key; here a query touches only the keys it
// sees. And for blocks with such a score: the matrix cores sum q k before the softmax scale, and
// that sum can pass fp32's range (keys of the type's lowest value) where the scaled one here does
// not.
template <class KMax, class KRow, class VRow>
__device__ __forceinline__ void extend_block_valu(const Params& P, int b, int h, int split, int q0, int q1, int k0,
                                                  int k1, KMax kmax, KRow k_row, VRow v_row) {
  const int g16 = threadIdx.x & 15;
#pragma unroll 1
  for (int i = q0 + (threadIdx.x >> 4); i < q1; i += GROUPS) {
    float q[8], o[8];
    const u32x4 qv = *reinterpret_cast<const u32x4*>(P.q + b * P.q_sb + i * P.q_ss + h * P.q_sh + 8 * g16);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      q[2 * e] = bf16lo(qv[e]) * P.scale_log2;
      q[2 * e + 1] = bf16hi(qv[e]) * P.scale_log2;
      o[2 * e] = o[2 * e + 1] = 0.f;
    }
    float m = -INFINITY, l = 0.f;
#pragma unroll 1
    for (int j = k0; j < min(k1, kmax(i)); ++j) {
      const u32x4 kv = *reinterpret_cast<const u32x4*>(k_row(j) + 8 * g16);
      const u32x4 vv = *reinterpret_cast<const u32x4*>(v_row(j) + 8 * g16);
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) s += q[2 * e] * bf16lo(kv[e]) + q[2 * e + 1] * bf16hi(kv[e]);
      s = row16_sum(s);
      const float mx = fmaxf(m, s), ref = max_ref(mx);
      const float alpha = __builtin_amdgcn_exp2f(m - ref), p = __builtin_amdgcn_exp2f(s - ref);
      m = mx;
      l = l * alpha + p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] = o[2 * e] * alpha + p * bf16lo(vv[e]);
        o[2 * e + 1] = o[2 * e + 1] * alpha + p * bf16hi(vv[e]);
      }
    }
    if (P.nsplit == 1) {
      const float inv = row_inv(kmax(i), l);
      *reinterpret_cast<bf16x8*>(P.out + b * P.o_sb + i * P.o_ss + h * P.o_sh + 8 * g16) =
          cvt8(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv, o[4] * inv, o[5] * inv, o[6] * inv, o[7] * inv);
    } else {
      float* dst = P.part + ((((int64_t)b * P.S + i) * P.H + h) * P.nsplit + split) * kPart;
      if (g16 == 0) *reinterpret_cast<f32x4*>(dst) = f32x4{m, l, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(dst + 4 + 8 * g16) = f32x4{o[0], o[1], o[2], o[3]};
      *reinterpret_cast<f32x4*>(dst + 8 + 8 * g16) = f32x4{o[4], o[5], o[6], o[7]};
    }
  }
}

template <int QW>
__global__ __launch_bounds__(NT, 2) void extend_kernel(Params P) {
  using G = ExtGeo<QW>;
  constexpr int KW = G::KW, TK = G::TK, TILE = G::TILE, NS = D / 16, NP = TK / 16;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int bad;   // some value row holds an infinity or NaN, or some score is one

  // unit u = (b, h, split); its query blocks sit 8 grid indices apart, on one XCD
  const int qb = (blockIdx.x >> 3) % P.nqb;
  const int u = (int)((blockIdx.x >> 3) / P.nqb) * 8 + (blockIdx.x & 7);
  if (u >= P.B * P.H * P.nsplit) return;
  const int split = u % P.nsplit, bh = u / P.nsplit;
  const int h = bh % P.H, b = bh / P.H;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = w % QW, kw = w / QW;
  const int len = cache_len(P, b);
  const int lk = min(P.Smax, len + P.s_new);      // keys in the cache after the append
  const int q0 = qb * 32 * QW;
  // query i sees keys [0, kmax(i))
  auto kmax = [&](int i) { return keys_seen(P, len, i); };
  const int per = ((lk + P.nsplit - 1) / P.nsplit + TK - 1) / TK * TK;   // keys per split, whole tiles
  const int k0 = split * per;
  const int k1 = min(kmax(min(P.S, q0 + 32 * QW) - 1), k0 + per);
  const int kall = kmax(q0);                      // keys below are seen by every query of the block
  const int qrow = q0 + 32 * qw + l32;            // this lane's query
  const bool active = q0 + 32 * qw < P.S;
  const int kq = min(k1, kmax(min(qrow, P.S - 1)));
  const int kend_w = active ? min(k1, kmax(min(P.S, q0 + 32 * qw + 32) - 1)) : 0;

  // row j of the keys or the values: cached, or one of the new rows
  const int n_old = P.fused ? len : 0x7fffffff;
  const bf16* const kc = P.kc + b * P.kc_sb + h * P.kc_sh;
  const bf16* const vc = P.vc + b * P.vc_sb + h * P.vc_sh;
  const bf16* const kn = P.fused ? P.k + b * P.k_sb + h * P.k_sh : nullptr;
  const bf16* const vn = P.fused ? P.v + b * P.v_sb + h * P.v_sh : nullptr;
  auto k_row = [&](int j) { return j < n_old ? kc + j * P.kc_ss : kn + (j - len) * P.k_ss; };
  auto v_row = [&](int j) { return j < n_old ? vc + j * P.vc_ss : vn + (j - len) * P.v_ss; };

  // this workgroup's share of the new rows goes into the caches (rows outside them are dropped)
  auto append_share = [&]() {
    if (!P.fused) return;
    const int parts = P.nqb * P.nsplit, part = qb * P.nsplit + split;
    for (int i = part + parts * (tid >> 5); i < P.S; i += parts * (NT / 32)) {
      const int row = len + i, c = 8 * (tid & 15);
      if (row < 0 || row >= P.Smax) continue;
      if (tid & 16)
        *reinterpret_cast<u32x4*>(P.vc + b * P.vc_sb + h * P.vc_sh + row * P.vc_ss + c) =
            *reinterpret_cast<const u32x4*>(vn + i * P.v_ss + c);
      else
        *reinterpret_cast<u32x4*>(P.kc + b * P.kc_sb + h * P.kc_sh + row * P.kc_ss + c) =
            *reinterpret_cast<const u32x4*>(kn + i * P.k_ss + c);
    }
  };

  // staging: thread = 16-byte chunk sch of rows srow + 16 r; V rows in permuted order
  const int srow = tid >> 4, sch = tid & 15, vrow = perm_row(srow);
  u32x4 ks[NP], vs[NP];
  const u32x4 zero = {0u, 0u, 0u, 0u};
  // tiles of cached rows (all but the last ones) through buffer loads off a uniform base:
  // 32-bit lane offsets, and rows from k1 on read as zero
  const bool small = P.kc_ss < (1 << 22) && P.vc_ss < (1 << 22);
  const uint32_t koff = (uint32_t)srow * (uint32_t)P.kc_ss * 2 + 16 * sch, koff16 = (uint32_t)P.kc_ss * 32;
  const uint32_t voff = (uint32_t)vrow * (uint32_t)P.vc_ss * 2 + 16 * sch, voff16 = (uint32_t)P.vc_ss * 32;
  auto load_kv = [&](int t0) {
    const int n = min(TK, k1 - t0);
    if (small && t0 + n <= n_old) {
      const __amdgpu_buffer_rsrc_t kr = make_rsrc(kc + t0 * P.kc_ss, rows_bytes(n, P.kc_ss, D));
      const __amdgpu_buffer_rsrc_t vr = make_rsrc(vc + t0 * P.vc_ss, rows_bytes(n, P.vc_ss, D));
#pragma unroll
      for (int r = 0; r < NP; ++r) {
        ks[r] = buf_load16(kr, koff + r * koff16);
        vs[r] = buf_load16(vr, voff + r * voff16);
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < NP; ++r) {
      const int jk = t0 + 16 * r + srow, jv = t0 + 16 * r + vrow;
      ks[r] = jk < k1 ? *reinterpret_cast<const u32x4*>(k_row(jk) + 8 * sch) : zero;
      vs[r] = jv < k1 ? *reinterpret_cast<const u32x4*>(v_row(jv) + 8 * sch) : zero;
    }
  };
  auto store_kv = [&](int buf) {
    char* base = smem + buf * G::BUF + srow * RS + sch * 16;
#pragma unroll
    for (int r = 0; r < NP; ++r) {
      *reinterpret_cast<u32x4*>(base + 16 * r * RS) = ks[r];
      *reinterpret_cast<u32x4*>(base + TILE + 16 * r * RS) = vs[r];
    }
    u16x2 m = {0, 0};
#pragma unroll
    for (int r = 0; r < NP; ++r) m = max_mag(m, vs[r]);
    if (m[0] >= 0x7f80 || m[1] >= 0x7f80) bad = 1;
  };

  float m_run = -INFINITY, l_run = 0.f;
  f32x16 oacc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[t][r] = 0.f;

  if (k0 < k1) {
    const int nt = (k1 - k0 + TK - 1) / TK;
    load_kv(k0);
    // Q^T fragments: lane holds query qrow, d = 16 s + 8 hh + 0..7 (rows past S: the last one, not stored)
    bf16x8 qf[NS];
    {
      const bf16* qp = P.q + b * P.q_sb + h * P.q_sh + min(qrow, P.S - 1) * P.q_ss + 8 * hh;
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
    }
    if (tid == 0) bad = 0;
    __syncthreads();
    store_kv(0);
#pragma unroll
    for (int s = 0; s < NS; ++s) settle(__builtin_bit_cast(u32x4, qf[s]));
    __syncthreads();
    const float c = P.scale_log2;
    for (int t = 0; t < nt; ++t) {
      const int buf = G::NBUF == 2 ? t & 1 : 0;
      load_kv(k0 + (t + 1) * TK);
      const int kk = k0 + t * TK + 32 * kw;   // first key of this wave's 32
      if (kk < kend_w) {
        const char* kt = smem + buf * G::BUF + (32 * kw + l32) * RS + hh * 16;
        const char* vt = smem + buf * G::BUF + TILE + 32 * kw * RS + xt_lane_off(lane);
        f32x16 sacc;
#pragma unroll
        for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
        bf16x8 ka[NS];
        ka[0] = *reinterpret_cast<const bf16x8*>(kt);
        ka[1] = *reinterpret_cast<const bf16x8*>(kt + 32);
#pragma unroll
        for (int s = 0; s < NS; ++s) {   // operands two steps ahead
          if (s + 2 < NS) ka[s + 2] = *reinterpret_cast<const bf16x8*>(kt + 32 * (s + 2));
          sched_fence();
          sacc = mfma32x32x16(ka[s], qf[s], sacc);
          sched_fence();
        }
        // key kk + 8 (r / 4) + 4 hh + r % 4 is seen iff it is below kq
        const int tk = kq - kk - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r) sacc[r] *= c;   // before the mask: the scale may have any sign
        if (kk + 32 > min(kall, k1)) {
#pragma unroll
          for (int r = 0; r < 16; ++r) sacc[r] = (8 * (r >> 2) + (r & 3) < tk) ? sacc[r] : -INFINITY;
        }
        float mx = sacc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sacc[r]);
        mx = halves_max(mx);
        if (__builtin_amdgcn_ballot_w64(mx > m_run) != 0) {
          const float m_new = fmaxf(m_run, mx);
          const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
          m_run = m_new;
          l_run *= alpha;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
        }
        const float m_use = max_ref(m_run);
        u32x4 xt[8];
        xt[0] = lds_read_xt(vt, 0, 0);
        xt[1] = lds_read_xt(vt, 0, 1);
        // 16 keys at a time: P's three terms (n = 0 first), times V
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          float e[8], ps = 0.f;
          bf16x8 pt[3];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            e[i] = __builtin_amdgcn_exp2f(sacc[8 * half + i] - m_use);
            ps += e[i];
          }
          l_run += ps;
#pragma unroll
          for (int n = 0; n < 3; ++n) {
            u32x4 w;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              w[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, e[2 * i + 1]),
                                           __builtin_bit_cast(uint32_t, e[2 * i]), 0x07060302u);
            pt[n] = __builtin_bit_cast(bf16x8, w);
#pragma unroll
            for (int i = 0; i < 8; ++i)   // exact
              e[i] -= __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, e[i]) & 0xffff0000u);
          }
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            const int x = 4 * half + dt;
            if (x + 2 < 8) xt[x + 2] = lds_read_xt(vt, (x + 2) / 4, (x + 2) % 4);
#pragma unroll
            for (int n = 0; n < 3; ++n) oacc[dt] = mfma32x32x16(__builtin_bit_cast(bf16x8, xt[x]), pt[n], oacc[dt]);
          }
        }
      }
      if (G::NBUF == 1) __syncthreads();
      if (t + 1 < nt) store_kv(G::NBUF == 2 ? buf ^ 1 : 0);
      __syncthreads();
    }
    l_run = halves_sum(l_run);
    // the KW waves of one query block: waves kw > 0 hand theirs to wave kw = 0
    if (KW > 1) {
      if (kw > 0) {
        float* area = reinterpret_cast<float*>(smem + (w - QW) * G::MERGE);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int m = 0; m < 4; ++m)
            *reinterpret_cast<f32x4*>(area + ((4 * dt + m) * 64 + lane) * 4) =
                f32x4{oacc[dt][4 * m], oacc[dt][4 * m + 1], oacc[dt][4 * m + 2], oacc[dt][4 * m + 3]};
        area[64 * 64 + lane] = m_run;
        area[65 * 64 + lane] = l_run;
      }
      __syncthreads();
      if (kw == 0) {
        float mo[KW], M = m_run;
#pragma unroll
        for (int g = 1; g < KW; ++g) {
          mo[g] = reinterpret_cast<const float*>(smem + (g * QW + qw - QW) * G::MERGE)[64 * 64 + lane];
          M = fmaxf(M, mo[g]);
        }
        mo[0] = m_run;
        m_run = M;
        float L = 0.f;
#pragma unroll
        for (int g = 0; g < KW; ++g) {
          const float* area = reinterpret_cast<const float*>(smem + (g * QW + qw - QW) * G::MERGE);
          const float wgt = mo[g] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mo[g] - M);
          L += wgt * (g == 0 ? l_run : area[65 * 64 + lane]);
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              if (g == 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) oacc[dt][4 * m + e] *= wgt;
              } else {
                const f32x4 x = *reinterpret_cast<const f32x4*>(area + ((4 * dt + m) * 64 + lane) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) oacc[dt][4 * m + e] += wgt * x[e];
              }
            }
        }
        l_run = L;
      }
    }
    // a score past the range upwards leaves NaN; one past it downwards (raw below -3.4e38) only
    // counts where every key that the query sees here scores about as low
    if (kw == 0 && active && min(k1, kmax(min(qrow, P.S - 1))) > k0 &&
        (l_run != l_run || m_run < 200.f - 3e38f * fabsf(P.scale_log2)))
      bad = 1;
    __syncthreads();
    if (bad) {
      extend_block_valu(P, b, h, split, q0, min(P.S, q0 + 32 * QW), k0, k1, kmax, k_row, v_row);
      append_share();
      return;
    }
  }
  if (kw == 0 && active) {
    if (P.nsplit == 1) {
      // whole rows through LDS
      const float inv = row_inv(kmax(min(qrow, P.S - 1)), l_run);
      char* wl = smem + qw * OUT_WAVE_BYTES;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          *reinterpret_cast<bf16x4*>(wl + l32 * OUT_RS + (32 * dt + 8 * m + 4 * hh) * 2) =
              cvt4(oacc[dt][4 * m] * inv, oacc[dt][4 * m + 1] * inv, oacc[dt][4 * m + 2] * inv,
                   oacc[dt][4 * m + 3] * inv);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int row = (lane >> 4) + 4 * r, i = q0 + 32 * qw + row;
        const u32x4 v = *reinterpret_cast<const u32x4*>(wl + row * OUT_RS + (lane & 15) * 16);
        if (i < P.S) *reinterpret_cast<u32x4*>(P.out + b * P.o_sb + i * P.o_ss + h * P.o_sh + 8 * (lane & 15)) = v;
      }
    } else if (qrow < P.S) {
      float* dst = P.part + ((((int64_t)b * P.S + qrow) * P.H + h) * P.nsplit + split) * kPart;
      if (hh == 0) *reinterpret_cast<f32x4*>(dst) = f32x4{m_run, l_run, 0.f, 0.f};
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          *reinterpret_cast<f32x4*>(dst + 4 + 32 * dt + 8 * m + 4 * hh) =
              f32x4{oacc[dt][4 * m], oacc[dt][4 * m + 1], oacc[dt][4 * m + 2], oacc[dt][4 * m + 3]};
    }
  }
  append_share();
}

// One wave per (b, i, h). Lane s weighs split s (its max and sum read by all lanes at
// once); then each half-wave adds every other split's o, lane % 32 holding four of the 128
// columns. Bound by memory latency: with a serial walk over the splits, which paid a round
// trip each, 12.9 us for 1024 rows x 8 splits and 7.0 us for 16 rows x 23; now 5.0 and 4.2.
__global__ __launch_bounds__(256) void combine_kernel(Params P) {
  const int64_t w = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (w >= (int64_t)P.B * P.S * P.H) return;
  const int h = (int)(w % P.H);
  const int i = (int)((w / P.H) % P.S);
  const int b = (int)(w / ((int64_t)P.H * P.S));
  const float* src = P.part + w * P.nsplit * kPart;
  float M = -INFINITY;
  for (int s = lane; s < P.nsplit; s += 64) M = fmaxf(M, src[s * kPart]);
  M = wave_max(M);
  float L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < P.nsplit; s0 += 64) {
    const int n = min(64, P.nsplit - s0);
    const float* sp = src + s0 * kPart;
    float wgt = 0.f;
    if (lane < n && sp[lane * kPart] != -INFINITY) {
      wgt = __builtin_amdgcn_exp2f(sp[lane * kPart] - M);
      L += wgt * sp[lane * kPart + 1];
    }
    for (int sb = 0; sb < n; sb += 16) {
      const int s1 = sb + (lane >> 5);
      // eight loads in flight; past the last split its partial again, not added (it may be inf)
      f32x4 o[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        o[u] = *reinterpret_cast<const f32x4*>(sp + min(s1 + 2 * u, n - 1) * kPart + 4 + 4 * (lane & 31));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const f32x4 x = acc + __shfl(wgt, s1 + 2 * u) * o[u];
        acc = s1 + 2 * u < n ? x : acc;
      }
    }
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) L += __shfl_xor(L, m);
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] += wave_xor32(acc[e]);
  const float inv = row_inv(keys_seen(P, cache_len(P, b), i), L);
  if (lane < 32)
    *reinterpret_cast<bf16x4*>(P.out + b * P.o_sb + i * P.o_ss + h * P.o_sh + 4 * lane) =
        cvt4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
}

}  // namespace kvc
}  // namespace prefixlm
