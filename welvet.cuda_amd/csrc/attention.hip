// MHA ModeSelf attention core with the reference's indexing
// (src/cuda/kernels.cu:470-631):
//   token t = b*seq + s sits at global position pos = t;
//   queries of batch b see key positions k_pos in [0, b*seq + seq) allowed by
//   the mask (:470-485), scored against the KV ring row k_pos % msl, which by
//   then holds the latest position p <= last = b*seq + seq - 1 with
//   p == k_pos (mod msl): p = last - ((last - k_pos) mod msl);
//   RoPE rotates Q and K at their global position (:487-504), ALiBi uses
//   k_pos (:526-533); softmax or sigmoid over the allowed keys (:603-619).
// The reference loop is serial f64 on one thread. Here head dims 32, 64 and
// 128 run on the matrix cores (k_attn_mfma, below) for every mask; the other
// head dims, and ALiBi under the sigmoid, take k_attention, where one wave
// handles one (token, head), keys are scored 64 at a time (one per lane), and
// the softmax is accumulated online in fp32. RoPE is applied by the Q and K
// projections' GEMM epilogue when they run on the large tiles, else by
// k_rope before either kernel.
#include "bf16.h"
#include "common.h"
#include "kernels.h"
#include "split.h"

namespace wv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool allow(int qp, int kp, const AttnArgs& a) {
  if (a.mask == 2) return true;
  if (a.mask == 3) {
    const int w = a.window > 0 ? a.window : a.msl;
    if (a.window_causal) return kp <= qp && kp >= qp - w + 1;
    const int d = qp > kp ? qp - kp : kp - qp;
    return d < w;
  }
  if (a.mask == 4) {
    if (qp < a.prefix_len && kp < a.prefix_len) return true;
    return kp <= qp;
  }
  return kp <= qp;
}

__device__ __forceinline__ double rope_angle(int t, int d, int hd, double theta) {
  return (double)t / pow(theta, (double)(2 * d) / (double)hd);
}

__global__ void k_rope_table(double* __restrict__ tab, int tokens, int hd, double theta) {
  const int half = hd / 2;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= tokens * half) return;
  const double ang = rope_angle(i / half, i % half, hd, theta);
  tab[2 * i] = cos(ang);
  tab[2 * i + 1] = sin(ang);
}

// Rotates the pair (d, d + hd/2) of every head of Q (num_heads) and K
// (num_kv) rows of token t by angle t / theta^(2d/hd), in f64 (cos and sin
// from the table when one is given).
__global__ void k_rope(float* __restrict__ q, float* __restrict__ k, int tokens, int heads,
                       int kv_heads, int hd, int q_stride, int kv_stride, double theta,
                       const double* __restrict__ tab) {
  const int t = blockIdx.x;
  const int half = hd / 2;
  const int per_tok = (heads + kv_heads) * half;
  for (int i = threadIdx.x; i < per_tok; i += blockDim.x) {
    const int h = i / half, d = i % half;
    float* row = h < heads ? q + (size_t)t * q_stride + (size_t)h * hd
                           : k + (size_t)t * kv_stride + (size_t)(h - heads) * hd;
    double c, s;
    if (tab) {
      c = tab[2 * (t * half + d)];
      s = tab[2 * (t * half + d) + 1];
    } else {
      const double ang = rope_angle(t, d, hd, theta);
      c = cos(ang), s = sin(ang);
    }
    const double a0 = row[d], a1 = row[d + half];
    row[d] = (float)(a0 * c - a1 * s);
    row[d + half] = (float)(a0 * s + a1 * c);
  }
}

constexpr int kMaxHdPerLane = 4;  // head_dim <= 256

// Attention of query token t, head h by one wave: keys scored 64 at a time
// (one per lane) against their ring rows, online softmax in fp32. qs: the
// query's hd values. Lane l ends with output dims l + 64 i in acc[i].
__device__ __forceinline__ void attend_token(const AttnArgs& a, int t, int h, int lane,
                                             const float* qs, float (&acc)[kMaxHdPerLane]) {
  const int b = t / a.seq;
  const int qp = t;
  const int kv_len = b * a.seq + a.seq;
  const int last = kv_len - 1;
  const int kvh = h / (a.heads / a.kv_heads);
  const int kvd = a.kv_stride;

  float m = -INFINITY, l = 0.0f;
#pragma unroll
  for (int i = 0; i < kMaxHdPerLane; ++i) acc[i] = 0.0f;
  int n_allowed = 0;

  double slope = 0.0;
  if (a.alibi) slope = pow(2.0, -(double)(h + 1) * 8.0 / (double)(a.heads > 0 ? a.heads : 1));

  for (int base = 0; base < kv_len; base += 64) {
    const int kp = base + lane;
    bool ok = kp < kv_len && allow(qp, kp, a);
    int p = 0;
    float s = -INFINITY;
    if (ok) {
      p = last - ((last - kp) % a.msl);
      const float* kr = a.k + (size_t)p * kvd + (size_t)kvh * a.hd;
      float dot = 0.0f;
      for (int d = 0; d < a.hd; d += 4) {
        const float4 kk = *reinterpret_cast<const float4*>(kr + d);
        dot = fmaf(qs[d], kk.x, dot);
        dot = fmaf(qs[d + 1], kk.y, dot);
        dot = fmaf(qs[d + 2], kk.z, dot);
        dot = fmaf(qs[d + 3], kk.w, dot);
      }
      double sc = (double)dot * a.scale;
      if (a.alibi) {
        const int dd = qp > kp ? qp - kp : kp - qp;
        sc += -slope * (double)dd;
      }
      s = (float)sc;
    }
    const unsigned long long mask_bits = __ballot(ok);
    n_allowed += __popcll(mask_bits);
    if (mask_bits == 0ull) continue;
    float w;
    if (a.sigmoid) {
      w = ok ? 1.0f / (1.0f + expf(-s)) : 0.0f;
    } else {
      float bm = s;
      for (int off = 32; off > 0; off >>= 1) bm = fmaxf(bm, __shfl_xor(bm, off, 64));
      const float nm = fmaxf(m, bm);
      const float corr = (m == -INFINITY) ? 0.0f : expf(m - nm);
      w = ok ? expf(s - nm) : 0.0f;
      float ws = w;
      for (int off = 32; off > 0; off >>= 1) ws += __shfl_xor(ws, off, 64);
      l = l * corr + ws;
#pragma unroll
      for (int i = 0; i < kMaxHdPerLane; ++i) acc[i] *= corr;
      m = nm;
    }
    // acc[d] += sum_j w_j V[p_j][d]; lane owns dims lane, lane+64, ...
    for (int j = 0; j < 64; ++j) {
      const float wj = __shfl(w, j, 64);
      if (((mask_bits >> j) & 1ull) == 0ull) continue;
      const int pj = __shfl(p, j, 64);
      const float* vr = a.v + (size_t)pj * kvd + (size_t)kvh * a.hd;
#pragma unroll
      for (int i = 0; i < kMaxHdPerLane; ++i) {
        const int d = lane + 64 * i;
        if (d < a.hd) acc[i] = fmaf(wj, vr[d], acc[i]);
      }
    }
  }
  const float inv = (a.sigmoid || n_allowed == 0) ? 1.0f : 1.0f / l;
#pragma unroll
  for (int i = 0; i < kMaxHdPerLane; ++i) acc[i] = n_allowed == 0 ? 0.0f : acc[i] * inv;
}

__global__ __launch_bounds__(64) void k_attention(AttnArgs a) {
  const int t = blockIdx.x;  // query token
  const int h = blockIdx.y;  // query head
  const int lane = threadIdx.x;
  const size_t row = (size_t)t * a.heads * a.hd + (size_t)h * a.hd;
  __shared__ float qs[256];
  for (int d = lane; d < a.hd; d += 64) qs[d] = a.q[(size_t)t * a.q_stride + (size_t)h * a.hd + d];
  __syncthreads();
  float acc[kMaxHdPerLane];
  attend_token(a, t, h, lane, qs, acc);
  float* out = a.out + row;
#pragma unroll
  for (int i = 0; i < kMaxHdPerLane; ++i) {
    const int d = lane + 64 * i;
    if (d < a.hd) out[d] = acc[i];
  }
}


// ---------------------------------------------------------------------------
// Matrix-core path. The plain form (causal and bidirectional masks without
// ALiBi) first; GEN, below, takes the other masks and ALiBi.
//
// Under the reference indexing a query of batch b scans key positions
// kp in [0, b*seq + seq), and kp reads ring row p = last - ((last - kp) mod
// msl), so only the rows p in [max(0, last - msl + 1), last] occur, row p
// once for every allowed kp == p (mod msl). The score of a key depends on
// its row only (no ALiBi), so the softmax over key positions equals a
// softmax over distinct rows with multiplicity weights:
//   bidirectional: c(p) = floor(p / msl) + 1 (every kp = p - i*msl >= 0),
//   causal:        c(p) - 1 when p > qp (only kp = p itself is masked out:
//                  p - msl <= last - msl < b*seq <= qp since msl >= seq).
// Scores and sums are the same function of the same values; only the fp32
// summation order differs from the per-position loop.
//
// A workgroup of 16, 8 or 4 waves (attn_waves_of) takes 16 queries per wave of
// one (batch, head) and walks the distinct rows in tiles of 64 (or 32) keys staged
// in LDS in matrix-core operand order, double-buffered through registers, one
// barrier per tile. Per 16-key block a wave runs
//   S^T = K Q^T  on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16, hd/32
//                steps), Q and K each split into two bf16 terms hi + lo
//                (x - hi - lo ~ 2^-17 |x|), and the three products down to
//                2^-16 relative kept (hh, hl, lh): the scores carry ~2^-16
//                relative accuracy. Lane l holds the scores of query l%16 for keys
//                4*(l/16) + i, i = 0..3;
//   O^T += V^T P^T: the same 4 values per lane are the B operand (MFMA k
//                index l/16 <-> key 4*(l/16) + j at step j), V^T the A
//                operand, so no transpose is needed.
// The scores of a whole tile (4 blocks) are formed first, so the online
// softmax (fp32, per query: max and sum over the 4 lanes that share a
// query, xor 16 / xor 32) and the rescaling of O happen once per 64 keys.
// The softmax runs in base 2 (scores scaled by log2 e, weights from the
// hardware exp2, within a few ulp of e^x).
//
// GEN (ALiBi, the window and prefix masks, rings shorter than a tile): row p
// stands for the positions p, p - msl, p - 2 msl, ... that lie in the
// query's range [lo, hi] (every mask is such a range). With an ALiBi slope s
// the positions at or below the query, kp0 - i msl for i < c, add
//   e^(score - s (qp - kp0)) (1 + r + ... + r^(c - 1)),  r = e^(-s msl),
// the same score with one factor, and a row above the query that may see it
// (kp = p) adds its own term. Q, K, P and V take three bf16 terms there (six
// products, down to 2^-24 relative): against 64 bits, with exact projections,
// the output is 1e-7 off, as the fp32 loop of k_attention that it replaces.
// That loop took one wave per (token, head) and one dependent V row per key:
// 3 x 701 tokens, 12 heads of 64 over 4 K/V heads, causal with ALiBi: the layer
// 1636 us, now 109 us (this kernel 71 us; its matrix-core work is 14 us,
// the softmax, the splits and the LDS traffic of two waves per SIMD the rest).
// Keys per LDS tile: 64; 32 for GEN at 128 head dims (three terms of 64 keys
// do not fit the LDS twice) and for the 4-wave workgroups whose 64 keys would
// take more than half the LDS.
constexpr int attn_keys(int hd, bool gen, int waves) {
  return (hd > 64 && (gen || waves == 4)) || (gen && waves == 4) ? 32 : 64;
}

// Positions [lo, hi] that the mask allows to query qp (allow() as a range).
__device__ __forceinline__ void key_range(const AttnArgs& a, int qp, int last, int& lo, int& hi) {
  lo = 0;
  hi = qp;
  if (a.mask == 2) {
    hi = last;
  } else if (a.mask == 3) {
    int w = a.window > 0 ? a.window : a.msl;
    w = w < (1 << 30) ? w : 1 << 30;
    lo = qp - w + 1 > 0 ? qp - w + 1 : 0;
    if (!a.window_causal) hi = qp + w - 1 < last ? qp + w - 1 : last;
  } else if (a.mask == 4 && qp < a.prefix_len) {
    const int p1 = a.prefix_len - 1 < last ? a.prefix_len - 1 : last;
    hi = p1 > qp ? p1 : qp;
  }
}

// Positions of ring row p allowed to query qp: `count` of them at or below
// the query, from `first` down in steps of msl (msl >= seq, so p - msl <= qp),
// and `above` = 1 when p itself lies above the query and is allowed.
__device__ __forceinline__ int key_count(const AttnArgs& a, int p, int qp, int last, int lo, int hi,
                                         float inv_msl, int& first, int& above) {
  above = 0;
  first = p;
  if (p > last) return 0;
  if (p > qp) {
    above = p <= hi ? 1 : 0;
    first = p - a.msl;
  }
  const int n = first - lo;
  if (n < 0) return 0;
  int c = (int)((float)n * inv_msl);  // n / msl, at most one off
  const int r = n - c * a.msl;
  c += (r >= a.msl ? 1 : 0) - (r < 0 ? 1 : 0);
  return c + 1;
}

// ALiBi over rings of fewer than kShortRing rows: 1 - r, formed in f32 with r =
// e^(-s msl) near 1, keeps too few digits at the flattest slope (2^-8): 4e-6 of a
// weight at 2 rows, from 16 on below the exponents' own rounding. SHORT takes
// r^c - 1 over r - 1 from expm1f instead, in kernels of its own (expm1f in the
// others costs them up to 5%, also where it is not run).
constexpr int kShortRing = 16;

// The ALiBi constants of a head: the slope in log2 units and, for the sums
// over a row's positions, x = log2 r and lginv = -log2(1 - r); SHORT: x = ln r
// and lginv = 1 / (r - 1).
struct Bias {
  float sl2, x, lginv;
};

// log2(1 + r + ... + r^(c - 1)); log2(c) without ALiBi.
template <bool SHORT>
__device__ __forceinline__ float log2_copies(int c, const Bias& s) {
  if constexpr (SHORT)
    return c <= 1 ? 0.0f : __builtin_amdgcn_logf(expm1f(s.x * (float)c) * s.lginv);
  if (s.sl2 == 0.0f) return __builtin_amdgcn_logf((float)c);
  return __builtin_amdgcn_logf(1.0f - __builtin_amdgcn_exp2f(s.x * (float)c)) + s.lginv;
}

// log2 of the weight that row p's positions add to e^score for query qp;
// -inf when none is allowed.
template <bool SHORT>
__device__ __forceinline__ float log2_weight(const AttnArgs& a, int p, int qp, int last, int lo,
                                             int hi, float inv_msl, const Bias& s) {
  int first, above;
  const int c = key_count(a, p, qp, last, lo, hi, inv_msl, first, above);
  if (s.sl2 == 0.0f) return __builtin_amdgcn_logf((float)(c + above));  // log2(0) = -inf
  const float below = c > 0 ? fmaf(-s.sl2, (float)(qp - first), log2_copies<SHORT>(c, s)) : -INFINITY;
  if (!above) return below;
  const float up = -s.sl2 * (float)(p - qp);
  const float m = fmaxf(up, below);
  return m + __builtin_amdgcn_logf(__builtin_amdgcn_exp2f(up - m) + __builtin_amdgcn_exp2f(below - m));
}

// acc + A B with both operands in T bf16 terms: the products a_i b_j with
// i + j < T, the smallest first.
template <int T>
__device__ __forceinline__ v4f mfma_terms(const bf16x8 (&a)[T], const bf16x8 (&b)[T], v4f acc) {
#pragma unroll
  for (int s = T - 1; s >= 0; --s)
#pragma unroll
    for (int i = s; i >= 0; --i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[s - i], acc, 0, 0, 0);
  return acc;
}

template <int HD, bool SIG, bool GEN, int WAVES, bool SHORT = false>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(WAVES == 4 ? (GEN && HD > 64 ? 1 : 2) : WAVES / 4, 8)))
void k_attn_mfma(AttnArgs a, int qblocks) {
  constexpr int KT = attn_keys(HD, GEN, WAVES);         // keys per tile
  constexpr int NB = KT / 16, NQ = KT / 32;             // 16-key blocks, 32-key groups
  constexpr int TT = GEN ? 3 : 2;                       // bf16 terms of Q, K, V and P
  constexpr int KS = HD / 32;                           // QK MFMA steps (32 head dims)
  constexpr int DT = HD / 16;                           // 16-wide head-dim tiles of O
  constexpr int kQB = 16 * WAVES;                       // queries per workgroup
  constexpr int NT = 64 * WAVES;                        // threads
  // K in bf16 operand order: [16-key block kb][step ks][term][lane][8]:
  // lane 16 g + c16 holds key 16 kb + c16, head dims 32 ks + 8 g + j
  constexpr int KBYTES = NB * KS * TT * 1024;
  // V in bf16 operand order: [32-key group q][head-dim tile dt][term][lane][8]
  constexpr int VBYTES = NQ * DT * TT * 1024;
  __shared__ __attribute__((aligned(16))) uint8_t ksb[2][KBYTES], vsb[2][VBYTES];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int b = blockIdx.x / qblocks, qb = blockIdx.x % qblocks;
  const int h = blockIdx.y;
  const int kvh = h / (a.heads / a.kv_heads);
  const int qd = a.heads * HD, kvd = a.kv_stride;
  const int last = b * a.seq + a.seq - 1;
  const int p_lo = last - a.msl + 1 > 0 ? last - a.msl + 1 : 0;
  const int s_q = qb * kQB + wave * 16 + c16;      // query within the sequence
  const bool q_ok = s_q < a.seq;
  const int qp = b * a.seq + (q_ok ? s_q : a.seq - 1);
  const bool causal = a.mask == 1;
  // score scales: softmax weights are 2^(s log2 e - max), in log2 units;
  // the sigmoid variant works in natural units
  const float scale_log2 = (float)(a.scale * 1.4426950408889634);
  const float scale_nat = (float)a.scale;
  // GEN: key positions [lo, hi] allowed to this lane's query, and the ALiBi
  // slope in log2 units
  int lo = 0, hi = 0;
  float inv_msl = 0.0f;
  Bias al = {0.0f, 0.0f, 0.0f};
  if constexpr (GEN) {
    key_range(a, qp, last, lo, hi);
    inv_msl = 1.0f / (float)a.msl;
    if (a.alibi) {
      al.sl2 = (float)(exp2(-(double)(h + 1) * 8.0 / (double)a.heads) * 1.4426950408889634);
      if constexpr (SHORT) {
        al.x = (float)(-exp2(-(double)(h + 1) * 8.0 / (double)a.heads) * (double)a.msl);
        al.lginv = 1.0f / expm1f(al.x);
      } else {
        al.x = -al.sl2 * (float)a.msl;
        al.lginv = -__builtin_amdgcn_logf(1.0f - __builtin_amdgcn_exp2f(al.x));
      }
    }
  }

  // Q operand: lane (query c16, group g), head dims 32 ks + 8 g + j, as
  // TT bf16 terms (each the rounded remainder of those before it)
  bf16x8 qop[KS][TT];
  {
    const float* qrow = a.q + (size_t)qp * a.q_stride + (size_t)h * HD;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const v4f q0 = *reinterpret_cast<const v4f*>(qrow + 32 * ks + 8 * g);
      const v4f q1 = *reinterpret_cast<const v4f*>(qrow + 32 * ks + 8 * g + 4);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        bf16x4 t[TT];
        split_bf16<TT>(half ? q1 : q0, t);
#pragma unroll
        for (int k = 0; k < TT; ++k)
#pragma unroll
          for (int j = 0; j < 4; ++j) qop[ks][k][4 * half + j] = t[k][j];
      }
    }
  }
  v4f o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = v4f{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.0f;

  // K rows of a tile in pair units: unit i = tid + NT u covers row
  // i / (HD/8) and the column quads c4 and c4 + HD/2, c4 = 4 (i % (HD/8)).
  // Rows past `last` are exact zeros (a tile wholly past it is a zero tile:
  // the loads stay unconditional).
  constexpr int UNITS = KT * HD / 8, PU = (UNITS + NT - 1) / NT;
  v4f kreg[2 * PU];
  auto load_k = [&](int t0) {
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const int i = tid + NT * u;
      if (UNITS % NT != 0 && i >= UNITS) break;  // whole waves (HD = 32)
      const int r = i / (HD / 8), c4 = (i % (HD / 8)) * 4;
      const int p = t0 + r, pc = p <= last ? p : last;
      const size_t off = (size_t)pc * kvd + (size_t)kvh * HD + c4;
      const v4f k0 = *reinterpret_cast<const v4f*>(a.k + off);
      const v4f k1 = *reinterpret_cast<const v4f*>(a.k + off + HD / 2);
      const v4f z = v4f{0.f, 0.f, 0.f, 0.f};
      kreg[2 * u] = p <= last ? k0 : z;
      kreg[2 * u + 1] = p <= last ? k1 : z;
    }
  };
  // V of a tile in units of 4 rows x 1 column: unit i = tid + NT u covers
  // rows 4 (i / HD) .. + 3 of column i % HD (every load instruction of a wave
  // reads whole rows), so that the 4 values, neighbours in the operand
  // order, are stored with one 8-byte write per term.
  constexpr int VUNITS = KT / 4 * HD, PV = (VUNITS + NT - 1) / NT;
  v4f vreg[PV];
  auto load_v = [&](int t0) {
#pragma unroll
    for (int u = 0; u < PV; ++u) {
      const int i = tid + NT * u;
      if (VUNITS % NT != 0 && i >= VUNITS) break;  // whole waves
      const float* src = a.v + (size_t)kvh * HD + i % HD;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int p = t0 + 4 * (i / HD) + e, pc = p <= last ? p : last;
        const float v = src[(size_t)pc * kvd];
        vreg[u][e] = p <= last ? v : 0.0f;
      }
    }
  };
  // K row r, head dims d..d+3 (d = c4 or c4 + HD/2, a multiple of 4) go to
  // block r / 16, step d / 32, lane 16 ((d / 8) % 4) + r % 16, elements
  // d % 8 .. + 3: one 8-byte store per term.
  auto store_k = [&](int buf) {
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const int i = tid + NT * u;
      if (UNITS % NT != 0 && i >= UNITS) break;
      const int r = i / (HD / 8), c4 = (i % (HD / 8)) * 4;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int d = c4 + half * (HD / 2);
        bf16x4 t[TT];
        split_bf16<TT>(kreg[2 * u + half], t);
        uint8_t* dst = ksb[buf] + (size_t)(((r >> 4) * KS + (d >> 5)) * TT) * 1024 +
                       (((d >> 3) & 3) * 16 + (r & 15)) * 16 + (d & 7) * 2;
#pragma unroll
        for (int term = 0; term < TT; ++term) *reinterpret_cast<bf16x4*>(dst + term * 1024) = t[term];
      }
    }
  };
  // V row r (key) and head dim d go to the bf16 A operand of the P V
  // products: 32-key group q = r / 32, and within it the lane group g and
  // element j that also hold that key's weight in the score layout (key
  // 16 kb + 4 g + i of the group <-> g, j = 4 kb + i); lane 16 g + d % 16 of
  // head-dim tile d / 16.
  auto store_v = [&](int buf) {
#pragma unroll
    for (int u = 0; u < PV; ++u) {
      const int i = tid + NT * u;
      if (VUNITS % NT != 0 && i >= VUNITS) break;
      const int d = i % HD, r4 = i / HD;  // rows 4 r4 ..: group q, j = 4 (rr / 16) + 0..3
      const int q = r4 >> 3, rr4 = r4 & 7;
      bf16x4 t[TT];
      split_bf16<TT>(vreg[u], t);
      uint8_t* dst = vsb[buf] + (size_t)((q * DT + (d >> 4)) * TT) * 1024 +
                     ((rr4 & 3) * 16 + (d & 15)) * 16 + (rr4 >> 2) * 8;
#pragma unroll
      for (int term = 0; term < TT; ++term) *reinterpret_cast<bf16x4*>(dst + term * 1024) = t[term];
    }
  };
  // S^T of a tile: blocks of 16 keys; K terms times Q terms, the small
  // products first: with two terms each the three down to 2^-16 relative, with
  // three the six down to 2^-24
  auto scores = [&](const uint8_t* kt, v4f (&sc)[NB]) {
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) {
      sc[kb] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const uint8_t* kp = kt + (size_t)((kb * KS + ks) * TT) * 1024 + lane * 16;
        bf16x8 k[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) k[t] = *reinterpret_cast<const bf16x8*>(kp + t * 1024);
        sc[kb] = mfma_terms<TT>(k, qop[ks], sc[kb]);
      }
    }
  };

  load_k(p_lo);
  load_v(p_lo);
  store_k(0);
  store_v(0);
  __syncthreads();

  // tile i in buffer i & 1; the loads of tile i+1 are issued into registers
  // before tile i's products and stored to the other buffer after them (it
  // was last read before the previous barrier). All loads are unconditional
  // (a tile past the range is a zero tile, stored but never read).
#pragma unroll 1
  for (int t0 = p_lo, cur = 0; t0 <= last; t0 += KT, cur ^= 1) {
    load_k(t0 + KT);
    load_v(t0 + KT);
    const uint8_t* vt = vsb[cur];
    // multiplicity base of the tile start: floor(t0 / msl) + 1 (msl >= KT
    // without GEN, so the tile crosses at most one multiple of msl)
    const int base0 = t0 / a.msl + 1;
    const int next_mult = base0 * a.msl;  // first p with a larger base
    // multiplicity of the row of key k (block kb, lane key i) for this query
    const float base0f = (float)base0;
    auto mult = [&](int kb, int i) {
      const int p = t0 + 16 * kb + 4 * g + i;
      if constexpr (GEN) {
        int first, above;
        const int c = key_count(a, p, qp, last, lo, hi, inv_msl, first, above);
        return (float)(c + above);
      }
      const float c = p <= last ? base0f + (p >= next_mult ? 1.0f : 0.0f) : 0.0f;
      return c - (causal && p > qp ? 1.0f : 0.0f);
    };
    // Most tiles give every key of the wave the same multiplicity: wholly
    // inside [p_lo, last], not crossing a multiple of msl, and wholly at or
    // below (c = base) or wholly above (c = base - 1, causal) the wave's 16
    // queries. cu is that value (wave-uniform), or -1 for per-key values; a
    // tile with cu == 0 adds nothing to this wave's queries. GEN: the same
    // from the first and the last query's ranges (both grow with the query);
    // first0 is the first position that the tile's first row stands for.
    const int kmax = t0 + KT - 1;
    const int qw0 = b * a.seq + qb * kQB + __builtin_amdgcn_readfirstlane(wave) * 16;
    int cu = -1, first0 = t0;
    if constexpr (GEN) {
      const int qw1 = qw0 + 15 < last ? qw0 + 15 : last;  // the wave's last query
      int l0, h0, l1, h1;
      key_range(a, qw0 < last ? qw0 : last, last, l0, h0);
      key_range(a, qw1, last, l1, h1);
      const bool above = t0 > qw1 && t0 > h1;
      if (kmax <= last && (kmax <= qw0 || above)) {
        first0 = above ? t0 - a.msl : t0;
        const int n0 = first0 - l1, n1 = first0 + KT - 1 - l0;  // least and largest
        if (n1 < 0) cu = 0;
        else if (n0 >= 0 && n0 / a.msl == n1 / a.msl) cu = n0 / a.msl + 1;
      }
    } else if (kmax <= last && next_mult > kmax) {
      if (!causal || kmax <= qw0) cu = base0;
      else if (t0 > qw0 + 15) cu = base0 - 1;
    }
    if (cu != 0) {  // wave-uniform
    v4f sc[NB];
    scores(ksb[cur], sc);
    float w[4 * NB];
    if constexpr (SIG) {
#pragma unroll
      for (int kb = 0; kb < NB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float c = cu > 0 ? (float)cu : mult(kb, i);
          w[4 * kb + i] = c > 0.0f ? c / (1.0f + expf(-sc[kb][i] * scale_nat)) : 0.0f;
        }
    } else {
      // base-2 scores with the multiplicity folded into the exponent
      // (c 2^x = 2^(x + log2 c)); masked keys at -inf
      float smax = -INFINITY;
      if (GEN && cu > 0) {
        // ALiBi: the distance to the row's first position, then the sum over
        // its cu positions as one factor (log2_copies)
        const float lc = log2_copies<SHORT>(cu, al);
        const float d0 = (float)(qp - first0 - 4 * g);
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float bias = fmaf(-al.sl2, d0 - (float)(16 * kb + i), lc);
            w[4 * kb + i] = fmaf(sc[kb][i], scale_log2, bias);
            smax = fmaxf(smax, w[4 * kb + i]);
          }
      } else if (GEN) {
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float bias = log2_weight<SHORT>(a, t0 + 16 * kb + 4 * g + i, qp, last, lo, hi, inv_msl, al);
            w[4 * kb + i] = bias > -INFINITY ? fmaf(sc[kb][i], scale_log2, bias) : -INFINITY;
            smax = fmaxf(smax, w[4 * kb + i]);
          }
      } else if (cu > 0) {
        const float lc = __builtin_amdgcn_logf((float)cu);
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            w[4 * kb + i] = sc[kb][i] * scale_log2 + lc;
            smax = fmaxf(smax, w[4 * kb + i]);
          }
      } else {
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float c = mult(kb, i);
            w[4 * kb + i] = c > 0.0f ? sc[kb][i] * scale_log2 + __builtin_amdgcn_logf(c) : -INFINITY;
            smax = fmaxf(smax, w[4 * kb + i]);
          }
      }
      smax = fmaxf(smax, __shfl_xor(smax, 16, 64));
      smax = fmaxf(smax, __shfl_xor(smax, 32, 64));
      const float nm = fmaxf(m, smax);
      const float nz = nm == -INFINITY ? 0.0f : nm;  // all masked so far: weights 0
      const float corr = __builtin_amdgcn_exp2f(m - nz);  // m = -inf: 0
      float ws = 0.0f;
#pragma unroll
      for (int i = 0; i < 4 * NB; ++i) {
        w[i] = __builtin_amdgcn_exp2f(w[i] - nz);
        ws += w[i];
      }
      ws += __shfl_xor(ws, 16, 64);
      ws += __shfl_xor(ws, 32, 64);
      l = l * corr + ws;
#pragma unroll
      for (int d = 0; d < DT; ++d) o[d] *= corr;
      m = nm;
    }
    // O^T += V^T P^T on the bf16 matrix cores, 32 keys per product, each
    // operand split into TT bf16 terms as the scores' operands (with two, the
    // dropped lo*lo product and the split leave ~2^-16 relative error).
    // Lane (query c16, group g) passes the weights it already holds: element
    // j of group g is key 16 (2q + j / 4) + 4g + j % 4 of the tile.
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      bf16x8 p[TT];
#pragma unroll
      for (int j2 = 0; j2 < 2; ++j2) {
        const float* wq = w + 4 * (2 * q + j2);
        bf16x4 t[TT];
        split_bf16<TT>(v4f{wq[0], wq[1], wq[2], wq[3]}, t);
#pragma unroll
        for (int term = 0; term < TT; ++term)
#pragma unroll
          for (int j = 0; j < 4; ++j) p[term][4 * j2 + j] = t[term][j];
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const uint8_t* vb = vt + (size_t)((q * DT + d) * TT) * 1024 + lane * 16;
        bf16x8 v[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) v[t] = *reinterpret_cast<const bf16x8*>(vb + t * 1024);
        o[d] = mfma_terms<TT>(v, p, o[d]);
      }
    }
    }
    store_k(cur ^ 1);
    store_v(cur ^ 1);
    __syncthreads();
  }
  // o[d]: lane holds query c16, head dims d*16 + 4g + i
  const float inv = SIG ? 1.0f : (l > 0.0f ? 1.0f / l : 0.0f);
  // with a.split (seq % 16 == 0: the wave's 16 queries are rows 16 rb ..
  // 16 rb + 15, all valid), the outputs are also staged in LDS, which the
  // K/V tiles no longer use after the loop's last barrier: 64 HD bytes per
  // wave, the first half of the waves in ksb and the others in vsb
  constexpr int HW = WAVES / 2;
  static_assert(HW * 64 * HD <= 2 * KBYTES && HW * 64 * HD <= 2 * VBYTES, "output staging");
  float* stg = reinterpret_cast<float*>(wave < HW ? &ksb[0][0] + wave * 64 * HD
                                                  : &vsb[0][0] + (wave - HW) * 64 * HD);
  bool redo = false;
  if constexpr (GEN) {
    // A key or value that is not finite (or near the f32 maximum, where a
    // bf16 term overflows) puts NaN into the products of every query of the
    // tile, also of those that may not see it: such a wave takes its queries
    // again, one by one over the allowed keys only.
    float t = SIG ? 0.0f : l - l;
    if (!SIG && !(l > 0.0f)) t = NAN;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i) t += o[d][i] - o[d][i];
    redo = __any(q_ok && t != 0.0f);
  }
  if (redo) {
    for (int j = 0; j < 16; ++j) {
      const int sj = qb * kQB + wave * 16 + j;
      if (sj >= a.seq) break;  // wave-uniform
      const int t = b * a.seq + sj;
      const size_t row = (size_t)t * qd + (size_t)h * HD;
      float acc[kMaxHdPerLane];
      attend_token(a, t, h, lane, a.q + (size_t)t * a.q_stride + (size_t)h * HD, acc);
#pragma unroll
      for (int i = 0; i < (HD + 63) / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < HD) {
          a.out[row + d] = acc[i];
          if (a.split) stg[j * HD + d] = acc[i];
        }
      }
    }
  }
  if (!q_ok) return;
  if (!redo) {
    float* out = a.out + (size_t)qp * qd + (size_t)h * HD;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const float4 v = make_float4(o[d][0] * inv, o[d][1] * inv, o[d][2] * inv, o[d][3] * inv);
      *reinterpret_cast<float4*>(out + d * 16 + 4 * g) = v;
      if (a.split) *reinterpret_cast<float4*>(stg + c16 * HD + d * 16 + 4 * g) = v;
    }
  }
  if (a.split && lane < 16 * (HD / 32)) {  // (the LDS operations of a wave run in order)
    // the head's 32-element blocks of row i16: operand lane i16 + 16 gq of
    // the O projection's 16 x 128 slice (rb, kc), gq = (h HD % 128) / 32 + gg,
    // split exactly as k_split splits the stored outputs
    const int i16 = lane & 15, gg = lane >> 4;
    float v[32];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float4 t = *reinterpret_cast<const float4*>(stg + i16 * HD + 32 * gg + 4 * q);
      v[4 * q] = t.x, v[4 * q + 1] = t.y, v[4 * q + 2] = t.z, v[4 * q + 3] = t.w;
    }
    const int col0 = h * HD, kc = col0 / 128, KC = qd / 128;
    const int rb = (qp - c16) / 16;
    const int vlane = i16 + 16 * ((col0 % 128) / 32 + gg);
    const GlobalU8 chunk = (GlobalU8)(a.split + (size_t)(rb * KC + kc) * kTerms * kFrag6Bytes);
    const GlobalU8 scales = (GlobalU8)(a.split + (size_t)kTerms * a.split_mpad * qd +
                                       (size_t)(rb * KC + kc) * kChunkScaleBytes);
    split_terms6<1, kTerms, false>(v, chunk, scales, vlane);
  }
}

}  // namespace

Status build_rope_table(double* tab, int tokens, int hd, double theta, hipStream_t st) {
  const int n = tokens * (hd / 2);
  if (n <= 0) return Status::ok();
  k_rope_table<<<(n + 255) / 256, 256, 0, st>>>(tab, tokens, hd, theta);
  return hip_status(hipGetLastError(), "rope table launch");
}

// The matrix-core kernel takes head dims 32, 64 and 128. Its GEN form takes
// what the plain one does not: ALiBi, the window and prefix masks, and rings
// shorter than a 64-key tile (whose multiplicities change within one). ALiBi
// with the sigmoid has no common factor per ring row and stays on
// k_attention.
static bool attention_fast(const AttnArgs& a) {
  return (a.hd == 32 || a.hd == 64 || a.hd == 128) && a.msl >= a.seq && a.seq > 0 &&
         a.tokens % a.seq == 0 && !(a.alibi && a.sigmoid);
}

static bool attention_general(const AttnArgs& a) {
  return a.alibi || (a.mask != 1 && a.mask != 2) || a.msl < 64;
}

bool attention_writes_split(const AttnArgs& a) {
  return attention_fast(a) && (a.heads * a.hd) % 256 == 0 && a.seq % 16 == 0;
}

template <int HD, bool SIG, bool GEN, int WAVES, bool SHORT = false>
static void attn_launch(const AttnArgs& a, hipStream_t st) {
  const int qblocks = (a.seq + 16 * WAVES - 1) / (16 * WAVES);
  const dim3 grid((unsigned)(a.tokens / a.seq * qblocks), (unsigned)a.heads);
  k_attn_mfma<HD, SIG, GEN, WAVES, SHORT><<<grid, 64 * WAVES, 0, st>>>(a, qblocks);
}

template <int HD, bool GEN>
static void attn_waves_of(const AttnArgs& a, hipStream_t st) {
  constexpr int most = HD <= 64 ? 16 : 8;
  if (a.sigmoid) return attn_launch<HD, true, GEN, most>(a, st);
  if constexpr (GEN) {
    // (a ring holds the sequence: one wave has all of its queries)
    if (a.alibi && a.msl < kShortRing) return attn_launch<HD, false, true, 4, true>(a, st);
  }
  const auto groups = [&](int waves) {
    return (int64_t)(a.tokens / a.seq) * a.heads * ((a.seq + 16 * waves - 1) / (16 * waves));
  };
  // The widest workgroup (each K/V tile staged once for more queries) that
  // still reaches three quarters of the 256 CUs, else 4 waves, one per SIMD.
  // Whole layers, us at 16 / 8 / 4 waves, head dim 64: 8 x 512 tokens, 16
  // heads (256, 512, 1024 workgroups) 115 / 118 / 135; 3 x 701, 12 heads with
  // ALiBi (108, 216, 396) 166 / 134 / 151; 1 x 1024, 16 heads (64, 128, 256)
  // 113 / 101 / 94; 2 x 300, 8 heads (32, 48, 80) 77 / 71 / 68.
  constexpr int64_t kFill = 192;
  if (groups(most) >= kFill) return attn_launch<HD, false, GEN, most>(a, st);
  if (most > 8 && groups(8) >= kFill) return attn_launch<HD, false, GEN, 8>(a, st);
  attn_launch<HD, false, GEN, 4>(a, st);
}

template <int HD>
static void attn_hd(const AttnArgs& a, hipStream_t st) {
  if (attention_general(a)) attn_waves_of<HD, true>(a, st);
  else attn_waves_of<HD, false>(a, st);
}

Status launch_attention(const AttnArgs& a, hipStream_t st) {
  if (a.hd > 64 * kMaxHdPerLane || a.hd % 4 != 0)
    return Status::err(kUnsupported, "attention: head_dim must be a multiple of 4 and <= 256");
  if (a.q_stride < a.heads * a.hd || a.kv_stride < a.kv_heads * a.hd ||
      ((a.q_stride | a.kv_stride) & 3) != 0)
    return Status::err(kInvalid, "attention: token strides");
  const bool fast = attention_fast(a);
  if (a.split && (!attention_writes_split(a) || a.split_mpad < a.tokens || a.split_mpad % 16 != 0))
    return Status::err(kInvalid, "attention: the output split needs the matrix-core path, "
                                 "heads * hd % 256 == 0 and seq % 16 == 0");
  if (a.rope) {
    k_rope<<<a.tokens, 256, 0, st>>>(const_cast<float*>(a.q), const_cast<float*>(a.k), a.tokens,
                                     a.heads, a.kv_heads, a.hd, a.q_stride, a.kv_stride,
                                     a.rope_theta, a.rope_tab);
    WV_HIP(hipGetLastError());
  }
  if (fast) {
    switch (a.hd) {
    case 32: attn_hd<32>(a, st); break;
    case 64: attn_hd<64>(a, st); break;
    default: attn_hd<128>(a, st); break;
    }
    return hip_status(hipGetLastError(), "attention launch");
  }
  dim3 grid(a.tokens, a.heads);
  k_attention<<<grid, 64, 0, st>>>(a);
  return hip_status(hipGetLastError(), "attention launch");
}

}  // namespace wv
