// Head routing of the 1.5-5B pattern attention (unified_judge, partern_attention.py:463-521)
// for gfx950.
//
//   probs_kernel       one wave per (head, 32 sampled query rows): S^T = K Q^T with
//                      v_mfma_f32_32x32x16_bf16 over all sampled keys (optional additive bias
//                      on the first keys), row max and sum in a first pass, then the
//                      probabilities of a key range written row-major (through LDS, 128-byte
//                      rows) in a second pass;
//   share_kernel       judge_sparsity (:468-476): per query row, the probability mass of its
//                      K largest entries (K-th largest found by a bit search on the fp32
//                      bit patterns, its last bits over the compacted bucket), one workgroup
//                      per row;
//   gram_kernel        judge_similarity (:477-514): for key frame f2, the Gram matrix
//                      G[f1][f3] = sum_{s1,s2} P[f1 s1][f2 s2] * P[f3 s1][f2 s2] of the
//                      frame-pair patterns (their inner products and norms), as partial sums
//                      over chunks of s1;
//   topk_mass_kernel   judge_sparsity as the Python layer runs it: the same masses with the
//                      scores recomputed by each of a few walks over the keys instead of written;
//   simgram_kernel     judge_similarity as the Python layer runs it: the Gram partials with
//                      the probabilities kept on chip;
//   gather_operands_kernel  sampled keys in matrix-operand order, for topk_mass_kernel;
//   finish_kernel      per head: mean share > 0.9 (sparse), mean cosine similarity of the
//                      patterns sharing a key frame > 0.9 (twice), and the routing decision.
#include <cmath>
#include <type_traits>

#include "sa_common.h"

namespace {

constexpr int kD = 64;
constexpr float kLog2e = 1.4426950408889634f;

typedef unsigned jd_u32x4 __attribute__((ext_vector_type(4)));
typedef float jd_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short jd_u16x2 __attribute__((ext_vector_type(2)));

__device__ inline sa_f32x16 score_tile_k(const jd_u32x4 (&kop)[4], const sa_bf16x8 (&qf)[4]) {
  sa_f32x16 t = {};
#pragma unroll
  for (int s = 0; s < 4; ++s)
    t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sa_bf16x8, kop[s]), qf[s], t, 0, 0, 0);
  return t;
}

__device__ inline void load_k(const uint16_t* kp, jd_u32x4 (&kop)[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) kop[s] = *reinterpret_cast<const jd_u32x4*>(kp + 16 * s);
}

__device__ inline sa_f32x16 score_tile(const uint16_t* kp, const sa_bf16x8 (&qf)[4]) {
  jd_u32x4 kop[4];
  load_k(kp, kop);
  return score_tile_k(kop, qf);
}

// ---------------------------------------------------------------------------------------
struct ProbArgs {
  const uint16_t* qs;  // [BH][rows_pad][64]
  const uint16_t* ks;  // [BH][keys_pad][64]
  int rows, rows_pad, keys, keys_pad;
  float scale_log2;
  int n_bias;
  float bias_log2;     // added to keys < n_bias (log2 domain)
  int c_lo, c_hi;      // key range written
  float* P;            // P[bh*p_bh + r*p_row + (key - c_lo)]
  int64_t p_bh, p_row;
  int ng;              // rows_pad / 32
  int vec_ok;          // 16-byte stores possible (P, strides and c_lo multiples of 4 floats)
  int64_t total;       // BH * ng
};

__global__ __launch_bounds__(256) void probs_kernel(ProbArgs a) {
  __shared__ float tile[4][32][36];  // [wave][query row][key], rows 16-byte aligned
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t wid = (int64_t)blockIdx.x * 4 + wave;
  if (wid >= a.total) return;  // no workgroup barriers below
  const int64_t bh = wid / a.ng;
  const int g = (int)(wid - bh * a.ng);
  const int col = lane & 31, hh = lane >> 5;
  sa_bf16x8 qf[4];
  {
    const uint16_t* qp = a.qs + (bh * a.rows_pad + 32 * g + col) * kD + 8 * hh;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = __builtin_bit_cast(sa_bf16x8, *reinterpret_cast<const jd_u32x4*>(qp + 16 * s));
  }
  const uint16_t* kbase = a.ks + (bh * a.keys_pad + col) * kD + 8 * hh;
  // Logits (log2 domain) of key tile kt; -inf past the keys. Whole tiles inside the key
  // range and on one side of the bias boundary need no per-element tests.
  auto logits = [&](const sa_f32x16& t, int kt, float (&x)[16]) {
    if (32 * kt + 32 <= a.keys && (32 * kt + 32 <= a.n_bias || 32 * kt >= a.n_bias)) {
      const float tb = 32 * kt < a.n_bias ? a.bias_log2 : 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = fmaf(t[i], a.scale_log2, tb);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = 32 * kt + 8 * (i >> 2) + 4 * hh + (i & 3);
        x[i] = key >= a.keys ? -INFINITY : fmaf(t[i], a.scale_log2, key < a.n_bias ? a.bias_log2 : 0.f);
      }
    }
  };
  float m = -INFINITY, l = 0.f;
  for (int kt = 0; kt < a.keys_pad / 32; ++kt) {
    const sa_f32x16 t = score_tile(kbase + (int64_t)kt * 32 * kD, qf);
    float x[16], tmax = -INFINITY;
    logits(t, kt, x);
#pragma unroll
    for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, x[i]);
    const float mn = fmaxf(m, tmax);
    if (mn != -INFINITY) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) sum += __builtin_amdgcn_exp2f(x[i] - mn);
      l = l * __builtin_amdgcn_exp2f(m - mn) + sum;
      m = mn;
    }
  }
  {
    const auto mo = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    const auto lo = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    const float m0 = __uint_as_float(mo[0]), m1 = __uint_as_float(mo[1]);
    const float M = fmaxf(m0, m1);
    l = __uint_as_float(lo[0]) * __builtin_amdgcn_exp2f(m0 - M) + __uint_as_float(lo[1]) * __builtin_amdgcn_exp2f(m1 - M);
    m = M;
  }
  const float inv = 1.f / l;
  const int row0 = 32 * g;
  const int c4 = lane & 7;  // lane writes keys 4*c4 .. 4*c4+3 of rows lane/8 + 8j
  for (int kt = a.c_lo / 32; kt * 32 < a.c_hi; ++kt) {
    const sa_f32x16 t = score_tile(kbase + (int64_t)kt * 32 * kD, qf);
    float x[16];
    logits(t, kt, x);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      tile[wave][col][8 * (i >> 2) + 4 * hh + (i & 3)] = __builtin_amdgcn_exp2f(x[i] - m) * inv;
    __builtin_amdgcn_wave_barrier();
    // 8 lanes per row: each store instruction writes 128 contiguous bytes of 8 rows.
    const int key0 = 32 * kt + 4 * c4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 8 * j + (lane >> 3);
      if (row0 + r >= a.rows) continue;
      float* dst = a.P + bh * a.p_bh + (int64_t)(row0 + r) * a.p_row;
      const float4 v = *reinterpret_cast<const float4*>(&tile[wave][r][4 * c4]);
      const int o = key0 - a.c_lo;  // column of key0 in P
      if (a.vec_ok && key0 >= a.c_lo && key0 + 4 <= a.c_hi) {
        // streamed: P is far larger than the caches, K stays resident
        __builtin_nontemporal_store(jd_f32x4{v.x, v.y, v.z, v.w}, reinterpret_cast<jd_f32x4*>(dst + o));
      } else {
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (key0 + u >= a.c_lo && key0 + u < a.c_hi) dst[o + u] = e[u];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// ---------------------------------------------------------------------------------------
// share_kernel: one workgroup per (bh, row) over n probabilities (n <= 16384).
struct ShareArgs {
  const float* P;
  int64_t p_bh, p_row;
  int rows, n, K;
  int vec_ok;  // P, p_bh and p_row multiples of 16 bytes
  float* share;  // [BH][rows]
  int64_t total;
};

__device__ inline uint32_t wave_sum_u(uint32_t x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}
__device__ inline float wave_sum_f(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// Thread t holds entries t, t + 256, ... (at most 64 of them) in registers. The K-th largest
// bit pattern (p >= 0: bit patterns order as the values) is the largest thr with
// #{v >= thr} >= K, found bit by bit from the top. The first kShareHi bits are searched over
// every entry. The entries that share those bits (the bucket) are then compacted into LDS in
// thread order, and one wave finishes the search over them; entries above the bucket always
// count. A bucket larger than kShareCap entries continues the search over every entry.
constexpr int kShareHi = 12;
constexpr int kShareCap = 2048;

__device__ inline uint32_t wave_incl_scan_u(uint32_t x, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  return x;
}

__global__ __launch_bounds__(256) void share_kernel(ShareArgs a) {
  constexpr int kPer = 64;
  __shared__ uint32_t part_u[2][4];
  __shared__ float part_f[4];
  __shared__ uint32_t buck[kShareCap];
  __shared__ uint32_t wtot[2][4];
  __shared__ uint32_t thr_out;
  const int64_t w = blockIdx.x;
  if (w >= a.total) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t bh = w / a.rows;
  const int r = (int)(w - bh * a.rows);
  const float* src = a.P + bh * a.p_bh + (int64_t)r * a.p_row;
  uint32_t v[kPer];  // 0 past n; the order of the entries does not matter below
  if (a.vec_ok) {    // 16-byte loads: entries 4t + 1024q .. +3
#pragma unroll
    for (int q = 0; q < kPer / 4; ++q) {
      const int i = 4 * t + 1024 * q;
      if (i + 4 <= a.n) {
        const uint4 u = *reinterpret_cast<const uint4*>(src + i);
        v[4 * q] = u.x;
        v[4 * q + 1] = u.y;
        v[4 * q + 2] = u.z;
        v[4 * q + 3] = u.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * q + e] = i + e < a.n ? __float_as_uint(src[i + e]) : 0u;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = t + 256 * j;
      v[j] = i < a.n ? __float_as_uint(src[i]) : 0u;
    }
  }
  // Counting step over every entry (double-buffered partials, one barrier per step).
  auto step = [&](uint32_t thr, int bit) {
    const uint32_t cand = thr | (1u << bit);
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) c += v[j] >= cand;
    c = wave_sum_u(c);
    if (lane == 0) part_u[bit & 1][wave] = c;
    __syncthreads();
    const uint32_t tot = part_u[bit & 1][0] + part_u[bit & 1][1] + part_u[bit & 1][2] + part_u[bit & 1][3];
    return tot >= (uint32_t)a.K ? cand : thr;
  };
  // The first kShareHi steps compare top bits only (their candidates' low 16 bits are zero),
  // two entries per register: the top halves of non-negative fp32 patterns are below 0x8000
  // and the candidates' at most 0x8000, so x < c is the sign bit of the 16-bit difference
  // x - c (packed subtract, shift and add; no compare results in VCC).
  jd_u16x2 hp[kPer / 2];
#pragma unroll
  for (int i = 0; i < kPer / 2; ++i)
    hp[i] = jd_u16x2{(unsigned short)(v[2 * i] >> 16), (unsigned short)(v[2 * i + 1] >> 16)};
  auto step_hi = [&](uint32_t thr, int bit) {
    const uint32_t cand = thr | (1u << bit);
    const unsigned short c16 = (unsigned short)(cand >> 16);
    const jd_u16x2 cc = {c16, c16};
    jd_u16x2 lt = {0, 0};
#pragma unroll
    for (int i = 0; i < kPer / 2; ++i) lt += (jd_u16x2)(hp[i] - cc) >> (unsigned short)15;
    uint32_t c = (uint32_t)kPer - ((uint32_t)lt.x + (uint32_t)lt.y);
    c = wave_sum_u(c);
    if (lane == 0) part_u[bit & 1][wave] = c;
    __syncthreads();
    const uint32_t tot = part_u[bit & 1][0] + part_u[bit & 1][1] + part_u[bit & 1][2] + part_u[bit & 1][3];
    return tot >= (uint32_t)a.K ? cand : thr;
  };
  static_assert(32 - kShareHi >= 16, "the packed steps need candidates with zero low 16 bits");
  uint32_t thr = 0;
  for (int bit = 31; bit >= 32 - kShareHi; --bit) thr = step_hi(thr, bit);
  // Bucket: entries whose top kShareHi bits equal thr's; above: entries with larger top bits.
  const uint32_t hi = thr >> (32 - kShareHi);
  uint32_t nb = 0, above = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint32_t tb = v[j] >> (32 - kShareHi);
    nb += tb == hi;
    above += tb > hi;
  }
  const uint32_t nb_incl = wave_incl_scan_u(nb, lane);
  const uint32_t above_w = wave_sum_u(above);
  if (lane == 63) wtot[0][wave] = nb_incl;
  if (lane == 0) wtot[1][wave] = above_w;
  __syncthreads();
  uint32_t nb_off = nb_incl - nb;
  for (int q = 0; q < wave; ++q) nb_off += wtot[0][q];
  const uint32_t nb_tot = wtot[0][0] + wtot[0][1] + wtot[0][2] + wtot[0][3];
  const uint32_t above_tot = wtot[1][0] + wtot[1][1] + wtot[1][2] + wtot[1][3];
  if (nb_tot <= (uint32_t)kShareCap) {
    uint32_t o = nb_off;
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if ((v[j] >> (32 - kShareHi)) == hi) buck[o++] = v[j];
    __syncthreads();
    if (wave == 0) {
      // want-th largest in the bucket, want = K - above_tot >= 1 (the top bits are maximal)
      const uint32_t want = (uint32_t)a.K - above_tot;
      uint32_t x[kShareCap / 64];
#pragma unroll
      for (int i = 0; i < kShareCap / 64; ++i) {
        const uint32_t idx = (uint32_t)(lane + 64 * i);
        x[i] = idx < nb_tot ? buck[idx] : 0u;  // 0 is below every candidate (it has bits set)
      }
      uint32_t th = thr;
      for (int bit = 31 - kShareHi; bit >= 0; --bit) {
        const uint32_t cand = th | (1u << bit);
        uint32_t c = 0;
#pragma unroll
        for (int i = 0; i < kShareCap / 64; ++i) c += x[i] >= cand;
        if (wave_sum_u(c) >= want) th = cand;
      }
      if (lane == 0) thr_out = th;
    }
    __syncthreads();
    thr = thr_out;
  } else {
    for (int bit = 31 - kShareHi; bit >= 0; --bit) thr = step(thr, bit);
  }
  // Mass above thr, plus thr for the ties needed to make K.
  float sum = 0.f;
  uint32_t gt = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    if (v[j] > thr) {
      sum += __uint_as_float(v[j]);
      ++gt;
    }
  }
  sum = wave_sum_f(sum);
  gt = wave_sum_u(gt);
  __syncthreads();
  if (lane == 0) {
    part_f[wave] = sum;
    part_u[0][wave] = gt;
  }
  __syncthreads();
  if (t == 0) {
    const float s4 = ((part_f[0] + part_f[1]) + part_f[2]) + part_f[3];
    const uint32_t g4 = part_u[0][0] + part_u[0][1] + part_u[0][2] + part_u[0][3];
    a.share[bh * a.rows + r] = s4 + (float)((int)a.K - (int)g4) * __uint_as_float(thr);
  }
}

// ---------------------------------------------------------------------------------------
// topk_mass_kernel: the share of judge_sparsity without written probabilities. One workgroup of
// eight waves per (bh, 32 query rows), lane column = row; wave w takes key tiles w, w + 8, ... of
// every walk over the keys, and each walk recomputes the scores (four MFMAs per 32 x 32 tile from
// keys in operand order, one coalesced 1 KB load each):
//   1: row maxima and minima;
//   2: e = exp2(x - max) and a histogram per row of e's bit pattern above the row's smallest
//      (linear in log2 e: 256 equal bins, LDS atomics whose bank is the row's), the row sum; the
//      bin of the K-th largest e follows from the counts. While that bin holds more than kTmCap
//      entries and spans more than one pattern, it is divided again by another walk;
//   3: the sum of e above the bin; the bin's entries go to a list, whose K-th largest is then
//      searched bit by bit by 16 lanes per row.
// The same selection as share_kernel's, on e instead of e / sum: share = (sum of the entries above
// the K-th, and it for the ties needed) / row sum. The list arrives in any order, so its sum is
// taken in fp64, which is exact for the entries of one bin: the result is the same every time.
// Bound: the scores' exp2, bins and sums, 0.7 G entries for 96 heads of 500 x 15 035, three
// times (a third walk more where the heads are peaked); writing and re-reading their 2.9 GB in fp32
// took 1.24 + 1.31 ms, this takes 0.87 (1.09 with a head's workgroups spread over the XCDs).
constexpr int kTmWaves = 8;
constexpr int kTmBins = 256;
constexpr int kTmCap = 256;

struct TopkMassArgs {
  const uint16_t* qs;   // [BH][rows_pad][64]
  const jd_u32x4* ks;   // [BH][n_tiles][4][64]: key operands (gather_operands_kernel)
  int rows, rows_pad, n, n_tiles, K;
  float scale_log2;
  float* share;  // [BH][rows]
  int ng;        // cdiv(rows, 32)
  int BH;
};

__global__ __launch_bounds__(64 * kTmWaves, 4) void topk_mass_kernel(TopkMassArgs a) {
  __shared__ uint32_t hist[kTmBins * 32];  // [bin][row]
  __shared__ uint32_t list[kTmCap * 32];   // [entry][row]
  __shared__ float wred[kTmWaves][2][32];  // the waves' partial maxima / minima / sums
  // Per row: the bin under division is patterns base .. base + width - 1, in kTmBins parts of
  // 2^shift; above = entries above it, count = entries in it, todo = still to be divided.
  __shared__ uint32_t base[32], width[32], shift[32], above[32], count[32], fill[32];
  __shared__ int todo[32];
  __shared__ int again;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int col = lane & 31, hh = lane >> 5;
  // A head's workgroups share an XCD, whose L2 then holds the head's keys (workgroups go round
  // robin over the eight XCDs).
  const int x8 = blockIdx.x >> 3;
  const int64_t bh = 8 * (int64_t)(x8 / a.ng) + (blockIdx.x & 7);
  const int row0 = 32 * (x8 % a.ng);
  if (bh >= a.BH) return;

  sa_bf16x8 qf[4];
  {
    const uint16_t* qp = a.qs + (bh * a.rows_pad + row0 + col) * kD + 8 * hh;  // rows_pad covers row0 + 31
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = __builtin_bit_cast(sa_bf16x8, *reinterpret_cast<const jd_u32x4*>(qp + 16 * s));
  }
  const jd_u32x4* kbase = a.ks + bh * a.n_tiles * 256 + lane;
  // f(tag: the whole tile exists, scores of a tile, entries that exist); entry i of a lane is key
  // 32 kt + 8 (i / 4) + 4 hh + i % 4.
  auto walk = [&](auto f) __attribute__((always_inline)) {
    jd_u32x4 kop[4], knext[4];
    if (wave < a.n_tiles) {
#pragma unroll
      for (int s = 0; s < 4; ++s) knext[s] = kbase[(int64_t)wave * 256 + 64 * s];
    }
    for (int kt = wave; kt < a.n_tiles; kt += kTmWaves) {
      const int kn = kt + kTmWaves < a.n_tiles ? kt + kTmWaves : kt;
#pragma unroll
      for (int s = 0; s < 4; ++s) kop[s] = knext[s];
#pragma unroll
      for (int s = 0; s < 4; ++s) knext[s] = kbase[(int64_t)kn * 256 + 64 * s];
      const int left = a.n - 32 * kt;
      const sa_f32x16 x = score_tile_k(kop, qf);
      if (left >= 32) f(std::true_type{}, x, left);
      else f(std::false_type{}, x, left);
    }
  };
  auto exists = [&](int left, int i) { return 8 * (i >> 2) + 4 * hh + (i & 3) < left; };
  // max / sum over the two lane halves, then over the waves in order.
  auto half = [&](float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return hh ? __uint_as_float(r[0]) : __uint_as_float(r[1]);  // the other half's value
  };

  // ---- 1: maxima and minima of the raw scores (the scale is positive).
  float mx = -INFINITY, mn = INFINITY;
  walk([&](auto whole, const sa_f32x16& x, int left) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (whole.value || exists(left, i)) {
        mx = fmaxf(mx, x[i]);
        mn = fminf(mn, x[i]);
      }
  });
  mx = fmaxf(mx, half(mx));
  mn = fminf(mn, half(mn));
  if (hh == 0) {
    wred[wave][0][col] = mx;
    wred[wave][1][col] = mn;
  }
  for (int i = t; i < kTmBins * 32; i += 64 * kTmWaves) hist[i] = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kTmWaves; ++w) {
    mx = fmaxf(mx, wred[w][0][col]);
    mn = fminf(mn, wred[w][1][col]);
  }
  // The difference is formed before the scaling: it is exactly 0 at the row's maximum, so e <= 1, the
  // bins' top, whatever the scores' size (mx * scale rounded first is off by 2^-14 at 1 024, and the
  // largest e by 344 patterns).
  auto e_of = [&](float x) { return __builtin_amdgcn_exp2f((x - mx) * a.scale_log2); };
  if (t < 32) {
    // Patterns from just below the smallest e to just above 1 (exp2 may round either way).
    const uint32_t lo = min(__float_as_uint(e_of(mn)), 0x3f800000u);
    const uint32_t b0 = lo > 64u ? lo - 64u : 0u;
    base[t] = b0;
    width[t] = row0 + t < a.rows ? 0x3f800040u - b0 : 0u;
    shift[t] = max(0, 32 - 8 - __clz((int)(0x3f800040u - b0)));
    above[t] = 0;
    count[t] = 0;
    todo[t] = row0 + t < a.rows;
    fill[t] = 0;
  }
  if (t == 0) again = 0;
  __syncthreads();

  // ---- 2: histograms until the K-th entry's bin fits the list.
  float l = 0.f;
  for (int round = 1;; ++round) {
    const uint32_t b0 = base[col], wd = width[col], sh = shift[col];
    if (round == 1) {
      walk([&](auto whole, const sa_f32x16& x, int left) __attribute__((always_inline)) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (whole.value || exists(left, i)) {
            const float e = e_of(x[i]);
            sum += e;
            const uint32_t d = __builtin_elementwise_sub_sat(__float_as_uint(e), b0) >> sh;
            atomicAdd(&hist[32 * min(d, (uint32_t)kTmBins - 1) + col], 1u);
          }
        l += sum;
      });
    } else {
      const bool open = todo[col] != 0;
      walk([&](auto whole, const sa_f32x16& x, int left) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const uint32_t d = __float_as_uint(e_of(x[i])) - b0;
          if (open && d < wd && (whole.value || exists(left, i))) atomicAdd(&hist[32 * (d >> sh) + col], 1u);
        }
      });
    }
    __syncthreads();
    // 16 lanes per row: lane s sums bins 16 s .. + 15, then the counts from the top.
    {
      const int r = t >> 4, s = t & 15;
      const bool mine = todo[r] != 0;
      uint32_t h[16], tot = 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        h[i] = hist[32 * (16 * s + i) + r];
        tot += h[i];
      }
      uint32_t suffix = tot;  // entries in this lane's bins and above
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_down((int)suffix, o, 16);
        if (s + o < 16) suffix += y;
      }
      const uint32_t need = (uint32_t)a.K - above[r];
      const uint32_t over = suffix - tot;  // entries above this lane's bins
      __syncthreads();                     // every lane has read above and todo
      if (mine && over < need && suffix >= need) {  // the K-th is in one of this lane's bins
        uint32_t run = over;
        int bin = 15;
        for (; bin > 0; --bin) {
          if (run + h[bin] >= need) break;
          run += h[bin];
        }
        above[r] += run;
        count[r] = h[bin];
        base[r] += (uint32_t)(16 * s + bin) << shift[r];
        width[r] = 1u << shift[r];
        todo[r] = h[bin] > (uint32_t)kTmCap && shift[r] > 0;
        if (todo[r]) {
          shift[r] = shift[r] > 8 ? shift[r] - 8 : 0;
          again = round;
        }
      }
    }
    for (int i = t; i < kTmBins * 32; i += 64 * kTmWaves) hist[i] = 0;
    __syncthreads();
    if (again != round) break;
  }
  // ---- 3: the sum above the bin and the bin's entries.
  const uint32_t b0 = base[col], wd = width[col];
  const bool listed = count[col] <= (uint32_t)kTmCap;  // else the bin is one pattern
  float sum_above = 0.f;
  walk([&](auto whole, const sa_f32x16& x, int left) __attribute__((always_inline)) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float e = e_of(x[i]);
      const uint32_t u = __float_as_uint(e);
      if (whole.value || exists(left, i)) {
        sum += u >= b0 + wd ? e : 0.f;
        if (u - b0 < wd && listed) {
          const uint32_t at = atomicAdd(&fill[col], 1u);
          if (at < (uint32_t)kTmCap) list[32 * at + col] = u;
        }
      }
    }
    sum_above += sum;
  });
  l += half(l);
  sum_above += half(sum_above);
  if (hh == 0) {
    wred[wave][0][col] = l;
    wred[wave][1][col] = sum_above;
  }
  __syncthreads();
  // 16 lanes per row: the K-th largest is the (K - above)-th of the list, or the bin's one pattern.
  {
    const int r = t >> 4, s = t & 15;
    const uint32_t need = (uint32_t)a.K - above[r];
    const uint32_t nl = min(fill[r], (uint32_t)kTmCap);
    uint32_t v[kTmCap / 16];
#pragma unroll
    for (int i = 0; i < kTmCap / 16; ++i) {
      const uint32_t at = (uint32_t)(16 * i + s);
      v[i] = at < nl ? list[32 * at + r] : 0u;
    }
    uint32_t thr = base[r];
    double extra = 0.0;
    uint32_t gt = 0;
    if (count[r] <= (uint32_t)kTmCap) {
      thr = 0;
      for (int bit = 30; bit >= 0; --bit) {
        const uint32_t cand = thr | (1u << bit);
        uint32_t c = 0;
#pragma unroll
        for (int i = 0; i < kTmCap / 16; ++i) c += v[i] >= cand;
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) c += (uint32_t)__shfl_xor((int)c, o);
        if (c >= need) thr = cand;
      }
#pragma unroll
      for (int i = 0; i < kTmCap / 16; ++i)
        if (v[i] > thr) {
          extra += (double)__uint_as_float(v[i]);
          ++gt;
        }
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) {
        extra += __shfl_xor(extra, o);
        gt += (uint32_t)__shfl_xor((int)gt, o);
      }
    }
    if (s == 0 && row0 + r < a.rows) {
      float tot = 0.f, top = 0.f;
#pragma unroll
      for (int w = 0; w < kTmWaves; ++w) {
        tot += wred[w][0][r];
        top += wred[w][1][r];
      }
      const float ties = (float)((int)need - (int)gt) * __uint_as_float(thr);
      a.share[bh * a.rows + row0 + r] = (top + ((float)extra + ties)) / tot;
    }
  }
}

// Key operands: rows idx of x (zeros for -1) in the order of v_mfma_f32_32x32x16_bf16's A operand,
// out[bh][row / 32][s][lane (col, hh)] = x[b][h][idx[row]][16 s + 8 hh .. + 7], col = row % 32.
struct GatherOpsArgs {
  const uint16_t* x;
  int64_t sb, sh, sl;
  int H, L;
  const int32_t* idx;
  int n_pad;
  jd_u32x4* out;
  int64_t total;  // B * H * n_pad * 8
};

__global__ __launch_bounds__(256) void gather_operands_kernel(GatherOpsArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.total) return;
  const int c = (int)(i & 7);  // 16-byte chunk of the row: 8 lanes read one row
  const int64_t rb = i >> 3;
  const int64_t bh = rb / a.n_pad;
  const int row = (int)(rb - bh * a.n_pad);
  const int64_t b = bh / a.H;
  const int h = (int)(bh - b * a.H);
  const int src = a.idx[row];
  jd_u32x4 v = {0u, 0u, 0u, 0u};
  if ((unsigned)src < (unsigned)a.L)
    v = *reinterpret_cast<const jd_u32x4*>(a.x + b * a.sb + h * a.sh + (int64_t)src * a.sl + 8 * c);
  a.out[((bh * (a.n_pad / 32) + row / 32) * 4 + (c >> 1)) * 64 + (c & 1) * 32 + (row & 31)] = v;
}

// ---------------------------------------------------------------------------------------
// gram_kernel: one workgroup per (bh, key frame f2, chunk of kGramChunk sample positions s1).
// Thread t takes columns s2 = t, t + 256, ... of frame f2 and accumulates, over its s1 chunk,
// the products of the F values P[f1*ns + s1][f2*ns + s2] (f1 = 0..F-1) of each column.
// Partial sums go to G_part[bh][f2][chunk][pair]; the finish kernel adds the chunks in order.
constexpr int kGramChunk = 8;

struct GramArgs {
  const float* P;
  int64_t p_bh, p_row;
  int ns, n_chunks;
  float* G;  // [BH][F][n_chunks][F*(F+1)/2]
  int64_t total;
};

template <int F>
__global__ __launch_bounds__(256) void gram_kernel(GramArgs a) {
  constexpr int NP = F * (F + 1) / 2;
  __shared__ float part[4][NP];
  const int64_t w = blockIdx.x;
  if (w >= a.total) return;
  const int t = threadIdx.x, wave = t >> 6;
  const int64_t bhf = w / a.n_chunks;
  const int chunk = (int)(w - bhf * a.n_chunks);
  const int64_t bh = bhf / F;
  const int f2 = (int)(bhf - bh * F);
  const int s1_lo = chunk * kGramChunk, s1_hi = min(a.ns, s1_lo + kGramChunk);
  float acc[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) acc[p] = 0.f;
  const float* base = a.P + bh * a.p_bh + (int64_t)f2 * a.ns;
  for (int s2 = t; s2 < a.ns; s2 += 256) {
    for (int s1 = s1_lo; s1 < s1_hi; ++s1) {
      float x[F];
#pragma unroll
      for (int f1 = 0; f1 < F; ++f1) x[f1] = base[(int64_t)(f1 * a.ns + s1) * a.p_row + s2];
      int p = 0;
#pragma unroll
      for (int f1 = 0; f1 < F; ++f1)
#pragma unroll
        for (int f3 = f1; f3 < F; ++f3) {
          acc[p] = fmaf(x[f1], x[f3], acc[p]);
          ++p;
        }
    }
  }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const float r = wave_sum_f(acc[p]);
    if ((t & 63) == 0) part[wave][p] = r;
  }
  __syncthreads();
  float* out = a.G + (bhf * a.n_chunks + chunk) * NP;
  for (int p = t; p < NP; p += 256) out[p] = ((part[0][p] + part[1][p]) + part[2][p]) + part[3][p];
}

// ---------------------------------------------------------------------------------------
// simgram_kernel: judge_similarity with the probabilities kept on chip. One wave per (bh,
// chunk of kGramChunk = 8 sample positions s1). Its three 32-column query groups hold the
// F frames' rows f1*ns + s1 of the 8 positions, 12 columns per position: flat column
// 32 g + col = 12 j + f1 for position j of the chunk (columns with f1 >= F and positions
// past ns are zero queries whose results are never used).
// Per key frame f2, e = exp2(x - m) of the frame's ns keys, 32 at a time, goes through LDS
// ([key][flat column]) and the products e[f1][k] e[f3][k] are summed by v_mfma_f32_4x4x1_16b_f32,
// in fp32: block b of its 16 is position b % 8 at key 2 i + b / 8, its A and B operands four of
// the position's 12 columns (lane l: block l / 4, column l % 4), so three LDS reads feed the six
// column-group pairs u <= w.
//   kOne: one walk over the keys. m is the row's maximum over the first key tile (text keys carry
//     the bias, as in probs_kernel), the row sums add up beside the products, and the products,
//     kept per position, wait in a workspace until the sums are known: G = sum over the positions
//     of inv[f1] inv[f3] (e e). A row sum above kSgSumMax (or NaN) walks the keys for the exact
//     maxima first and starts again.
//   otherwise (no workspace): a first walk for the row sums, then normalised products.
// Bound: issue of scaling, exp2 and sums (VALU) and of the products, 3 G elements for 96 heads
// of 5 500 x 5 724, which do not overlap with this MFMA shape. Measured there, per judge: two
// walks with the products as 66 FMAs per (position, key) 2.2 ms, with MFMA products 1.85,
// one walk 1.44 (MFMA pipes busy 42 %).
struct SimGramArgs {
  const uint16_t* qs;  // [BH][rows_pad][64], row f*ns + s
  const uint16_t* ks;  // [BH][keys_pad][64], T text keys then F*ns sampled keys
  int ns, T, keys, keys_pad, rows_pad;
  float scale_log2, bias_log2;
  float* G;  // [BH][F][n_chunks][NP]
  int n_chunks;
  int64_t total;  // BH * n_chunks
  float* ws;      // kOne: [total][F][4 kPairs][32] unnormalised products
};

constexpr int kSgWidth = 12;                            // columns per position (F <= 12)
constexpr int kSgGroups = kGramChunk * kSgWidth / 32;  // query groups per wave
static_assert(kGramChunk * kSgWidth == 32 * kSgGroups, "positions fill whole query groups");
// LDS row stride (floats) of the e tile [key][flat column]: the product reads (8 positions x 4
// columns, 12 apart) of one key cover 32 of the 64 banks once.
constexpr int kSgStride = 32 * kSgGroups + 4;
constexpr float kSgSumMax = 0x1p60f;  // a product sum is at most the square of a row sum
constexpr int sg_pairs(int F) { return ((F + 3) / 4) * ((F + 3) / 4 + 1) / 2; }

__device__ inline sa_f32x4 mfma4x4(float a, float b, sa_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

template <int F, bool kOne>
__global__ __launch_bounds__(256, 2) void simgram_kernel(SimGramArgs a) {
  static_assert(F >= 1 && F <= 12, "frames");
  constexpr int NP = F * (F + 1) / 2;
  constexpr int kQuads = (F + 3) / 4;   // 4-column groups of a position
  constexpr int kPairs = sg_pairs(F);  // group pairs u <= w
  __shared__ __attribute__((aligned(16))) float lds[4][32 * kSgStride];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t wid = (int64_t)blockIdx.x * 4 + wave;
  if (wid >= a.total) return;  // no workgroup barriers below
  const int64_t bh = wid / a.n_chunks;
  const int chunk = (int)(wid - bh * a.n_chunks);
  const int col = lane & 31, hh = lane >> 5;
  float* L = lds[wave];

  sa_bf16x8 qf[kSgGroups][4];
#pragma unroll
  for (int g = 0; g < kSgGroups; ++g) {
    const int flat = 32 * g + col;
    const int s1 = chunk * kGramChunk + flat / kSgWidth, f1 = flat % kSgWidth;
    const bool ok = f1 < F && s1 < a.ns;
    const uint16_t* qp = a.qs + (bh * a.rows_pad + (ok ? f1 * a.ns + s1 : 0)) * kD + 8 * hh;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const jd_u32x4 w = ok ? *reinterpret_cast<const jd_u32x4*>(qp + 16 * s) : jd_u32x4{0u, 0u, 0u, 0u};
      qf[g][s] = __builtin_bit_cast(sa_bf16x8, w);
    }
  }

  float m[kSgGroups], l[kSgGroups];
  const uint16_t* kbase = a.ks + (bh * a.keys_pad + col) * kD + 8 * hh;
  // Row sums over key tiles [kt0, kt1) of the whole key list, keys >= end left out. kRunning: the
  // maxima follow the tiles; else they stay as they are.
  auto stats = [&](auto running_tag, int kt0, int kt1, int end) __attribute__((always_inline)) {
    constexpr bool kRunning = decltype(running_tag)::value;
    if (kt0 >= kt1) return;
    jd_u32x4 kop[4], knext[4];
    load_k(kbase + (int64_t)kt0 * 32 * kD, knext);
    for (int kt = kt0; kt < kt1; ++kt) {
#pragma unroll
      for (int s = 0; s < 4; ++s) kop[s] = knext[s];
      load_k(kbase + (int64_t)min(kt + 1, kt1 - 1) * 32 * kD, knext);  // in flight over this tile
      const bool uniform = 32 * kt + 32 <= end && (32 * kt + 32 <= a.T || 32 * kt >= a.T);
      const float tb = 32 * kt < a.T ? a.bias_log2 : 0.f;
#pragma unroll
      for (int g = 0; g < kSgGroups; ++g) {
        const sa_f32x16 t = score_tile_k(kop, qf[g]);
        if (!kRunning && uniform) {
          const float off = tb - m[g];
          float sum = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) sum += __builtin_amdgcn_exp2f(fmaf(t[i], a.scale_log2, off));
          l[g] += sum;
          continue;
        }
        float x[16], tmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = 32 * kt + 8 * (i >> 2) + 4 * hh + (i & 3);
          x[i] = key >= end ? -INFINITY : fmaf(t[i], a.scale_log2, key < a.T ? a.bias_log2 : 0.f);
        }
        if (kRunning) {
#pragma unroll
          for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, x[i]);
          const float mn = fmaxf(m[g], tmax);
          l[g] *= m[g] == mn ? 1.f : __builtin_amdgcn_exp2f(m[g] - mn);
          m[g] = mn;
        }
        if (m[g] != -INFINITY) {
          float sum = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) sum += __builtin_amdgcn_exp2f(x[i] - m[g]);
          l[g] += sum;
        }
      }
    }
  };
  // Both halves of a row's keys take one maximum, so that their sums add up directly.
  auto merge_max = [&]() {
#pragma unroll
    for (int g = 0; g < kSgGroups; ++g) {
      const auto mo = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[g]), __float_as_uint(m[g]), false, false);
      const float M = fmaxf(__uint_as_float(mo[0]), __uint_as_float(mo[1]));
      if (m[g] != M) l[g] *= __builtin_amdgcn_exp2f(m[g] - M);
      m[g] = M;
    }
  };
  auto reset = [&]() {
#pragma unroll
    for (int g = 0; g < kSgGroups; ++g) {
      m[g] = -INFINITY;
      l[g] = 0.f;
    }
  };
  float inv[kSgGroups];
  auto finish = [&]() {  // inv = 1 / row sum; true when a sum left the range (it is at least 1: the row's maximum of a tile)
    bool bad = false;
#pragma unroll
    for (int g = 0; g < kSgGroups; ++g) {
      const auto lo = __builtin_amdgcn_permlane32_swap(__float_as_uint(l[g]), __float_as_uint(l[g]), false, false);
      const float lt = __uint_as_float(lo[0]) + __uint_as_float(lo[1]);
      bad |= !(lt <= kSgSumMax);
      inv[g] = 1.f / lt;
    }
    return __ballot(bad) != 0;
  };
  const int n_tiles = a.keys_pad / 32;

  // Lane l reads column 4 u + l % 4 of position (l / 4) % 8 at key 2 i + l / 32.
  float* wp = L + 4 * hh * kSgStride + col;
  const float* rp = L + hh * kSgStride + kSgWidth * ((lane >> 2) & 7) + (lane & 3);
  const int n_kt = (a.ns + 31) / 32;
  // Products of key frame f2 (kOne: unnormalised, and the frame's part of the row sums).
  auto frame = [&](int f2, sa_f32x4 (&acc)[kPairs]) __attribute__((always_inline)) {
    const int frame0 = a.T + f2 * a.ns;
#pragma unroll
    for (int p = 0; p < kPairs; ++p) acc[p] = sa_f32x4{0.f, 0.f, 0.f, 0.f};
    auto load_frame = [&](int t, jd_u32x4 (&k4)[4]) {
      load_k(a.ks + (bh * a.keys_pad + min(frame0 + 32 * t + col, a.keys_pad - 1)) * kD + 8 * hh, k4);
    };
    jd_u32x4 kop[4], knext[4];
    load_frame(0, knext);
    for (int t = 0; t < n_kt; ++t) {
#pragma unroll
      for (int s = 0; s < 4; ++s) kop[s] = knext[s];
      load_frame(min(t + 1, n_kt - 1), knext);  // in flight over this tile
      const int left = a.ns - 32 * t;  // keys of the frame from this tile on
#pragma unroll
      for (int g = 0; g < kSgGroups; ++g) {
        sa_f32x16 e = score_tile_k(kop, qf[g]);
#pragma unroll
        for (int i = 0; i < 16; ++i) e[i] = __builtin_amdgcn_exp2f(fmaf(e[i], a.scale_log2, -m[g]));
        if (left < 32) {  // keys past the frame count for nothing
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (8 * (i >> 2) + 4 * hh + (i & 3) >= left) e[i] = 0.f;
        }
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (kOne) sum += e[i];
          else e[i] *= inv[g];
          wp[(8 * (i >> 2) + (i & 3)) * kSgStride + 32 * g] = e[i];
        }
        if (kOne) l[g] += sum;
      }
      __builtin_amdgcn_wave_barrier();
      // Operands of four steps are read while the previous four's products run.
      float x[2][4][kQuads];
      auto read4 = [&](int blk, float (&y)[4][kQuads]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int u = 0; u < kQuads; ++u) y[i][u] = rp[2 * (4 * blk + i) * kSgStride + 4 * u];
      };
      read4(0, x[0]);
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        if (blk < 3) read4(blk + 1, x[(blk + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          int p = 0;
#pragma unroll
          for (int u = 0; u < kQuads; ++u)
#pragma unroll
            for (int w = u; w < kQuads; ++w) {
              acc[p] = mfma4x4(x[blk & 1][i][u], x[blk & 1][i][w], acc[p]);
              ++p;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  // G of key frame f2 from v(p, i): the product sum of column 4 u + i and column 4 w + lane % 4 of
  // the lane's position (p = the pair u <= w), added over the 8 positions.
  auto write_g = [&](int f2, auto v) __attribute__((always_inline)) {
    float* out = a.G + ((bh * F + f2) * a.n_chunks + chunk) * NP;
    int p = 0;
#pragma unroll
    for (int u = 0; u < kQuads; ++u)
#pragma unroll
      for (int w = u; w < kQuads; ++w) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float sum = v(p, u, w, i);
#pragma unroll
          for (int o = 4; o < 32; o <<= 1) sum += __shfl_xor(sum, o);
          const int f1 = 4 * u + i, f3 = 4 * w + (lane & 3);
          if (lane < 4 && f1 <= f3 && f3 < F) out[f1 * F - f1 * (f1 - 1) / 2 + (f3 - f1)] = sum;
        }
        ++p;
      }
  };
  // Columns that are no sample (f1 >= F, positions past ns) weigh nothing.
  auto drop_unused = [&]() {
#pragma unroll
    for (int g = 0; g < kSgGroups; ++g) {
      const int flat = 32 * g + col;
      if (!(chunk * kGramChunk + flat / kSgWidth < a.ns && flat % kSgWidth < F)) inv[g] = 0.f;
    }
  };
  sa_f32x4 acc[kPairs];
  if constexpr (!kOne) {
    reset();
    stats(std::true_type{}, 0, n_tiles, a.keys);
    merge_max();
    finish();
    drop_unused();
    for (int f2 = 0; f2 < F; ++f2) {
      frame(f2, acc);
      write_g(f2, [&](int p, int, int, int i) { return acc[p][i] + __shfl_xor(acc[p][i], 32); });
    }
  } else {
    float* ws = a.ws + wid * (F * 4 * kPairs * 32);
    // Maxima over the first tile (after a failed walk: over every key), then the text keys' part of
    // the sums, then every frame's products to ws and its sums to l.
    for (int tiles = 1;; tiles = n_tiles) {
      reset();
      stats(std::true_type{}, 0, tiles, a.keys);
      merge_max();
#pragma unroll
      for (int g = 0; g < kSgGroups; ++g) l[g] = 0.f;
      stats(std::false_type{}, 0, (a.T + 31) / 32, a.T);
      for (int f2 = 0; f2 < F; ++f2) {
        frame(f2, acc);
#pragma unroll
        for (int p = 0; p < kPairs; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float sum = acc[p][i] + __shfl_xor(acc[p][i], 32);
            if (lane < 32) ws[(f2 * 4 * kPairs + 4 * p + i) * 32 + lane] = sum;
          }
      }
      if (!finish() || tiles == n_tiles) break;
    }
    drop_unused();
    // The rows' factors by flat column. Below every lane reads the products that lanes 0 .. 31 stored to
    // ws: a wave's accesses to memory take effect in its program order, so no wait is needed.
#pragma unroll
    for (int g = 0; g < kSgGroups; ++g)
      if (hh == 0) L[32 * g + col] = inv[g];
    __builtin_amdgcn_wave_barrier();
    const float* fp = L + kSgWidth * ((lane >> 2) & 7);
    float fa[kQuads * 4], fb[kQuads];  // factors of the position's columns and of 4 w + lane % 4
#pragma unroll
    for (int c = 0; c < 4 * kQuads; ++c) fa[c] = fp[c];
#pragma unroll
    for (int w = 0; w < kQuads; ++w) fb[w] = fp[4 * w + (lane & 3)];
    for (int f2 = 0; f2 < F; ++f2) {
      float e[4 * kPairs];
#pragma unroll
      for (int p = 0; p < 4 * kPairs; ++p) e[p] = ws[(f2 * 4 * kPairs + p) * 32 + (lane & 31)];
      write_g(f2, [&](int p, int u, int w, int i) { return e[4 * p + i] * fa[4 * u + i] * fb[w]; });
    }
  }
}

// ---------------------------------------------------------------------------------------
struct FinishArgs {
  const float* share;  // [BH][rows] or null
  const float* G1;     // [BH][F][n_chunks][NP] partials or null
  const float* G2;
  int BH, rows, F, n_chunks;
  float sparse_thr, sim_thr;
  float* share_mean;  // [BH]
  float* col1;        // [BH]
  float* col2;        // [BH]
  int32_t* use;       // [BH]
};

// Block sum over the 256 threads in a fixed order (per-wave shuffles, then the four waves).
__device__ float block_sum(float x, float* red /* LDS [4] */) {
  x = wave_sum_f(x);
  const int t = threadIdx.x;
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = x;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

// Mean cosine similarity of the patterns sharing a key frame, from one head's Gram partials:
// col = mean over f2 of mean over (f1, f3) of G[f2][f1][f3] / sqrt(G[f2][f1][f1] G[f2][f3][f3]).
__device__ float col_sim(const float* Gp, int F, int n_chunks, float* gs /* LDS [F * NP] */, float* red) {
  const int t = threadIdx.x;
  const int NP = F * (F + 1) / 2;
  __syncthreads();
  for (int e = t; e < F * NP; e += 256) {
    const int f2 = e / NP, p = e - f2 * NP;
    // Added in chunk order, eight loads at a time.
    const float* gp = Gp + (int64_t)f2 * n_chunks * NP + p;
    float s = 0.f;
    int c = 0;
    for (; c + 8 <= n_chunks; c += 8) {
      float y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = gp[(int64_t)(c + i) * NP];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += y[i];
    }
    for (; c < n_chunks; ++c) s += gp[(int64_t)c * NP];
    gs[e] = s;
  }
  __syncthreads();
  auto at = [&](const float* g, int i, int j) {
    if (i > j) {
      const int tmp = i;
      i = j;
      j = tmp;
    }
    return g[i * F - i * (i - 1) / 2 + (j - i)];
  };
  float part = 0.f;
  for (int u = t; u < F * F * F; u += 256) {
    const int f2 = u / (F * F), f1 = (u / F) % F, f3 = u % F;
    const float* g = gs + f2 * NP;
    part += at(g, f1, f3) / sqrtf(at(g, f1, f1) * at(g, f3, f3));
  }
  return block_sum(part, red) / (float)(F * F * F);
}

// One 256-thread workgroup per head.
__global__ __launch_bounds__(256) void finish_kernel(FinishArgs a) {
  __shared__ float gs[12 * 78];
  __shared__ float red[4];
  const int bh = blockIdx.x;
  if (bh >= a.BH) return;
  const int t = threadIdx.x;
  float s = 0.f;
  if (a.share) {
    for (int r = t; r < a.rows; r += 256) s += a.share[(int64_t)bh * a.rows + r];
    s = block_sum(s, red) / (float)a.rows;
  }
  const int NP = a.F * (a.F + 1) / 2;
  const int64_t gstride = (int64_t)a.F * a.n_chunks * NP;
  const float c1 = a.G1 ? col_sim(a.G1 + bh * gstride, a.F, a.n_chunks, gs, red) : 0.f;
  const float c2 = a.G2 ? col_sim(a.G2 + bh * gstride, a.F, a.n_chunks, gs, red) : 0.f;
  if (t == 0) {
    a.share_mean[bh] = s;
    a.col1[bh] = c1;
    a.col2[bh] = c2;
    a.use[bh] = (!(s > a.sparse_thr) && c1 > a.sim_thr && c2 > a.sim_thr) ? 1 : 0;
  }
}

}  // namespace

extern "C" int sa_sampled_probs(const uint16_t* q_rows, const uint16_t* k_rows, int BH, int rows, int rows_pad,
                                int keys, int keys_pad, float sm_scale, int n_bias, float bias, int c_lo, int c_hi,
                                float* P, int64_t p_bh_stride, int64_t p_row_stride, void* stream) {
  const char* fn = "sa_sampled_probs";
  SA_REQUIRE(q_rows && k_rows && P, "%s: null pointer", fn);
  SA_REQUIRE(reinterpret_cast<uintptr_t>(q_rows) % 16 == 0 && reinterpret_cast<uintptr_t>(k_rows) % 16 == 0,
             "%s: q_rows/k_rows must be 16-byte aligned", fn);
  SA_REQUIRE(BH > 0 && rows > 0 && keys > 0, "%s: bad shape", fn);
  SA_REQUIRE(rows_pad % 32 == 0 && rows_pad >= rows && keys_pad % 32 == 0 && keys_pad >= keys,
             "%s: rows_pad/keys_pad must be multiples of 32 covering rows/keys", fn);
  SA_REQUIRE(0 <= c_lo && c_lo < c_hi && c_hi <= keys, "%s: bad key range [%d, %d)", fn, c_lo, c_hi);
  SA_REQUIRE(std::isfinite(sm_scale) && sm_scale > 0.f, "%s: bad sm_scale", fn);
  SA_REQUIRE(p_row_stride >= c_hi - c_lo, "%s: p_row_stride too small", fn);
  ProbArgs a;
  a.qs = q_rows; a.ks = k_rows; a.rows = rows; a.rows_pad = rows_pad; a.keys = keys; a.keys_pad = keys_pad;
  a.scale_log2 = sm_scale * kLog2e; a.n_bias = n_bias; a.bias_log2 = bias * kLog2e;
  a.c_lo = c_lo; a.c_hi = c_hi; a.P = P; a.p_bh = p_bh_stride; a.p_row = p_row_stride;
  a.ng = rows_pad / 32; a.total = (int64_t)BH * a.ng;
  a.vec_ok = (reinterpret_cast<uintptr_t>(P) % 16 == 0 && p_row_stride % 4 == 0 && p_bh_stride % 4 == 0 &&
              c_lo % 4 == 0) ? 1 : 0;
  hipLaunchKernelGGL(probs_kernel, dim3((unsigned)((a.total + 3) / 4)), dim3(256), 0, sa::as_stream(stream), a);
  return sa::check_launch(fn);
}

extern "C" int sa_topk_share(const float* P, int64_t p_bh_stride, int64_t p_row_stride, int BH, int rows, int n,
                             int K, float* share, void* stream) {
  const char* fn = "sa_topk_share";
  SA_REQUIRE(P && share, "%s: null pointer", fn);
  SA_REQUIRE(BH > 0 && rows > 0 && n > 0 && K >= 1 && K <= n, "%s: bad shape (1 <= K <= n)", fn);
  if (n > 16384) return sa::fail(SA_ERR_UNSUPPORTED, "%s: n=%d > 16384", fn, n);
  ShareArgs a;
  a.P = P; a.p_bh = p_bh_stride; a.p_row = p_row_stride; a.rows = rows; a.n = n; a.K = K; a.share = share;
  a.vec_ok = (reinterpret_cast<uintptr_t>(P) % 16 == 0 && p_bh_stride % 4 == 0 && p_row_stride % 4 == 0) ? 1 : 0;
  a.total = (int64_t)BH * rows;
  hipLaunchKernelGGL(share_kernel, dim3((unsigned)a.total), dim3(256), 0, sa::as_stream(stream), a);
  return sa::check_launch(fn);
}

extern "C" int sa_gather_key_operands(const uint16_t* x, const int64_t strides[3], int B, int H, int L, int D,
                                      const int32_t* idx, int n_pad, uint16_t* out, void* stream) {
  const char* fn = "sa_gather_key_operands";
  SA_REQUIRE(x && strides && idx && out, "%s: null pointer", fn);
  SA_REQUIRE(B > 0 && H > 0 && L > 0 && n_pad > 0 && n_pad % 32 == 0, "%s: bad shape (n_pad a multiple of 32)", fn);
  if (D != kD) return sa::fail(SA_ERR_UNSUPPORTED, "%s: head_dim %d (64)", fn, D);
  SA_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
             "%s: x/out must be 16-byte aligned", fn);
  for (int i = 0; i < 3; ++i)
    if (strides[i] % 8 != 0) return sa::fail(SA_ERR_UNSUPPORTED, "%s: strides must be multiples of 8 elements", fn);
  GatherOpsArgs a;
  a.x = x; a.sb = strides[0]; a.sh = strides[1]; a.sl = strides[2]; a.H = H; a.L = L; a.idx = idx; a.n_pad = n_pad;
  a.out = reinterpret_cast<jd_u32x4*>(out);
  a.total = (int64_t)B * H * n_pad * 8;
  SA_REQUIRE((a.total + 255) / 256 < (1LL << 31), "%s: grid too large", fn);
  hipLaunchKernelGGL(gather_operands_kernel, dim3((unsigned)((a.total + 255) / 256)), dim3(256), 0,
                     sa::as_stream(stream), a);
  return sa::check_launch(fn);
}

extern "C" int sa_topk_mass(const uint16_t* q_rows, const uint16_t* k_ops, int BH, int rows, int rows_pad, int n,
                            int n_pad, float sm_scale, int K, float* share, void* stream) {
  const char* fn = "sa_topk_mass";
  SA_REQUIRE(q_rows && k_ops && share, "%s: null pointer", fn);
  SA_REQUIRE(reinterpret_cast<uintptr_t>(q_rows) % 16 == 0 && reinterpret_cast<uintptr_t>(k_ops) % 16 == 0,
             "%s: q_rows/k_ops must be 16-byte aligned", fn);
  SA_REQUIRE(BH > 0 && rows > 0 && n > 0 && K >= 1 && K <= n, "%s: bad shape (1 <= K <= n)", fn);
  SA_REQUIRE(rows_pad % 32 == 0 && rows_pad >= rows && n_pad % 32 == 0 && n_pad >= n,
             "%s: rows_pad/n_pad must be multiples of 32 covering rows/n", fn);
  SA_REQUIRE(std::isfinite(sm_scale) && sm_scale > 0.f, "%s: bad sm_scale", fn);
  if (n > 16384) return sa::fail(SA_ERR_UNSUPPORTED, "%s: n=%d > 16384", fn, n);
  TopkMassArgs a;
  a.qs = q_rows; a.ks = reinterpret_cast<const jd_u32x4*>(k_ops); a.rows = rows; a.rows_pad = rows_pad;
  a.n = n; a.n_tiles = n_pad / 32; a.K = K; a.scale_log2 = sm_scale * kLog2e; a.share = share;
  a.ng = (rows + 31) / 32;
  a.BH = BH;
  const int64_t grid = ((int64_t)BH + 7) / 8 * 8 * a.ng;
  SA_REQUIRE(grid < (1LL << 31), "%s: grid too large", fn);
  hipLaunchKernelGGL(topk_mass_kernel, dim3((unsigned)grid), dim3(64 * kTmWaves), 0, sa::as_stream(stream), a);
  return sa::check_launch(fn);
}

extern "C" int sa_pattern_gram(const float* P, int64_t p_bh_stride, int64_t p_row_stride, int BH, int F, int ns,
                               float* G, void* stream) {
  const char* fn = "sa_pattern_gram";
  SA_REQUIRE(P && G, "%s: null pointer", fn);
  SA_REQUIRE(BH > 0 && ns > 0 && ns <= 512, "%s: bad shape (ns <= 512)", fn);
  SA_REQUIRE(F >= 1 && F <= 12, "%s: frames %d outside [1, 12]", fn, F);
  GramArgs a;
  a.P = P; a.p_bh = p_bh_stride; a.p_row = p_row_stride; a.ns = ns; a.G = G;
  a.n_chunks = (ns + kGramChunk - 1) / kGramChunk;
  a.total = (int64_t)BH * F * a.n_chunks;
  const dim3 g((unsigned)a.total), blk(256);
  hipStream_t s = sa::as_stream(stream);
  switch (F) {
#define SA_GRAM_CASE(n)\
  case n:              \
    hipLaunchKernelGGL(gram_kernel<n>, g, blk, 0, s, a);\
    break;
    SA_GRAM_CASE(1) SA_GRAM_CASE(2) SA_GRAM_CASE(3) SA_GRAM_CASE(4) SA_GRAM_CASE(5) SA_GRAM_CASE(6)
    SA_GRAM_CASE(7) SA_GRAM_CASE(8) SA_GRAM_CASE(9) SA_GRAM_CASE(10) SA_GRAM_CASE(11) SA_GRAM_CASE(12)
#undef SA_GRAM_CASE
  }
  return sa::check_launch(fn);
}

extern "C" int sa_pattern_judge_finish(const float* share, const float* G1, const float* G2, int BH, int rows, int F,
                                       int ns, float sparse_thr, float sim_thr, float* share_mean, float* col1, float* col2,
                                       int32_t* use, void* stream) {
  const char* fn = "sa_pattern_judge_finish";
  SA_REQUIRE(share_mean && col1 && col2 && use, "%s: null output", fn);
  SA_REQUIRE(BH > 0 && rows > 0 && F >= 1 && F <= 12 && ns > 0, "%s: bad shape", fn);
  FinishArgs a;
  a.share = share; a.G1 = G1; a.G2 = G2; a.BH = BH; a.rows = rows; a.F = F;
  a.n_chunks = (ns + kGramChunk - 1) / kGramChunk;
  a.sparse_thr = sparse_thr; a.sim_thr = sim_thr; a.share_mean = share_mean; a.col1 = col1; a.col2 = col2; a.use = use;
  hipLaunchKernelGGL(finish_kernel, dim3((unsigned)BH), dim3(256), 0, sa::as_stream(stream), a);
  return sa::check_launch(fn);
}

namespace {

int launch_sim_gram(const uint16_t* q_rows, const uint16_t* k_rows, int BH, int F, int ns, int T, int rows_pad,
                    int keys_pad, float sm_scale, float bias, float* G, float* ws, void* stream, const char* fn) {
  SA_REQUIRE(q_rows && k_rows && G, "%s: null pointer", fn);
  SA_REQUIRE(reinterpret_cast<uintptr_t>(q_rows) % 16 == 0 && reinterpret_cast<uintptr_t>(k_rows) % 16 == 0,
             "%s: q_rows/k_rows must be 16-byte aligned", fn);
  SA_REQUIRE(BH > 0 && F >= 1 && F <= 12 && ns > 0 && T >= 0, "%s: bad shape (1 <= F <= 12)", fn);
  SA_REQUIRE(rows_pad % 32 == 0 && rows_pad >= F * ns && keys_pad % 32 == 0 && keys_pad >= T + F * ns,
             "%s: rows_pad/keys_pad must be multiples of 32 covering F*ns / T+F*ns", fn);
  SA_REQUIRE(std::isfinite(sm_scale) && sm_scale > 0.f && std::isfinite(bias), "%s: bad sm_scale/bias", fn);
  SimGramArgs a;
  a.qs = q_rows; a.ks = k_rows; a.ns = ns; a.T = T; a.keys = T + F * ns; a.keys_pad = keys_pad; a.rows_pad = rows_pad;
  a.scale_log2 = sm_scale * kLog2e; a.bias_log2 = bias * kLog2e; a.G = G;
  a.n_chunks = (ns + kGramChunk - 1) / kGramChunk;
  a.total = (int64_t)BH * a.n_chunks;
  a.ws = ws;
  const dim3 grid((unsigned)((a.total + 3) / 4)), blk(256);
  hipStream_t s = sa::as_stream(stream);
  switch (F) {
#define SA_SG_CASE(n)                                                              \
  case n:                                                                          \
    if (ws) hipLaunchKernelGGL((simgram_kernel<n, true>), grid, blk, 0, s, a);     \
    else hipLaunchKernelGGL((simgram_kernel<n, false>), grid, blk, 0, s, a);       \
    break;
    SA_SG_CASE(1) SA_SG_CASE(2) SA_SG_CASE(3) SA_SG_CASE(4) SA_SG_CASE(5) SA_SG_CASE(6)
    SA_SG_CASE(7) SA_SG_CASE(8) SA_SG_CASE(9) SA_SG_CASE(10) SA_SG_CASE(11) SA_SG_CASE(12)
#undef SA_SG_CASE
  }
  return sa::check_launch(fn);
}

}  // namespace

extern "C" int sa_pattern_sim_gram(const uint16_t* q_rows, const uint16_t* k_rows, int BH, int F, int ns, int T,
                                   int rows_pad, int keys_pad, float sm_scale, float bias, float* G, void* stream) {
  return launch_sim_gram(q_rows, k_rows, BH, F, ns, T, rows_pad, keys_pad, sm_scale, bias, G, nullptr, stream,
                         "sa_pattern_sim_gram");
}

extern "C" int sa_pattern_sim_gram_workspace(int BH, int F, int ns, int64_t* bytes) {
  const char* fn = "sa_pattern_sim_gram_workspace";
  SA_REQUIRE(bytes, "%s: null bytes", fn);
  SA_REQUIRE(BH > 0 && F >= 1 && F <= 12 && ns > 0, "%s: bad shape (1 <= F <= 12)", fn);
  *bytes = (int64_t)BH * ((ns + kGramChunk - 1) / kGramChunk) * F * 4 * sg_pairs(F) * 32 * 4;
  return sa::ok();
}

extern "C" int sa_pattern_sim_gram_ws(const uint16_t* q_rows, const uint16_t* k_rows, int BH, int F, int ns, int T,
                                      int rows_pad, int keys_pad, float sm_scale, float bias, float* G,
                                      void* workspace, int64_t workspace_bytes, void* stream) {
  const char* fn = "sa_pattern_sim_gram_ws";
  int64_t need = 0;
  if (int rc = sa_pattern_sim_gram_workspace(BH, F, ns, &need)) return rc;
  SA_REQUIRE(workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "%s: workspace null or not 16-byte aligned",
             fn);
  SA_REQUIRE(workspace_bytes >= need, "%s: workspace of %lld bytes < %lld", fn, (long long)workspace_bytes,
             (long long)need);
  return launch_sim_gram(q_rows, k_rows, BH, F, ns, T, rows_pad, keys_pad, sm_scale, bias, G,
                         static_cast<float*>(workspace), stream, fn);
}
