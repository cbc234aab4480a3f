// Block-sparse attention forward for fp32 q, k, v: the reference kernel takes any float type
// (utils/block_sparse_attn_kernel.py:52-209: tl.dot of the loaded tiles, P cast to v's dtype,
// :107, i.e. kept in fp32 here). Same list contract as sa_block_sparse_fwd (attn_fwd.hip);
// head dim 64 or 128, no key bias. A pooling mode serves attn_with_pooling in fp32
// (utils/attn_pooling_kernel.py:230-287, which computes in fp32): each row's largest scaled
// logit per 32- or 64-key column and its log2-sum-exp2 are stored for the pooled-map reduce,
// with grouped key heads and a causal diagonal tile.
//
// One wave computes one 64-row query block with v_mfma_f32_16x16x4_f32 (head dim 128: two
// 64-wide halves of d in the S contraction, eight 16-row d blocks of O^T). Operand layouts of
// that instruction: A (16 x 4) lane l holds A[l % 16][l / 16], B (4 x 16) lane l holds
// B[l / 16][l % 16], D (16 x 16) lane l holds D[4 (l / 16) + i][l % 16], i < 4. Both
// contractions use an order of their index that keeps each lane's operands contiguous:
//   S^T = K Q^T over d: k-slot g = l / 16 and step s take d = 16 g + s, so lane l reads 16
//     consecutive floats of one K row and of one Q row;
//   O^T = V^T P^T over the 64 keys of a tile: 16-key group kb16, k-slot g and step i take key
//     16 kb16 + 4 g + i, which is where the S^T output already holds P (D row 4 g + i), so P
//     is the B operand in place; the A operand is V[key][d] for d = 16 dblk + l % 16.
// A sum over d (or over keys) in any order is the same sum; only the fp32 rounding order
// differs from a sequential loop. The running row maximum is kept per 64-key tile (exact
// rescale, no threshold), P = exp2(S * scale * log2(e) - m) in fp32, row sums in fp32.
// Keys past Lk and list entries outside [0, nkb) get P = 0; their K/V loads are clamped to
// the last key row, so every load is inside the tensors.
//
// With a workspace, bsa_fwd_f32_terms_kernel computes the same products on the bf16 matrix
// core, 16 times the fp32 one's rate: every operand is split exactly into three bf16 terms
// (x = hi + mid + lo, 8 significand bits each) and each product takes the six term products
// down to 2^-18 of the largest (hi.hi, hi.mid, mid.hi, mid.mid, hi.lo, lo.hi; the dropped ones
// are below 2^-26), accumulated in fp32. See that kernel below.
#include <type_traits>

#include "sa_common.h"

#include <cmath>

namespace {

constexpr int kBlk = 64;     // rows per query block == keys per key block
constexpr int kWavesF32 = 4;  // independent waves per workgroup
constexpr float kLog2eF32 = 1.4426950408889634f;

struct F32Args {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  int64_t q_sb, q_sh, q_sl;
  int64_t k_sb, k_sh, k_sl;
  int64_t v_sb, v_sh, v_sl;
  int64_t o_sb, o_sh, o_sl;
  int H, Lq, Lk, nqb, nkb;
  int n_items;
  const int32_t* order;  // dispatch slot -> item, -1 = idle; may be null
  int n_slots;
  const int32_t* kv_idx;
  const int32_t* kv_cnt;
  int max_cnt;
  int list_bh_stride;  // list row = bh * list_bh_stride + qb (0: lists shared by heads)
  float scale_log2;    // sm_scale * log2(e)
  int kv_rep;          // query heads per key/value head
  int causal;          // the tile of key block qb masks keys past the query (Lq == Lk)
  // Pooling (kPool 32 or 64): the row's maximum scaled logit (log2 domain) per kPool-key
  // column to pool_r[((bh * nqb + row / 64) * pool_ncol + column) * 64 + row % 64] and its
  // log2-sum-exp2 to pool_lse[bh * pool_lpad + row].
  float* pool_r;
  int pool_ncol;
  float* pool_lse;
  int pool_lpad;
  // bsa_fwd_f32_terms_kernel: the split operands and the per-key-block flags (f32_terms_kernel).
  const uint8_t* planes;
  const uint4* flags;
  int plain_after;  // bsa_fwd_f32_kernel follows for the heads flagged kTermSkip
};

__device__ inline sa_f32x4 mfma16x4(float a, float b, sa_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// max / sum over the four lanes r, r + 16, r + 32, r + 48 (the k-slots of one MFMA column).
__device__ inline float slot_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}
__device__ inline float slot_sum(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

// One wave's fp32 pass over list positions it0, it0 + step, ... of query block qb: rows
// 64 qb + row0 + (0 .. 16 kJ - 1). Leaves O^T (unnormalised), the running maxima and this
// lane's row-sum parts in acc, m and l.
template <int kD, int kPool, int kJ>
__device__ __forceinline__ void f32_rows(const F32Args& a, int bh, int qb, int row0, int it0, int step, int lane,
                                         sa_f32x4 (&acc)[kD / 16][kJ], float (&m)[kJ], float (&l)[kJ]) {
  constexpr int kHalf = kD / 64;   // 64-wide halves of d
  constexpr int kDB = kD / 16;     // 16-row d blocks of O^T
  const int b = bh / a.H;
  const int h = bh - b * a.H;
  const int hk = a.kv_rep > 1 ? h / a.kv_rep : h;
  const int r = lane & 15;  // MFMA row of A, column of B and D
  const int g = lane >> 4;  // MFMA k-slot

  const int64_t list_row = (int64_t)bh * a.list_bh_stride + qb;
  int cnt = a.kv_cnt[list_row];
  cnt = cnt < 0 ? 0 : (cnt > a.max_cnt ? a.max_cnt : cnt);
  const __attribute__((address_space(4))) int32_t* list =
      (const __attribute__((address_space(4))) int32_t*)(a.kv_idx + list_row * a.max_cnt);

  const float* qbase = a.q + b * a.q_sb + h * a.q_sh;
  const float* khead = a.k + b * a.k_sb + hk * a.k_sh;
  const float* vhead = a.v + b * a.v_sb + hk * a.v_sh;

  // Q^T B operands: qop[j][hf][s] = Q[qb * 64 + row0 + 16 j + r][64 hf + 16 g + s] (rows clamped
  // into Lq; the clamped rows are never stored).
  float qop[kJ][kHalf][16];
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const int row = min(qb * kBlk + row0 + 16 * j + r, a.Lq - 1);
#pragma unroll
    for (int hf = 0; hf < kHalf; ++hf) {
      const float4* p = reinterpret_cast<const float4*>(qbase + (int64_t)row * a.q_sl + 64 * hf + 16 * g);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float4 w = p[c];
        qop[j][hf][4 * c] = w.x;
        qop[j][hf][4 * c + 1] = w.y;
        qop[j][hf][4 * c + 2] = w.z;
        qop[j][hf][4 * c + 3] = w.w;
      }
    }
  }

  // acc[dblk][j]: O^T[16 dblk + 4 g + i][16 j + r]; m, l per query column j (log2 domain).
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    m[j] = -INFINITY;
    l[j] = 0.f;
#pragma unroll
    for (int dblk = 0; dblk < kDB; ++dblk) acc[dblk][j] = sa_f32x4{0.f, 0.f, 0.f, 0.f};
  }

  for (int it = it0; it < cnt; it += step) {
    const int kb = list[it];
    const bool ok = (unsigned)kb < (unsigned)a.nkb;
    const int key0 = ok ? kb * kBlk : 0;
    const int nvalid = ok ? min(kBlk, a.Lk - key0) : 0;
    const bool diag = kPool != 0 && a.causal && kb == qb;  // causal lists exist for pooling only

    // ---- S^T[16 kb16 + 4 g + i][16 j + r] in S[kb16][j][i].
    sa_f32x4 S[4][kJ];
#pragma unroll
    for (int kb16 = 0; kb16 < 4; ++kb16) {
      const int key = min(key0 + 16 * kb16 + r, a.Lk - 1);
      float kop[kHalf][16];
#pragma unroll
      for (int hf = 0; hf < kHalf; ++hf) {
        const float4* p = reinterpret_cast<const float4*>(khead + (int64_t)key * a.k_sl + 64 * hf + 16 * g);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float4 w = p[c];
          kop[hf][4 * c] = w.x;
          kop[hf][4 * c + 1] = w.y;
          kop[hf][4 * c + 2] = w.z;
          kop[hf][4 * c + 3] = w.w;
        }
      }
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        sa_f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int hf = 0; hf < kHalf; ++hf)
#pragma unroll
          for (int s = 0; s < 16; ++s) t = mfma16x4(kop[hf][s], qop[j][hf][s], t);
        S[kb16][j] = t;
      }
    }

    // ---- Masks (keys past Lk; keys past the query on the causal diagonal tile), pooled
    // column maxima, running maximum per query, then P = exp2(S * sc - m) in place and the
    // row sums.
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      float mx = -INFINITY;
#pragma unroll
      for (int kb16 = 0; kb16 < 4; ++kb16)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kk = 16 * kb16 + 4 * g + i;
          if (kk >= nvalid || (kPool != 0 && diag && kk > row0 + 16 * j + r)) S[kb16][j][i] = -INFINITY;
          mx = fmaxf(mx, S[kb16][j][i]);
        }
      if constexpr (kPool != 0) {
        if (ok) {
          constexpr int kCols = kBlk / kPool;  // columns per tile
#pragma unroll
          for (int cc = 0; cc < kCols; ++cc) {
            float x = -INFINITY;
#pragma unroll
            for (int kb16 = cc * (4 / kCols); kb16 < (cc + 1) * (4 / kCols); ++kb16)
#pragma unroll
              for (int i = 0; i < 4; ++i) x = fmaxf(x, S[kb16][j][i]);
            x = slot_max(x) * a.scale_log2;  // scale > 0
            if (g == 0)
              a.pool_r[(((int64_t)bh * a.nqb + qb) * a.pool_ncol + kb * kCols + cc) * kBlk + row0 +
                     16 * j + r] = x;
          }
        }
      }
      const float cand = slot_max(mx) * a.scale_log2;  // scale > 0
      const float m_new = fmaxf(m[j], cand);
      if (m_new != -INFINITY) {  // otherwise nothing is accumulated yet and every P is 0
        const float alpha = exp2f(m[j] - m_new);  // 0 when m = -inf
        m[j] = m_new;
        l[j] *= alpha;
#pragma unroll
        for (int dblk = 0; dblk < kDB; ++dblk) acc[dblk][j] *= alpha;
      }
      const float mu = m[j] == -INFINITY ? 0.f : m[j];
#pragma unroll
      for (int kb16 = 0; kb16 < 4; ++kb16)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = exp2f(fmaf(S[kb16][j][i], a.scale_log2, -mu));  // -inf -> 0
          S[kb16][j][i] = p;
          l[j] += p;
        }
    }

    // ---- O^T += V^T P^T: key 16 kb16 + 4 g + i, A = V[key][16 dblk + r], B = P in place.
#pragma unroll
    for (int kb16 = 0; kb16 < 4; ++kb16)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = min(key0 + 16 * kb16 + 4 * g + i, a.Lk - 1);
        const float* vrow = vhead + (int64_t)key * a.v_sl + r;
        float vop[kDB];
#pragma unroll
        for (int dblk = 0; dblk < kDB; ++dblk) vop[dblk] = vrow[16 * dblk];
#pragma unroll
        for (int dblk = 0; dblk < kDB; ++dblk)
#pragma unroll
          for (int j = 0; j < kJ; ++j) acc[dblk][j] = mfma16x4(vop[dblk], S[kb16][j][i], acc[dblk][j]);
      }
  }
}

// Epilogue of one wave: out = acc / l; an empty list writes 0. Pooling: the row's log2-sum-exp2.
template <int kD, int kPool, int kJ>
__device__ __forceinline__ void f32_store(const F32Args& a, int bh, int qb, int row0, int lane,
                                          const sa_f32x4 (&acc)[kD / 16][kJ], const float (&m)[kJ],
                                          const float (&l)[kJ]) {
  const int b = bh / a.H;
  const int h = bh - b * a.H;
  const int r = lane & 15, g = lane >> 4;
  float* obase = a.o + b * a.o_sb + h * a.o_sh;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const float l_tot = slot_sum(l[j]);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const int row = qb * kBlk + row0 + 16 * j + r;
    if constexpr (kPool != 0) {
      if (g == 0) a.pool_lse[(int64_t)bh * a.pool_lpad + row] = (m[j] == -INFINITY ? 0.f : m[j]) + log2f(l_tot);
    }
    if (row < a.Lq) {
      float* orow = obase + (int64_t)row * a.o_sl;
#pragma unroll
      for (int dblk = 0; dblk < kD / 16; ++dblk) {
        const sa_f32x4 A = acc[dblk][j];
        *reinterpret_cast<float4*>(orow + 16 * dblk + 4 * g) = make_float4(A[0] * inv, A[1] * inv, A[2] * inv, A[3] * inv);
      }
    }
  }
}

// Bits of |x| (see f32_terms_kernel).
constexpr uint32_t kTermMax = 0x5d800000u;  // 2^60
constexpr uint32_t kTermMin = 0x17800000u;  // 2^-80: 2^18 products that lose 2^-126 lose 2^-28 of a value
constexpr uint32_t kTermSkip = 0xffffffffu;  // no |x| has these bits

template <int kD, int kPool>
__global__ __launch_bounds__(64 * kWavesF32, kD == 64 ? 2 : 1) void bsa_fwd_f32_kernel(F32Args a) {
  static_assert(kD == 64 || kD == 128, "head dim 64 or 128");
  static_assert(kPool == 0 || kPool == 32 || kPool == 64, "pooling columns of 32 or 64 keys");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = blockIdx.x * kWavesF32 + wave;
  if (slot >= a.n_slots) return;
  const int item = __builtin_amdgcn_readfirstlane(a.order ? order_item(a.order, slot) : slot);
  if (item < 0 || item >= a.n_items) return;
  const int bh = item / a.nqb;
  const int qb = item - bh * a.nqb;
  // Behind bsa_fwd_f32_terms_kernel: the heads that it left (plain lists, so kv_rep = 1).
  if (a.flags && a.flags[(int64_t)bh * a.nkb].x != kTermSkip) return;
  sa_f32x4 acc[kD / 16][4];
  float m[4], l[4];
  f32_rows<kD, kPool, 4>(a, bh, qb, 0, 0, 1, lane, acc, m, l);
  f32_store<kD, kPool, 4>(a, bh, qb, 0, lane, acc, m, l);
}

// ---------------------------------------------------------------------------------------
// Split operands. f32_terms_kernel writes, per key/value head and 64-key block, the three bf16
// terms of the block's K and V in the order in which bsa_fwd_f32_terms_kernel consumes them:
// per 32-key chunk c, groups of six 1 KB operands (16 bytes per lane, lane l at 16 l), so that
// every operand load is one coalesced 1 KB read and takes no LDS:
//   K group i (d steps s = 2 i, 2 i + 1 of 16): operand 3 (s % 2) + term, lane (col, hh) holds
//     K[32 c + col][16 s + 8 hh .. + 7], the A operand of S^T = K Q^T;
//   V group (u, dp) (16 keys from 32 c + 16 u, d chunks dc = 2 dp, 2 dp + 1 of 32): operand
//     3 (dc % 2) + term, lane (col, hh) holds V[32 c + 16 u + 8 (j / 4) + 4 hh + j % 4]
//     [32 dc + col], j < 8: the A operand of O^T = V^T P^T for the key slots in which S^T leaves P.
// Rows past Lk are zero. flags[head * nkb + block] = the largest |k| of the block's two chunks
// and the largest |v| of its two chunks (fp32 bits), or kTermMax where one of a chunk's values is
// not 0 but below kTermMin. The attention takes the split operands only where all are below
// kTermMax: no inf or NaN, no product near overflow, and every value's low term (2^-16 of it) and
// its products with probabilities far enough above 2^-126. Other heads run in fp32. (One value
// decides for its head: a column or block of small values beside ordinary ones would lose its
// low terms however large the head's maximum is.)
// A head whose lists hold too few tiles to be worth the pass (terms_min_tiles4) is only flagged
// (kTermSkip) and runs in fp32.

template <int kD>
struct TermLayout {
  static constexpr int kGroup = 6 * 1024;                  // bytes per group
  static constexpr int kKGroups = kD / 32;                 // K groups per 32-key chunk
  static constexpr int kGroups = kKGroups + 2 * (kD / 64);  // all groups per chunk
  static constexpr int kTile = 2 * kGroups * kGroup;        // bytes per 64-key block: 768 kD
};

typedef unsigned f32_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 f32_bf16x2 __attribute__((ext_vector_type(2)));

__device__ inline uint32_t pack_bf16(float x0, float x1) {  // round to nearest even
  const f32_bf16x2 r = {(__bf16)x0, (__bf16)x1};
  return __builtin_bit_cast(uint32_t, r);
}

// The three bf16 terms of x0 and x1, packed: each remainder is exact in fp32, and the last one
// has at most 8 significand bits, so hi + mid + lo = x (above bf16's subnormals).
__device__ inline void split3(float x0, float x1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = pack_bf16(x0, x1);
  const float a0 = x0 - __uint_as_float(hi << 16), a1 = x1 - __uint_as_float(hi & 0xffff0000u);
  mid = pack_bf16(a0, a1);
  lo = pack_bf16(a0 - __uint_as_float(mid << 16), a1 - __uint_as_float(mid & 0xffff0000u));
}

__device__ inline uint32_t abs_bits(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// Largest and, 0 apart, smallest |x| of a wave's operands.
struct TermRange {
  uint32_t hi = 0u, lo1 = 0xffffffffu;  // lo1: the smallest less one, so that 0 counts as the largest
  __device__ void add(float x) {
    const uint32_t b = abs_bits(x);
    hi = max(hi, b);
    lo1 = min(lo1, b - 1u);
  }
  __device__ uint32_t flag() const { return lo1 < kTermMin - 1u ? max(hi, kTermMax) : hi; }
};

__device__ inline uint32_t wave_max_u(uint32_t x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = max(x, (uint32_t)__shfl_xor((int)x, o));
  return x;
}

struct TermArgs {
  const float* k;
  const float* v;
  int64_t k_sb, k_sh, k_sl;
  int64_t v_sb, v_sh, v_sl;
  int Hk, Lk, nkb;
  const int32_t* kv_cnt;  // [B * Hk][nqb] list lengths, or null: every block is split
  int nqb, max_cnt;
  int min_tiles4;  // listed tiles per four key blocks from which splitting pays,
  int together;    // by the launch's mean, unless a head is far off; else by each head's
  uint32_t lists;  // B * Hk * nqb
  uint8_t* planes;
  uint32_t* flags;  // [B * Hk * nkb][4]
};

// One workgroup per (head, key block): waves 0, 1 split the K chunks, waves 2, 3 the V chunks.
// HBM-bound: 512 kD bytes read and 768 kD written per block.
template <int kD>
__global__ __launch_bounds__(256) void f32_terms_kernel(TermArgs a) {
  typedef TermLayout<kD> Lay;
  __shared__ int64_t tiles[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t blk = blockIdx.x;
  const int bh = (int)(blk / a.nkb);
  const int kb = (int)(blk - (int64_t)bh * a.nkb);
  if (a.kv_cnt) {
    auto count = [&](int64_t row) { return min(max(a.kv_cnt[row], 0), a.max_cnt); };
    int64_t n = 0;
    for (int i = threadIdx.x; i < a.nqb; i += 256) n += count((int64_t)bh * a.nqb + i);
    // 64 of the launch's lists, at scattered places, the same in every wave.
    int64_t m = a.together ? count((uint32_t)lane * 2654435761u % a.lists) : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      n += __shfl_xor(n, o);
      m += __shfl_xor(m, o);
    }
    if (lane == 0) tiles[wave] = n;
    __syncthreads();
    int min4 = a.min_tiles4;
    if (a.together) min4 = m * a.nqb * 4 < (int64_t)min4 * a.nkb * 64 ? max(min4, 12) : min(min4, 5);
    if (4 * (tiles[0] + tiles[1] + tiles[2] + tiles[3]) < min4 * (int64_t)a.nkb) {
      if (threadIdx.x < 4) a.flags[blk * 4 + threadIdx.x] = kTermSkip;
      return;
    }
  }
  const int b = bh / a.Hk, h = bh - b * a.Hk;
  const int col = lane & 31, hh = lane >> 5;
  const int c = wave & 1;
  const int key0 = kb * kBlk + 32 * c;
  uint8_t* dst = a.planes + blk * Lay::kTile + c * Lay::kGroups * Lay::kGroup + 16 * lane;
  TermRange range;
  auto put = [&](int group, int operand, const float (&x)[8]) {
    f32_u32x4 t[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t hi, mid, lo;
      split3(x[2 * i], x[2 * i + 1], hi, mid, lo);
      t[0][i] = hi;
      t[1][i] = mid;
      t[2][i] = lo;
      range.add(x[2 * i]);
      range.add(x[2 * i + 1]);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *reinterpret_cast<f32_u32x4*>(dst + group * Lay::kGroup + (operand + p) * 1024) = t[p];
  };
  if (wave < 2) {
    const int key = key0 + col;
    const float* row = a.k + b * a.k_sb + h * a.k_sh + (int64_t)min(key, a.Lk - 1) * a.k_sl + 8 * hh;
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) {
      const float4 x0 = *reinterpret_cast<const float4*>(row + 16 * s);
      const float4 x1 = *reinterpret_cast<const float4*>(row + 16 * s + 4);
      float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = key < a.Lk ? x[j] : 0.f;
      put(s >> 1, 3 * (s & 1), x);
    }
  } else {
    const float* base = a.v + b * a.v_sb + h * a.v_sh + col;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int dc = 0; dc < kD / 32; ++dc) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int key = key0 + 16 * u + 8 * (j >> 2) + 4 * hh + (j & 3);
          const float y = base[(int64_t)min(key, a.Lk - 1) * a.v_sl + 32 * dc];
          x[j] = key < a.Lk ? y : 0.f;
        }
        put(Lay::kKGroups + u * (kD / 64) + (dc >> 1), 3 * (dc & 1), x);
      }
  }
  const uint32_t flag = wave_max_u(range.flag());
  if (lane == 0) a.flags[blk * 4 + wave] = flag;
}

__device__ inline sa_f32x16 mfma_bf16(f32_u32x4 x, f32_u32x4 y, sa_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sa_bf16x8, x), __builtin_bit_cast(sa_bf16x8, y),
                                                 c, 0, 0, 0);
}

// max / sum of x over lanes l and l ^ 32.
__device__ inline float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float half_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// fp32 attention on split operands. A wave owns 32 kG query rows (head dim 64: a whole 64-row
// block, 128: half of one) and walks its tiles in 32-key chunks with v_mfma_f32_32x32x16_bf16:
// six MFMAs per fp32 product block, smallest terms first, S^T and O^T accumulated in fp32; the
// softmax is the fp32 kernel's (running maximum, P and row sums in fp32; P is split like the
// other operands). Each S takes 6 kD / 16 rounded accumulations and O^T 24 per 64 keys, where
// the fp32 MFMA's fmaf chains take kD and 64.
//   kKW = 1: four waves of a workgroup own four units (query blocks or halves);
//   kKW = 4: they share one unit, wave w taking list positions w, w + 4, ..., and merge their
//     partials through LDS: for launches too small to fill the card otherwise.
// Bound: the matrix core (192 MFMAs, 6 144 cycles per 64 x 64 tile at head dim 64, against 512
// and 16 384 in fp32). Q's hi terms stay in registers, mid and lo in LDS (16 KB per wave), K and
// V operands are loaded straight from the split planes, kRing groups ahead, so two waves fit a
// SIMD and one's softmax runs beside the other's MFMAs. Measured, splitting included: [2, 30,
// 17776, 64] with a fifth of the blocks 9.61 -> 5.24 ms (1 130 TFLOP/s of bf16 products; the
// MFMA pipes busy 69 % at a power-limited 1.54 GHz, the largest bf16 matrix products on the card
// reach 1 380), the same at head dim 128 with 15 heads 11.9 -> 7.8 ms (there a wave's 32 rows
// load each operand for half the MFMAs, 64 bytes per cycle and CU, the vector cache's rate), and
// [1, 2, 2048, 64] with a quarter of the blocks 153 -> 37 us. Error against a 64-bit softmax 9.6e-7
// where the fp32 MFMA's was 1.1e-6 (2-norm, relative).
template <int kD, int kPool, int kKW>
__global__ __launch_bounds__(256, 2) void bsa_fwd_f32_terms_kernel(F32Args a) {
  static_assert(kD == 64 || kD == 128, "head dim 64 or 128");
  static_assert(kPool == 0 || kPool == 32 || kPool == 64, "pooling columns of 32 or 64 keys");
  static_assert(kKW == 1 || kKW == 4, "waves per unit");
  typedef TermLayout<kD> Lay;
  constexpr int kG = kD == 64 ? 2 : 1;   // 32-row query groups per wave
  constexpr int kHalvesQ = 2 / kG;       // units per query block
  constexpr int kRows = 32 * kG;
  constexpr int kDS = kD / 16, kDC = kD / 32;
  constexpr int kNG = Lay::kGroups;
  constexpr int kRing = 2;  // operand groups in registers (a deeper ring spills at head dim 128)
  static_assert(kNG % kRing == 0, "the ring's slots are static");
  constexpr int kUnitsWg = 4 / kKW;
  constexpr int kWgs = 4 * kHalvesQ / kUnitsWg;  // workgroups per dispatch group (4 slots)
  // Per wave: Q mid and lo operands, [term][g][s] of 1 KB; later its partial [kRows][kD].
  __shared__ __attribute__((aligned(1024))) f32_u32x4 q_lds[4][2 * kG * kDS * 64];
  __shared__ float ml_lds[kKW == 4 ? 4 : 1][2][kRows];
  static_assert(sizeof(q_lds[0]) == kRows * kD * sizeof(float), "a partial fits the Q operands' space");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hh = lane >> 5;
  // Dispatch group w (four slots of the work order) stays on XCD w % 8.
  const int x = blockIdx.x;
  const int w8 = 8 * (x / (8 * kWgs)) + (x & 7);
  const int unit = 4 * kHalvesQ * w8 + ((x >> 3) % kWgs) * kUnitsWg + (kKW == 1 ? wave : 0);
  const int slot = unit / kHalvesQ;
  if (slot >= a.n_slots) return;  // kKW = 4: the same for every wave of the workgroup
  const int item = __builtin_amdgcn_readfirstlane(a.order ? order_item(a.order, slot) : slot);
  if (item < 0 || item >= a.n_items) return;
  const int row0 = (unit % kHalvesQ) * kRows;
  const int bh = item / a.nqb;
  const int qb = item - bh * a.nqb;
  const int b = bh / a.H;
  const int h = bh - b * a.H;
  const int hk = a.kv_rep > 1 ? h / a.kv_rep : h;
  const int bhk = b * (a.H / a.kv_rep) + hk;
  const int it0 = kKW == 1 ? 0 : wave;

  const int64_t list_row = (int64_t)bh * a.list_bh_stride + qb;
  int cnt = a.kv_cnt[list_row];
  cnt = cnt < 0 ? 0 : (cnt > a.max_cnt ? a.max_cnt : cnt);
  const __attribute__((address_space(4))) int32_t* list =
      (const __attribute__((address_space(4))) int32_t*)(a.kv_idx + list_row * a.max_cnt);

  const uint4* fl = a.flags + (int64_t)bhk * a.nkb;
  f32_u32x4 qhi[kG][kDS];
  f32_u32x4* ql = q_lds[wave];
  bool use_terms = (uint32_t)__builtin_amdgcn_readfirstlane((int)fl[0].x) != kTermSkip;
  if (!use_terms && a.plain_after) return;
  if (use_terms) {
    // The flags of the head's blocks and of this wave's query rows.
    uint32_t worst = 0u;
    TermRange range;
    for (int j = 0; j < a.nkb; j += 64) {
      const uint4 f = fl[min(j + lane, a.nkb - 1)];
      worst = max(worst, max(max(f.x, f.y), max(f.z, f.w)));
    }
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      const int row = min(qb * kBlk + row0 + 32 * g + col, a.Lq - 1);  // clamped rows are never stored
      const float* p = a.q + b * a.q_sb + h * a.q_sh + (int64_t)row * a.q_sl + 8 * hh;
#pragma unroll
      for (int s = 0; s < kDS; ++s) {
        const float4 x0 = *reinterpret_cast<const float4*>(p + 16 * s);
        const float4 x1 = *reinterpret_cast<const float4*>(p + 16 * s + 4);
        const float y[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        f32_u32x4 mid, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t t0, t1, t2;
          split3(y[2 * i], y[2 * i + 1], t0, t1, t2);
          qhi[g][s][i] = t0;
          mid[i] = t1;
          lo[i] = t2;
          range.add(y[2 * i]);
          range.add(y[2 * i + 1]);
        }
        ql[(g * kDS + s) * 64 + lane] = mid;
        ql[((kG + g) * kDS + s) * 64 + lane] = lo;
      }
    }
    use_terms = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max_u(max(worst, range.flag()))) < kTermMax;
  }

  float* part = reinterpret_cast<float*>(q_lds[wave]);  // kKW = 4: [row][16-byte chunk ^ row % 16]
  if (!use_terms) {
    // In passes of 16 kJ rows, which fit beside this kernel's registers.
    constexpr int kJ = 2;
    for (int r0 = 0; r0 < kRows; r0 += 16 * kJ) {
      sa_f32x4 acc[kD / 16][kJ];
      float m[kJ], l[kJ];
      f32_rows<kD, kPool, kJ>(a, bh, qb, row0 + r0, it0, kKW, lane, acc, m, l);
      if constexpr (kKW == 1) {
        f32_store<kD, kPool, kJ>(a, bh, qb, row0 + r0, lane, acc, m, l);
      } else {
        const int r = lane & 15, g = lane >> 4;
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
          const int row = r0 + 16 * j + r;
          const float l_tot = slot_sum(l[j]);
#pragma unroll
          for (int dblk = 0; dblk < kD / 16; ++dblk)
            *reinterpret_cast<sa_f32x4*>(part + row * kD + 4 * ((4 * dblk + g) ^ (row & 15))) = acc[dblk][j];
          if (g == 0) {
            ml_lds[wave][0][row] = m[j];
            ml_lds[wave][1][row] = l_tot;
          }
        }
      }
    }
  } else {
    sa_f32x16 acc[kDC][kG];
    float m[kG], l[kG];
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      m[g] = -INFINITY;
      l[g] = 0.f;
#pragma unroll
      for (int dc = 0; dc < kDC; ++dc) acc[dc][g] = sa_f32x16{};
    }
    const uint8_t* head = a.planes + (int64_t)bhk * a.nkb * Lay::kTile;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(head), (short)0, (int)((uint32_t)a.nkb * Lay::kTile), 0x00020000);
    f32_u32x4 ring[kRing][6];
    auto load_group = [&](f32_u32x4 (&r)[6], uint32_t off) __attribute__((always_inline)) {
#pragma unroll
      for (int o = 0; o < 6; ++o)
        r[o] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * lane + 1024 * (o & 3), off + 4096 * (o >> 2), 0);
    };
    auto tile_off = [&](int kb) -> uint32_t {  // an entry outside the grid reads block 0 (masked out)
      return __builtin_amdgcn_readfirstlane(((unsigned)kb < (unsigned)a.nkb ? (uint32_t)kb : 0u) * Lay::kTile);
    };
    int kb = it0 < cnt ? list[it0] : 0;
    uint32_t off = tile_off(kb);
    if (it0 < cnt) {
#pragma unroll
      for (int i = 0; i < kRing; ++i) load_group(ring[i], off + i * Lay::kGroup);
    }
    for (int it = it0; it < cnt; it += kKW) {
      // Past the end the prefetch re-reads the current tile.
      const int kb_next = it + kKW < cnt ? list[it + kKW] : kb;
      const uint32_t off_next = tile_off(kb_next);
      const bool ok = (unsigned)kb < (unsigned)a.nkb;
      const int nvalid = ok ? min(kBlk, a.Lk - kb * kBlk) : 0;
      const bool diag = kPool != 0 && a.causal && kb == qb;
      float pmax[kG];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        // ---- S^T: S[g] element e is key 32 c + 8 (e / 4) + 4 hh + e % 4, row 32 g + col.
        sa_f32x16 S[kG];
#pragma unroll
        for (int g = 0; g < kG; ++g) S[g] = sa_f32x16{};
#pragma unroll
        for (int i = 0; i < Lay::kKGroups; ++i) {
          f32_u32x4(&r)[6] = ring[i % kRing];
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            const int s = 2 * i + s2;
            asm volatile("" ::: "memory");  // the LDS operands are read here, not kept in registers
            f32_u32x4 qm[kG], qo[kG];
#pragma unroll
            for (int g = 0; g < kG; ++g) {
              qm[g] = ql[(g * kDS + s) * 64 + lane];
              qo[g] = ql[((kG + g) * kDS + s) * 64 + lane];
            }
            const f32_u32x4 khi = r[3 * s2], kmid = r[3 * s2 + 1], klo = r[3 * s2 + 2];
#pragma unroll
            for (int g = 0; g < kG; ++g) S[g] = mfma_bf16(klo, qhi[g][s], S[g]);
#pragma unroll
            for (int g = 0; g < kG; ++g) S[g] = mfma_bf16(kmid, qm[g], S[g]);
#pragma unroll
            for (int g = 0; g < kG; ++g) S[g] = mfma_bf16(khi, qo[g], S[g]);
#pragma unroll
            for (int g = 0; g < kG; ++g) S[g] = mfma_bf16(kmid, qhi[g][s], S[g]);
#pragma unroll
            for (int g = 0; g < kG; ++g) S[g] = mfma_bf16(khi, qm[g], S[g]);
#pragma unroll
            for (int g = 0; g < kG; ++g) S[g] = mfma_bf16(khi, qhi[g][s], S[g]);
          }
          const int next = c * kNG + i + kRing;  // (never past this tile: K groups come first)
          load_group(r, off + next * Lay::kGroup);
          __builtin_amdgcn_sched_barrier(0x38f);  // loads stay where they are issued
        }
        // ---- Masks, pooled column maxima, running maximum, P = exp2(S * sc - m), row sums.
        if (nvalid < kBlk || diag) {
#pragma unroll
          for (int g = 0; g < kG; ++g)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int kk = 32 * c + 8 * (e >> 2) + 4 * hh + (e & 3);
              if (kk >= nvalid || (diag && kk > row0 + 32 * g + col)) S[g][e] = -INFINITY;
            }
        }
        float cand[kG];
        bool raise = false;
#pragma unroll
        for (int g = 0; g < kG; ++g) {
          float mx = fmaxf(S[g][0], S[g][1]);
#pragma unroll
          for (int e = 2; e < 16; e += 2) mx = fmaxf(fmaxf(mx, S[g][e]), S[g][e + 1]);
          cand[g] = half_max(mx) * a.scale_log2;  // scale > 0
          raise |= cand[g] > m[g];
        }
        if constexpr (kPool != 0) {
          // Lane l stores row l of the block (kG = 2), or lanes hh = 0 their unit's rows.
          const int cc = kPool == 32 ? c : 0;
#pragma unroll
          for (int g = 0; g < kG; ++g) pmax[g] = (kPool == 32 || c == 0) ? cand[g] : fmaxf(pmax[g], cand[g]);
          if (ok && (kPool == 32 || c == 1)) {
            constexpr int kCols = kBlk / kPool;
            float* rp = a.pool_r + (((int64_t)bh * a.nqb + qb) * a.pool_ncol + kb * kCols + cc) * kBlk + row0;
            if (kG == 2) rp[lane] = hh ? pmax[kG - 1] : pmax[0];
            else if (hh == 0) rp[col] = pmax[0];
          }
        }
        if (__ballot(raise) != 0) {
#pragma unroll
          for (int g = 0; g < kG; ++g) {
            const float m_new = fmaxf(m[g], cand[g]);
            const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[g] - m_new);
            m[g] = m_new;
            l[g] *= alpha;
#pragma unroll
            for (int dc = 0; dc < kDC; ++dc) acc[dc][g] *= alpha;
          }
        }
#pragma unroll
        for (int g = 0; g < kG; ++g) {
          const float mu = m[g] == -INFINITY ? 0.f : m[g];
          float sum = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float p = __builtin_amdgcn_exp2f(fmaf(S[g][e], a.scale_log2, -mu));  // -inf -> 0
            S[g][e] = p;
            sum += p;
          }
          l[g] += sum;
        }
        // ---- O^T += V^T P^T over the chunk's two 16-key steps.
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32_u32x4 P[kG][3];
#pragma unroll
          for (int g = 0; g < kG; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              uint32_t t0, t1, t2;
              split3(S[g][8 * u + 2 * i], S[g][8 * u + 2 * i + 1], t0, t1, t2);
              P[g][0][i] = t0;
              P[g][1][i] = t1;
              P[g][2][i] = t2;
            }
#pragma unroll
          for (int dp = 0; dp < kDC / 2; ++dp) {
            const int i = Lay::kKGroups + u * (kDC / 2) + dp;
            f32_u32x4(&r)[6] = ring[i % kRing];
#pragma unroll
            for (int d2 = 0; d2 < 2; ++d2) {
              const int dc = 2 * dp + d2;
              const f32_u32x4 vhi = r[3 * d2], vmid = r[3 * d2 + 1], vlo = r[3 * d2 + 2];
#pragma unroll
              for (int g = 0; g < kG; ++g) acc[dc][g] = mfma_bf16(vlo, P[g][0], acc[dc][g]);
#pragma unroll
              for (int g = 0; g < kG; ++g) acc[dc][g] = mfma_bf16(vmid, P[g][1], acc[dc][g]);
#pragma unroll
              for (int g = 0; g < kG; ++g) acc[dc][g] = mfma_bf16(vhi, P[g][2], acc[dc][g]);
#pragma unroll
              for (int g = 0; g < kG; ++g) acc[dc][g] = mfma_bf16(vmid, P[g][0], acc[dc][g]);
#pragma unroll
              for (int g = 0; g < kG; ++g) acc[dc][g] = mfma_bf16(vhi, P[g][1], acc[dc][g]);
#pragma unroll
              for (int g = 0; g < kG; ++g) acc[dc][g] = mfma_bf16(vhi, P[g][0], acc[dc][g]);
            }
            const int next = c * kNG + i + kRing;
            load_group(r, next < 2 * kNG ? off + next * Lay::kGroup : off_next + (next - 2 * kNG) * Lay::kGroup);
            __builtin_amdgcn_sched_barrier(0x38f);
          }
        }
      }
      kb = kb_next;
      off = off_next;
    }
    // ---- Epilogue: element 4 q4 + j of acc[dc][g] is d = 32 dc + 8 q4 + 4 hh + j.
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      const float l_tot = half_sum(l[g]);
      const int lrow = 32 * g + col;
      if constexpr (kKW == 1) {
        const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        const int row = qb * kBlk + row0 + lrow;
        if constexpr (kPool != 0) {
          if (hh == 0) a.pool_lse[(int64_t)bh * a.pool_lpad + row] = (m[g] == -INFINITY ? 0.f : m[g]) + log2f(l_tot);
        }
        if (row < a.Lq) {
          float* orow = a.o + b * a.o_sb + h * a.o_sh + (int64_t)row * a.o_sl;
#pragma unroll
          for (int dc = 0; dc < kDC; ++dc)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
              const sa_f32x16& A = acc[dc][g];
              *reinterpret_cast<float4*>(orow + 32 * dc + 8 * q4 + 4 * hh) =
                  make_float4(A[4 * q4] * inv, A[4 * q4 + 1] * inv, A[4 * q4 + 2] * inv, A[4 * q4 + 3] * inv);
            }
        }
      } else {
#pragma unroll
        for (int dc = 0; dc < kDC; ++dc)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const sa_f32x16& A = acc[dc][g];
            *reinterpret_cast<sa_f32x4*>(part + lrow * kD + 4 * ((8 * dc + 2 * q4 + hh) ^ (lrow & 15))) =
                sa_f32x4{A[4 * q4], A[4 * q4 + 1], A[4 * q4 + 2], A[4 * q4 + 3]};
          }
        if (hh == 0) {
          ml_lds[wave][0][lrow] = m[g];
          ml_lds[wave][1][lrow] = l_tot;
        }
      }
    }
  }
  if constexpr (kKW == 4) {
    // Merge in wave order: out = sum_w 2^(m_w - M) acc_w / sum_w 2^(m_w - M) l_w.
    __syncthreads();
    constexpr int kChunks = kD / 4;
    for (int t = threadIdx.x; t < kRows * kChunks; t += 256) {
      const int lrow = t / kChunks, ch = t % kChunks;
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < 4; ++w) M = fmaxf(M, ml_lds[w][0][lrow]);
      float L = 0.f;
      sa_f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float mw = ml_lds[w][0][lrow];
        const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);  // no key of this row: nothing
        const sa_f32x4 p = *reinterpret_cast<const sa_f32x4*>(
            reinterpret_cast<const float*>(q_lds[w]) + lrow * kD + 4 * (ch ^ (lrow & 15)));
        L += f * ml_lds[w][1][lrow];
        o += f * p;
      }
      const float inv = L > 0.f ? 1.f / L : 0.f;
      const int row = qb * kBlk + row0 + lrow;
      if constexpr (kPool != 0) {
        if (ch == 0) a.pool_lse[(int64_t)bh * a.pool_lpad + row] = (M == -INFINITY ? 0.f : M) + log2f(L);
      }
      if (row < a.Lq) {
        float* orow = a.o + b * a.o_sb + h * a.o_sh + (int64_t)row * a.o_sl;
        *reinterpret_cast<float4*>(orow + 4 * ch) = make_float4(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
      }
    }
  }
}

}  // namespace

namespace {

int64_t terms_blocks(int B, int Hk, int Lk) { return (int64_t)B * Hk * sa::cdiv(Lk, kBlk); }

template <int kD, int kPool>
void launch_terms_pool(const F32Args& a, hipStream_t s) {
  // Up to three rounds of the card's 2 048 waves, four waves share each unit (64 query rows, 32
  // at head dim 128); measured, one wave against four per unit: 64 units 78 / 43 us, 504 154 / 84,
  // 2 400 361 / 310, 5 640 717 / 690 (head dim 128: 784 / 771), 7 500 729 / 733, and 16 680 with
  // few tiles each 1 241 / 1 354.
  constexpr int64_t kSharedUnits = 6144;
  constexpr int kHalvesQ = kD == 64 ? 1 : 2;
  const int64_t groups = (a.n_slots + 3) / 4;
  const bool shared = (int64_t)a.n_items * kHalvesQ <= kSharedUnits;
  const int64_t wgs = shared ? 4 * kHalvesQ : kHalvesQ;  // workgroups per dispatch group
  const dim3 grid((unsigned)((groups + 7) / 8 * 8 * wgs)), blk(256);
  if (shared) hipLaunchKernelGGL((bsa_fwd_f32_terms_kernel<kD, kPool, 4>), grid, blk, 0, s, a);
  else hipLaunchKernelGGL((bsa_fwd_f32_terms_kernel<kD, kPool, 1>), grid, blk, 0, s, a);
}

// Heads with few tiles are not worth splitting k and v (12 D bytes per key). At head dim 64:
//   up to kTermsAlways query blocks every head is split: the workgroups are too few for its cost to show
//     ([1, 4, 2048] of one tile per key block 17.8 us, the fp32 kernel 17.6, of 1.6 tiles 22.5 / 56.8);
//   up to kTermsInline a head of fewer than 3/2 tiles per key block runs in fp32 where it is, four waves
//     sharing a unit: [1, 8, 4096] of 1.3 tiles 32 us (fp32 kernel 49), but of one tile 23 (19), [1, 16,
//     4096] 42 (23);
//   beyond, bsa_fwd_f32_kernel follows for such heads (one wave per unit; 3-7 us where there are none),
//     and all heads go by the launch's mean unless one is far from it: with heads on both sides of the line
//     each kernel leaves most of the card idle ([2, 30, 3000] of 1.8 tiles 176 us, all on one side 134).
// Measured there by tiles per key block, 1 / 1.6 / 2 / 3 (us; the fp32 kernel alone, with every head
// below 3/2 inline, and this): [2, 30, 3000] 50, 115, 131, 197 / 110, 153, 127, 140 / 61, 125, 135, 148;
// [1, 30, 8192] 66, 137, 172, 231 / 143, 186, 172, 191 / 79, 151, 185, 200; [2, 30, 17776] 275, 464,
// 557, 769 / 327, 587, 581, 661 / 305, 494, 586, 677.
// Head dim 128 keeps 3/2 and one kernel at all sizes: its fp32 kernel fits one wave per SIMD, and [1, 15,
// 17776] of one tile takes it 199 us where the inline path takes 174.
constexpr int64_t kTermsAlways = 128;
constexpr int64_t kTermsInline = 1024;
int terms_min_tiles4(int64_t units) { return units <= 2048 ? 6 : units <= 3072 ? 7 : units <= 6144 ? 8 : 9; }

template <int kD>
int launch_terms(F32Args& a, int B, void* ws, int pool_cols, void* stream, const char* fn) {
  const int Hk = a.H / a.kv_rep;
  const int64_t blocks = terms_blocks(B, Hk, a.Lk);
  TermArgs t;
  t.k = a.k; t.v = a.v;
  t.k_sb = a.k_sb; t.k_sh = a.k_sh; t.k_sl = a.k_sl;
  t.v_sb = a.v_sb; t.v_sh = a.v_sh; t.v_sl = a.v_sl;
  t.Hk = Hk; t.Lk = a.Lk; t.nkb = a.nkb;
  t.kv_cnt = a.list_bh_stride ? a.kv_cnt : nullptr;  // lists shared by the heads are dense
  t.nqb = a.nqb; t.max_cnt = a.max_cnt;
  if (kD == 64 && a.n_items <= kTermsAlways) t.kv_cnt = nullptr;
  t.together = kD == 64 && t.kv_cnt && a.n_items > kTermsInline;
  t.min_tiles4 = t.together ? terms_min_tiles4(a.n_items) : 6;
  t.lists = (uint32_t)B * Hk * a.nqb;
  a.plain_after = t.together;
  t.planes = static_cast<uint8_t*>(ws);
  t.flags = reinterpret_cast<uint32_t*>(t.planes + blocks * TermLayout<kD>::kTile);
  hipStream_t s = sa::as_stream(stream);
  hipLaunchKernelGGL(f32_terms_kernel<kD>, dim3((unsigned)blocks), dim3(256), 0, s, t);
  if (int rc = sa::check_launch(fn)) return rc;
  a.planes = t.planes;
  a.flags = reinterpret_cast<const uint4*>(t.flags);
  if (pool_cols == 32) launch_terms_pool<kD, 32>(a, s);
  else if (pool_cols == 64) launch_terms_pool<kD, 64>(a, s);
  else launch_terms_pool<kD, 0>(a, s);
  if (a.plain_after) {
    if (int rc = sa::check_launch(fn)) return rc;
    const dim3 grid((unsigned)(a.n_slots / kWavesF32)), blk(64 * kWavesF32);
    hipLaunchKernelGGL((bsa_fwd_f32_kernel<kD, 0>), grid, blk, 0, s, a);
  }
  return sa::check_launch(fn);
}

// Checks a terms workspace; blocks of one head are addressed with 32-bit offsets.
int check_terms(int B, int Hk, int Lk, int D, const void* ws, int64_t ws_bytes, const char* fn) {
  SA_REQUIRE(ws, "%s: null workspace", fn);
  SA_REQUIRE(reinterpret_cast<uintptr_t>(ws) % 256 == 0, "%s: workspace not 256-byte aligned", fn);
  const int64_t need = sa::attn_f32_terms_bytes(B, Hk, Lk, D);
  SA_REQUIRE(ws_bytes >= need, "%s: workspace of %lld bytes < %lld", fn, (long long)ws_bytes, (long long)need);
  if ((int64_t)sa::cdiv(Lk, kBlk) * 768 * D > 0x7fffffffLL || terms_blocks(B, Hk, Lk) >= (1LL << 31))
    return sa::fail(SA_ERR_UNSUPPORTED, "%s: Lk=%d too long for the split operands", fn, Lk);
  return SA_OK;
}

int launch_f32(const float* q, const int64_t q_strides[3], const float* k, const int64_t k_strides[3],
               const float* v, const int64_t v_strides[3], float* out, const int64_t out_strides[3], int B, int H,
               int Lq, int Lk, int D, const int32_t* kv_idx, const int32_t* kv_cnt, int max_cnt, bool lists_shared,
               float sm_scale, const int32_t* work_order, int64_t n_slots, int kv_rep, bool causal, int pool_cols,
               float* pool_r, float* pool_lse, void* terms_ws, void* stream, const char* fn) {
  SA_REQUIRE(q && k && v && out && q_strides && k_strides && v_strides && out_strides && kv_idx && kv_cnt,
             "%s: null pointer", fn);
  SA_REQUIRE(B > 0 && H > 0 && Lq > 0 && Lk > 0, "%s: bad shape B=%d H=%d Lq=%d Lk=%d", fn, B, H, Lq, Lk);
  if (D != 64 && D != 128) return sa::fail(SA_ERR_UNSUPPORTED, "%s: head_dim %d (64 or 128)", fn, D);
  SA_REQUIRE(max_cnt > 0, "%s: max_cnt must be > 0", fn);
  SA_REQUIRE(std::isfinite(sm_scale) && sm_scale > 0.f, "%s: sm_scale must be finite and > 0", fn);
  SA_REQUIRE(kv_rep >= 1 && H % kv_rep == 0, "%s: kv_rep=%d must divide H=%d", fn, kv_rep, H);
  SA_REQUIRE(!causal || (Lq == Lk && pool_cols), "%s: causal needs Lq == Lk and pooling", fn);
  const void* ptrs[4] = {q, k, v, out};
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0)
      return sa::fail(SA_ERR_UNSUPPORTED, "%s: tensor base not 16-byte aligned", fn);
  const int64_t* strides[4] = {q_strides, k_strides, v_strides, out_strides};
  for (const int64_t* st : strides)
    for (int i = 0; i < 3; ++i)
      if (st[i] % 4 != 0) return sa::fail(SA_ERR_UNSUPPORTED, "%s: strides must be multiples of 4 elements", fn);
  const int nqb = sa::cdiv(Lq, kBlk);
  const int64_t n_items = (int64_t)B * H * nqb;
  SA_REQUIRE(n_items < (1LL << 30), "%s: too many query blocks", fn);
  if (work_order) {
    SA_REQUIRE(n_slots > 0 && n_slots % kWavesF32 == 0, "%s: n_slots must be a positive multiple of 4", fn);
  } else {
    n_slots = (n_items + kWavesF32 - 1) / kWavesF32 * kWavesF32;
  }
  SA_REQUIRE(n_slots / kWavesF32 < (1LL << 31), "%s: grid too large", fn);
  F32Args a;
  a.q = q; a.k = k; a.v = v; a.o = out;
  a.q_sb = q_strides[0]; a.q_sh = q_strides[1]; a.q_sl = q_strides[2];
  a.k_sb = k_strides[0]; a.k_sh = k_strides[1]; a.k_sl = k_strides[2];
  a.v_sb = v_strides[0]; a.v_sh = v_strides[1]; a.v_sl = v_strides[2];
  a.o_sb = out_strides[0]; a.o_sh = out_strides[1]; a.o_sl = out_strides[2];
  a.H = H; a.Lq = Lq; a.Lk = Lk; a.nqb = nqb; a.nkb = sa::cdiv(Lk, kBlk);
  a.n_items = (int)n_items;
  a.order = work_order;
  a.n_slots = (int)n_slots;
  a.kv_idx = kv_idx; a.kv_cnt = kv_cnt; a.max_cnt = max_cnt;
  a.list_bh_stride = lists_shared ? 0 : nqb;
  a.scale_log2 = sm_scale * kLog2eF32;
  a.kv_rep = kv_rep;
  a.causal = causal ? 1 : 0;
  a.pool_r = pool_r;
  a.pool_ncol = pool_cols ? a.nkb * (kBlk / pool_cols) : 0;
  a.pool_lse = pool_lse;
  a.pool_lpad = nqb * kBlk;
  a.planes = nullptr;
  a.flags = nullptr;
  a.plain_after = 0;
  SA_REQUIRE(pool_cols == 0 || (pool_r && pool_lse), "%s: pooling needs its buffers", fn);
  if (terms_ws) return D == 64 ? launch_terms<64>(a, B, terms_ws, pool_cols, stream, fn)
                               : launch_terms<128>(a, B, terms_ws, pool_cols, stream, fn);
  const dim3 grid((unsigned)(n_slots / kWavesF32)), blk(64 * kWavesF32);
  hipStream_t s = sa::as_stream(stream);
  if (D == 64) {
    if (pool_cols == 32) hipLaunchKernelGGL((bsa_fwd_f32_kernel<64, 32>), grid, blk, 0, s, a);
    else if (pool_cols == 64) hipLaunchKernelGGL((bsa_fwd_f32_kernel<64, 64>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((bsa_fwd_f32_kernel<64, 0>), grid, blk, 0, s, a);
  } else {
    if (pool_cols == 32) hipLaunchKernelGGL((bsa_fwd_f32_kernel<128, 32>), grid, blk, 0, s, a);
    else if (pool_cols == 64) hipLaunchKernelGGL((bsa_fwd_f32_kernel<128, 64>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((bsa_fwd_f32_kernel<128, 0>), grid, blk, 0, s, a);
  }
  return sa::check_launch(fn);
}

}  // namespace

namespace sa {
int64_t attn_f32_terms_bytes(int B, int Hk, int Lk, int D) { return terms_blocks(B, Hk, Lk) * (768LL * D + 16); }

// fp32 attention in pooling mode for the pooled-map entry point (attn_fwd.hip).
int attn_f32_pooling(const float* q, const int64_t q_strides[3], const float* k, const int64_t k_strides[3],
                     const float* v, const int64_t v_strides[3], float* out, const int64_t out_strides[3], int B,
                     int H, int L, int D, const int32_t* kv_idx, const int32_t* kv_cnt, int max_cnt, int kv_rep,
                     bool causal, float sm_scale, int pool_cols, float* pool_r, float* pool_lse, void* terms_ws,
                     void* stream, const char* fn) {
  return launch_f32(q, q_strides, k, k_strides, v, v_strides, out, out_strides, B, H, L, L, D, kv_idx, kv_cnt,
                    max_cnt, true, sm_scale, nullptr, 0, kv_rep, causal, pool_cols, pool_r, pool_lse, terms_ws, stream,
                    fn);
}
}  // namespace sa

extern "C" int sa_block_sparse_fwd_f32(const float* q, const int64_t q_strides[3], const float* k,
                                       const int64_t k_strides[3], const float* v, const int64_t v_strides[3],
                                       float* out, const int64_t out_strides[3], int B, int H, int Lq, int Lk, int D,
                                       const int32_t* kv_idx, const int32_t* kv_cnt, int max_cnt,
                                       const float* key_bias, const int64_t bias_strides[2], float sm_scale,
                                       const int32_t* work_order, int64_t n_slots, void* stream) {
  const char* fn = "sa_block_sparse_fwd_f32";
  (void)bias_strides;
  if (key_bias) return sa::fail(SA_ERR_UNSUPPORTED, "%s: key_bias (bf16 and fp16 only)", fn);
  return launch_f32(q, q_strides, k, k_strides, v, v_strides, out, out_strides, B, H, Lq, Lk, D, kv_idx, kv_cnt,
                    max_cnt, false, sm_scale, work_order, n_slots, 1, false, 0, nullptr, nullptr, nullptr, stream, fn);
}

extern "C" int sa_block_sparse_fwd_f32_terms_workspace(int B, int H, int Lk, int D, int64_t* bytes) {
  const char* fn = "sa_block_sparse_fwd_f32_terms_workspace";
  SA_REQUIRE(bytes, "%s: null bytes", fn);
  SA_REQUIRE(B > 0 && H > 0 && Lk > 0, "%s: bad shape B=%d H=%d Lk=%d", fn, B, H, Lk);
  if (D != 64 && D != 128) return sa::fail(SA_ERR_UNSUPPORTED, "%s: head_dim %d (64 or 128)", fn, D);
  *bytes = sa::attn_f32_terms_bytes(B, H, Lk, D);
  return sa::ok();
}

extern "C" int sa_block_sparse_fwd_f32_terms(const float* q, const int64_t q_strides[3], const float* k,
                                             const int64_t k_strides[3], const float* v, const int64_t v_strides[3],
                                             float* out, const int64_t out_strides[3], int B, int H, int Lq, int Lk,
                                             int D, const int32_t* kv_idx, const int32_t* kv_cnt, int max_cnt,
                                             float sm_scale, const int32_t* work_order, int64_t n_slots,
                                             void* workspace, int64_t workspace_bytes, void* stream) {
  const char* fn = "sa_block_sparse_fwd_f32_terms";
  SA_REQUIRE(B > 0 && H > 0 && Lk > 0, "%s: bad shape B=%d H=%d Lk=%d", fn, B, H, Lk);
  if (D != 64 && D != 128) return sa::fail(SA_ERR_UNSUPPORTED, "%s: head_dim %d (64 or 128)", fn, D);
  if (int rc = check_terms(B, H, Lk, D, workspace, workspace_bytes, fn)) return rc;
  return launch_f32(q, q_strides, k, k_strides, v, v_strides, out, out_strides, B, H, Lq, Lk, D, kv_idx, kv_cnt,
                    max_cnt, false, sm_scale, work_order, n_slots, 1, false, 0, nullptr, nullptr, workspace, stream, fn);
}
