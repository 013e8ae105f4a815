// attn_fp32.hip — fp32 attention forward and backward on the matrix cores,
// for every d_head in 1..128 and any 4-byte alignment.
//
// The fp16 MFMA kernels cover d_head = 64 with 16-byte aligned tensors. These
// kernels take everything else with the reference's full precision: operands,
// products, probabilities and sums are fp32 (v_mfma_f32_16x16x4_f32, 32 cycles
// for 2048 FLOP: 157 TFLOP/s on the chip, which bounds them).
//
// One unit of work is a 16 x 16 tile of the score matrix. The products are
// transposed as in the fp16 kernels, so that the scores leave the MFMA in the
// layout the next product takes as its B operand, register for register: in
// the result, lane l holds column l%16 and rows 4*(l/16) + r in register r; in
// the next product, step r contracts the four rows 4*g + r (g = 0..3), lane
// group g supplying its row. Two layouts of a 16-row operand tile:
//   * row fragments (contraction over d): lane l holds row l%16, values
//     16*i + 4*(l/16) + 0..3 of block i — one 16-byte load per block;
//   * column fragments (contraction over the rows): step r, lane l holds row
//     4*(l/16) + r and, for blocks 4c .. 4c+3, values 64*c + 4*(l%16) + 0..3 —
//     one 16-byte load for four blocks. The N = DBLK%4 last blocks take values
//     64*(DBLK/4) + N*(l%16) + 0..N-1. col_of() gives the value a block and
//     row of the result stand for.
// DBLK = ceil(d_head / 16); values at or past d_head are zero in row fragments
// and belong to rows of the result that are not stored in column fragments.
//
// The waves of a workgroup own the same 16 (or 32) rows and split the rows they
// stream among themselves, and add their results through LDS at the end: with
// d_head 128 one tile takes 2048 cycles, and a 1024-row head has only 64 row
// blocks, so splitting by rows alone would leave most of the 1024 SIMDs idle.
// No wave shares a streamed row with another of its workgroup, so the forward's
// operands go straight from L2 to registers, without LDS or barriers.
#include "dfattn_internal.h"

#include <type_traits>

namespace dfattn {
namespace {

constexpr int kRows = 16;  // rows of a tile
// ln 2 - kLn2, so that lse = top * (kLn2 + kLn2Lo) + ln(sum) is rounded once, at
// the end: 4.42e-8 from 64 bits on average over d_head 16 .. 128 at S = 64 .. 512,
// 4.88e-8 with the log2 domain's sum times kLn2.
constexpr float kLn2Lo = -1.90465421e-09f;

// fp32 vectors at any 4-byte alignment.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Max / sum over the four lanes l%16 + 16*g that share a result column.
__device__ __forceinline__ float column_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return pair_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float column_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return pair_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// One [S, H*D] operand as seen by a head.
struct Shape {
  int S, D, ld, hoff;
};

// Descriptor of the 16 rows from row0 (uniform) of one head: loads past row S-1
// and past the last row's d_head values return zero. (n_heads <= 65535: 16
// rows span at most 2^29 bytes.)
__device__ __forceinline__ auto tile_rsrc(const float *X, int row0, const Shape &s) {
  const int rows = uniform_clamp0<kRows>(s.S - row0);
  const unsigned nrec = rows > 0 ? (unsigned)((rows - 1) * s.ld + s.D) * 4u : 0u;
  return buffer_rsrc(X + (size_t)min(row0, s.S) * s.ld + s.hoff, nrec);
}

template <int DBLK>
__device__ __forceinline__ void load_row_frags(const float *X, int row0, const Shape &s, int lane, f32x4 (&f)[DBLK]) {
  const auto rs = tile_rsrc(X, row0, s);
  const int off = ((lane & 15) * s.ld + 4 * (lane >> 4)) * 4;
#pragma unroll
  for (int i = 0; i < DBLK; ++i)
    f[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 64 * i, 0, 0));
}
// Zeroes the values of the last block at or past d_head (the next head's, when
// d_head is not a multiple of 16).
template <int DBLK>
__device__ __forceinline__ void trim_row_frags(const Shape &s, int lane, f32x4 (&f)[DBLK]) {
  if (s.D == 16 * DBLK) return;
  const int left = s.D - 16 * (DBLK - 1) - 4 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j >= left) f[DBLK - 1][j] = 0.f;
}

// The value (column of the tensor) that row m of result block blk stands for.
template <int DBLK>
__device__ __forceinline__ int col_of(int blk, int m) {
  constexpr int CF = DBLK / 4, N = DBLK % 4;
  return blk < 4 * CF ? 64 * (blk >> 2) + 4 * m + (blk & 3) : 64 * CF + N * m + (blk - 4 * CF);
}

// Column fragments of the 16 rows from row0, f[r][blk], straight from memory.
template <int DBLK>
__device__ __forceinline__ void load_col_frags(const float *X, int row0, const Shape &s, int lane,
                                               float (&f)[4][DBLK]) {
  constexpr int CF = DBLK / 4, N = DBLK % 4;
  const auto rs = tile_rsrc(X, row0, s);
  const int n16 = lane & 15;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int off = (4 * (lane >> 4) + r) * s.ld * 4;
#pragma unroll
    for (int c = 0; c < CF; ++c) {
      const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + (64 * c + 4 * n16) * 4, 0, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j) f[r][4 * c + j] = v[j];
    }
    const int rest = off + (64 * CF + N * n16) * 4;
    if constexpr (N == 1) {
      f[r][4 * CF] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, rest, 0, 0));
    } else if constexpr (N == 2) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, rest, 0, 0);
#pragma unroll
      for (int j = 0; j < 2; ++j) f[r][4 * CF + j] = __uint_as_float(v[j]);
    } else if constexpr (N == 3) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b96(rs, rest, 0, 0);
#pragma unroll
      for (int j = 0; j < 3; ++j) f[r][4 * CF + j] = __uint_as_float(v[j]);
    }
  }
}

// A masked pair of a diagonal tile has weight 0, which the MFMA turns into NaN
// where the streamed row holds an infinity or NaN that the other row must not
// see. Such a tile is left out of the second product: its weights
// w[16*z + k][own row] go to LDS, and when a workgroup stores its result it
// adds the visible pairs' products to block `b` here, rows from memory.
// (Rows past S need no such care: they read as zeros.)
template <int DBLK, class Visible>
__device__ __forceinline__ f32x4 diagonal_products(const float (*w)[kRows], int n_rows, const float *X, int row0,
                                                   const Shape &s, int lane, int b, Visible visible) {
  f32x4 o = f32x4{};
  for (int k = 0; k < n_rows && row0 + k < s.S; ++k)
    if (visible(k)) {
      const float *x = X + (size_t)(row0 + k) * s.ld + s.hoff;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = col_of<DBLK>(b, 4 * (lane >> 4) + r);
        if (d < s.D) o[r] += w[k][lane & 15] * x[d];
      }
    }
  return o;
}
// Whether any value of a tile's fragments (in any lane) is infinite or NaN.
template <class T, int N>
__device__ __forceinline__ bool any_nonfinite(const T (&f)[N]) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (unsigned j = 0; j < sizeof(T) / sizeof(float); ++j) bad |= !(fabsf(f[i][j]) < INFINITY);
  return __any(bad);
}

// ------------------------------------------------------------------ forward
// A workgroup of NW waves owns 16 query rows of one head; wave w takes the key
// tiles w, w + NW, ... (16*KS keys each):
//   S^T (keys x queries) = K . Q^T,  O^T (d x queries) += V^T . P^T.
// K of the wave's next tile is fetched during the softmax and the second
// product, V of this one during the first. The online softmax works in the
// log2 domain and moves its reference point only when a score exceeds it by
// more than 8 (P stays below 2^8, the sums are fp32). Four waves a workgroup:
// three workgroups share a CU (two above d_head 80), so that one's loads and merge
// run beside another's products (eight waves measured 15-25 % slower at S = 1000).
// Measured: H = 12, S = 1000, d_head 80 causal 29.4 us (607 us with one wave
// per row on the vector unit); H = 8, d_head 128: S = 1024 causal 29.1 us (620
// us), S = 4096 full 592 us = 116 TFLOP/s of the 157 the fp32 MFMA has (537 us
// with every load taken out of the loop).
template <int DBLK, int NW, int KS>
__global__ __launch_bounds__(64 * NW) void fwd_fp32_kernel(const float *__restrict__ Q, const float *__restrict__ K,
                                                           const float *__restrict__ V, float *__restrict__ O,
                                                           float *__restrict__ LSE, int H, int S, int D, float c2,
                                                           int causal, int n_blocks, int fold) {
  constexpr int kTileKeys = kRows * KS;
  __shared__ __attribute__((aligned(16))) f32x4 o_lds[NW][DBLK][64];
  __shared__ float m_lds[NW][kRows], l_lds[NW][kRows];
  __shared__ float diag_w[kTileKeys][kRows];  // see diagonal_products
  __shared__ int diag_wave;                   // the wave whose diagonal tile is in diag_w, or -1
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (The division runs on the vector unit.)
  const int idx = __builtin_amdgcn_readfirstlane(linear_block() / H), head = linear_block() - idx * H;
  if (idx >= n_blocks) return;
  const Shape sh{S, D, H * D, head * D};

  // Longest query blocks first under causal masking; with `fold` the second
  // half of the workgroups takes the short blocks in ascending order.
  const int n_long = (n_blocks + 1) / 2;
  const int q0 = (!causal ? idx : fold && idx >= n_long ? idx - n_long : n_blocks - 1 - idx) * kRows;
  const int kv_end = causal ? min(S, q0 + kRows) : S;
  const int n_tiles = (kv_end + kTileKeys - 1) / kTileKeys;
  // Keys below n_clear are visible to every row of the block; no key at or
  // above lim + 1 is to this lane's.
  const int n_clear = causal ? q0 + 1 : S;
  const int lim = causal ? min(q0 + col, S - 1) : S - 1;

  f32x4 qf[DBLK], acc[DBLK], kf[KS][DBLK];
  float m = -INFINITY, l = 0.f;
  load_row_frags<DBLK>(Q, q0, sh, lane, qf);
#pragma unroll
  for (int z = 0; z < KS; ++z) load_row_frags<DBLK>(K, wave * kTileKeys + kRows * z, sh, lane, kf[z]);
#pragma unroll
  for (int b = 0; b < DBLK; ++b) acc[b] = f32x4{};
  trim_row_frags<DBLK>(sh, lane, qf);
  // A hidden key's score is an infinity that c2 turns into -inf, so a c2 of 0 goes
  // into Q instead. (Masking after the scale costs the loop 2 %.)
  if (c2 == 0.f) {
#pragma unroll
    for (int b = 0; b < DBLK; ++b) qf[b] *= c2;
    c2 = 1.f;
  }
  const float hidden = c2 < 0.f ? INFINITY : -INFINITY;

  for (int t = wave; t < n_tiles; t += NW) {
    const int k0 = t * kTileKeys;
    float vf[KS][4][DBLK];
#pragma unroll
    for (int z = 0; z < KS; ++z) load_col_frags<DBLK>(V, k0 + kRows * z, sh, lane, vf[z]);
    // Scores: register r of s[z] is key k0 + 16 z + 4 g + r.
    f32x4 s[KS];
#pragma unroll
    for (int z = 0; z < KS; ++z) {
      trim_row_frags<DBLK>(sh, lane, kf[z]);
      s[z] = f32x4{};
    }
#pragma unroll
    for (int i = 0; i < DBLK; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int z = 0; z < KS; ++z) s[z] = mfma16(kf[z][i][j], qf[i][j], s[z]);
#pragma unroll
    for (int z = 0; z < KS; ++z)
      load_row_frags<DBLK>(K, (t + NW) * kTileKeys + kRows * z, sh, lane, kf[z]);

    const bool masked = k0 + kTileKeys > n_clear;
    if (masked) {
#pragma unroll
      for (int z = 0; z < KS; ++z)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + kRows * z + 4 * g + r > lim) s[z][r] = hidden;
    }
    // P = 2^(s c2 - m); the exact column maximum and the rescale only when a
    // score lies more than 8 above the reference point (or none is set).
    const float m_use = m == -INFINITY ? 0.f : m;
    float top = -INFINITY;
    f32x4 x[KS];
#pragma unroll
    for (int z = 0; z < KS; ++z)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[z][r] = fmaf(s[z][r], c2, -m_use);
        top = fmaxf(top, x[z][r]);
      }
    if (__any(top > 8.f || m == -INFINITY)) {
      const float m_new = fmaxf(m, m_use + column_max(top));
      const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - m_new);
      const float use = m_new == -INFINITY ? 0.f : m_new;
      l *= alpha;
#pragma unroll
      for (int b = 0; b < DBLK; ++b) acc[b] *= alpha;
#pragma unroll
      for (int z = 0; z < KS; ++z)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[z][r] = fmaf(s[z][r], c2, -use);
      m = m_new;
    }
#pragma unroll
    for (int z = 0; z < KS; ++z)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[z][r] = fast_exp2(x[z][r]);
        l += s[z][r];
      }
    if (causal && t == n_tiles - 1) {  // the diagonal tile, its wave's last
      bool bad = false;
#pragma unroll
      for (int z = 0; z < KS; ++z) bad |= any_nonfinite(vf[z]);
      if (lane == 0) diag_wave = bad ? wave : -1;
      if (bad) {
#pragma unroll
        for (int z = 0; z < KS; ++z)
#pragma unroll
          for (int r = 0; r < 4; ++r) diag_w[kRows * z + 4 * g + r][col] = s[z][r];
        break;
      }
    }
#pragma unroll
    for (int z = 0; z < KS; ++z)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int b = 0; b < DBLK; ++b) acc[b] = mfma16(vf[z][r][b], s[z][r], acc[b]);
  }

  // Merge the waves: each writes (m, l, O); wave w then finishes the result
  // blocks w, w + NW, ....
  const float lsum = column_sum(l);
  if (g == 0) {
    m_lds[wave][col] = m;
    l_lds[wave][col] = lsum;
  }
#pragma unroll
  for (int b = 0; b < DBLK; ++b) o_lds[wave][b][lane] = acc[b];
  __syncthreads();
  for (int b = wave; b < DBLK; b += NW) {
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) top = fmaxf(top, m_lds[w][col]);
    const float use = top == -INFINITY ? 0.f : top;
    float sum = 0.f;
    f32x4 o = f32x4{};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = fast_exp2(m_lds[w][col] - use);
      sum += a * l_lds[w][col];
      o += a * o_lds[w][b][lane];
    }
    if (causal && diag_wave >= 0) {
      const int k0 = (n_tiles - 1) * kTileKeys;
      o += fast_exp2(m_lds[diag_wave][col] - use) *
           diagonal_products<DBLK>(diag_w, kTileKeys, V, k0, sh, lane, b, [&](int k) { return k0 + k <= lim; });
    }
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    const int q = q0 + col;
    if (q < S) {
      float *row = O + (size_t)q * sh.ld + sh.hoff;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = col_of<DBLK>(b, 4 * g + r);
        if (d < D) row[d] = o[r] * inv;
      }
      if (LSE != nullptr && b == 0 && g == 0)
        LSE[(size_t)head * S + q] = sum > 0.f ? fmaf(top, kLn2, fmaf(top, kLn2Lo, logf(sum))) : -INFINITY;
    }
  }
}

// ----------------------------------------------------------------- backward
// Delta_i = dO_i . O_i, [H, S]: 16 lanes per (row, head).
__global__ __launch_bounds__(256) void delta_fp32_kernel(const float *__restrict__ O, const float *__restrict__ dO,
                                                         float *__restrict__ delta, int H, int S, int D) {
  const size_t i = (size_t)linear_block() * 16 + (threadIdx.x >> 4);  // row * H + head
  const int c = threadIdx.x & 15;
  float a = 0.f;
  if (i < (size_t)S * H)
    for (int d = c; d < D; d += 16) a = fmaf(O[i * D + d], dO[i * D + d], a);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
  if (i < (size_t)S * H && c == 0) delta[(i % H) * S + i / H] = a;
}

struct BwdFp32 {
  const float *Q, *K, *V, *dO, *lse, *delta;
  float *dQ, *dK, *dV;
  int H, S, D, n_blocks, causal;
  float scale;
};

constexpr int kBwdWaves = 4;  // two workgroups per CU (eight waves, one workgroup: 122 against 102 us, see below)
// Row stride in floats of an LDS tile: 16*DBLK + 4 keeps row-fragment stores
// (16 rows at one column) and column-fragment reads (rows 4 g + r) on
// different banks.
template <int DBLK>
constexpr int kLdsLd = 16 * DBLK + 4;

// One item: KV: dK and dV of the 16 keys from row0, streaming query tiles;
// else dQ of the 16 queries from row0, streaming key tiles. `own` are the
// item's rows (K and V, or Q and dO), `x`, `y` the streamed ones (Q and dO, or
// K and V):
//   s = x . own1^T, dp = y . own2^T         (streamed rows x own rows)
//   P = exp(scale s - lse), dS = P (dp - Delta)
//   acc1 += x^T dS (dK or dQ), and KV: acc2 += y^T P (dV).
// The streamed tile's row fragments arrive in registers (fetched during the
// previous tile's second products), feed the first products and are stored to
// the wave's own LDS tile, from which the second products read them by
// columns.
template <int DBLK, bool KV>
__device__ __forceinline__ void bwd_item(const BwdFp32 &a, int head, int row0, float *lds,
                                         float (*diag_w)[kRows][kRows], int *diag_bad) {
  constexpr int LD = kLdsLd<DBLK>, CF = DBLK / 4, N = DBLK % 4, kOuts = KV ? 2 : 1;
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int S = a.S;
  const Shape sh{S, a.D, a.H * a.D, head * a.D};
  const float *X = KV ? a.Q : a.K, *Y = KV ? a.dO : a.V;
  const float *lse = a.lse + (size_t)head * S, *delta = a.delta + (size_t)head * S;
  float *xt = lds + (size_t)wave * 2 * kRows * LD, *yt = xt + kRows * LD;

  f32x4 own1[DBLK], own2[DBLK], xf[DBLK], yf[DBLK], acc1[DBLK], acc2[DBLK];
  load_row_frags<DBLK>(KV ? a.K : a.Q, row0, sh, lane, own1);
  load_row_frags<DBLK>(KV ? a.V : a.dO, row0, sh, lane, own2);
  const int own = row0 + col;  // this lane's own row
  float own_lse = 0.f, own_delta = 0.f;
  if (!KV && own < S) {
    own_lse = lse[own];
    own_delta = delta[own];
  }
  const int n_tiles = (S + kRows - 1) / kRows;
  const int own_tile = row0 / kRows;
  const int t0 = (KV && a.causal ? own_tile : 0) + wave, t1 = !KV && a.causal ? own_tile + 1 : n_tiles;
#pragma unroll
  for (int b = 0; b < DBLK; ++b) acc1[b] = acc2[b] = f32x4{};
  load_row_frags<DBLK>(X, t0 * kRows, sh, lane, xf);
  load_row_frags<DBLK>(Y, t0 * kRows, sh, lane, yf);
  f32x4 row_lse = f32x4{}, row_delta = f32x4{};
  auto load_stats = [&](int t) {
    if (KV) {
      const int r0 = min(t * kRows, S);
      const unsigned nrec = (unsigned)uniform_clamp0<kRows>(S - t * kRows) * 4u;
      row_lse = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer_rsrc(lse + r0, nrec), 16 * g, 0, 0));
      row_delta =
          __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer_rsrc(delta + r0, nrec), 16 * g, 0, 0));
    }
  };
  load_stats(t0);
  trim_row_frags<DBLK>(sh, lane, own1);
  trim_row_frags<DBLK>(sh, lane, own2);

  // Second product: acc += tile^T . w, tile by columns from LDS.
  auto columns = [&](const float *tile, int r, float (&f)[DBLK]) {
    const float *row = tile + (4 * g + r) * LD;
#pragma unroll
    for (int c = 0; c < CF; ++c) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(row + 64 * c + 4 * col);
#pragma unroll
      for (int j = 0; j < 4; ++j) f[4 * c + j] = v[j];
    }
#pragma unroll
    for (int j = 0; j < N; ++j) f[4 * CF + j] = row[64 * CF + N * col + j];
  };
  for (int t = t0; t < t1; t += kBwdWaves) {
    trim_row_frags<DBLK>(sh, lane, xf);
    trim_row_frags<DBLK>(sh, lane, yf);
    const bool diagonal = a.causal && t == own_tile, masked = diagonal || (t + 1) * kRows > S;
    bool bad = false;
    if (diagonal) {
      bad = any_nonfinite(xf);
      if (KV) bad |= any_nonfinite(yf);
      if (lane == 0) *diag_bad = bad;
    }
#pragma unroll
    for (int i = 0; i < DBLK; ++i) {
      *reinterpret_cast<f32x4 *>(xt + col * LD + 16 * i + 4 * g) = xf[i];
      if (KV) *reinterpret_cast<f32x4 *>(yt + col * LD + 16 * i + 4 * g) = yf[i];
    }
    f32x4 s = f32x4{}, dp = f32x4{};
#pragma unroll
    for (int i = 0; i < DBLK; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s = mfma16(xf[i][j], own1[i][j], s);
        dp = mfma16(yf[i][j], own2[i][j], dp);
      }
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 tl = row_lse, td = row_delta;
    const int next = t + kBwdWaves;
    load_row_frags<DBLK>(X, next * kRows, sh, lane, xf);
    load_row_frags<DBLK>(Y, next * kRows, sh, lane, yf);
    load_stats(next);
    // Register r is streamed row t*16 + 4 g + r.
    auto visible = [&](int k) {  // streamed row t*16 + k against this lane's own row
      const int row = t * kRows + k;
      return row < S && (!a.causal || (KV ? own <= row : row <= own));
    };
    f32x4 ds;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float lr = KV ? tl[r] : own_lse, dr = KV ? td[r] : own_delta;
      s[r] = fast_exp2(fmaf(s[r], a.scale, -lr) * kLog2e);
      ds[r] = s[r] * (dp[r] - dr);
      if (masked && !visible(4 * g + r)) s[r] = ds[r] = 0.f;
    }
    // The wave's own stores are complete (same-wave LDS order) and visible.
    __builtin_amdgcn_wave_barrier();
    if (bad) {
      // See diagonal_products; the second products below run on a tile of zeros
      // (leaving them out of this pass instead costs the compiler 18+ registers).
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        diag_w[0][4 * g + r][col] = ds[r];
        if (KV) diag_w[1][4 * g + r][col] = s[r];
      }
#pragma unroll 1
      for (int i = 0; i < 4 * DBLK; ++i) {
        xt[col * LD + 4 * i + g] = 0.f;
        if (KV) yt[col * LD + 4 * i + g] = 0.f;
      }
      ds = s = f32x4{};
    }
    // Each step's fragments are read during the step before it; the scheduling
    // barriers keep the reads of later steps from filling the registers.
    constexpr int kSteps = 4 * kOuts;  // step = kOuts * r + (0: acc1, 1: acc2)
    float f[2][DBLK];
    columns(xt, 0, f[0]);
#pragma unroll
    for (int step = 0; step < kSteps; ++step) {
      const int nxt = step + 1;
      if (nxt < kSteps) columns(nxt % kOuts ? yt : xt, nxt / kOuts, f[nxt & 1]);
      const bool second = step % kOuts != 0;
      const float w = second ? s[step / kOuts] : ds[step / kOuts];
#pragma unroll
      for (int b = 0; b < DBLK; ++b) {
        if (second)
          acc2[b] = mfma16(f[step & 1][b], w, acc2[b]);
        else
          acc1[b] = mfma16(f[step & 1][b], w, acc1[b]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_wave_barrier();
  }

  // Add the waves' results in wave order; wave w finishes result blocks w, w + 4, ....
  f32x4 *part = reinterpret_cast<f32x4 *>(lds);
  __syncthreads();  // the tiles are no longer read
#pragma unroll
  for (int b = 0; b < DBLK; ++b) {
    part[(wave * kOuts * DBLK + b) * 64 + lane] = acc1[b];
    if (KV) part[(wave * kOuts * DBLK + DBLK + b) * 64 + lane] = acc2[b];
  }
  __syncthreads();
  for (int item = wave; item < kOuts * DBLK; item += kBwdWaves) {
    f32x4 o = part[item * 64 + lane];
#pragma unroll
    for (int w = 1; w < kBwdWaves; ++w) o += part[(w * kOuts * DBLK + item) * 64 + lane];
    const bool second = item >= DBLK;
    const int b = second ? item - DBLK : item;
    if (a.causal && *diag_bad)
      o += diagonal_products<DBLK>(diag_w[second ? 1 : 0], kRows, second ? Y : X, row0, sh, lane, b,
                                   [&](int k) { return KV ? col <= k : k <= col; });
    float *out = second ? a.dV : (KV ? a.dK : a.dQ);
    const float f = second ? 1.f : a.scale;
    if (own < S) {
      float *row = out + (size_t)own * sh.ld + sh.hoff;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = col_of<DBLK>(b, 4 * g + r);
        if (d < a.D) row[d] = o[r] * f;
      }
    }
  }
}

// One workgroup per item, longest first: for rank r = 0, 1, ... the dK/dV item
// of key block r (under causal masking it streams n_blocks - r query tiles)
// and the dQ item of query block n_blocks-1-r (as many key tiles), for every
// head. No atomics: S and dP are computed in both kinds of item (7 products
// instead of 5), and every sum has one order.
// Measured at H = 8, S = 1024, d_head 128 causal: 102 us (4800 us with one wave
// per row on the vector unit and dK, dV by atomics); S = 4096 full: 2.2 ms =
// 109 TFLOP/s of the seven products.
template <int DBLK>
__global__ __launch_bounds__(64 * kBwdWaves) void bwd_fp32_kernel(BwdFp32 a) {
  __shared__ __attribute__((aligned(16))) float lds[kBwdWaves * 2 * kRows * kLdsLd<DBLK>];
  __shared__ float diag_w[2][kRows][kRows];  // see diagonal_products: dS and P of the diagonal tile
  __shared__ int diag_bad;
  const int item = __builtin_amdgcn_readfirstlane(linear_block() / a.H), head = linear_block() - item * a.H;
  if (item >= 2 * a.n_blocks) return;
  if ((item & 1) == 0)
    bwd_item<DBLK, true>(a, head, (item >> 1) * kRows, lds, diag_w, &diag_bad);
  else
    bwd_item<DBLK, false>(a, head, (a.n_blocks - 1 - (item >> 1)) * kRows, lds, diag_w, &diag_bad);
}

// Calls fn.template operator()<DBLK>() for DBLK = ceil(d_head / 16).
template <class Fn>
void with_dblk(int d_head, Fn fn) {
  switch ((d_head + 15) / 16) {
    case 1: fn(std::integral_constant<int, 1>{}); break;
    case 2: fn(std::integral_constant<int, 2>{}); break;
    case 3: fn(std::integral_constant<int, 3>{}); break;
    case 4: fn(std::integral_constant<int, 4>{}); break;
    case 5: fn(std::integral_constant<int, 5>{}); break;
    case 6: fn(std::integral_constant<int, 6>{}); break;
    case 7: fn(std::integral_constant<int, 7>{}); break;
    default: fn(std::integral_constant<int, 8>{}); break;
  }
}

}  // namespace

hipError_t launch_fwd_fp32(const float *q, const float *k, const float *v, float *o, float *lse, int n_heads,
                           int seq_len, int d_head, float scale, bool causal, hipStream_t stream) {
  with_dblk(d_head, [&](auto n) {
    constexpr int DBLK = decltype(n)::value, KS = DBLK <= 4 ? 2 : 1, NW = 4;
    const int n_blocks = (seq_len + kRows - 1) / kRows;
    const size_t grid = (size_t)n_blocks * n_heads;
    // When every workgroup is resident at once (three per CU on 256 CUs; two above
    // d_head 80, where the rule's last third is not) there is no later round to
    // fill the gaps of the long ones: the short half in ascending order then lands
    // beside them (29.1 against 34.9 us at H = 8, S = 1024, d_head 128). Larger
    // grids run longest first (94 against 107 us at S = 2048).
    const int fold = causal && grid <= 768 ? 1 : 0;
    hipLaunchKernelGGL((fwd_fp32_kernel<DBLK, NW, KS>), linear_grid(grid), dim3(64 * NW), 0, stream, q, k, v, o, lse,
                       n_heads, seq_len, d_head, scale * kLog2e, causal ? 1 : 0, n_blocks, fold);
  });
  return hipGetLastError();
}

hipError_t launch_bwd_fp32(const float *q, const float *k, const float *v, const float *o, const float *d_o,
                           const float *lse, float *delta, float *d_q, float *d_k, float *d_v, int n_heads,
                           int seq_len, int d_head, float scale, bool causal, hipStream_t stream) {
  const size_t rows = (size_t)n_heads * seq_len;
  hipLaunchKernelGGL(delta_fp32_kernel, linear_grid((rows + 15) / 16), dim3(256), 0, stream, o, d_o, delta,
                     n_heads, seq_len, d_head);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  BwdFp32 a{q, k, v, d_o, lse, delta, d_q, d_k, d_v, n_heads, seq_len, d_head, (seq_len + kRows - 1) / kRows,
            causal ? 1 : 0, scale};
  with_dblk(d_head, [&](auto n) {
    constexpr int DBLK = decltype(n)::value;
    hipLaunchKernelGGL((bwd_fp32_kernel<DBLK>), linear_grid((size_t)2 * a.n_blocks * n_heads), dim3(64 * kBwdWaves),
                       0, stream, a);
  });
  return hipGetLastError();
}

}  // namespace dfattn
