// gpt2_linear.hip — the linear layers' products on gfx950 matrix cores, fp32
// in and out: y = x W^T + b (with GELU), dx = dy W (times GELU's derivative)
// and dW = dy^T x (reference: linear_into, linear_backward_into,
// darkforest-core/src/engine/static_gpt2.rs:1353-1357, 1441-1451).
//
// Each operand value is split as it is staged into two bf16 terms, hi = bf16(v)
// and lo = bf16(v - hi), and a product is lo hi' + hi lo' + hi hi' summed in
// fp32: at most 2^-16 of a value is lost, and 4.4e-6 of the result's norm on random data
// against float64, the same as the library's fast fp32 path. A bf16 product
// runs at 7 times the fp32 matrix rate, so three cost less than half.
//
// Bound: latency from one contraction step to the next (LDS reads, matrix
// products, the next step's loads and their split), with one tile per CU. So
// a tile's waves are many and small: waves of 32 rows by 64 or 96 columns, and
// KW groups of waves that take alternate steps, each through its own LDS
// blocks (64-row waves with half the LDS traffic measured 31 us where these
// take 24; loads two steps ahead instead of one changed nothing).
// In a graph, this kernel and the library's tuned solution: [1024, 768] x
// [768, 3072] 23.9 us (0.61 PFLOP/s of bf16 products) and 25.9; [1024, 768] x
// [768, 768] 10.3 and 15.2; dW of [2304, 768] over 1024 rows 21.0 and 29.7. In
// GPT-2 small's step, with bias and GELU: fc1 forward 29.2 us and 34.3 for
// GEMM and bias_gelu, fc2's input gradient 29.6 and 34.0.
#include "dfattn_internal.h"
#include "dfattn_status.h"
#include "dfgpt2.h"
#include "gpt2_device.h"

#include <algorithm>
#include <climits>
#include <cstdint>
#include <initializer_list>
#include <string>

namespace dfattn {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

constexpr int kTerms = 2;        // bf16 terms of a value
constexpr int kB = 32;           // rows of a block, and contraction values per step
constexpr int kBlock = kB * kB;  // values of a staged block and term

__device__ __forceinline__ f32x16 mfma_bf16(bf16x8_t a, bf16x8_t b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// An operand's block: 32 rows (of C's rows or columns) by 32 contraction values,
// in LDS as kTerms bf16 tiles of 64-byte rows. KC: [rows][k] in memory (k
// contiguous) and LDS, its 16-byte granules swizzled so that one granule of 16
// rows covers all banks; else [k][rows] in both, read transposed (four rows of
// 16 columns from each of two lane groups cover all banks as they lie).
template <bool KC>
struct Operand {
  const float *p;
  int ld, rows, k;
  static __device__ __forceinline__ int off(int line, int g) {
    return line * kB + ((KC ? g ^ ((line >> 2) & 3) : g) << 3);
  }
  // Lane's 8 values of half h (16 lines) of the block of rows row0 at k0:
  // line 16h + lane/4, values 8*(lane%4) .. +7. Values past the operand read as zeros.
  __device__ __forceinline__ void load(int row0, int k0, int h, int lane, float4 (&x)[2]) const {
    const int line = 16 * h + (lane >> 2), v = 8 * (lane & 3);
    const int l0 = KC ? row0 : k0, v0 = KC ? k0 : row0;             // first line, first value
    const int n_lines = KC ? rows : k, n_values = KC ? k : rows;
    const int lines = min(n_lines - l0, kB);
    const auto rs = buffer_rsrc(p + (size_t)min(l0, n_lines) * ld, lines > 0 ? (unsigned)((lines - 1) * ld + n_values) * 4u : 0u);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = v0 + v + 4 * i;
      x[i] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(rs, c < n_values ? (line * ld + c) * 4 : 0x7ffffffc, 0, 0));
      // A line's last load may hold the next line's first values: those of a
      // contraction line count, those past C's edge are not stored.
      if (KC && (k & 3) && k0 + kB > k) {
        if (c + 1 >= k) x[i].y = 0.f;
        if (c + 2 >= k) x[i].z = 0.f;
        if (c + 3 >= k) x[i].w = 0.f;
      }
    }
  }
  static __device__ __forceinline__ void store(__bf16 *block, int h, int lane, const float4 (&x)[2]) {
    const f32x2_t v[4] = {{x[0].x, x[0].y}, {x[0].z, x[0].w}, {x[1].x, x[1].y}, {x[1].z, x[1].w}};
    u32x4_t term[kTerms];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f32x2_t r = v[i];
#pragma unroll
      for (int n = 0; n < kTerms; ++n) {
        const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2_t));
        term[n][i] = u;
        if (n + 1 < kTerms) r = f32x2_t{r.x - __uint_as_float(u << 16), r.y - __uint_as_float(u & 0xffff0000u)};
      }
    }
    const int o = off(16 * h + (lane >> 2), lane & 3);
#pragma unroll
    for (int n = 0; n < kTerms; ++n) *reinterpret_cast<u32x4_t *>(block + n * kBlock + o) = term[n];
  }
  // Fragment of a term's block, step ks: lane c + 32*hh holds row c, k = 16*ks + 8*hh + 0..7.
  static __device__ __forceinline__ bf16x8_t frag(const __bf16 *t, int ks, int lane) {
    const int c = lane & 31, hh = lane >> 5;
    if constexpr (KC) return *reinterpret_cast<const bf16x8_t *>(t + off(c, 2 * ks + hh));
    // Lane r of each 16 reads 4 values of k = k0 + r/4; the result holds column i of four k.
    typedef __attribute__((address_space(3))) const __bf16 lds_bf16;
    const int r = lane & 15;
    lds_bf16 *b = (lds_bf16 *)t + (16 * ks + 8 * hh + (r >> 2)) * kB + 16 * ((lane >> 4) & 1) + 4 * (r & 3);
    const i16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)b);
    const i16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(b + 4 * kB));
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    return __builtin_bit_cast(bf16x8_t, i16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]});
  }
};

enum Epilogue {
  kPlain,     // C = sum
  kBias,      // C = sum + e[column]
  kBiasGelu,  // C = sum + e[column], out2 = gelu(C)
  kGeluGrad,  // C = sum * gelu'(e), e as C
};

// C [M][N] = A B over K. A workgroup computes 32*BM x 32*BN of C with KW groups
// of BM waves; group g takes the contraction steps g, g + KW, ... through LDS
// blocks of its own, its wave w the 32 rows 32*w .. and all the columns, and the
// groups' sums are added at the end in group order.
template <bool AKC, bool BKC, int BM, int BN, int KW, Epilogue EP>
__global__ __launch_bounds__(64 * BM * KW) void gemm_kernel(const float *__restrict__ A, const float *__restrict__ B,
                                                            float *__restrict__ C, const float *__restrict__ e,
                                                            float *__restrict__ out2, int M, int N, int K, int lda,
                                                            int ldb, int tiles_n, int n_tiles) {
  constexpr int kStage = (BM + BN) * kTerms * kBlock;
  constexpr int kHalves = 2 * (BM + BN), kPer = (kHalves + BM - 1) / BM;  // half blocks per step, and per wave
  constexpr int kSums = KW > 1 ? KW * BM * BN * 16 * 64 * 4 : 0;
  constexpr int kRing = KW * 2 * kStage * 2;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[kRing > kSums ? kRing : kSums];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wv / BM, wave = wv % BM;
  __bf16 *ring = reinterpret_cast<__bf16 *>(lds_raw) + (size_t)grp * 2 * kStage;
  int t = blockIdx.x;
  if (n_tiles % 8 == 0) t = (t & 7) * (n_tiles >> 3) + (t >> 3);
  const int tm = __builtin_amdgcn_readfirstlane(t / tiles_n), tn = t - tm * tiles_n;
  const int m0 = tm * kB * BM, n0 = tn * kB * BN;
  const Operand<AKC> a{A, lda, M, K};
  const Operand<BKC> b{B, ldb, N, K};

  const int steps = ((K + kB - 1) / kB + KW - 1) / KW;  // of every group
  float4 x[kPer][2];
  auto load = [&](int s) {
    const int k0 = (s * KW + grp) * kB;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int hb = wave + BM * i;  // half block: A's first, then B's
      if (hb < 2 * BM)
        a.load(m0 + kB * (hb >> 1), k0, hb & 1, lane, x[i]);
      else if (hb < kHalves)
        b.load(n0 + kB * ((hb >> 1) - BM), k0, hb & 1, lane, x[i]);
    }
  };
  auto store = [&](int st) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int hb = wave + BM * i;
      __bf16 *block = ring + st * kStage + (hb >> 1) * kTerms * kBlock;
      if (hb < 2 * BM)
        Operand<AKC>::store(block, hb & 1, lane, x[i]);
      else if (hb < kHalves)
        Operand<BKC>::store(block, hb & 1, lane, x[i]);
    }
  };
  f32x16 acc[BN];
#pragma unroll
  for (int j = 0; j < BN; ++j) acc[j] = f32x16{};
  load(0);
  store(0);
  load(1);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const __bf16 *cur = ring + (s & 1) * kStage;
    if (s + 1 < steps) {
      store((s + 1) & 1);
      if (s + 2 < steps) load(s + 2);
    }
#pragma unroll
    for (int ks = 0; ks < kB / 16; ++ks) {
      bf16x8_t fa[kTerms];
#pragma unroll
      for (int n = 0; n < kTerms; ++n) fa[n] = Operand<AKC>::frag(cur + (wave * kTerms + n) * kBlock, ks, lane);
#pragma unroll
      for (int j = 0; j < BN; ++j) {
        bf16x8_t fb[kTerms];
#pragma unroll
        for (int n = 0; n < kTerms; ++n)
          fb[n] = Operand<BKC>::frag(cur + ((BM + j) * kTerms + n) * kBlock, ks, lane);
        // Smallest products first.
#pragma unroll
        for (int o = kTerms - 1; o >= 0; --o)
#pragma unroll
          for (int n = 0; n <= o; ++n) acc[j] = mfma_bf16(fa[n], fb[o - n], acc[j]);
      }
    }
    __syncthreads();
  }
  const int c = lane & 31, hh = lane >> 5;
  // Rows and column of registers 4q .. 4q+3 of block j: row0 + i, col.
  auto row0 = [&](int q) { return m0 + kB * wave + 8 * q + 4 * hh; };
  auto col_of = [&](int j) { return n0 + kB * j + c; };
  auto out = [&](int j, int q, f32x4 v, f32x4 x) {  // x: GELU's inputs
    const int col = col_of(j);
    if (col >= N) return;
    const float bias = EP == kBias || EP == kBiasGelu ? e[col] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (row0(q) + i >= M) break;
      const size_t at = (size_t)(row0(q) + i) * N + col;
      if constexpr (EP == kGeluGrad) {
        C[at] = gelu_grad(v[i], x[i]);
      } else {
        const float y = EP == kPlain ? v[i] : v[i] + bias;
        C[at] = y;
        if constexpr (EP == kBiasGelu) out2[at] = gelu_f(y);
      }
    }
  };
  constexpr int kQuads = BN * 4, kMine = (kQuads + KW - 1) / KW;  // of a wave, and those it finishes
  f32x4 x_in[kMine] = {};
  if constexpr (EP == kGeluGrad) {  // on their way while the groups' sums are exchanged
#pragma unroll
    for (int p = 0; p < kMine; ++p) {
      const int q = grp + KW * p, col = col_of(q >> 2);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (q < kQuads && col < N && row0(q & 3) + i < M) x_in[p][i] = e[(size_t)(row0(q & 3) + i) * N + col];
    }
  }
  f32x4 *part = reinterpret_cast<f32x4 *>(lds_raw) + (size_t)wave * kQuads * 64 + lane;
  constexpr int kGroup = BM * kQuads * 64;
#pragma unroll
  for (int j = 0; j < BN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      part[grp * kGroup + (j * 4 + q) * 64] = f32x4{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
  __syncthreads();
#pragma unroll
  for (int p = 0; p < kMine; ++p) {
    const int q = grp + KW * p;
    if (q >= kQuads) break;
    f32x4 v = part[q * 64];
#pragma unroll
    for (int g = 1; g < KW; ++g) v += part[g * kGroup + q * 64];
    out(q >> 2, q & 3, v, x_in[p]);
  }
}

int ceil_div(int a, int b) { return (a + b - 1) / b; }

struct Gemm {
  const float *A, *B;
  float *C;
  const float *e;
  float *out2;
  int M, N, K, lda, ldb;
};

template <bool AKC, bool BKC, Epilogue EP, int BM, int BN, int KW>
bool launch_tile(const Gemm &g, hipStream_t stream) {
  const int tn = ceil_div(g.N, kB * BN);
  const int64_t tiles = (int64_t)ceil_div(g.M, kB * BM) * tn;
  if (tiles * 64 * BM * KW > UINT_MAX) return false;  // threads of a launch
  const int n = (int)tiles;
  hipLaunchKernelGGL((gemm_kernel<AKC, BKC, BM, BN, KW, EP>), dim3((unsigned)n), dim3(64 * BM * KW), 0, stream, g.A, g.B,
                     g.C, g.e, g.out2, g.M, g.N, g.K, g.lda, g.ldb, tn, n);
  return true;
}

// The tile: each CU runs one at a time, so a product takes ceil(tiles / 256)
// times a tile's time, which measures (us at K = 768) 22 for 128 x 96, 14 for
// 128 x 64 and 10 for 64 x 64, however many run. M x N of 1024 x 3072: 23, 30
// and 36 us; 2304 x 768 (K = 1024): 23, 19 and 24; 1024 x 768: 18, 14 and 10.
template <bool AKC, bool BKC, Epilogue EP>
int launch_gemm(const char *fn, const Gemm &g, hipStream_t stream) {
  // Row offsets inside a block stay in int.
  if (g.lda >= 1 << 24 || g.ldb >= 1 << 24 || g.M > INT_MAX - 512 || g.N > INT_MAX - 512 || g.K > INT_MAX - 512)
    return record_error(DFATTN_ERR_OVERFLOW, std::string(fn) + ": shape is too large");
  auto cost = [&](int m, int n, int tile) {
    return ((int64_t)ceil_div(g.M, m) * ceil_div(g.N, n) + 255) / 256 * tile;
  };
  const int64_t large = cost(128, 96, 11), medium = cost(128, 64, 7), small = cost(64, 64, 5);
  const bool fits = small <= medium && small <= large ? launch_tile<AKC, BKC, EP, 2, 2, 4>(g, stream)
                    : medium <= large                 ? launch_tile<AKC, BKC, EP, 4, 2, 2>(g, stream)
                                                      : launch_tile<AKC, BKC, EP, 4, 3, 2>(g, stream);
  if (!fits) return record_error(DFATTN_ERR_OVERFLOW, std::string(fn) + ": shape is too large");
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? DFATTN_OK : record_error(DFATTN_ERR_HIP, std::string(fn) + ": " + hipGetErrorString(err));
}

// rows == 0 leaves nothing to compute, or sums over nothing.
int check(const char *fn, uint32_t rows, uint32_t in, uint32_t out, std::initializer_list<const void *> data,
          std::initializer_list<const void *> optional) {
  if (in == 0 || out == 0) return record_error(DFATTN_ERR_SHAPE, std::string(fn) + ": features must be >= 1");
  if (rows > (uint32_t)INT_MAX || in > (uint32_t)INT_MAX || out > (uint32_t)INT_MAX)
    return record_error(DFATTN_ERR_OVERFLOW, std::string(fn) + ": shape is too large");
  for (const void *p : data)
    if (p == nullptr && rows > 0) return record_error(DFATTN_ERR_NULL_POINTER, std::string(fn) + ": null pointer");
  for (const auto &list : {data, optional})
    for (const void *p : list)
      if (reinterpret_cast<uintptr_t>(p) % 4 != 0)
        return record_error(DFATTN_ERR_MISALIGNED, std::string(fn) + ": pointer not 4-byte aligned");
  return DFATTN_OK;
}

}  // namespace
}  // namespace dfattn

using namespace dfattn;

extern "C" int dfgpt2_linear_forward(const float *x, const float *w, const float *bias, float *out, float *gelu_out,
                                     uint32_t rows, uint32_t in_features, uint32_t out_features, hipStream_t stream) {
  const char *fn = "dfgpt2_linear_forward";
  if (int st = check(fn, rows, in_features, out_features, {x, w, bias, out}, {gelu_out}); st != DFATTN_OK) return st;
  if (rows == 0) return DFATTN_OK;
  const Gemm g{x, w, out, bias, gelu_out, (int)rows, (int)out_features, (int)in_features, (int)in_features,
               (int)in_features};
  return gelu_out != nullptr ? launch_gemm<true, true, kBiasGelu>(fn, g, stream)
                             : launch_gemm<true, true, kBias>(fn, g, stream);
}

extern "C" int dfgpt2_linear_backward_input(const float *grad_out, const float *w, const float *gelu_in, float *grad_x,
                                            uint32_t rows, uint32_t in_features, uint32_t out_features,
                                            hipStream_t stream) {
  const char *fn = "dfgpt2_linear_backward_input";
  if (int st = check(fn, rows, in_features, out_features, {grad_out, w, grad_x}, {gelu_in}); st != DFATTN_OK) return st;
  if (rows == 0) return DFATTN_OK;
  const Gemm g{grad_out, w, grad_x, gelu_in, nullptr, (int)rows, (int)in_features, (int)out_features,
               (int)out_features, (int)in_features};
  return gelu_in != nullptr ? launch_gemm<true, false, kGeluGrad>(fn, g, stream)
                            : launch_gemm<true, false, kPlain>(fn, g, stream);
}

extern "C" int dfgpt2_linear_backward_weight(const float *grad_out, const float *x, float *grad_w, uint32_t rows,
                                             uint32_t in_features, uint32_t out_features, hipStream_t stream) {
  const char *fn = "dfgpt2_linear_backward_weight";
  if (int st = check(fn, rows, in_features, out_features, {grad_out, x}, {grad_w}); st != DFATTN_OK) return st;
  if (grad_w == nullptr) return record_error(DFATTN_ERR_NULL_POINTER, std::string(fn) + ": null pointer");
  const Gemm g{grad_out, x, grad_w, nullptr, nullptr, (int)out_features, (int)in_features, (int)rows,
               (int)out_features, (int)in_features};
  return launch_gemm<false, false, kPlain>(fn, g, stream);
}
