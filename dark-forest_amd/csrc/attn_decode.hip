// attn_decode.hip — single-query attention against a KV cache (autoregressive
// decode), gfx950.
//
// Reference: attention_fused.cu:551-615 (kernel_fused_mha_decode_kv), 622-745
// (split-K kernel and its reduction), 800-1090 (paged pools, fp32 and bf16).
// Per head h and cached keys t = 0 .. L-1 (row t of the cache, or of the pool
// through the block table): out = softmax_t(scale * q.k_t) . v_t, computed as
// an online softmax; nothing is written when L is 0.
//
// The work is split over the key range: workgroup (h, c) takes keys
// [c*chunk, min(L, (c+1)*chunk)) and either writes the normalised output
// (one chunk) or the chunk's partial (m, l, unnormalised o) in the reference's
// split-K layout (m, l: [H, n_chunks]; o: [H, n_chunks, D]), which
// decode_reduce_kernel merges with the logsumexp identity.
//
// decode_kernel: 8 waves; each wave takes groups of keys. Its loads are coalesced
// rows: LPR lanes (8, 16 or 32, the smallest power of two >= D/4) read 4 values
// each (16 bytes fp32, 8 bytes bf16) of one row, 64/LPR rows per load, all of a
// group's K and V loads before the first wait. The score of a row is reduced
// over its lanes, gathered through LDS so that lane r holds key r for the
// softmax, and P goes back through LDS to the V lanes. Rows that are not 4-value
// aligned (D % 4 != 0, or an odd base) load value by value.
// decode_few_kernel: caches of up to three keys, one wave per head.
#include "dfattn_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace dfattn {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kDecWaves = 8;
constexpr int kDecThreads = 64 * kDecWaves;

struct DecodeArgs {
  const float *q;            // [H*D]
  const void *k, *v;         // rows of H*D values (fp32, or bf16 bit patterns)
  const int32_t *table;      // logical page -> physical block; null: contiguous cache
  int page_size;
  int H, L, D;
  float scale;
  int chunk, n_chunks;
  float *out, *lse;                  // n_chunks == 1
  float *part_m, *part_l, *part_o;   // n_chunks > 1
};

__device__ __forceinline__ size_t cache_row(const DecodeArgs &a, int t) {
  if (a.table == nullptr) return (size_t)t;
  return (size_t)a.table[t / a.page_size] * (size_t)a.page_size + (size_t)(t % a.page_size);
}

// 4 consecutive values of a cache row: the raw bits (fp32: the floats; bf16:
// four bf16 in the low 8 bytes), loaded without conversion so that every
// load of a group is issued before the first wait, and widened later. A
// call reads each cache row once, and a long cache is larger than the
// caches: the loads are nontemporal (streaming), which measured 10-11 %
// faster at 131072 rows than cached loads.
typedef unsigned raw2_t __attribute__((ext_vector_type(2)));
typedef unsigned raw4_t __attribute__((ext_vector_type(4)));
template <bool BF16>
__device__ __forceinline__ uint4 load4_raw(const void *base, size_t elem) {
  if constexpr (BF16) {
    const raw2_t u = __builtin_nontemporal_load(
        reinterpret_cast<const raw2_t *>(reinterpret_cast<const unsigned short *>(base) + elem));
    return make_uint4(u.x, u.y, 0u, 0u);
  } else {
    const raw4_t u =
        __builtin_nontemporal_load(reinterpret_cast<const raw4_t *>(reinterpret_cast<const float *>(base) + elem));
    return make_uint4(u.x, u.y, u.z, u.w);
  }
}
template <bool BF16>
__device__ __forceinline__ float4 widen4(uint4 r) {
  if constexpr (BF16)
    return make_float4(__builtin_bit_cast(float, r.x << 16), __builtin_bit_cast(float, r.x & 0xffff0000u),
                       __builtin_bit_cast(float, r.y << 16), __builtin_bit_cast(float, r.y & 0xffff0000u));
  else
    return __builtin_bit_cast(float4, r);
}

// The same for rows without that alignment: value by value, the values at or
// past D (clamped loads) zeroed in widen4_any.
template <bool BF16>
__device__ __forceinline__ uint4 load4_any(const void *base, size_t row, int d0, int D) {
  unsigned u[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const size_t e = row + min(d0 + j, D - 1);
    u[j] = BF16 ? (unsigned)reinterpret_cast<const unsigned short *>(base)[e] << 16
                : reinterpret_cast<const unsigned *>(base)[e];
  }
  return make_uint4(u[0], u[1], u[2], u[3]);
}
__device__ __forceinline__ float4 widen4_any(uint4 r, int d0, int D) {
  const float4 v = __builtin_bit_cast(float4, r);
  return make_float4(d0 < D ? v.x : 0.f, d0 + 1 < D ? v.y : 0.f, d0 + 2 < D ? v.z : 0.f, d0 + 3 < D ? v.w : 0.f);
}

template <int CTRL>
__device__ __forceinline__ float add_dpp(float x) {
  return x + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
// Sum over each aligned group of LPR lanes, in every lane of the group: DPP
// moves within the row of 16 lanes (rotations by 8, 4, 2, 1, or for 8 lanes
// two swaps within the quad and the half-row mirror), full-rate VALU instead
// of LDS-pipe permutes, and for 32 lanes one permlane16 swap.
template <int LPR>
__device__ __forceinline__ float group_sum(float x) {
  if constexpr (LPR == 8) return add_dpp<0x141>(add_dpp<0x4e>(add_dpp<0xb1>(x)));
  x = add_dpp<0x121>(add_dpp<0x122>(add_dpp<0x124>(add_dpp<0x128>(x))));
  if constexpr (LPR == 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return x;
}

// Writes one chunk's (m, l, o) — m and the scores in the log2 domain — as the
// normalised output and logsumexp (one chunk) or as the chunk's partial in the
// reference's layout (m converted to the natural-log domain).
__device__ __forceinline__ void write_chunk(const DecodeArgs &a, int h, int c, int d, float m2, float l,
                                            float o) {
  if (a.n_chunks == 1) {
    a.out[(size_t)h * a.D + d] = l > 0.f ? o / l : 0.f;
    if (d == 0 && a.lse) a.lse[h] = l > 0.f ? (m2 + __builtin_log2f(l)) * kLn2 : -INFINITY;
  } else {
    const size_t slot = (size_t)h * a.n_chunks + c;
    a.part_o[slot * a.D + d] = o;
    if (d == 0) {
      a.part_m[slot] = m2 * kLn2;
      a.part_l[slot] = l;
    }
  }
}

// How a row lies on its lanes: it fills them (D = 4 * LPR), it leaves some out,
// or its 4-value pieces are not aligned (any D).
enum Rows { kFull, kPartial, kUnaligned };

// Bound by HBM (K and V are read once) or, for short caches, by latency: one
// group's loads are all in flight before its first wait. Against one wave per
// chunk taking one key at a time, any D but 64 (H, keys): 274 -> 4.5 us (4, 509,
// D 32 bf16 paged), 368 -> 10.6 us (7, 18490, D 32 bf16 paged), 527 -> 14 us (8,
// 4096, D 128 fp32), 7.0 ms -> 395 us (16, 131072, D 128 fp32: 5.4 TB/s).
// Row and key bounds checked at run time in every group cost a 1024-key decode
// 0.8 of 8.0 us: D = 32, 64 and 128 have kernels of their own, and only the
// last group of a chunk has key bounds. There the V of rows past the end is
// masked; leaving them out by a branch per load cost the wave with the last group
// 0.2-0.5 us (12 heads, 300 keys of D 64 fp32: 6.6 us, now 6.2).
template <bool BF16, bool PAGED, int LPR, Rows ROWS>
__global__ __launch_bounds__(kDecThreads) void decode_kernel(DecodeArgs a) {
  constexpr int kRowsPerLoad = 64 / LPR;
  constexpr int kLoads = LPR == 8 ? 8 : 16;           // K (and V) loads per group and lane
  constexpr int kGroup = kRowsPerLoad * kLoads;       // keys per group: 64, 64, 32
  constexpr int kCols = 4 * LPR;
  constexpr bool VEC = ROWS != kUnaligned;
  // Physical rows of 32-bit size but for the narrowest rows, which a GPU could hold more of.
  using row_t = std::conditional_t<LPR == 8, size_t, unsigned>;
  __shared__ float s_lds[kDecWaves][kGroup];   // scores, then P, of the wave's group
  __shared__ row_t row_lds[kDecWaves][kGroup];  // paged: the group's physical rows
  __shared__ float m_lds[kDecWaves], l_lds[kDecWaves];
  __shared__ __attribute__((aligned(16))) float o_lds[kDecWaves][kCols];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int sub = lane / LPR, d0 = 4 * (lane % LPR);  // row kRowsPerLoad*j + sub of a group, columns d0 .. +3
  const int h = blockIdx.y;
  const int D = ROWS == kFull ? kCols : a.D;
  const size_t dm = (size_t)a.H * D, hoff = (size_t)h * D;
  // Lanes past the row's values read column 0 and add nothing.
  const bool on = d0 < D;
  const size_t col = hoff + (on ? d0 : 0);
  float4 q4;
  if constexpr (VEC)
    q4 = *reinterpret_cast<const float4 *>(a.q + col);
  else
    q4 = widen4_any(load4_any<false>(a.q, hoff, d0, D), d0, D);
  const float c2 = a.scale * kLog2e;

  for (int c = blockIdx.x;;) {
    const int t0 = c * a.chunk, t1 = min(a.L, t0 + a.chunk);
    float m = -INFINITY, l = 0.f;
    float4 o4 = make_float4(0.f, 0.f, 0.f, 0.f);
    // One group: keys g0 .. g0+kGroup-1, the last group's only those below t1.
    auto group = [&](int g0, auto last) {
      constexpr bool kLast = decltype(last)::value;
      const int n = kLast ? t1 - g0 : kGroup;
      // Paged: lane r looks up the physical row of key g0 + r once, for every lane.
      if constexpr (PAGED) {
        if (lane < kGroup) row_lds[wave][lane] = (row_t)cache_row(a, g0 + (kLast ? min(lane, n - 1) : lane));
        __builtin_amdgcn_wave_barrier();
      }
      // Rows past the last key read its row instead, so every load is unconditional.
      uint4 kr[kLoads], vr[kLoads];
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        int r = kRowsPerLoad * j + sub;
        if (kLast) r = min(r, n - 1);
        const size_t row = PAGED ? (size_t)row_lds[wave][r] : (size_t)(g0 + r);
        if constexpr (VEC) {
          kr[j] = load4_raw<BF16>(a.k, row * dm + col);
          vr[j] = load4_raw<BF16>(a.v, row * dm + col);
        } else {
          kr[j] = load4_any<BF16>(a.k, row * dm + hoff, d0, D);
          vr[j] = load4_any<BF16>(a.v, row * dm + hoff, d0, D);
        }
      }
      auto widen = [&](uint4 x) {
        if constexpr (VEC)
          return widen4<BF16>(x);
        else
          return widen4_any(x, d0, D);
      };
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const float4 k4 = widen(kr[j]);
        const float part = q4.x * k4.x + q4.y * k4.y + q4.z * k4.z + q4.w * k4.w;
        const float s = group_sum<LPR>(on ? part : 0.f);
        if (d0 == 0) s_lds[wave][kRowsPerLoad * j + sub] = s;
      }
      __builtin_amdgcn_wave_barrier();
      // Online softmax over the group, lane r = key g0 + r.
      const bool valid = lane < kGroup && (!kLast || lane < n);
      const float s2 = valid ? s_lds[wave][lane % kGroup] * c2 : -INFINITY;
      const float m_new = fmaxf(m, wave_max(s2));
      const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
      const float p = valid ? __builtin_amdgcn_exp2f(s2 - m_new) : 0.f;
      l = l * alpha + p;
      m = m_new;
      __builtin_amdgcn_wave_barrier();
      if (lane < kGroup) s_lds[wave][lane] = p;
      __builtin_amdgcn_wave_barrier();
      o4.x *= alpha;
      o4.y *= alpha;
      o4.z *= alpha;
      o4.w *= alpha;
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const float pj = s_lds[wave][kRowsPerLoad * j + sub];
        if (kLast) {
          // (The last key's value, read for the rows past it, may be infinite: 0 * inf is NaN.)
          const unsigned keep = (unsigned)((kRowsPerLoad * j + sub - n) >> 31);
          vr[j] = make_uint4(vr[j].x & keep, vr[j].y & keep, vr[j].z & keep, vr[j].w & keep);
        }
        const float4 v4 = widen(vr[j]);
        o4.x += pj * v4.x;
        o4.y += pj * v4.y;
        o4.z += pj * v4.z;
        o4.w += pj * v4.w;
      }
      __builtin_amdgcn_wave_barrier();
    };
    int g0 = t0 + kGroup * wave;
    for (; g0 + kGroup <= t1; g0 += kGroup * kDecWaves) group(g0, std::false_type{});
    if (g0 < t1) group(g0, std::true_type{});

    // The wave's (m, l, o): l summed over lanes, o over the rows of a load.
    l = wave_sum(l);
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) {
      o4.x += __shfl_xor(o4.x, off, 64);
      o4.y += __shfl_xor(o4.y, off, 64);
      o4.z += __shfl_xor(o4.z, off, 64);
      o4.w += __shfl_xor(o4.w, off, 64);
    }
    if (lane == 0) {
      m_lds[wave] = m;
      l_lds[wave] = l;
    }
    if (sub == 0) *reinterpret_cast<float4 *>(&o_lds[wave][d0]) = o4;
    __syncthreads();
    if (tid < kCols && tid < D) {
      // Merge the waves (a wave with no keys has m = -inf and weight 0).
      float mm = -INFINITY;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) mm = fmaxf(mm, m_lds[w]);
      float ll = 0.f, oo = 0.f;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) {
        const float f = m_lds[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_lds[w] - mm);
        ll += f * l_lds[w];
        oo += f * o_lds[w][tid];
      }
      write_chunk(a, h, c, tid, mm, ll, oo);
    }
    // Another chunk only where a grid cannot hold them all.
    c += gridDim.x;
    if (c >= a.n_chunks) break;
    __syncthreads();
  }
}

// A cache of at most kFewKeys keys: one wave per head, lane d holding columns d and
// d + 64, keys one at a time. The kernel above takes 3.2-4.9 us for any cache this
// short (a group of loads, the exchanges between lanes and waves); this one 2.3-3.0
// us for one key and 0.5 us for each more (12 heads, D 80 fp32: 2.9 and 4.5 us for
// one, 3.9 and 4.5 for three, 4.5 and 4.5 for four). At D 64 the two meet at one.
constexpr int kFewKeys = 3;
template <bool BF16>
__global__ __launch_bounds__(64) void decode_few_kernel(DecodeArgs a) {
  const int lane = threadIdx.x, h = blockIdx.x, D = a.D;
  const size_t dm = (size_t)a.H * D, hoff = (size_t)h * D;
  auto load = [&](const void *p, size_t e) {
    return BF16 ? __uint_as_float((unsigned)reinterpret_cast<const unsigned short *>(p)[e] << 16)
                : reinterpret_cast<const float *>(p)[e];
  };
  const bool in0 = lane < D, in1 = lane + 64 < D;
  const float q0 = in0 ? a.q[hoff + lane] : 0.f, q1 = in1 ? a.q[hoff + lane + 64] : 0.f;
  const float c2 = a.scale * kLog2e;
  float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
  for (int t = 0; t < a.L; ++t) {
    const size_t base = cache_row(a, t) * dm + hoff;
    float s = 0.f;
    if (in0) s += q0 * load(a.k, base + lane);
    if (in1) s += q1 * load(a.k, base + lane + 64);
    s = wave_sum(s) * c2;
    const float m_new = fmaxf(m, s);
    const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
    const float p = s == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s - m_new);
    l = l * alpha + p;
    m = m_new;
    o0 = o0 * alpha + (in0 ? p * load(a.v, base + lane) : 0.f);
    o1 = o1 * alpha + (in1 ? p * load(a.v, base + lane + 64) : 0.f);
  }
  if (in0) write_chunk(a, h, 0, lane, m, l, o0);
  if (in1) write_chunk(a, h, 0, lane + 64, m, l, o1);
}

template <int LPR, Rows ROWS>
void launch_decode_rows(const DecodeArgs &a, bool bf16, dim3 grid, hipStream_t stream) {
  const bool paged = a.table != nullptr;
  if (bf16 && paged)
    hipLaunchKernelGGL((decode_kernel<true, true, LPR, ROWS>), grid, dim3(kDecThreads), 0, stream, a);
  else if (bf16)
    hipLaunchKernelGGL((decode_kernel<true, false, LPR, ROWS>), grid, dim3(kDecThreads), 0, stream, a);
  else if (paged)
    hipLaunchKernelGGL((decode_kernel<false, true, LPR, ROWS>), grid, dim3(kDecThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((decode_kernel<false, false, LPR, ROWS>), grid, dim3(kDecThreads), 0, stream, a);
}

// Merges the split-K partials of one head (attention_fused.cu:712-757):
// m = max_c m_c, l = sum_c l_c exp(m_c - m), out = sum_c exp(m_c - m) o_c / l.
// Chunks whose m_c is not above -FLT_MAX hold no key and are skipped. 512
// threads per head: the chunks are strided over the threads (and, for o,
// over 8 groups of 64 columns), so the partial loads are independent of each
// other instead of one chained loop.
constexpr int kRedThreads = 512;
__device__ __forceinline__ float block_reduce(float v, float *scratch, bool is_max) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = is_max ? wave_max(v) : wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float r = scratch[0];
#pragma unroll
  for (int w = 1; w < kRedThreads / 64; ++w) r = is_max ? fmaxf(r, scratch[w]) : r + scratch[w];
  return r;
}

__global__ __launch_bounds__(kRedThreads) void decode_reduce_kernel(const float *__restrict__ part_m,
                                                                    const float *__restrict__ part_l,
                                                                    const float *__restrict__ part_o,
                                                                    float *__restrict__ out, float *__restrict__ lse,
                                                                    int n_chunks, int D) {
  __shared__ float scratch[kRedThreads / 64];
  __shared__ float w_lds[kRedThreads];
  __shared__ float acc_lds[kRedThreads / 64][128];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, grp = tid >> 6;
  constexpr int kGroups = kRedThreads / 64;
  constexpr int kPre = 8;  // o values a lane loads before the weights are known
  const float *pm = part_m + (size_t)h * n_chunks;
  const float *pl = part_l + (size_t)h * n_chunks;
  const float *po = part_o + (size_t)h * n_chunks * D;
  constexpr float kNoKey = -3.402823466e38f;  // -FLT_MAX, the reference's empty-chunk mark
  // Every load of the first kRedThreads chunks is issued at once: thread c
  // takes chunk c's (m, l); lane d of group g takes o[c][d] of chunks
  // c = g + 8i, i < kPre.
  const bool mine = tid < n_chunks;
  const float m_c = mine ? pm[tid] : -INFINITY, l_c = mine ? pl[tid] : 0.f;
  float o0[kPre], o1[kPre];
#pragma unroll
  for (int i = 0; i < kPre; ++i) {
    const int cc = grp + kGroups * i;
    o0[i] = cc < n_chunks && lane < D ? po[(size_t)cc * D + lane] : 0.f;
    o1[i] = cc < n_chunks && lane + 64 < D ? po[(size_t)cc * D + lane + 64] : 0.f;
  }
  float mm = m_c;
  for (int cc = tid + kRedThreads; cc < n_chunks; cc += kRedThreads) mm = fmaxf(mm, pm[cc]);
  mm = block_reduce(mm, scratch, true);
  const float w_c = m_c > kNoKey ? __expf(m_c - mm) : 0.f;
  w_lds[tid] = w_c;
  float ll = w_c * l_c;
  for (int cc = tid + kRedThreads; cc < n_chunks; cc += kRedThreads)
    if (pm[cc] > kNoKey) ll += pl[cc] * __expf(pm[cc] - mm);
  ll = block_reduce(ll, scratch, false);  // (its barriers also publish w_lds)
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int i = 0; i < kPre; ++i) {
    const int cc = grp + kGroups * i;
    if (cc < kRedThreads) {
      a0 += w_lds[cc] * o0[i];
      a1 += w_lds[cc] * o1[i];
    }
  }
  for (int cc = grp + kGroups * kPre; cc < n_chunks; cc += kGroups) {
    const float m2 = pm[cc];
    const float w = cc < kRedThreads ? w_lds[cc] : (m2 > kNoKey ? __expf(m2 - mm) : 0.f);
    if (lane < D) a0 += w * po[(size_t)cc * D + lane];
    if (lane + 64 < D) a1 += w * po[(size_t)cc * D + lane + 64];
  }
  acc_lds[grp][lane] = a0;
  acc_lds[grp][lane + 64] = a1;
  __syncthreads();
  if (grp == 0) {
    const float inv = ll > 0.f ? 1.f / ll : 0.f;
    for (int d = lane; d < D; d += 64) {
      float o = 0.f;
#pragma unroll
      for (int g = 0; g < kGroups; ++g) o += acc_lds[g][d];
      out[(size_t)h * D + d] = o * inv;
    }
    if (lane == 0 && lse) lse[h] = ll > 0.f ? mm + __logf(ll) : -INFINITY;
  }
}

}  // namespace

hipError_t launch_decode(const float *q, const void *k, const void *v, const int32_t *block_table,
                         int page_size, bool bf16, float *out, float *lse, int n_heads, int cur_len,
                         int d_head, float scale, int chunk, float *part_m, float *part_l, float *part_o,
                         bool aligned, hipStream_t stream) {
  DecodeArgs a;
  a.q = q;
  a.k = k;
  a.v = v;
  a.table = block_table;
  a.page_size = page_size > 0 ? page_size : 1;
  a.H = n_heads;
  a.L = cur_len;
  a.D = d_head;
  a.scale = scale;
  a.chunk = chunk >= cur_len || part_m == nullptr ? cur_len : chunk;
  a.n_chunks = (cur_len + a.chunk - 1) / a.chunk;
  a.out = out;
  a.lse = lse;
  a.part_m = part_m;
  a.part_l = part_l;
  a.part_o = part_o;
  if (cur_len <= kFewKeys && a.n_chunks == 1 && !(d_head == 64 && aligned)) {
    if (bf16)
      hipLaunchKernelGGL(decode_few_kernel<true>, dim3((unsigned)n_heads), dim3(64), 0, stream, a);
    else
      hipLaunchKernelGGL(decode_few_kernel<false>, dim3((unsigned)n_heads), dim3(64), 0, stream, a);
    return hipGetLastError();
  }
  const dim3 grid((unsigned)std::min(a.n_chunks, 1 << 20), (unsigned)n_heads);
  // 8 lanes to a row up to 32 values, 16 up to 64, 32 up to 128.
  auto with_lanes = [&](auto lpr) {
    constexpr int LPR = decltype(lpr)::value;
    if (!aligned)
      launch_decode_rows<LPR, kUnaligned>(a, bf16, grid, stream);
    else if (d_head == 4 * LPR)
      launch_decode_rows<LPR, kFull>(a, bf16, grid, stream);
    else
      launch_decode_rows<LPR, kPartial>(a, bf16, grid, stream);
  };
  if (d_head <= 32)
    with_lanes(std::integral_constant<int, 8>{});
  else if (d_head <= 64)
    with_lanes(std::integral_constant<int, 16>{});
  else
    with_lanes(std::integral_constant<int, 32>{});
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || a.n_chunks == 1) return err;
  hipLaunchKernelGGL(decode_reduce_kernel, dim3((unsigned)n_heads), dim3(kRedThreads), 0, stream, part_m, part_l,
                     part_o, out, lse, a.n_chunks, d_head);
  return hipGetLastError();
}

}  // namespace dfattn
