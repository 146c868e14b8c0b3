// Row permutation passes fused with layer norms (gfx950): the gather of the node features into
// Hilbert order before the mesh transformer's layers together with the first block's layer
// norm, and the final layer norm with its per-member affine together with the scatter back
// (patch.py:244, 274-276, 288-292). The second pass without a permutation is each block's
// conditioned layer norm, optionally with the residual add in front of it (patch.py:240-253).
//
// Both passes are HBM-bound streaming: one wave per row, 16 bytes per lane per load, so each
// wave-wide load or store covers 1 KB of one row. A row stays in registers between its
// statistics and its outputs, so every byte is read once. Statistics are float32: the mean
// first, then the biased variance of the centred values, both as fixed-order wave sums.
#include "rows_kernels.h"

#include "fwn_attn.h"

namespace fwn {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;  // rows per workgroup, one per wave

// Bit reinterpretation of a vector element. The element is passed by value: clang's
// __builtin_bit_cast applied to a subscripted ext_vector lvalue (v[e]) reads element 0 for
// every e (seen with this ROCm's hipcc), so it is never applied to v[e] directly.
__device__ __forceinline__ float as_float(uint32_t u) { return __builtin_bit_cast(float, u); }

template <typename T>
struct Vec;

template <>
struct Vec<float> {
  static constexpr int E = 4;  // elements per 16-byte vector
  __device__ __forceinline__ static void unpack(const u32x4& v, float (&f)[E]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = as_float(v[e]);
  }
  __device__ __forceinline__ static u32x4 pack(const float (&f)[E]) {
    return u32x4{__builtin_bit_cast(uint32_t, f[0]), __builtin_bit_cast(uint32_t, f[1]),
                 __builtin_bit_cast(uint32_t, f[2]), __builtin_bit_cast(uint32_t, f[3])};
  }
};

template <>
struct Vec<uint16_t> {  // bfloat16 bits
  static constexpr int E = 8;
  __device__ __forceinline__ static void unpack(const u32x4& v, float (&f)[E]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f[2 * k] = as_float(v[k] << 16);
      f[2 * k + 1] = as_float(v[k] & 0xffff0000u);
    }
  }
  __device__ __forceinline__ static u32x4 pack(const float (&f)[E]) {  // round to nearest even
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t lo = __builtin_bit_cast(uint16_t, (__bf16)f[2 * k]);
      const uint32_t hi = __builtin_bit_cast(uint16_t, (__bf16)f[2 * k + 1]);
      v[k] = lo | (hi << 16);
    }
    return v;
  }
};

// A row is read once by a pass: its loads are non-temporal, so that they do not push other rows out of
// the caches. Outputs are what the program's next kernel reads: they are stored through the caches
// while what a pass writes stays in the 256 MB memory-side cache, and non-temporally (NT) above. NT is a
// template parameter: of two stores in the branches of a run-time choice the compiler makes one, without
// the hint. Producer, pass and consumer of [1, n, 768], us for the pass and the consumer, plain stores
// / non-temporal:
//   gather (two outputs), a tensor of 96 MB: float32 102 / 106, bf16 113 / 125; 126 MB 148 / 148, 155 / 144;
//     160 MB 197 / 180, 204 / 189; 240 MB 288 / 266, 286 / 267; 480 MB 571 / 553, 547 / 514
//   scatter (one output): 126 MB 91 / 98, 109 / 120; 176 MB 128 / 128, 158 / 160; 240 MB 186 / 171, 223 / 210
//   residual add and norm (two outputs): 126 MB 135 / 144, 149 / 154; 160 MB 184 / 172, 199 / 188
//   gather's gradient: 240 MB 264 / 273, 287 / 296; 320 MB 363 / 363, 397 / 398; 480 MB 563 / 547, 613 / 599
//   scatter's gradient: 160 MB 148 / 158, 192 / 198; 240 MB 228 / 227, 280 / 280; 320 MB 306 / 296, 373 / 363.
// With plain loads scatter and the gradients are 5 to 15% slower from 126 MB up. The float32 gather with
// non-temporal stores takes them: up to 200 MB it is faster so (144 MB 166 for 174, 160 MB 180 for 184; at
// 320 MB 361 for 355).
constexpr uint64_t kStreamBytes = 256ull << 20;      // bytes written from which a pass stores non-temporally
constexpr uint64_t kStreamOneBytes = 192ull << 20;   // the same of a forward pass with one output

template <bool NT = true>
__device__ __forceinline__ u32x4 load16(const void* p) {
  if constexpr (NT) return __builtin_nontemporal_load((const u32x4*)p);
  return *(const u32x4*)p;
}
template <bool NT>
__device__ __forceinline__ void store16(void* p, const u32x4& v) {
  if constexpr (NT)
    __builtin_nontemporal_store(v, (u32x4*)p);
  else
    *(u32x4*)p = v;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// Loads one row (VPL vectors per lane, vector lane + 64k) and returns its mean and 1/std. With
// `row2`, the row is row + row2, added in float32 and rounded once to T (as a separate
// elementwise add would store it); v then holds that sum and the statistics are the sum's.
template <typename T, int VPL, bool NT = true>
__device__ __forceinline__ void load_row(const T* row, bool ok, int nv, int channels, float eps, int lane,
                                         u32x4 (&v)[VPL], float (&f)[VPL][Vec<T>::E], float& mean, float& rstd,
                                         const T* row2 = nullptr) {
  constexpr int E = Vec<T>::E;
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    const int idx = lane + 64 * k;
    v[k] = u32x4{0u, 0u, 0u, 0u};
    if (ok && idx < nv) v[k] = load16<NT>(row + (size_t)idx * E);
    Vec<T>::unpack(v[k], f[k]);
    if (row2) {
      u32x4 w = u32x4{0u, 0u, 0u, 0u};
      if (ok && idx < nv) w = load16<NT>(row2 + (size_t)idx * E);
      float g[E];
      Vec<T>::unpack(w, g);
#pragma unroll
      for (int e = 0; e < E; ++e) f[k][e] += g[e];
      v[k] = Vec<T>::pack(f[k]);
      Vec<T>::unpack(v[k], f[k]);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) sum += f[k][e];
  }
  mean = wave_sum(sum) / (float)channels;
  float sq = 0.f;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    if (lane + 64 * k >= nv) continue;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float c = f[k][e] - mean;
      sq = fmaf(c, c, sq);
    }
  }
  const float var = wave_sum(sq) / (float)channels;
  rstd = __builtin_amdgcn_rsqf(var + eps);
}

template <typename T, int VPL, bool NT>
__global__ void __launch_bounds__(64 * kWaves) gather_norm_kernel(RowArgs a) {
  constexpr int E = Vec<T>::E;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (row >= (int64_t)a.batch * a.n) return;  // whole waves leave together
  const int64_t b = row / a.n, i = row - b * a.n;
  const int64_t src = a.perm[i];
  const bool ok = src >= 0 && src < a.n;
  const size_t c = (size_t)a.channels;
  const int nv = a.channels / E;
  u32x4 v[VPL];
  float f[VPL][E];
  float mean, rstd;
  constexpr bool NTL = !(NT && sizeof(T) == 4);
  load_row<T, VPL, NTL>((const T*)a.x + (size_t)(b * a.n + (ok ? src : 0)) * c, ok, nv, a.channels, a.eps, lane, v, f,
                        mean, rstd);
  T* xo = (T*)a.x_out + (size_t)row * c;
  T* no = a.norm_out ? (T*)a.norm_out + (size_t)row * c : nullptr;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    const int idx = lane + 64 * k;
    if (idx >= nv) continue;
    store16<NT>(xo + (size_t)idx * E, v[k]);
    if (no) {
      float y[E];
#pragma unroll
      for (int e = 0; e < E; ++e) y[e] = (f[k][e] - mean) * rstd;
      store16<NT>(no + (size_t)idx * E, Vec<T>::pack(y));
    }
  }
}

// ADD: a.addend is added to x first and the sum written to a.x_out (a compile-time switch, so
// the plain pass carries no test for it).
template <typename T, int VPL, bool ADD, bool NT>
__global__ void __launch_bounds__(64 * kWaves) norm_scatter_kernel(RowArgs a) {
  constexpr int E = Vec<T>::E;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (row >= (int64_t)a.batch * a.n) return;
  const int64_t b = row / a.n, i = row - b * a.n;
  const int64_t dst = a.perm ? a.perm[i] : i;  // no permutation: the conditioned layer norm alone
  if (dst < 0 || dst >= a.n) return;
  const size_t c = (size_t)a.channels;
  const int nv = a.channels / E;
  u32x4 v[VPL];
  float f[VPL][E];
  float mean, rstd;
  load_row<T, VPL>((const T*)a.x + (size_t)row * c, true, nv, a.channels, a.eps, lane, v, f, mean, rstd,
                   ADD ? (const T*)a.addend + (size_t)row * c : nullptr);
  if constexpr (ADD) {  // the sum x + addend, in place of x's row (the whole row is in registers)
    T* so = (T*)a.x_out + (size_t)row * c;
#pragma unroll
    for (int k = 0; k < VPL; ++k)
      if (lane + 64 * k < nv) store16<NT>(so + (size_t)(lane + 64 * k) * E, v[k]);
  }
  T* o = (T*)a.out + (size_t)(b * a.n + dst) * c;
  const float* mul = a.mul ? a.mul + (size_t)b * c : nullptr;
  const float* add = a.add ? a.add + (size_t)b * c : nullptr;
#pragma unroll
  for (int k = 0; k < VPL; ++k) {
    const int idx = lane + 64 * k;
    if (idx >= nv) continue;
    float y[E];
#pragma unroll
    for (int e = 0; e < E; ++e) y[e] = (f[k][e] - mean) * rstd;
    if (mul) {
#pragma unroll
      for (int q = 0; q < E / 4; ++q) {
        const u32x4 m = *(const u32x4*)(mul + (size_t)idx * E + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] *= as_float(m[e]);
      }
    }
    if (add) {
#pragma unroll
      for (int q = 0; q < E / 4; ++q) {
        const u32x4 m = *(const u32x4*)(add + (size_t)idx * E + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] += as_float(m[e]);
      }
    }
    store16<NT>(o + (size_t)idx * E, Vec<T>::pack(y));
  }
}

template <typename T, int VPL, bool NT>
hipError_t launch_tvn(RowPass pass, const RowArgs& a, hipStream_t stream) {
  const int64_t rows = (int64_t)a.batch * a.n;
  const dim3 grid((unsigned)((rows + kWaves - 1) / kWaves)), block(64 * kWaves);
  if (pass == RowPass::kGatherNorm)
    hipLaunchKernelGGL((gather_norm_kernel<T, VPL, NT>), grid, block, 0, stream, a);
  else if (a.addend)
    hipLaunchKernelGGL((norm_scatter_kernel<T, VPL, true, NT>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((norm_scatter_kernel<T, VPL, false, NT>), grid, block, 0, stream, a);
  return hipGetLastError();
}

template <typename T, int VPL>
hipError_t launch_tv(RowPass pass, const RowArgs& a, hipStream_t stream) {
  return a.stream ? launch_tvn<T, VPL, true>(pass, a, stream) : launch_tvn<T, VPL, false>(pass, a, stream);
}

template <typename T>
hipError_t launch_t(RowPass pass, const RowArgs& a, hipStream_t stream) {
  const int per_lane = (a.channels / Vec<T>::E + 63) / 64;  // 16-byte vectors per lane
  if (per_lane <= 1) return launch_tv<T, 1>(pass, a, stream);
  if (per_lane <= 2) return launch_tv<T, 2>(pass, a, stream);
  if (per_lane <= 3) return launch_tv<T, 3>(pass, a, stream);
  if (per_lane <= 4) return launch_tv<T, 4>(pass, a, stream);
  if (per_lane <= 8) return launch_tv<T, 8>(pass, a, stream);
  if (per_lane <= 16) return launch_tv<T, 16>(pass, a, stream);
  return hipErrorInvalidValue;
}

// ------------------------------------------------------------------------------------------
// Backward of both passes (autograd of patch.py:240-253, 274-276, 288-292; JAX differentiates the
// reference's own). One wave per row: x and the gradients are read once, the statistics are
// recomputed in registers, and the input gradient is written once, so the pass is bound by HBM as
// the forward is (3 or 4 tensors of traffic). The per-channel sums of the affine's gradients stay in
// each lane's registers over all rows of its wave (a strided share of one batch member's rows), are
// added over the workgroup's waves in LDS and go out as one partial row per workgroup, which
// sums_kernel adds; both orders are fixed. At [1, 40962, 768] float32: with the sums 76 + 6 us (378 MB,
// 5.0 TB/s), gather_norm's 81 us (504 MB, its scattered rows written whole; 6.2 TB/s); bf16 with sums
// and the residual's gradient 58 + 6 us. The same gradients as torch operations took 15 to 25
// launches: a gather, scatter and their gradients 1.64 -> 0.33 ms, a block's training pass by
// 1.5 ms.
constexpr int kSumGroups = 16;  // partial rows added in parallel by sums_kernel's workgroup

__device__ __forceinline__ void wave_sum2(float& x, float& y) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    x += __shfl_xor(x, o);
    y += __shfl_xor(y, o);
  }
}

template <typename T, int VPL, bool SUMS, bool NT>
__global__ void __launch_bounds__(64 * kWaves) norm_bwd_kernel(RowBwdArgs a) {
  constexpr int E = Vec<T>::E;
  extern __shared__ float sums[];  // SUMS: [2][channels]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int b = (int)blockIdx.x / a.blocks, blk = (int)blockIdx.x - b * a.blocks;
  const size_t c = (size_t)a.channels, base = (size_t)b * a.n;
  const int nv = a.channels / E;
  const float inv_c = 1.f / (float)a.channels;
  const float* mul = a.mul ? a.mul + (size_t)b * c : nullptr;
  float sm[SUMS ? VPL : 1][E], sa[SUMS ? VPL : 1][E];
  if constexpr (SUMS) {
#pragma unroll
    for (int k = 0; k < VPL; ++k)
#pragma unroll
      for (int e = 0; e < E; ++e) sm[k][e] = sa[k][e] = 0.f;
  }
  for (int64_t i = (int64_t)blk * kWaves + wave; i < a.n; i += (int64_t)a.blocks * kWaves) {
    const int64_t src = a.perm_grad ? a.perm_grad[i] : i, dst = a.perm_out ? a.perm_out[i] : i;
    const bool has = a.g_norm && (uint64_t)src < (uint64_t)a.n;
    const T* gn = (const T*)a.g_norm + (base + (size_t)(has ? src : 0)) * c;
    const T* gr = a.g_res ? (const T*)a.g_res + (base + (size_t)i) * c : nullptr;
    u32x4 gv[VPL], rv[VPL];
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int idx = lane + 64 * k;
      gv[k] = rv[k] = u32x4{0u, 0u, 0u, 0u};
      if (has && idx < nv) gv[k] = load16(gn + (size_t)idx * E);
      if (gr && idx < nv) rv[k] = load16(gr + (size_t)idx * E);
    }
    u32x4 v[VPL];
    float f[VPL][E];
    float mean, rstd;
    load_row<T, VPL>((const T*)a.x + (base + (size_t)i) * c, true, nv, a.channels, a.eps, lane, v, f, mean, rstd);
    float g[VPL][E], s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int idx = lane + 64 * k;
      Vec<T>::unpack(gv[k], g[k]);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        f[k][e] = (f[k][e] - mean) * rstd;
        if constexpr (SUMS) {
          sm[k][e] = fmaf(g[k][e], f[k][e], sm[k][e]);
          sa[k][e] += g[k][e];
        }
      }
      if (mul && idx < nv) {
#pragma unroll
        for (int q = 0; q < E / 4; ++q) {
          const u32x4 m = *(const u32x4*)(mul + (size_t)idx * E + 4 * q);
#pragma unroll
          for (int e = 0; e < 4; ++e) g[k][4 * q + e] *= as_float(m[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        s1 += g[k][e];
        s2 = fmaf(g[k][e], f[k][e], s2);
      }
    }
    wave_sum2(s1, s2);
    const float m1 = s1 * inv_c, m2 = s2 * inv_c;
    if ((uint64_t)dst >= (uint64_t)a.n) continue;
    T* out = (T*)a.gx + (base + (size_t)dst) * c;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int idx = lane + 64 * k;
      if (idx >= nv) continue;
      float r[E], y[E];
      Vec<T>::unpack(rv[k], r);
#pragma unroll
      for (int e = 0; e < E; ++e) y[e] = fmaf(rstd, g[k][e] - m1 - f[k][e] * m2, r[e]);
      store16<NT>(out + (size_t)idx * E, Vec<T>::pack(y));
    }
  }
  if constexpr (SUMS) {
    for (int w = 0; w < kWaves; ++w) {
      if (wave == w) {
#pragma unroll
        for (int k = 0; k < VPL; ++k) {
          const int idx = lane + 64 * k;
          if (idx >= nv) continue;
#pragma unroll
          for (int e = 0; e < E; ++e) {
            float* p = sums + (size_t)idx * E + e;
            p[0] = w == 0 ? sm[k][e] : p[0] + sm[k][e];
            p[c] = w == 0 ? sa[k][e] : p[c] + sa[k][e];
          }
        }
      }
      __syncthreads();
    }
    float* part = a.part + (size_t)blockIdx.x * 2 * c;
    for (int j = threadIdx.x; j < 2 * a.channels; j += 64 * kWaves) part[j] = sums[j];
  }
}

// g_mul and g_add from the partial rows: 64 columns per workgroup, kSumGroups strided shares of a
// batch member's partial rows, added in LDS.
__global__ void __launch_bounds__(64 * kSumGroups) sums_kernel(RowBwdArgs a) {
  __shared__ float red[kSumGroups][64];
  const int lane = threadIdx.x & 63, grp = (int)threadIdx.x >> 6;
  const int cols = 2 * a.channels, per = (cols + 63) / 64;
  const int b = (int)blockIdx.x / per, j = ((int)blockIdx.x - b * per) * 64 + lane;
  float s = 0.f;
  if (j < cols) {
    const float* p = a.part + (size_t)b * a.blocks * cols + j;
#pragma unroll 8
    for (int r = grp; r < a.blocks; r += kSumGroups) s += p[(size_t)r * cols];
  }
  red[grp][lane] = s;
  __syncthreads();
  if (grp != 0 || j >= cols) return;
#pragma unroll
  for (int r = 1; r < kSumGroups; ++r) s += red[r][lane];
  if (j < a.channels)
    a.g_mul[(size_t)b * a.channels + j] = s;
  else
    a.g_add[(size_t)b * a.channels + j - a.channels] = s;
}

// ------------------------------------------------------------------------------------------
// The conditioning of several norms in one launch: one thread per output column, its weight row read
// straight from memory (64 bytes at 32 bf16 conditioning features; read once for 4 batch members).
// Bound by launches, not by bytes: each norm's own GEMM, add and two casts are four or five launches.
// 49 norms of 768 channels, issued back to back: 1.7 to 2.0 ms norm by norm, 58 us here (most of it
// the host's); the refinement-6 forward of a 24-layer transformer, which has 48 of its 49 norms in the
// launch (block 0's first is projected by itself), 30.04 -> 29.84 ms.
template <typename T>
__device__ __forceinline__ float load_one(const void* p, size_t i) {
  if constexpr (sizeof(T) == 4) {
    return ((const float*)p)[i];
  } else {
    return as_float((uint32_t)((const uint16_t*)p)[i] << 16);
  }
}

template <typename T>
__global__ void __launch_bounds__(256) cond_kernel(CondArgs a) {
  const int cols = 2 * a.channels, per = (cols + 255) / 256;
  const int l = (int)blockIdx.x / per, j = ((int)blockIdx.x - l * per) * 256 + (int)threadIdx.x;
  if (j >= cols) return;
  const void* w = a.weight[l];
  const float first = load_one<T>(a.bias[l], (size_t)j) + (j < a.channels ? 1.f : 0.f);
  float* out = (j < a.channels ? a.mul + j : a.add + (j - a.channels)) + (size_t)l * a.batch * a.channels;
  constexpr int MEMBERS = 4;  // one pass over the weight row for this many batch members
  for (int b0 = 0; b0 < a.batch; b0 += MEMBERS) {
    const int nb = a.batch - b0 < MEMBERS ? a.batch - b0 : MEMBERS;
    float sum[MEMBERS] = {};
#pragma unroll 8
    for (int k = 0; k < a.cond_size; ++k) {
      const float wk = load_one<T>(w, (size_t)j * a.cond_size + k);
#pragma unroll
      for (int m = 0; m < MEMBERS; ++m)
        sum[m] = fmaf(wk, load_one<T>(a.cond, (size_t)(b0 + (m < nb ? m : 0)) * a.cond_size + k), sum[m]);
    }
#pragma unroll
    for (int m = 0; m < MEMBERS; ++m)
      if (m < nb) out[(size_t)(b0 + m) * a.channels] = sum[m] + first;
  }
}

template <typename T, int VPL, bool NT>
hipError_t launch_bwd_tvn(const RowBwdArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)a.blocks * (unsigned)a.batch), block(64 * kWaves);
  if (!a.part) {
    hipLaunchKernelGGL((norm_bwd_kernel<T, VPL, false, NT>), grid, block, 0, stream, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL((norm_bwd_kernel<T, VPL, true, NT>), grid, block, 2 * (unsigned)a.channels * sizeof(float), stream, a);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  const unsigned per = (2u * (unsigned)a.channels + 63u) / 64u;
  hipLaunchKernelGGL(sums_kernel, dim3(per * (unsigned)a.batch), dim3(64 * kSumGroups), 0, stream, a);
  return hipGetLastError();
}

template <typename T, int VPL>
hipError_t launch_bwd_tv(const RowBwdArgs& a, hipStream_t stream) {
  return a.stream ? launch_bwd_tvn<T, VPL, true>(a, stream) : launch_bwd_tvn<T, VPL, false>(a, stream);
}

template <typename T>
hipError_t launch_bwd_t(const RowBwdArgs& a, hipStream_t stream) {
  const int per_lane = (a.channels / Vec<T>::E + 63) / 64;
  if (per_lane <= 1) return launch_bwd_tv<T, 1>(a, stream);
  if (per_lane <= 2) return launch_bwd_tv<T, 2>(a, stream);
  if (per_lane <= 3) return launch_bwd_tv<T, 3>(a, stream);
  if (per_lane <= 4) return launch_bwd_tv<T, 4>(a, stream);
  if (per_lane <= 8) return launch_bwd_tv<T, 8>(a, stream);
  if constexpr (Vec<T>::E == 4) return launch_bwd_tv<T, 16>(a, stream);  // float32, up to 4,096 channels
  return hipErrorInvalidValue;
}

// Bytes of one [batch, n, channels] tensor.
uint64_t tensor_bytes(int dtype, int64_t batch, int64_t n, int64_t channels) {
  return (uint64_t)(batch * n) * (uint64_t)(channels * (dtype == FWN_F32 ? 4 : 2));
}

}  // namespace

hipError_t launch_rows(RowPass pass, int dtype, const RowArgs& args, hipStream_t stream) {
  RowArgs a = args;
  if ((int64_t)a.batch * a.n == 0) return hipSuccess;
  const uint64_t bytes = tensor_bytes(dtype, a.batch, a.n, a.channels);
  const bool two = pass == RowPass::kGatherNorm ? a.norm_out != nullptr : a.addend != nullptr;
  a.stream = two ? 2 * bytes >= kStreamBytes : bytes >= kStreamOneBytes;
  return dtype == FWN_F32 ? launch_t<float>(pass, a, stream) : launch_t<uint16_t>(pass, a, stream);
}

// Four rows per wave at least (with sums: each workgroup writes a partial row), and about four
// workgroups per CU over the whole call; without sums twice as many, one row per wave for small calls.
int32_t rows_bwd_blocks(int32_t batch, int32_t n, bool sums) {
  const int64_t rows = sums ? 4 * kWaves : kWaves, most = sums ? 1024 : 2048;
  const int64_t want = ((int64_t)n + rows - 1) / rows, cap = most / (batch > 0 ? batch : 1);
  const int64_t blocks = want < cap ? want : cap;
  return (int32_t)(blocks > 1 ? blocks : 1);
}

hipError_t launch_cond(int dtype, const CondArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)a.count * ((2u * (unsigned)a.channels + 255u) / 256u)), block(256);
  if (dtype == FWN_F32)
    hipLaunchKernelGGL(cond_kernel<float>, grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL(cond_kernel<uint16_t>, grid, block, 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_rows_bwd(int dtype, const RowBwdArgs& args, hipStream_t stream) {
  RowBwdArgs a = args;
  a.stream = tensor_bytes(dtype, a.batch, a.n, a.channels) >= kStreamBytes;
  return dtype == FWN_F32 ? launch_bwd_t<float>(a, stream) : launch_bwd_t<uint16_t>(a, stream);
}

}  // namespace fwn
