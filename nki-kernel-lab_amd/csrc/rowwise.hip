// Row-wise kernels: fused softmax, three-pass softmax, RMSNorm, SwiGLU.
//
// These are HBM-bound: every input byte is read once and every output byte
// written once (the three-pass softmax deliberately round-trips its fp32
// intermediates through HBM, as the reference's unfused kernel does).
//
// Outputs are written with non-temporal (streaming) stores, which reach HBM
// faster than write-back stores for data the kernel never reads again.
//
// Layout: a row is held in registers by 1, 4 or 16 wavefronts (pick_row), each
// lane with NV 16-byte vectors, so it is read from HBM exactly once and the
// reductions are wavefront shuffles (and one LDS exchange per reduction when
// several wavefronts share the row).  Rows whose length, stride or base is off
// 16 bytes are read and written with the same 16-byte instructions at the
// element's own alignment (gfx950 takes them at any address); the elements
// ahead of the row's first 64-byte boundary and its last ones go one to a
// lane.  One wavefront per row with element loads and three sweeps took 315 us
// for the softmax of 1000 x 20000 fp32 and 336 of 66 x 31363, inputs rotated
// through twice the last-level cache (276 and 173 with them in the cache);
// sixteen wavefronts holding the row take 26.8 (6.0 TB/s) and 7.7 (24.0 and 6.3).
// Rows past 65536 elements take the looped kernels, which re-read the row (from
// L2) once per pass.
#include <math.h>

#include <type_traits>

#include "common.h"

namespace nkl {

constexpr int kRowsPerBlock = 4;

// 16 bytes at the alignment of T only.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));

__device__ __forceinline__ u32x4 ld16_any(const float* p) { return *reinterpret_cast<const u32x4_a4*>(p); }
__device__ __forceinline__ u32x4 ld16_any(const bf16* p) { return *reinterpret_cast<const u32x4_a2*>(p); }
__device__ __forceinline__ void unpack16(u32x4 t, float (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(t[i]);
}
__device__ __forceinline__ void unpack16(u32x4 t, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[2 * i] = bf16lo(t[i]), v[2 * i + 1] = bf16hi(t[i]);
}

// E elements at p as fp32 values (AL: p is 16-byte aligned).
template <bool AL, typename T, int E>
__device__ __forceinline__ void load_row_vec(const T* p, float (&v)[E]) {
  if constexpr (AL)
    load16(p, v);
  else
    unpack16(ld16_any(p), v);
}

// E fp32 values to p as T (E = 4 or 8), streaming.
template <bool AL, typename T, int E>
__device__ __forceinline__ void store_row_vec(T* p, const float (&v)[E]) {
  if constexpr (AL) {
    store_vec_nt<E>(p, v);
  } else if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < E; i += 4) {
      const u32x4 t = {__float_as_uint(v[i]), __float_as_uint(v[i + 1]), __float_as_uint(v[i + 2]),
                       __float_as_uint(v[i + 3])};
      __builtin_nontemporal_store(t, reinterpret_cast<u32x4_a4*>(p + i));
    }
  } else {
    auto pack = [](float a, float b) {
      if constexpr (std::is_same<T, bf16>::value)
        return pack_bf16x2(a, b);
      else
        return pack_f16x2(a, b);
    };
    if constexpr (E == 8) {
      const u32x4 t = {pack(v[0], v[1]), pack(v[2], v[3]), pack(v[4], v[5]), pack(v[6], v[7])};
      __builtin_nontemporal_store(t, reinterpret_cast<u32x4_a2*>(p));
    } else {
      const u32x2 t = {pack(v[0], v[1]), pack(v[2], v[3])};
      __builtin_nontemporal_store(t, reinterpret_cast<u32x2_a2*>(p));
    }
  }
}

// Elements of a row ahead of its first 64-byte boundary in y: the vectors start
// there, so that whole-vector stores do not straddle lines (4097 x 2049 bf16
// softmax 7.6 us, 8.0 with vectors from the row's first element; 500 x 20001
// fp32 17.3, 17.8 from the first 16-byte boundary).
template <typename T>
__device__ __forceinline__ int row_head(const T* y, int cols) {
  return min(cols, (int)((0u - (unsigned)(uintptr_t)y) % 64 / sizeof(T)));
}

// max / sum over the WPR wavefronts of a row (WPR > 1: the whole workgroup;
// `red` is one of the kernel's LDS arrays, used once).
template <int WPR>
__device__ __forceinline__ float row_max(float v, float* red) {
  v = wave_max(v);
  if constexpr (WPR > 1) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < WPR; ++i) v = fmaxf(v, red[i]);
  }
  return v;
}
template <int WPR>
__device__ __forceinline__ float row_sum(float v, float* red) {
  v = wave_sum(v);
  if constexpr (WPR > 1) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < WPR; ++i) v += red[i];
  }
  return v;
}

// ------------------------------------------------------------- softmax --
// nkilab/kernels/norm.py:65-89: neg_max = -max(x); e = exp(x + neg_max) with
// the row sum in fp32; rinv = 1 / sum; y = e * rinv rounded once.
// Wavefronts per SIMD the compiler makes room for: two 1024-thread workgroups a
// CU where their rows' registers (32 values a lane) allow it (softmax, rotated
// inputs, us, in brackets inputs in the cache: 1000 x 20000 fp32 30.8 -> 26.8 (30.4
// -> 24.0), 1000 x 32768 bf16 27.3 -> 22.7).  The unaligned form would spill (500 x
// 20001 16.5 -> 18.3 (15.7 -> 18.2)).
constexpr int row_waves(int wpr, int nv, int e, bool al) { return al && wpr == 16 && nv * e <= 32 ? 8 : 1; }

template <typename T, int WPR, int NV, bool AL>
__global__ __launch_bounds__(WPR == 1 ? 256 : 64 * WPR, row_waves(WPR, NV, VecE<T>::value, AL)) void softmax_vec_kernel(const T* __restrict__ x,
                                                                                T* __restrict__ y, int rows, int cols,
                                                                                long ldx, long ldy) {
  constexpr int E = VecE<T>::value;
  __shared__ float red[2][WPR];
  const int t = WPR == 1 ? threadIdx.x & 63 : threadIdx.x;
  const int row = WPR == 1 ? blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6) : blockIdx.x;
  if (row >= rows) return;  // WPR > 1: one row per workgroup, never taken
  const T* xr = x + (long)row * ldx;
  T* yr = y + (long)row * ldy;
  const int head = AL ? 0 : NV == 0 ? cols : row_head(yr, cols);
  const int nvec = (cols - head) / E, edge = AL ? 0 : cols - nvec * E;
  // Edge element of lane t < edge: the row's first head, then its last ones.
  const int te = t < head ? t : nvec * E + t;
  float v[NV > 0 ? NV : 1][E];
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int vi = n * 64 * WPR + t;
    if (vi < nvec) {
      load_row_vec<AL>(xr + head + vi * E, v[n]);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) v[n][e] = -INFINITY;
    }
  }
  float tv = -INFINITY;
  if (t < edge) tv = to_f32(xr[te]);
  float mx = tv;
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < E; ++e) mx = fmaxf(mx, v[n][e]);
  mx = row_max<WPR>(mx, red[0]);
  const float mx2 = mx * kLog2e;
  float sum = 0.f;
  if constexpr (!AL) sum = tv = fast_exp2(fmaf(tv, kLog2e, -mx2));
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      v[n][e] = fast_exp2(fmaf(v[n][e], kLog2e, -mx2));
      sum += v[n][e];
    }
  sum = row_sum<WPR>(sum, red[1]);
  const float rinv = 1.0f / sum;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int vi = n * 64 * WPR + t;
    if (vi < nvec) {
      float o[E];
#pragma unroll
      for (int e = 0; e < E; ++e) o[e] = v[n][e] * rinv;
      store_row_vec<AL>(yr + head + vi * E, o);
    }
  }
  if (t < edge) yr[te] = from_f32<T>(tv * rinv);
}

// Rows too long for registers: one 1024-thread workgroup per row, three sweeps
// over the row.
template <typename T>
__global__ __launch_bounds__(1024) void softmax_loop_kernel(const T* __restrict__ x, T* __restrict__ y, int cols,
                                                            long ldx, long ldy) {
  constexpr int E = VecE<T>::value;
  __shared__ float red[2][16];
  const T* xr = x + (long)blockIdx.x * ldx;
  T* yr = y + (long)blockIdx.x * ldy;
  const int t = threadIdx.x, nvec = cols / E, tail = cols - nvec * E;
  float v[E];
  float tv = -INFINITY;
  if (t < tail) tv = to_f32(xr[(long)nvec * E + t]);
  float mx = tv;
  for (int vi = t; vi < nvec; vi += 1024) {
    load_row_vec<false>(xr + (long)vi * E, v);
#pragma unroll
    for (int e = 0; e < E; ++e) mx = fmaxf(mx, v[e]);
  }
  mx = row_max<16>(mx, red[0]);
  const float mx2 = mx * kLog2e;
  float sum = tv = fast_exp2(fmaf(tv, kLog2e, -mx2));
  for (int vi = t; vi < nvec; vi += 1024) {
    load_row_vec<false>(xr + (long)vi * E, v);
#pragma unroll
    for (int e = 0; e < E; ++e) sum += fast_exp2(fmaf(v[e], kLog2e, -mx2));
  }
  sum = row_sum<16>(sum, red[1]);
  const float rinv = 1.0f / sum;
  for (int vi = t; vi < nvec; vi += 1024) {
    load_row_vec<false>(xr + (long)vi * E, v);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = fast_exp2(fmaf(v[e], kLog2e, -mx2)) * rinv;
    store_row_vec<false>(yr + (long)vi * E, v);
  }
  if (t < tail) yr[(long)nvec * E + t] = from_f32<T>(tv * rinv);
}

// ---------------------------------------------------- three-pass softmax --
// nkilab/kernels/norm.py:22-62.  Pass 1: m = max(x) -> HBM.  Pass 2:
// e = exp(x - m) (fp32, -> HBM) and s = sum(e) -> HBM.  Pass 3: y = e / s.
template <typename T>
__global__ __launch_bounds__(256) void softmax_pass1_kernel(const T* __restrict__ x, float* __restrict__ m,
                                                            int rows, int cols, long ldx) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* xr = x + (long)row * ldx;
  float mx = -INFINITY;
  for (int c = lane; c < cols; c += kWave) mx = fmaxf(mx, to_f32(xr[c]));
  mx = wave_max(mx);
  if (lane == 0) m[row] = mx;
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_pass2_kernel(const T* __restrict__ x, const float* __restrict__ m,
                                                            float* __restrict__ e, float* __restrict__ s,
                                                            int rows, int cols, long ldx) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* xr = x + (long)row * ldx;
  float* er = e + (long)row * cols;
  const float mr = m[row];
  float sum = 0.f;
  for (int c = lane; c < cols; c += kWave) {
    const float t = fast_exp2((to_f32(xr[c]) - mr) * kLog2e);
    er[c] = t;
    sum += t;
  }
  sum = wave_sum(sum);
  if (lane == 0) s[row] = sum;
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_pass3_kernel(const float* __restrict__ e, const float* __restrict__ s,
                                                            T* __restrict__ y, int rows, int cols, long ldy) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* er = e + (long)row * cols;
  T* yr = y + (long)row * ldy;
  const float sr = s[row];
  for (int c = lane; c < cols; c += kWave) yr[c] = from_f32<T>(er[c] / sr);
}

// ------------------------------------------------------------- RMSNorm --
// nkilab/kernels/norm.py:92-118: ssq = sum(x^2) (fp32); ms = ssq * (1/D) + eps;
// rstd = rsqrt(ms); xn = x * rstd (fp32); y = xn * w rounded once.
// E weight elements of type TW as fp32 values.
template <bool AL, int E>
__device__ __forceinline__ void load_w(const float* p, float (&v)[E]) {
#pragma unroll
  for (int i = 0; i < E; i += 4) {
    float t[4];
    load_row_vec<AL>(p + i, t);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[i + k] = t[k];
  }
}
template <bool AL, int E>
__device__ __forceinline__ void load_w(const bf16* p, float (&v)[E]) {
  if constexpr (E == 8) {
    load_row_vec<AL>(p, v);
  } else {
    static_assert(E == 4, "4 or 8 weights per vector");
    const u32x2 t = AL ? *reinterpret_cast<const u32x2*>(p) : *reinterpret_cast<const u32x2_a2*>(p);
    v[0] = bf16lo(t[0]), v[1] = bf16hi(t[0]), v[2] = bf16lo(t[1]), v[3] = bf16hi(t[1]);
  }
}

template <typename TI, typename TW, typename TO, int WPR, int NV, bool AL>
__global__ __launch_bounds__(WPR == 1 ? 256 : 64 * WPR, row_waves(WPR, NV, VecE<TI>::value, AL)) void rmsnorm_vec_kernel(
    const TI* __restrict__ x, const TW* __restrict__ w, TO* __restrict__ y, int rows, int cols, long ldx, long ldy,
    float inv_d, float eps) {
  constexpr int E = VecE<TI>::value;
  __shared__ float red[WPR];
  const int t = WPR == 1 ? threadIdx.x & 63 : threadIdx.x;
  const int row = WPR == 1 ? blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6) : blockIdx.x;
  if (row >= rows) return;  // WPR > 1: one row per workgroup, never taken
  const TI* xr = x + (long)row * ldx;
  TO* yr = y + (long)row * ldy;
  const int head = AL ? 0 : NV == 0 ? cols : row_head(yr, cols);
  const int nvec = (cols - head) / E, edge = AL ? 0 : cols - nvec * E;
  // Edge element of lane t < edge: the row's first head, then its last ones.
  const int te = t < head ? t : nvec * E + t;
  const bool two = NV == 0 && t + kWave < cols;  // (a row of edge elements alone: two a lane)
  float v[NV > 0 ? NV : 1][E];
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int vi = n * 64 * WPR + t;
    if (vi < nvec) {
      load_row_vec<AL>(xr + head + vi * E, v[n]);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) v[n][e] = 0.f;
    }
  }
  float tv = 0.f, tv2 = 0.f;
  if (t < edge) tv = to_f32(xr[te]);
  if (two) tv2 = to_f32(xr[t + kWave]);
  float ssq = fmaf(tv2, tv2, tv * tv);
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < E; ++e) ssq = fmaf(v[n][e], v[n][e], ssq);
  ssq = row_sum<WPR>(ssq, red);
  const float rstd = __frsqrt_rn(fmaf(ssq, inv_d, eps));
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int vi = n * 64 * WPR + t;
    if (vi < nvec) {
      float wv[E];
      load_w<AL>(w + head + vi * E, wv);
      float o[E];
#pragma unroll
      for (int e = 0; e < E; ++e) o[e] = (v[n][e] * rstd) * wv[e];
      store_row_vec<AL>(yr + head + vi * E, o);
    }
  }
  if (t < edge) yr[te] = from_f32<TO>((tv * rstd) * to_f32(w[te]));
  if (two) yr[t + kWave] = from_f32<TO>((tv2 * rstd) * to_f32(w[t + kWave]));
}

// Rows too long for registers: one 1024-thread workgroup per row, two sweeps.
template <typename TI, typename TW, typename TO>
__global__ __launch_bounds__(1024) void rmsnorm_loop_kernel(const TI* __restrict__ x, const TW* __restrict__ w,
                                                            TO* __restrict__ y, int cols, long ldx, long ldy,
                                                            float inv_d, float eps) {
  constexpr int E = VecE<TI>::value;
  __shared__ float red[16];
  const TI* xr = x + (long)blockIdx.x * ldx;
  TO* yr = y + (long)blockIdx.x * ldy;
  const int t = threadIdx.x, nvec = cols / E, tail = cols - nvec * E;
  float v[E];
  float tv = 0.f;
  if (t < tail) tv = to_f32(xr[(long)nvec * E + t]);
  float ssq = tv * tv;
  for (int vi = t; vi < nvec; vi += 1024) {
    load_row_vec<false>(xr + (long)vi * E, v);
#pragma unroll
    for (int e = 0; e < E; ++e) ssq = fmaf(v[e], v[e], ssq);
  }
  ssq = row_sum<16>(ssq, red);
  const float rstd = __frsqrt_rn(fmaf(ssq, inv_d, eps));
  for (int vi = t; vi < nvec; vi += 1024) {
    float wv[E];
    load_row_vec<false>(xr + (long)vi * E, v);
    load_w<false>(w + (long)vi * E, wv);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = (v[e] * rstd) * wv[e];
    store_row_vec<false>(yr + (long)vi * E, v);
  }
  if (t < tail) yr[(long)nvec * E + t] = from_f32<TO>((tv * rstd) * to_f32(w[(long)nvec * E + t]));
}

// -------------------------------------------------------------- SwiGLU --
// nkilab/kernels/norm.py:121-136: a = silu(g) in fp32; y = a * u rounded once
// (silu is in common.h, shared with the GEMM's gate/up epilogue).

// Each thread handles UNROLL 16-byte vectors spaced a grid-width apart.
template <typename T, int UNROLL>
__global__ __launch_bounds__(256) void swiglu_vec_kernel(const T* __restrict__ g, const T* __restrict__ u,
                                                         T* __restrict__ y, long nvec) {
  constexpr int E = VecE<T>::value;
  const long stride = (long)gridDim.x * blockDim.x;
  const long base = (long)blockIdx.x * blockDim.x + threadIdx.x;
  float gv[UNROLL][E], uv[UNROLL][E];
#pragma unroll
  for (int r = 0; r < UNROLL; ++r) {
    const long vi = base + r * stride;
    if (vi < nvec) {
      load16(g + vi * E, gv[r]);
      load16(u + vi * E, uv[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < UNROLL; ++r) {
    const long vi = base + r * stride;
    if (vi < nvec) {
      float o[E];
#pragma unroll
      for (int e = 0; e < E; ++e) o[e] = silu(gv[r][e]) * uv[r][e];
      store_vec_nt<E>(y + vi * E, o);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void swiglu_tail_kernel(const T* __restrict__ g, const T* __restrict__ u,
                                                          T* __restrict__ y, long start, long n) {
  const long i = start + (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = from_f32<T>(silu(to_f32(g[i])) * to_f32(u[i]));
}

// ------------------------------------------------------------ dispatch --
static bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Wavefronts per row and vectors per lane (a power of two) that hold a row of
// nvec 16-byte vectors in registers; nv = 0 when it is longer than 16
// wavefronts hold (64 values a lane).
//
// One wavefront holds up to 16 vectors a lane; four share the row when that
// fills the chip sooner: from 4 vectors a lane while every row's workgroup
// fits one round (2048 of 256 threads; rotated inputs, us, one wavefront /
// four: softmax 1536 x 2048 bf16 5.2 / 4.7, RMSNorm 5.2 / 4.3, 2048 x 2048
// fp32 -> fp16 6.3 / 5.7; past one round one wavefront is level or ahead: 3000
// x 2048 bf16 softmax 5.7 / 6.3).  Sixteen vectors a lane turn at `deep_rows`
// (fp32 softmax 1024 x 4096 7.6 / 6.0 but 1536 x 4096 9.0 / 9.7).  128 values a
// lane (16 vectors in 16 bits) always go to four times the wavefronts (bf16
// softmax 4096 x 8192 25.2 / 21.0; four / sixteen: 1000 x 32768 24.1 / 22.7,
// RMSNorm 31.8 / 22.2).
struct RowPlan {
  int wpr, nv;
};
// Short unaligned rows: one element a lane of one wavefront (RMSNorm: up to
// two), no vectors.  300000 rows in the last-level cache, us, with vectors /
// without: softmax bf16 x 3 54.3 / 39.7, x 17 62.0 / 43.0, x 64 62.6 / 45.8,
// fp32 x 17 54.7 / 43.5, but 65536 x 64 12.5 / 13.8; RMSNorm bf16 x 17 53.3 / 39.1,
// x 65 67.4 / 55.3, x 127 68.4 / 57.0, fp32 x 63 57.0 / 42.9; where y's rows all
// start on 64 bytes and fill both elements, bf16 x 96 53.4 / 60.9.
constexpr RowPlan kShortRow{1, 0};

template <typename T>
static RowPlan pick_row(int rows, int cols, int deep_rows) {
  constexpr int E = VecE<T>::value;
  const int nvec = cols / E;  // full vectors: the edges of an unaligned row ride in one more register
  for (int wpr : {1, 4, 16}) {
    const int cap = wpr == 16 ? 64 / E : 16;
    for (int nv = 1; nv <= cap; nv *= 2) {
      if (nvec > nv * 64 * wpr) continue;
      const bool more = nv * E > 64 || (wpr == 1 && nv >= 4 && rows <= (nv == 16 ? deep_rows : 2048));
      return more ? RowPlan{4 * wpr, nv / 4} : RowPlan{wpr, nv};
    }
  }
  return RowPlan{16, 0};
}

// Calls f(wpr, nv) with the plan's values as compile-time constants; false
// when the plan is the looped kernel's.
template <typename T, typename F>
static bool with_row_plan(RowPlan p, F f) {
#define NKL_ROW(W, N)                                                        \
  if (p.wpr == W && p.nv == N) {                                             \
    f(std::integral_constant<int, W>{}, std::integral_constant<int, N>{});   \
    return true;                                                             \
  }
  NKL_ROW(1, 0) NKL_ROW(1, 1) NKL_ROW(1, 2) NKL_ROW(1, 4) NKL_ROW(1, 8)
  if constexpr (VecE<T>::value == 4) { NKL_ROW(1, 16) }
  NKL_ROW(4, 1) NKL_ROW(4, 2) NKL_ROW(4, 4) NKL_ROW(4, 8)
  if constexpr (VecE<T>::value == 4) { NKL_ROW(4, 16) NKL_ROW(16, 16) } else { NKL_ROW(16, 4) }
  NKL_ROW(16, 8)
#undef NKL_ROW
  return false;
}

// Calls f(first row, rows, grid) for the launches of a row kernel: one, unless
// its threads pass HIP's limit (16.8M rows of 256 threads).
template <typename F>
static void for_row_launches(int rows, int rows_per_wg, int threads, F f) {
  const long step = kMaxGridThreads / threads * rows_per_wg;
  for (long r = 0; r < rows; r += step) {
    const int n = (int)min(step, rows - r);
    f(r, n, dim3((unsigned)(((long)n + rows_per_wg - 1) / rows_per_wg)));
  }
}

template <typename T>
static int softmax_launch_plan(RowPlan plan, const void* x, void* y, int rows, int cols, long ldx, long ldy,
                               hipStream_t st) {
  constexpr int E = VecE<T>::value;
  const T* xp = static_cast<const T*>(x);
  T* yp = static_cast<T*>(y);
  const bool al = cols % E == 0 && ldx % E == 0 && ldy % E == 0 && aligned16(x) && aligned16(y);
  if (!al && cols * sizeof(T) <= 128) plan = kShortRow;
  const bool done = with_row_plan<T>(plan, [&](auto W, auto N) {
    constexpr int WPR = decltype(W)::value, NV = decltype(N)::value, NT = WPR == 1 ? 256 : 64 * WPR;
    for_row_launches(rows, WPR == 1 ? kRowsPerBlock : 1, NT, [&](long r, int n, dim3 grid) {
      if (al)
        softmax_vec_kernel<T, WPR, NV, true><<<grid, dim3(NT), 0, st>>>(xp + r * ldx, yp + r * ldy, n, cols, ldx, ldy);
      else
        softmax_vec_kernel<T, WPR, NV, false><<<grid, dim3(NT), 0, st>>>(xp + r * ldx, yp + r * ldy, n, cols, ldx, ldy);
    });
  });
  if (!done)
    for_row_launches(rows, 1, 1024, [&](long r, int, dim3 grid) {
      softmax_loop_kernel<T><<<grid, dim3(1024), 0, st>>>(xp + r * ldx, yp + r * ldy, cols, ldx, ldy);
    });
  return check_launch("nkl_softmax");
}
template <typename T>
static int softmax_launch(const void* x, void* y, int rows, int cols, long ldx, long ldy, hipStream_t st) {
  return softmax_launch_plan<T>(pick_row<T>(rows, cols, 1280), x, y, rows, cols, ldx, ldy, st);
}

template <typename TI, typename TW, typename TO>
static int rmsnorm_launch_plan(RowPlan plan, const void* x, const void* w, void* y, int rows, int cols, long ldx,
                               long ldy, float eps, hipStream_t st) {
  constexpr int E = VecE<TI>::value;
  const TI* xp = static_cast<const TI*>(x);
  const TW* wp = static_cast<const TW*>(w);
  TO* yp = static_cast<TO*>(y);
  // The multiplier 1/D is the fp32 value nearest the exact quotient.
  const float inv_d = (float)(1.0 / (double)cols);
  const bool al = cols % E == 0 && ldx % E == 0 && ldy % E == 0 && aligned16(x) && aligned16(w) && aligned16(y);
  if (!al && cols * sizeof(TI) <= 256 && (cols <= kWave || ldy * sizeof(TO) % 64)) plan = kShortRow;
  const bool done = with_row_plan<TI>(plan, [&](auto W, auto N) {
    constexpr int WPR = decltype(W)::value, NV = decltype(N)::value, NT = WPR == 1 ? 256 : 64 * WPR;
    for_row_launches(rows, WPR == 1 ? kRowsPerBlock : 1, NT, [&](long r, int n, dim3 grid) {
      if (al)
        rmsnorm_vec_kernel<TI, TW, TO, WPR, NV, true><<<grid, dim3(NT), 0, st>>>(xp + r * ldx, wp, yp + r * ldy, n, cols,
                                                                                 ldx, ldy, inv_d, eps);
      else
        rmsnorm_vec_kernel<TI, TW, TO, WPR, NV, false><<<grid, dim3(NT), 0, st>>>(xp + r * ldx, wp, yp + r * ldy, n,
                                                                                  cols, ldx, ldy, inv_d, eps);
    });
  });
  if (!done)
    for_row_launches(rows, 1, 1024, [&](long r, int, dim3 grid) {
      rmsnorm_loop_kernel<TI, TW, TO><<<grid, dim3(1024), 0, st>>>(xp + r * ldx, wp, yp + r * ldy, cols, ldx, ldy, inv_d,
                                                                   eps);
    });
  return check_launch("nkl_rmsnorm");
}
template <typename TI, typename TW, typename TO>
static int rmsnorm_launch(const void* x, const void* w, void* y, int rows, int cols, long ldx, long ldy, float eps,
                          hipStream_t st) {
  return rmsnorm_launch_plan<TI, TW, TO>(pick_row<TI>(rows, cols, 2048), x, w, y, rows, cols, ldx, ldy, eps, st);
}

template <typename T>
static int swiglu_launch(const void* g, const void* u, void* y, long n, hipStream_t st) {
  constexpr int E = VecE<T>::value;
  // Two vectors of each input per thread.  In bench.py's harness at 4096 x
  // 2048 bf16 one per thread was no faster (10.8 against 10.7 us), four
  // slower, and per-workgroup contiguous chunks (with or without an
  // XCD-aware order) slower still.
  constexpr int UNROLL = 2;
  const T* gp = static_cast<const T*>(g);
  const T* up = static_cast<const T*>(u);
  T* yp = static_cast<T*>(y);
  long done = 0;
  if (aligned16(g) && aligned16(u) && aligned16(y)) {
    const long nvec = n / E;
    if (nvec > 0) {
      const long threads = (nvec + UNROLL - 1) / UNROLL;
      const long blocks = (threads + 255) / 256;
      swiglu_vec_kernel<T, UNROLL><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(gp, up, yp, nvec);
    }
    done = nvec * E;
  }
  if (done < n) {
    const long rem = n - done;
    swiglu_tail_kernel<T><<<dim3((unsigned)((rem + 255) / 256)), dim3(256), 0, st>>>(gp, up, yp, done, n);
  }
  return check_launch("nkl_swiglu");
}

// Streaming copy with the row kernels' loads and non-temporal stores and none
// of their arithmetic: each lane reads kCopyUnroll 16-byte chunks one grid
// span apart, then writes them.  Two per lane is the fastest of 1, 2, 4 and 8
// (and of per-workgroup contiguous chunks) at 16 - 128 MiB on MI355X.  It
// measures the HBM ceiling the row kernels' roofline is read against at the
// same size.
constexpr int kCopyUnroll = 2;
__global__ __launch_bounds__(256) void stream_copy_kernel(const u32x4* __restrict__ x, u32x4* __restrict__ y, long n) {
  const long base = (long)blockIdx.x * 256 + threadIdx.x, span = (long)gridDim.x * 256;
  u32x4 v[kCopyUnroll];
#pragma unroll
  for (int k = 0; k < kCopyUnroll; ++k) {
    const long i = base + k * span;
    v[k] = i < n ? x[i] : u32x4{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int k = 0; k < kCopyUnroll; ++k) {
    const long i = base + k * span;
    if (i < n) __builtin_nontemporal_store(v[k], y + i);
  }
}

// ------------------------------------------------------ hi/lo bf16 split --
// y[r, c] = bf16(x[r, c]) and y[r, cols + c] = bf16(x[r, c] - bf16(x[r, c])):
// an fp32 activation as two bf16 values whose sum carries 16 significand
// bits.  A GEMM over [hi | lo] (K doubled) against a bf16 weight stacked
// twice along K then accumulates x . w in fp32 to about 2^-17 of x: the
// decoder block runs its projections on bf16 MFMA at fp32 accuracy.
// One thread per 4 consecutive columns of a row (cols % 4 == 0, aligned rows).
__global__ __launch_bounds__(256) void split_bf16_kernel(const float* __restrict__ x, bf16* __restrict__ y, int rows,
                                                         int cols, long ldx, long ldy) {
  const int q = cols / 4;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)rows * q) return;
  const int r = (int)(i / q), c = 4 * (int)(i % q);
  float v[4];
  load16(x + (long)r * ldx + c, v);
  float hi[4], lo[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    hi[e] = (float)(bf16)v[e];
    lo[e] = v[e] - hi[e];  // exact in fp32
  }
  store_vec<4>(y + (long)r * ldy + c, hi);
  store_vec<4>(y + (long)r * ldy + cols + c, lo);
}

}  // namespace nkl

using namespace nkl;

static int check_rows(const char* fn, int rows, int cols, long ldx, long ldy) {
  if (rows < 0 || cols < 0) return set_error(NKL_EINVAL, "%s: negative shape (%d, %d)", fn, rows, cols);
  if (rows > 0 && cols > 0 && (ldx < cols || ldy < cols))
    return set_error(NKL_EINVAL, "%s: leading dimension (%ld, %ld) smaller than cols %d", fn, ldx, ldy, cols);
  return NKL_OK;
}

extern "C" int nkl_softmax(const void* x, void* y, int rows, int cols, long ldx, long ldy, int dtype,
                           void* stream) {
  int rc = check_rows("nkl_softmax", rows, cols, ldx, ldy);
  if (rc) return rc;
  if (rows == 0 || cols == 0) return NKL_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NKL_F32) return softmax_launch<float>(x, y, rows, cols, ldx, ldy, st);
  if (dtype == NKL_BF16) return softmax_launch<bf16>(x, y, rows, cols, ldx, ldy, st);
  return set_error(NKL_EDTYPE, "nkl_softmax: unsupported dtype %d", dtype);
}

extern "C" size_t nkl_softmax_unfused_workspace_bytes(int rows, int cols) {
  if (rows <= 0 || cols <= 0) return 0;
  const size_t r = ((size_t)rows * 4 + 255) / 256 * 256;
  return 2 * r + (size_t)rows * (size_t)cols * 4;
}

extern "C" int nkl_softmax_unfused(const void* x, void* y, void* workspace, size_t workspace_bytes, int rows,
                                   int cols, long ldx, long ldy, int dtype, void* stream) {
  int rc = check_rows("nkl_softmax_unfused", rows, cols, ldx, ldy);
  if (rc) return rc;
  if (rows == 0 || cols == 0) return NKL_OK;
  const size_t need = nkl_softmax_unfused_workspace_bytes(rows, cols);
  if (!workspace || workspace_bytes < need)
    return set_error(NKL_EWORKSPACE, "nkl_softmax_unfused: workspace of %zu bytes needed, %zu given", need,
                     workspace_bytes);
  const size_t r = ((size_t)rows * 4 + 255) / 256 * 256;
  float* m = static_cast<float*>(workspace);
  float* s = reinterpret_cast<float*>(static_cast<char*>(workspace) + r);
  float* e = reinterpret_cast<float*>(static_cast<char*>(workspace) + 2 * r);
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((rows + kRowsPerBlock - 1) / kRowsPerBlock), block(256);
  if (dtype == NKL_F32) {
    softmax_pass1_kernel<float><<<grid, block, 0, st>>>(static_cast<const float*>(x), m, rows, cols, ldx);
    softmax_pass2_kernel<float><<<grid, block, 0, st>>>(static_cast<const float*>(x), m, e, s, rows, cols, ldx);
    softmax_pass3_kernel<float><<<grid, block, 0, st>>>(e, s, static_cast<float*>(y), rows, cols, ldy);
  } else if (dtype == NKL_BF16) {
    softmax_pass1_kernel<bf16><<<grid, block, 0, st>>>(static_cast<const bf16*>(x), m, rows, cols, ldx);
    softmax_pass2_kernel<bf16><<<grid, block, 0, st>>>(static_cast<const bf16*>(x), m, e, s, rows, cols, ldx);
    softmax_pass3_kernel<bf16><<<grid, block, 0, st>>>(e, s, static_cast<bf16*>(y), rows, cols, ldy);
  } else {
    return set_error(NKL_EDTYPE, "nkl_softmax_unfused: unsupported dtype %d", dtype);
  }
  return check_launch("nkl_softmax_unfused");
}

extern "C" int nkl_rmsnorm_ex(const void* x, const void* w, void* y, int rows, int cols, long ldx, long ldy,
                              float eps, int dtype_in, int dtype_w, int dtype_out, void* stream) {
  int rc = check_rows("nkl_rmsnorm", rows, cols, ldx, ldy);
  if (rc) return rc;
  if (rows == 0 || cols == 0) return NKL_OK;
  if (dtype_w != NKL_F32 && dtype_w != NKL_BF16)
    return set_error(NKL_EDTYPE, "nkl_rmsnorm: unsupported weight dtype %d", dtype_w);
  hipStream_t st = (hipStream_t)stream;
  const bool wf = dtype_w == NKL_F32;
  if (dtype_in == NKL_F32 && dtype_out == NKL_F32)
    return wf ? rmsnorm_launch<float, float, float>(x, w, y, rows, cols, ldx, ldy, eps, st)
              : rmsnorm_launch<float, bf16, float>(x, w, y, rows, cols, ldx, ldy, eps, st);
  if (dtype_in == NKL_BF16 && dtype_out == NKL_BF16)
    return wf ? rmsnorm_launch<bf16, float, bf16>(x, w, y, rows, cols, ldx, ldy, eps, st)
              : rmsnorm_launch<bf16, bf16, bf16>(x, w, y, rows, cols, ldx, ldy, eps, st);
  if (dtype_in == NKL_F32 && dtype_out == NKL_BF16)
    return wf ? rmsnorm_launch<float, float, bf16>(x, w, y, rows, cols, ldx, ldy, eps, st)
              : rmsnorm_launch<float, bf16, bf16>(x, w, y, rows, cols, ldx, ldy, eps, st);
  if (dtype_in == NKL_F32 && dtype_out == NKL_F16)
    return wf ? rmsnorm_launch<float, float, f16>(x, w, y, rows, cols, ldx, ldy, eps, st)
              : rmsnorm_launch<float, bf16, f16>(x, w, y, rows, cols, ldx, ldy, eps, st);
  return set_error(NKL_EDTYPE, "nkl_rmsnorm: unsupported dtype pair (%d -> %d)", dtype_in, dtype_out);
}

extern "C" int nkl_rmsnorm(const void* x, const void* w, void* y, int rows, int cols, long ldx, long ldy,
                           float eps, int dtype_in, int dtype_out, void* stream) {
  return nkl_rmsnorm_ex(x, w, y, rows, cols, ldx, ldy, eps, dtype_in, dtype_in, dtype_out, stream);
}

extern "C" int nkl_swiglu(const void* g, const void* u, void* y, long n, int dtype, void* stream) {
  if (n < 0) return set_error(NKL_EINVAL, "nkl_swiglu: negative length %ld", n);
  if (n == 0) return NKL_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NKL_F32) return swiglu_launch<float>(g, u, y, n, st);
  if (dtype == NKL_BF16) return swiglu_launch<bf16>(g, u, y, n, st);
  if (dtype == NKL_F16) return swiglu_launch<f16>(g, u, y, n, st);
  return set_error(NKL_EDTYPE, "nkl_swiglu: unsupported dtype %d", dtype);
}

extern "C" int nkl_stream_copy(const void* x, void* y, long nbytes, void* stream) {
  if (nbytes < 0 || nbytes % 16 != 0)
    return set_error(NKL_EINVAL, "nkl_stream_copy: %ld bytes is not a non-negative multiple of 16", nbytes);
  if (nbytes == 0) return NKL_OK;
  if (!x || !y || ((uintptr_t)x & 15u) || ((uintptr_t)y & 15u))
    return set_error(NKL_EINVAL, "nkl_stream_copy: null or non-16-byte-aligned pointer");
  const long n = nbytes / 16;
  const long grid = (n + kCopyUnroll * 256 - 1) / (kCopyUnroll * 256);
  if (grid > 0x7fffffffL) return set_error(NKL_EINVAL, "nkl_stream_copy: %ld bytes is too large", nbytes);
  stream_copy_kernel<<<dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream>>>(static_cast<const u32x4*>(x),
                                                                                   static_cast<u32x4*>(y), n);
  return check_launch("nkl_stream_copy");
}

extern "C" int nkl_split_bf16(const void* x, void* y, int rows, int cols, long ldx, long ldy, void* stream) {
  if (rows < 0 || cols < 0) return set_error(NKL_EINVAL, "nkl_split_bf16: negative shape (%d, %d)", rows, cols);
  if (rows == 0 || cols == 0) return NKL_OK;
  if (cols % 4 || ldx % 4 || ldy % 4 || ldx < cols || ldy < 2L * cols || ((uintptr_t)x & 15u) || ((uintptr_t)y & 7u))
    return set_error(NKL_EINVAL,
                     "nkl_split_bf16: cols %d and leading dimensions (%ld, %ld) must be multiples of 4 with "
                     "ldx >= cols, ldy >= 2 cols; x 16-byte and y 8-byte aligned", cols, ldx, ldy);
  const long n = (long)rows * (cols / 4);
  split_bf16_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(
      static_cast<const float*>(x), static_cast<bf16*>(y), rows, cols, ldx, ldy);
  return check_launch("nkl_split_bf16");
}
