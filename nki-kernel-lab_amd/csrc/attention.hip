// Causal attention on gfx950.
//
// Argument checks, workspaces and C entries of the flash kernels (flash_*.hip;
// fp32: flash_f32.hip).
//
// attention_naive -- the reference's unfused variant: scores and
// probabilities are materialised in a caller-provided workspace, using the
// GEMM kernels for Q.K^T and P.V and a masked row softmax in between.
#include <math.h>

#include "attention.h"

namespace nkl {


// ------------------------------------------------ naive (unfused) path --
// nkilab/kernels/attention.py:35-89, pass 2: scores (already Q.K^T) are
// scaled and causally masked, then a row softmax writes P in the input dtype.
template <typename T>
__global__ __launch_bounds__(256) void masked_softmax_kernel(float* __restrict__ sc, T* __restrict__ pr, int H,
                                                             int S, float scale) {
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);  // (h, q) flattened
  if (row >= (long)H * S) return;
  const int q = (int)(row % S);
  float* srow = sc + row * S;
  T* prow = pr + row * S;
  float mx = -INFINITY;
  for (int c = lane; c < S; c += kWave) {
    const float s = c > q ? -INFINITY : srow[c] * scale;
    srow[c] = s;
    mx = fmaxf(mx, s);
  }
  mx = wave_max(mx);
  float sum = 0.f;
  for (int c = lane; c < S; c += kWave) sum += fast_exp2((srow[c] - mx) * kLog2e);
  sum = wave_sum(sum);
  const float rinv = 1.0f / sum;
  for (int c = lane; c < S; c += kWave) prow[c] = from_f32<T>(fast_exp2((srow[c] - mx) * kLog2e) * rinv);
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace nkl

using namespace nkl;

constexpr long kMaxRowStride = 1L << 21;

static int check_attn(const char* fn, const void* q, const void* k, const void* v, const void* o, int H, int S,
                      int d, int dtype, const long* strides) {
  if (H < 0 || S < 0) return set_error(NKL_EINVAL, "%s: negative shape H=%d S=%d", fn, H, S);
  if (d < 1 || d > 128) return set_error(NKL_EINVAL, "%s: head dim d=%d outside [1, 128]", fn, d);
  if (dtype != NKL_F32 && dtype != NKL_BF16 && dtype != NKL_F16)
    return set_error(NKL_EDTYPE, "%s: unsupported dtype %d", fn, dtype);
  const int E = dtype == NKL_F32 ? 4 : 8;
  if (d % E != 0)
    return set_error(NKL_EINVAL, "%s: d=%d must be a multiple of %d (pad the head dim on the host)", fn, d, E);
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o))
    return set_error(NKL_EINVAL, "%s: q/k/v/o must be 16-byte aligned", fn);
  if (H > 0 && S > 0 && (!q || !k || !v || !o)) return set_error(NKL_EINVAL, "%s: null q/k/v/o", fn);
  // Head strides (even entries) up to 2^24 elements; row strides (odd) up to
  // 2^21, so that the kernels' 32-bit byte offsets within a block of up to 256
  // rows stay below 2^30 -- the offset at which a copy of a chunk past d reads
  // zeros from outside every buffer.
  for (int i = 0; i < 8; ++i) {
    const long lim = i % 2 ? kMaxRowStride : 1L << 24;
    if (strides[i] % E != 0)
      return set_error(NKL_EINVAL, "%s: stride %ld is not a multiple of %d elements", fn, strides[i], E);
    if (strides[i] < 0 || strides[i] > lim)
      return set_error(NKL_EINVAL, "%s: %s stride %ld outside [0, %ld]", fn, i % 2 ? "row" : "head", strides[i], lim);
  }
  return NKL_OK;
}

static int flash_entry(const char* fn, const void* q, const void* k, const void* v, void* o, void* workspace,
                       size_t workspace_bytes, int* counters, size_t counter_bytes, bool ws_entry, int H, int Hkv,
                       int S, int d, const long* st8, float scale, int dtype, void* stream) {
  int rc = check_attn(fn, q, k, v, o, H, S, d, dtype, st8);
  if (rc) return rc;
  if (Hkv < 1 || H % Hkv != 0)
    return set_error(NKL_EINVAL, "%s: H=%d query heads do not divide into Hkv=%d K/V heads", fn, H, Hkv);
  if (H == 0 || S == 0) return NKL_OK;
  AttnArgs a{q, k, v, o, H, S, d, st8[0], st8[1], st8[2], st8[3], st8[4], st8[5], st8[6], st8[7], scale * kLog2e,
             H / Hkv, dtype == NKL_F16 ? 1 : 0};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NKL_BF16 || dtype == NKL_F16) {
    if (!ws_entry) return flash_bf16_launch(a, nullptr, 0, nullptr, 0, st);
    // Shapes that need no scratch (size 0) accept a null workspace.
    if (!workspace && flash_bf16_workspace_bytes(H, S, d, dtype == NKL_F16) > 0)
      return set_error(NKL_EWORKSPACE, "%s: null workspace", fn);
    return flash_bf16_launch(a, workspace, workspace_bytes, counters, counter_bytes, st);
  }
  return flash_f32_launch(a, st);
}

extern "C" int nkl_flash_attn_causal(const void* q, const void* k, const void* v, void* o, int H, int S, int d,
                                     long q_sh, long q_ss, long k_sh, long k_ss, long v_sh, long v_ss, long o_sh,
                                     long o_ss, float scale, int dtype, void* stream) {
  const long strides[8] = {q_sh, q_ss, k_sh, k_ss, v_sh, v_ss, o_sh, o_ss};
  return flash_entry("nkl_flash_attn_causal", q, k, v, o, nullptr, 0, nullptr, 0, false, H, H > 0 ? H : 1, S, d,
                     strides, scale, dtype, stream);
}

extern "C" size_t nkl_flash_attn_causal_workspace_bytes(int H, int S, int d, int dtype) {
  if (dtype != NKL_BF16 && dtype != NKL_F16) return 0;
  return flash_bf16_workspace_bytes(H, S, d, dtype == NKL_F16);
}

extern "C" size_t nkl_flash_attn_causal_counter_bytes(int H, int S, int dtype) {
  if (dtype != NKL_BF16 && dtype != NKL_F16) return 0;
  return flash_bf16_counter_bytes(H, S);
}

extern "C" int nkl_flash_attn_causal_ws(const void* q, const void* k, const void* v, void* o, void* workspace,
                                        size_t workspace_bytes, int* counters, size_t counter_bytes, int H, int S,
                                        int d, long q_sh, long q_ss, long k_sh, long k_ss, long v_sh, long v_ss,
                                        long o_sh, long o_ss, float scale, int dtype, void* stream) {
  const long strides[8] = {q_sh, q_ss, k_sh, k_ss, v_sh, v_ss, o_sh, o_ss};
  return flash_entry("nkl_flash_attn_causal_ws", q, k, v, o, workspace, workspace_bytes, counters, counter_bytes,
                     true, H, H > 0 ? H : 1, S, d, strides, scale, dtype, stream);
}

extern "C" int nkl_flash_attn_causal_gqa(const void* q, const void* k, const void* v, void* o, void* workspace,
                                         size_t workspace_bytes, int* counters, size_t counter_bytes, int H, int Hkv,
                                         int S, int d, long q_sh, long q_ss, long k_sh, long k_ss, long v_sh,
                                         long v_ss, long o_sh, long o_ss, float scale, int dtype, void* stream) {
  const long strides[8] = {q_sh, q_ss, k_sh, k_ss, v_sh, v_ss, o_sh, o_ss};
  return flash_entry("nkl_flash_attn_causal_gqa", q, k, v, o, workspace, workspace_bytes, counters, counter_bytes,
                     true, H, Hkv, S, d, strides, scale, dtype, stream);
}

// Scratch of the allocation-free entry point: kNoAllocPartBytes of partial
// states, then kNoAllocCounterBytes of arrival counters.  Each GPU the library
// runs on holds its own copy from the first call until the process ends.  In
// host code the array's name is not a device address: kernels and fills get
// the per-device address hipGetSymbolAddress returns.
constexpr size_t kNoAllocPartBytes = (size_t)64 << 20;
constexpr size_t kNoAllocCounterBytes = (size_t)1 << 20;
constexpr int kNoAllocMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocPartBytes + kNoAllocCounterBytes];
static void* scratch_addr[kNoAllocMaxDevices];

static __global__ void zero_words_kernel(int* p, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0;
}

// The current device's copy of `scratch`, looked up once per device.  Two
// threads racing on a device's first call both store the same address.
static int scratch_of_current_device(const char* fn, unsigned char** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kNoAllocMaxDevices)
    return set_error(NKL_ELAUNCH, "%s: no usable current device (%d)", fn, dev);
  void* p = __atomic_load_n(&scratch_addr[dev], __ATOMIC_ACQUIRE);
  if (!p) {
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(NKL_ELAUNCH, "%s: hipGetSymbolAddress(scratch) failed on device %d: %s", fn, dev,
                       hipGetErrorString(e));
    __atomic_store_n(&scratch_addr[dev], p, __ATOMIC_RELEASE);
  }
  *out = static_cast<unsigned char*>(p);
  return NKL_OK;
}

extern "C" int nkl_flash_attn_causal_noalloc(const void* q, const void* k, const void* v, void* o, int H, int Hkv,
                                             int S, int d, long q_sh, long q_ss, long k_sh, long k_ss, long v_sh,
                                             long v_ss, long o_sh, long o_ss, float scale, int dtype, void* stream) {
  const char* fn = "nkl_flash_attn_causal_noalloc";
  const long strides[8] = {q_sh, q_ss, k_sh, k_ss, v_sh, v_ss, o_sh, o_ss};
  int rc = check_attn(fn, q, k, v, o, H, S, d, dtype, strides);
  if (rc) return rc;
  if ((dtype != NKL_BF16 && dtype != NKL_F16) || H == 0 || S == 0)  // no scratch on these paths
    return flash_entry(fn, q, k, v, o, nullptr, 0, nullptr, 0, true, H, Hkv, S, d, strides, scale, dtype, stream);
  const size_t need = flash_bf16_workspace_bytes(H, S, d, dtype == NKL_F16);
  // One counter per 64-query block (the smallest block) covers every schedule.
  const size_t need_c = need ? (size_t)H * ((S + 63) / 64) * 4 : 0;
  if (need > kNoAllocPartBytes || need_c > kNoAllocCounterBytes)
    return set_error(NKL_EWORKSPACE,
                     "%s: H=%d S=%d d=%d needs %zu bytes of partial states and %zu of counters; the static scratch "
                     "holds %zu and %zu (use nkl_flash_attn_causal_gqa with a workspace)",
                     fn, H, S, d, need, need_c, kNoAllocPartBytes, kNoAllocCounterBytes);
  unsigned char* base = nullptr;
  if ((rc = scratch_of_current_device(fn, &base))) return rc;
  int* counters = reinterpret_cast<int*>(base + kNoAllocPartBytes);
  if (need_c > 0) {
    // The kernels leave the counters zero; clear them anyway, with a kernel
    // (not a memset node) so that the call can be captured in a graph.
    const long n = (long)(need_c / 4);
    zero_words_kernel<<<dim3((unsigned)((n + 255) / 256 < 64 ? (n + 255) / 256 : 64)), dim3(256), 0,
                        (hipStream_t)stream>>>(counters, n);
    if ((rc = check_launch(fn))) return rc;
  }
  return flash_entry(fn, q, k, v, o, need ? base : nullptr, need, counters, need_c, true, H, Hkv, S, d, strides,
                     scale, dtype, stream);
}

extern "C" int nkl_flash_attn_configure(int kernel, int schedule, int qb, int cpb) {
  return flash_bf16_configure(kernel, schedule, qb, cpb);
}

extern "C" int nkl_flash_attn_configure_polls(int polls) { return flash_bf16_configure_polls(polls); }

extern "C" int nkl_flash_attn_plan_check(int H, int S, int d, int dtype, long* info) {
  if (dtype != NKL_BF16 && dtype != NKL_F16)
    return set_error(NKL_EDTYPE, "nkl_flash_attn_plan_check: the 16-bit kernels only (dtype %d)", dtype);
  return flash_bf16_plan_check(H, S, d, dtype == NKL_F16, info);
}

extern "C" size_t nkl_attention_naive_workspace_bytes(int H, int S, int dtype) {
  if (H <= 0 || S <= 0) return 0;
  const size_t n = (size_t)H * S * S;
  const size_t sc = (n * 4 + 255) / 256 * 256;
  return sc + n * (dtype == NKL_F32 ? 4 : 2);
}

static int naive_entry(const char* fn, const void* q, const void* k, const void* v, void* o, void* workspace,
                       size_t workspace_bytes, int H, int Hkv, int S, int d, const long* st8, float scale, int dtype,
                       void* stream) {
  int rc = check_attn(fn, q, k, v, o, H, S, d, dtype, st8);
  if (rc) return rc;
  if (Hkv < 1 || H % Hkv != 0)
    return set_error(NKL_EINVAL, "%s: H=%d query heads do not divide into Hkv=%d K/V heads", fn, H, Hkv);
  if (H == 0 || S == 0) return NKL_OK;
  const size_t need = nkl_attention_naive_workspace_bytes(H, S, dtype);
  if (!workspace || workspace_bytes < need)
    return set_error(NKL_EWORKSPACE, "%s: workspace of %zu bytes needed, %zu given", fn, need, workspace_bytes);
  const long q_sh = st8[0], q_ss = st8[1], k_sh = st8[2], k_ss = st8[3], v_sh = st8[4], v_ss = st8[5],
             o_sh = st8[6], o_ss = st8[7];
  const size_t n = (size_t)H * S * S;
  float* sc = static_cast<float*>(workspace);
  char* pr = static_cast<char*>(workspace) + (n * 4 + 255) / 256 * 256;
  const size_t esz = dtype == NKL_F32 ? 4 : 2;
  hipStream_t st = (hipStream_t)stream;
  const long SS = (long)S * S;
  const int G = H / Hkv;
  // Query head h = kvh * G + g uses K/V head kvh.  For each g, the heads
  // g, G + g, ... form one batched GEMM over the K/V heads (batch strides
  // G times the query / score / output strides).
  // pass 1: scores[h] = Q[h] . K[h / G]^T (fp32)
  for (int g = 0; g < G; ++g) {
    rc = nkl_gemm(static_cast<const char*>(q) + g * q_sh * esz, k, sc + g * SS, nullptr, S, S, d, q_ss, k_ss, S, 0, 1,
                  Hkv, G * q_sh, k_sh, G * SS, 0, dtype, NKL_F32, NKL_GEMM_BLOCKED, stream);
    if (rc) return rc;
  }
  // pass 2: scale, mask, row softmax -> P
  const dim3 grid((unsigned)(((long)H * S + 3) / 4)), block(256);
  if (dtype == NKL_BF16)
    masked_softmax_kernel<bf16><<<grid, block, 0, st>>>(sc, reinterpret_cast<bf16*>(pr), H, S, scale);
  else if (dtype == NKL_F16)
    masked_softmax_kernel<f16><<<grid, block, 0, st>>>(sc, reinterpret_cast<f16*>(pr), H, S, scale);
  else
    masked_softmax_kernel<float><<<grid, block, 0, st>>>(sc, reinterpret_cast<float*>(pr), H, S, scale);
  rc = check_launch(fn);
  if (rc) return rc;
  // pass 3: O[h] = P[h] . V[h / G]
  for (int g = 0; g < G; ++g) {
    rc = nkl_gemm(pr + g * SS * esz, v, static_cast<char*>(o) + g * o_sh * esz, nullptr, S, d, S, S, v_ss, o_ss, 0,
                  0, Hkv, G * SS, v_sh, G * o_sh, 0, dtype, dtype, NKL_GEMM_BLOCKED, stream);
    if (rc) return rc;
  }
  return NKL_OK;
}

extern "C" int nkl_attention_naive(const void* q, const void* k, const void* v, void* o, void* workspace,
                                   size_t workspace_bytes, int H, int S, int d, long q_sh, long q_ss, long k_sh,
                                   long k_ss, long v_sh, long v_ss, long o_sh, long o_ss, float scale, int dtype,
                                   void* stream) {
  const long strides[8] = {q_sh, q_ss, k_sh, k_ss, v_sh, v_ss, o_sh, o_ss};
  return naive_entry("nkl_attention_naive", q, k, v, o, workspace, workspace_bytes, H, H > 0 ? H : 1, S, d, strides,
                     scale, dtype, stream);
}

extern "C" int nkl_attention_naive_gqa(const void* q, const void* k, const void* v, void* o, void* workspace,
                                       size_t workspace_bytes, int H, int Hkv, int S, int d, long q_sh, long q_ss,
                                       long k_sh, long k_ss, long v_sh, long v_ss, long o_sh, long o_ss, float scale,
                                       int dtype, void* stream) {
  const long strides[8] = {q_sh, q_ss, k_sh, k_ss, v_sh, v_ss, o_sh, o_ss};
  return naive_entry("nkl_attention_naive_gqa", q, k, v, o, workspace, workspace_bytes, H, Hkv, S, d, strides, scale,
                     dtype, stream);
}
