// Causal flash attention in fp32: 16x16x4 fp32 MFMA, every sum, score and
// probability in 32 bits.
//
// One 512-thread workgroup per 64-query block (32-query on small grids) of a
// head, heaviest blocks first: the dispatcher hands the light ones to the CUs
// that end early.  Its eight wavefronts are 2 query groups x 4 key groups:
// wavefront (qg, kg) owns queries 32 qg .. + 31 (16 qg .. + 15) and keys 16 kg .. + 15 of every step of 64 keys, with a
// running state (max, sum, O) of its own; the four key groups of a query group
// are merged through LDS at the end.  Each SIMD so holds two wavefronts, one's
// softmax beside the other's MFMAs, on a grid of twice the 128-query blocks.
//
// K and V rows are copied global -> LDS by the buffer unit, one step ahead,
// into two stages.  Everything is computed transposed, so that a lane works on
// two queries (halves h of its group) and nothing is shuffled between the
// products:
//     S^T = K . Q^T    a K fragment is one b128 read, 4 elements of d for four
//                      MFMAs (lane group g supplies d = 16 ks + 4 g + j to MFMA
//                      j) and both halves; Q^T is held in registers.
//     O^T = V^T . P^T  MFMA i takes key 4 g + i from lane group g, which is
//                      where S^T left its probability; a V fragment is one b128
//                      read of a key's row, d = 4 r .. 4 r + 3 of lane r for
//                      four 16-row blocks of O^T (row r of block b is d = 4 r +
//                      b), so that a lane ends up with contiguous runs of O.
// K rows are swizzled by 16-byte chunks (chunk c of row r at c ^ swz(r)), which
// keeps the 16-row reads free of bank conflicts; V reads are whole rows.
//
// (A second kernel further down takes many short heads.)
//
// Bound by the fp32 MFMAs (256 flop per clock and CU; a step is 8192 cycles of
// them per SIMD, 3.5 of its 4.5 us): 16 x 2048 x 128 281 -> 171 us (101 TFLOP/s),
// 8/2 x 4096 x 128 551 -> 320, 4 x 300 x 64 24.5 -> 10.9, against 64-query
// workgroups of four 16-query wavefronts that read one 4-byte operand per MFMA.
// Of the rest, the copies take 0.3 us a step and the softmax, which the second
// wavefront hides only in part, 0.3.
#include <math.h>

#include "attention.h"

namespace nkl {

namespace {

constexpr int kKB = 64;                     // keys of a step
constexpr unsigned kPastEnd = 0x80000000u;  // a buffer offset past every range: the lane reads zeros

template <int D>
__device__ __forceinline__ int k_swz(int row) {
  return D == 32 ? (row >> 1) & 7 : row & 15;
}

__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace

// NHF: 16-query halves of a query group (2: 64-query blocks, 1: 32-query ones).
template <int D, int NHF>
__global__ __launch_bounds__(512) void flash_f32_kernel(AttnArgs p) {
  constexpr int kQB = 32 * NHF;
  constexpr int ROWB = D * 4, TILEB = kKB * ROWB, STAGEB = 2 * TILEB;  // K then V
  constexpr int CPT = TILEB / 1024 / 8;                                // copies per wavefront and tile
  constexpr int NKS = D / 16;                                          // K fragments (and 16-row blocks of O^T)
  constexpr int NB = D >= 64 ? 4 : 2, NH = NKS / NB;                   // blocks per V read, V reads per key
  __shared__ __align__(16) unsigned char lds[2 * STAGEB];
  __shared__ float ml[8][NHF][16][2];  // (max, sum) per wavefront, half and query

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qg = w & 1, kg = w >> 1;
  const int g = lane >> 4, r = lane & 15;
  const int S = p.S;

  const int nqb = (S + kQB - 1) / kQB;
  const int h = blockIdx.x % p.H;
  const int q0 = (nqb - 1 - blockIdx.x / p.H) * kQB;
  const int qw = q0 + 16 * NHF * qg;  // first query of this wavefront
  const float* Q = static_cast<const float*>(p.q) + (long)h * p.q_sh;
  const float* K = static_cast<const float*>(p.k) + (long)(h / p.group) * p.k_sh;  // shared K/V head (GQA)
  const float* V = static_cast<const float*>(p.v) + (long)(h / p.group) * p.v_sh;
  float* O = static_cast<float*>(p.o) + (long)h * p.o_sh;

  // Copy u of this wavefront, 1024 bytes of a tile, lane l's 16 bytes at 16 l:
  // u < CPT of a K tile, then of a V tile.
  unsigned off[2 * CPT];
  int crow[CPT];
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int b = (w * CPT + u) * 1024 + lane * 16;
    const int row = b / ROWB, pc = b % ROWB / 16, kc = pc ^ k_swz<D>(row);
    crow[u] = row;
    off[u] = 4 * kc < p.d ? (unsigned)(4 * ((long)row * p.k_ss + 4 * kc)) : kPastEnd;
    off[CPT + u] = 4 * pc < p.d ? (unsigned)(4 * ((long)row * p.v_ss + 4 * pc)) : kPastEnd;
  }
  // K tiles at lds, V tiles after both of them.
  auto copy1 = [&](bool isv, int src, int s, int u) __attribute__((always_inline)) {
    const int k0 = src * kKB, rows = min(kKB, S - k0);
    const long ss = isv ? p.v_ss : p.k_ss;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((isv ? V : K) + (long)k0 * ss), (short)0, (int)(4 * ((rows - 1) * ss + p.d)), 0x00020000);
    const unsigned dst = opaque_lds_addr(lds) + (isv ? 2 * TILEB : 0) + (s & 1) * TILEB + (w * CPT + u) * 1024;
    const unsigned o = crow[u] < rows ? off[isv ? CPT + u : u] : kPastEnd;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, lds_ptr(dst), 16, (int)o, 0, 0, 0);
  };
  auto copy = [&](bool isv, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) copy1(isv, s, s, u);
  };
  // Every wavefront's LDS reads are done (its copies still in flight).
  auto lds_done_barrier = [&]() __attribute__((always_inline)) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
  // Every wavefront's copies have landed and its LDS accesses are done.
  auto step_barrier = [&]() __attribute__((always_inline)) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };

  const int ns = (min(q0 + kQB, S) - 1) / kKB + 1;  // steps up to the diagonal
  copy(false, 0);
  copy(true, 0);
  if (ns > 1) copy(false, 1);
  // Q^T: lane (r, g) holds Q[qw + 16 hf + r][16 ks + 4 g + j].
  floatx4 qf[NHF][NKS];
#pragma unroll
  for (int hf = 0; hf < NHF; ++hf) {
    const int q = qw + 16 * hf + r;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int d = 16 * ks + 4 * g;
      qf[hf][ks] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (q < S && d < p.d) qf[hf][ks] = *reinterpret_cast<const floatx4*>(Q + (long)q * p.q_ss + d);
    }
  }

  float m[NHF], l[NHF];  // l: this lane's share
  floatx4 o[NHF][NKS];
#pragma unroll
  for (int hf = 0; hf < NHF; ++hf) {
    m[hf] = -INFINITY, l[hf] = 0.f;
#pragma unroll
    for (int b = 0; b < NKS; ++b) o[hf][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  const int krow = 16 * kg + r;  // this lane's K row of a step
  const int swz = k_swz<D>(krow);
  // Whether any key of this wavefront's step s is at or before its last query.
  auto active = [&](int s) __attribute__((always_inline)) { return s < ns && s * kKB + 16 * kg < qw + 16 * NHF; };
  // Scores of step s: sc[hf][i] for key s kKB + 16 kg + 4 g + i, query qw + 16 hf + r.
  auto qk = [&](int s, int ks, floatx4 (&sc)[NHF]) __attribute__((always_inline)) {
    const floatx4 a =
        *reinterpret_cast<const floatx4*>(lds + (s & 1) * TILEB + krow * ROWB + (((4 * ks + g) ^ swz) << 4));
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int hf = 0; hf < NHF; ++hf)
        sc[hf] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], qf[hf][ks][j], sc[hf], 0, 0, 0);
  };
  float mx[NHF];
  // Element i of both halves: scale, causal mask, running maximum of the step.
  auto mask_max = [&](int s, int i, floatx4 (&sc)[NHF]) __attribute__((always_inline)) {
    const int key = s * kKB + 16 * kg + 4 * g + i;
#pragma unroll
    for (int hf = 0; hf < NHF; ++hf) {
      const float x = key > qw + 16 * hf + r ? -INFINITY : sc[hf][i] * p.c;
      sc[hf][i] = x;
      mx[hf] = i == 0 ? x : fmaxf(mx[hf], x);
    }
  };
  float mu[NHF];  // the maximum the step's exponents are taken against
  // The step's maxima over the wavefront's keys; O and the sum follow when one grew.
  auto raise_max = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int hf = 0; hf < NHF; ++hf) {
      const float mn = fmaxf(m[hf], max_xor32(max_xor16(mx[hf])));
      if (__any(mn > m[hf])) {
        // (no key yet: m is -inf, l and O are 0)
        const float corr = m[hf] == -INFINITY ? 0.f : fast_exp2(m[hf] - mn);
        l[hf] *= corr;
#pragma unroll
        for (int b = 0; b < NKS; ++b) o[hf][b] *= corr;
        m[hf] = mn;
      }
      mu[hf] = mn == -INFINITY ? 0.f : mn;  // every key masked so far: p = 0
    }
  };

  // Pipeline over steps: the exponentials of step s beside the QK^T MFMAs of
  // step s + 1, then mask and maximum of step s + 1 beside the PV MFMAs of
  // step s.  K tile s + 2 and V tile s + 1 are copied meanwhile, into the
  // tiles read last in step s - 1.
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 sc[NHF];
#pragma unroll
  for (int hf = 0; hf < NHF; ++hf) sc[hf] = zero;
  step_barrier();
  if (active(0)) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qk(0, ks, sc);
#pragma unroll
    for (int i = 0; i < 4; ++i) mask_max(0, i, sc);
    raise_max();
  }
  lds_done_barrier();
#pragma unroll 1
  for (int s = 0; s < ns; ++s) {
    const bool next = active(s + 1);
    floatx4 nx[NHF];
#pragma unroll
    for (int hf = 0; hf < NHF; ++hf) nx[hf] = zero;
    if (active(s)) {
      auto exps = [&](int x0, int x1) __attribute__((always_inline)) {
#pragma unroll
        for (int x = x0; x < x1; ++x) {
          const int hf = x % NHF, i = x / NHF;
          sc[hf][i] = fast_exp2(sc[hf][i] - mu[hf]);
          l[hf] += sc[hf][i];
        }
      };
      // Copies of the next tiles, CPT of V tile s + 1 and of K tile s + 2 (the
      // last one again when there is none): spread over the MFMAs, as each
      // holds the wavefront's issue for a while.
      const int k2 = min(s + 2, ns - 1);
      if (next) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          qk(s + 1, ks, nx);
          exps(4 * NHF * ks / NKS, 4 * NHF * (ks + 1) / NKS);
#pragma unroll
          for (int u = 2 * CPT * ks / NKS; u < 2 * CPT * (ks + 1) / NKS; ++u)
            u < CPT ? copy1(true, s + 1, s + 1, u) : copy1(false, k2, s + 2, u - CPT);
        }
      } else {
        exps(0, 4 * NHF);
        if (s + 1 < ns) copy(true, s + 1);  // (that step is the last one)
      }
      typedef float vfrag __attribute__((ext_vector_type(NB)));
      vfrag va[2][NH];
      auto vread = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NH; ++n)
          va[i & 1][n] = *reinterpret_cast<const vfrag*>(lds + 2 * TILEB + (s & 1) * TILEB +
                                                         (16 * kg + 4 * g + i) * ROWB + 64 * NB * n + 4 * NB * r);
      };
      vread(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < 3) vread(i + 1);
        __builtin_amdgcn_sched_barrier(0);  // a key's fragments are read one key ahead
#pragma unroll
        for (int n = 0; n < NH; ++n)
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int hf = 0; hf < NHF; ++hf)
              o[hf][n * NB + b] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(va[i & 1][n][b], sc[hf][i], o[hf][n * NB + b], 0, 0, 0);
        mask_max(s + 1, i, nx);
      }
      if (next) raise_max();
#pragma unroll
      for (int hf = 0; hf < NHF; ++hf) sc[hf] = nx[hf];
    }
    step_barrier();
  }

  // Merge the four key groups: states through LDS, then wavefront kg finishes
  // every fourth run of 4 NB values of d per lane.
  floatx4* ob = reinterpret_cast<floatx4*>(lds);
#pragma unroll
  for (int hf = 0; hf < NHF; ++hf) {
    l[hf] = sum_xor32(sum_xor16(l[hf]));
    if (g == 0) ml[w][hf][r][0] = m[hf], ml[w][hf][r][1] = l[hf];
#pragma unroll
    for (int b = 0; b < NKS; ++b) ob[(w * NHF * NKS + hf * NKS + b) * 64 + lane] = o[hf][b];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NHF * NH; ++t) {
    if (t % 4 != kg) continue;
    const int hf = t / NH, n = t % NH;
    float wt[4], M = -INFINITY, L = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) M = fmaxf(M, ml[2 * k + qg][hf][r][0]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      wt[k] = fast_exp2(ml[2 * k + qg][hf][r][0] - M);
      L = fmaf(wt[k], ml[2 * k + qg][hf][r][1], L);
    }
    const float linv = 1.0f / L;
    floatx4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        acc[b] += wt[k] * ob[((2 * k + qg) * NHF * NKS + hf * NKS + n * NB + b) * 64 + lane];
    }
    const int q = qw + 16 * hf + r;
    if (q < S) {
      float* orow = O + (long)q * p.o_ss;
#pragma unroll
      for (int e = 0; e < 4; e += 4 / NB) {
        // Row 4 g + e of the blocks: d = 16 NB n + NB (4 g + e) + b.
        const int d = 16 * NB * n + NB * (4 * g + e);
        float v[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = acc[x % NB][e + x / NB] * linv;
        if (d < p.d) store_vec<4>(orow + d, v);
      }
    }
  }
}

// The kernel for many short heads: one 256-thread workgroup per 64-query block
// of a head, heaviest blocks first, four wavefronts of 16 queries each, steps of
// 32 keys staged through registers into two padded stages (68 KB at D = 128, 35
// at 64, 18 at 32), so that two, three or five workgroups share a CU and hide
// each other's starts, waits and ends, and a ragged last step is half as long.
// S^T and O^T as in the kernel above, one 4-byte LDS read per MFMA; a block's
// state stays with its wavefronts, nothing is merged.  O is summed over every
// fourth group of 16 keys apart, as the other kernel's key groups do: one sum is
// up to 5% faster, at 128 x 2048 x 32 with 3.7e-7 from 64 bits where four, and the
// other kernel, have 2.5e-7.
template <int D>
__global__ __launch_bounds__(256, D == 128 ? 2 : D == 64 ? 3 : 5) void flash_f32_short_kernel(AttnArgs p) {
  constexpr int NC = 4;  // sums of O
  constexpr int kQB = 64, kKS = 32, CPR = D / 4, LD = D + 4, NCH = kKS * CPR / 256, ND = D / 16, NQF = D / 4;
  __shared__ float Ks[2][kKS * LD];
  __shared__ float Vs[2][kKS * LD];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int S = p.S;

  const int nqb = (S + kQB - 1) / kQB;
  const int h = blockIdx.x % p.H;
  const int q0 = (nqb - 1 - blockIdx.x / p.H) * kQB;
  const int qw = q0 + 16 * w, q = qw + r;  // this wavefront's first query, this lane's query
  const float* Q = static_cast<const float*>(p.q) + (long)h * p.q_sh;
  const float* K = static_cast<const float*>(p.k) + (long)(h / p.group) * p.k_sh;  // shared K/V head (GQA)
  const float* V = static_cast<const float*>(p.v) + (long)(h / p.group) * p.v_sh;
  float* O = static_cast<float*>(p.o) + (long)h * p.o_sh;

  // Q^T: lane (r, g) holds Q[q][4 f + g].
  float qf[NQF];
#pragma unroll
  for (int f = 0; f < NQF; ++f) qf[f] = q < S && 4 * f + g < p.d ? Q[(long)q * p.q_ss + 4 * f + g] : 0.f;

  uint4 rk[NCH], rv[NCH];
  auto gload = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = tid + 256 * i, key = k0 + c / CPR, cc = (c % CPR) * 4;
      rk[i] = ld16_or_zero(K, (long)key * p.k_ss + cc, key < S && cc < p.d);
      rv[i] = ld16_or_zero(V, (long)key * p.v_ss + cc, key < S && cc < p.d);
    }
  };
  auto lstore = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = tid + 256 * i, at = c / CPR * LD + (c % CPR) * 4;
      *reinterpret_cast<uint4*>(&Ks[buf][at]) = rk[i];
      *reinterpret_cast<uint4*>(&Vs[buf][at]) = rv[i];
    }
  };

  float m = -INFINITY, l[2] = {0.f, 0.f};  // l: this lane's share
  floatx4 o[NC][ND];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int b = 0; b < ND; ++b) o[c][b] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int ns = (min(q0 + kQB, S) - 1) / kKS + 1;  // steps up to the diagonal
  const int q_last = qw + 15;
  gload(0);
  lstore(0);
  __syncthreads();
  auto step = [&](int s, int buf) __attribute__((always_inline)) {
    const int k0 = s * kKS;
    if (s + 1 < ns) gload(k0 + kKS);
    // S^T = K . Q^T, element i of sc[kb] for key k0 + 16 kb + 4 g + i; the
    // 16-key groups past the wavefront's last query are left out.
    floatx4 sc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      sc[kb] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (k0 + 16 * kb <= q_last) {
#pragma unroll
        for (int f = 0; f < NQF; ++f)
          sc[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ks[buf][(16 * kb + r) * LD + 4 * f + g], qf[f], sc[kb], 0, 0, 0);
      }
    }
    const bool diag = k0 + kKS - 1 > qw;
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = diag && k0 + 16 * kb + 4 * g + i > q ? -INFINITY : sc[kb][i] * p.c;
        sc[kb][i] = x;
        mx = fmaxf(mx, x);
      }
    const float mn = fmaxf(m, max_xor32(max_xor16(mx)));
    // (no key yet: m is -inf, l and O are 0; every key masked so far: p = 0)
    const float mu = mn == -INFINITY ? 0.f : mn;
    if (__any(mn > m)) {
      const float corr = m == -INFINITY ? 0.f : fast_exp2(m - mn);
      l[0] *= corr, l[1] *= corr;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int b = 0; b < ND; ++b) o[c][b] *= corr;
      m = mn;
    }
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[kb][i] = fast_exp2(sc[kb][i] - mu);
        sum += sc[kb][i];
      }
    l[buf] += sum;
    // O^T += V^T . P^T
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      if (k0 + 16 * kb > q_last) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < ND; ++b)
          o[2 * buf + kb][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              Vs[buf][(16 * kb + 4 * g + i) * LD + 16 * b + r], sc[kb][i], o[2 * buf + kb][b], 0, 0, 0);
    }
    if (s + 1 < ns) lstore(buf ^ 1);
    __syncthreads();
  };
#pragma unroll 1
  for (int s = 0; s < ns; s += 2) {
    step(s, 0);
    if (s + 1 < ns) step(s + 1, 1);
  }

  const float linv = 1.0f / sum_xor32(sum_xor16(l[0] + l[1]));
  if (q < S) {
    float* orow = O + (long)q * p.o_ss;
#pragma unroll
    for (int b = 0; b < ND; ++b) {
      const int d = 16 * b + 4 * g;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = o[0][b][i];
#pragma unroll
        for (int c = 1; c < NC; ++c) v[i] += o[c][b][i];
        v[i] *= linv;
      }
      if (d < p.d) store_vec<4>(orow + d, v);
    }
  }
}

// One launch over all heads, unless their threads pass HIP's limit: then
// over ranges of heads, each of whole groups or within one group.
template <typename F>
static void launch_heads(const AttnArgs& a, int qb, int threads, F kernel, hipStream_t st) {
  const long nqb = ((long)a.S + qb - 1) / qb, fit = kMaxGridThreads / threads / nqb;
  for (long h = 0, n; h < a.H; h += n) {
    n = min(fit > 1 ? fit : 1, a.H - h);
    AttnArgs p = a;
    if (n < a.H && a.group > 1) {
      const long left = a.group - h % a.group;  // heads left of the group of head h
      if (left < a.group || n < a.group)
        n = min(n, left), p.group = (int)n;
      else
        n -= n % a.group;
    }
    p.H = (int)n;
    p.q = static_cast<const float*>(a.q) + h * a.q_sh;
    p.k = static_cast<const float*>(a.k) + h / a.group * a.k_sh;
    p.v = static_cast<const float*>(a.v) + h / a.group * a.v_sh;
    p.o = static_cast<float*>(a.o) + h * a.o_sh;
    kernel<<<dim3((unsigned)(nqb * n)), dim3(threads), 0, st>>>(p);
  }
}

// Whether the kernel for many short heads leads the 64-query one: by the heads,
// which with short sequences are the rounds of workgroups, up to the length
// where the 64-query kernel's steps win them back (heads x positions, us, short /
// 64-query).
// d <= 32: at any length from enough blocks on: 256 x 200 17.2 / 19.3, 1024 x 64
// 11.1 / 12.1, 8192 x 16 31 / 68, 96 x 900 68 / 70, 128 x 2048 343 / 377, 32 x 6000
// 714 / 766; but 256 x 128 9.7 / 8.8, 128 x 512 32 / 31, 32 x 4096 375 / 363.
// d <= 64: 512 x 100 23 / 25, 384 x 200 44 / 46, 1024 x 384 231 / 236, 4096 x 16 31 /
// 57, 640 x 64 15.6 / 17.5; but 320 x 200 level, 512 x 64 12.6 / 12.0, 1024 x 600 575
// / 570.
// d <= 128: 1024 x 16 18.5 / 34, 256 x 100 24 / 31, 144 x 200 42 / 47, 256 x 800 498 /
// 524; but 128 x 100 19.4 / 16.6, 256 x 1024 level.  With somewhat fewer heads where
// the 64-query kernel's last step would be half empty, and past 256: 128 x 200 35 /
// 41, 128 x 300 52 / 59, but 128 x 256 41.7 / 40.9.
template <int D>
static bool many_short(int H, int S) {
  const long blocks = (long)H * ((S - 1) / 64 + 1);
  if (D == 32) return blocks >= (H >= 256 ? 768 : H >= 64 ? 1400 : 2200);
  if (D == 64) return H >= 384 && S <= (H >= 512 ? 384 : 300) && (S <= 32 || S > 64 || H >= 640);
  return (H >= 144 && S <= 800) || (H >= 112 && S > 128 && S <= 384 && ((S - 1) % 64 < 32 || S > 256));
}

template <int D>
static void launch(const AttnArgs& a, hipStream_t st) {
  // 32-query blocks where 64-query ones leave half the CUs idle: half the MFMAs
  // of a step per workgroup (us, 64 / 32: 4 x 300 x 64 17.8 / 10.9, 1 x 4096 x
  // 128 290 / 161, 2 x 100 x 128 15.7 / 9.5).
  const long n64 = ((long)a.S + 63) / 64;
  if (n64 * a.H <= 128)
    launch_heads(a, 32, 512, flash_f32_kernel<D, 1>, st);
  else if (many_short<D>(a.H, a.S))
    launch_heads(a, 64, 256, flash_f32_short_kernel<D>, st);
  else
    launch_heads(a, 64, 512, flash_f32_kernel<D, 2>, st);
}

int flash_f32_launch(const AttnArgs& a, hipStream_t st) {
  if (a.d <= 32)
    launch<32>(a, st);
  else if (a.d <= 64)
    launch<64>(a, st);
  else
    launch<128>(a, st);
  return check_launch("nkl_flash_attn_causal");
}

}  // namespace nkl
