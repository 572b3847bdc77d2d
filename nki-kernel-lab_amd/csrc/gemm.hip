// GEMM: C = A . op(B) (+ R) on 32x32 MFMA tiles with fp32 accumulation.
//
// gemm_dma_kernel, the hot path: operands of 16-byte chunks (bf16, fp16 and
// fp32) staged by the buffer unit, tiles from 32x32 to 256x256.
// gemm_reg_kernel: any alignment, staged through registers; fp32 products with
// a short K too.
// gemm_pack_kernel, gemm_reduce_kernel: with a workspace (nkl_gemm_ws), large
// unaligned 16-bit products copy their operands into aligned rows for the
// first kernel, and few-tile products with a long K split it over workgroups.
//
// Naive kernel (variant "naive", and unaligned products with next to no K):
// each wavefront computes one 32x32 tile of C
// reading its operands straight from global memory at every K step -- no
// on-chip reuse, like the reference's matmul_naive.
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "common.h"

namespace nkl {

// Epilogues of the LDS-DMA kernel.
enum Epi {
  kEpiElem = 0,    // one element per lane per store (any alignment)
  kEpiStaged = 1,  // tile staged in LDS, 16 bytes per lane per store
  kEpiSwiglu = 2,  // staged; adjacent 32-column tiles are gate and up: C = silu(gate) * up, N / 2 columns
};

struct GemmArgs {
  const void* A;
  const void* B;
  void* C;
  const void* R;
  int M, N, K;
  long lda, ldb, ldc, ldr;
  long sA, sB, sC, sR;
  int epi;  // Epi (the LDS-DMA kernel; the other kernels store elements)
  int Nc;   // columns stored: N, or fewer when packed operands pad N
  int Kall; // 0, or the whole K of a product split over the batch index: entry z takes K columns from z K
  int padded;  // rows along K hold zeros up to a multiple of 16 bytes past K
  const void* B2;  // GU kernels: the up weight (B the gate weight; N their 32-row groups taken in turn)
  long ldb2;
};

// Workgroup tile index -> (tile_m, tile_n).  Consecutive workgroup ids are
// dispatched round-robin over the 8 XCDs; the remap gives each XCD a
// contiguous range of tiles, walked in groups of GROUP_M tile-rows so the
// A and B stripes a group touches stay in that XCD's L2.
__device__ __forceinline__ void tile_coords(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  int id = bid;
  if (total % 8 == 0) id = (bid % 8) * (total / 8) + bid / 8;
  constexpr int GROUP_M = 8;
  const int group_size = GROUP_M * tiles_n;
  const int group = id / group_size;
  const int first_m = group * GROUP_M;
  const int gm = min(tiles_m - first_m, GROUP_M);
  const int in_group = id - group * group_size;
  tm = first_m + in_group % gm;
  tn = in_group / gm;
}

// One wavefront per 32x32 tile of C, four per workgroup; operands are read
// from global memory at every K step with per-element bounds checks.
template <typename T, typename TO, bool BT>
__global__ __launch_bounds__(256) void gemm_naive_kernel(GemmArgs p) {
  using MF = Mfma32<T>;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int tiles_n = (p.N + 31) / 32;
  const int tile = blockIdx.x * 4 + wid;
  const int tm = tile / tiles_n, tn = tile % tiles_n;
  if (tm * 32 >= p.M) return;
  const int bz = blockIdx.z;
  const T* A = static_cast<const T*>(p.A) + (long)bz * p.sA;
  const T* B = static_cast<const T*>(p.B) + (long)bz * p.sB;
  TO* C = static_cast<TO*>(p.C) + (long)bz * p.sC;
  const TO* R = p.R ? static_cast<const TO*>(p.R) + (long)bz * p.sR : nullptr;
  const int lr = lane & 31, lg = lane >> 5;
  const int arow = tm * 32 + lr, bcol = tn * 32 + lr;
  floatx16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  for (int k0 = 0; k0 < p.K; k0 += MF::MK) {
    T av[MF::KPER], bv[MF::KPER];
#pragma unroll
    for (int j = 0; j < MF::KPER; ++j) {
      const int k = k0 + lg * MF::KPER + j;
      const bool kin = k < p.K;
      av[j] = (kin && arow < p.M) ? A[(long)arow * p.lda + k] : from_f32<T>(0.f);
      if constexpr (BT)
        bv[j] = (kin && bcol < p.N) ? B[(long)bcol * p.ldb + k] : from_f32<T>(0.f);
      else
        bv[j] = (kin && bcol < p.N) ? B[(long)k * p.ldb + bcol] : from_f32<T>(0.f);
    }
    typename MF::frag af, bfr;
    if constexpr (MF::KPER == 1) {
      af = av[0];
      bfr = bv[0];
    } else {
#pragma unroll
      for (int j = 0; j < MF::KPER; ++j) {
        af[j] = av[j];
        bfr[j] = bv[j];
      }
    }
    acc = MF::mma(af, bfr, acc);
  }
  const int col = tn * 32 + lr;
  if (col >= p.N) return;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int row = tm * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
    if (row < p.M) {
      float vv = acc[e];
      if (R) vv += to_f32(R[(long)row * p.ldr + col]);
      C[(long)row * p.ldc + col] = from_f32<TO>(vv);
    }
  }
}

// 16 bytes at the alignment of their element only.
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef u32x4_t u32x4_al2 __attribute__((aligned(2)));
typedef u32x4_t u32x4_al4 __attribute__((aligned(4)));

// ----------------------------------------------------- GEMM, LDS-DMA staged --
//
// Operand tiles are copied global -> LDS by the buffer unit
// (buffer_load ... lds, lane l's 16 bytes at the instruction's LDS base + 16 l)
// into a ring of NS stages, NS - 1 K-steps ahead of use, so that even a small
// GEMM (1024^3, 256 workgroups of 64x64) keeps enough loads in flight to cover
// the memory latency.  Every staged tile is made of 128-byte rows (64 bf16 of
// K for A and for B given as [N, K]; 64 columns of N for B given as [K, N],
// in sub-tiles of 64 columns) whose 16-byte chunks are swizzled: chunk c of
// row r sits at chunk c ^ g_swz(r).  The swizzle keeps the 16-row b128
// fragment reads (A, B^T) and the 4-row transposed b64 reads (B as [K, N],
// read with ds_read_b64_tr_b16) free of bank conflicts.  One barrier per
// K-step; WGM x WGN wavefronts of 32x32x16 MFMA tiles.
//
// fp32 runs the same pipeline over the same bytes: a 16-byte fragment is 4
// elements of K for four 32x32x2 MFMAs (lane group lg supplies k = 4 lg + j to
// MFMA j, the same order in A and B), and B as [K, N] stays row-major in LDS
// and is read 4 bytes at a time.  Its MFMAs take 64 cycles each, so the loop is
// bound by them: 2048^3 222 -> 131 us (B^T; [K, N] 133) against 111 us of MFMA
// time, 128x128 tiles in two K groups; a 64 x 64 wavefront tile without the
// copies, or without the fragment reads, takes 125 and 128.  The register-staged
// kernel takes 150 to 160 there.
//
// 2 x 2 wavefronts (256 threads, one per SIMD) for tiles up to 128 x 128;
// 2 x 4 (512 threads, two per SIMD) for 256-row tiles.  A 128 x 128 tile
// stages 32 KB per K-step for 2 MFLOP, ~64 B/clk per CU at the MFMA rate --
// all an L2 channel set delivers; a 256 x 256 tile stages half that per flop.
// With two 64 KB stages the next K-step's copies have one K-step (32 MFMAs
// per wavefront, two wavefronts per SIMD) to land.

namespace {

// K elements per stage (128-byte rows).
template <typename T>
constexpr int kBK = 128 / (int)sizeof(T);

__device__ __forceinline__ int g_swz(int r) { return (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | ((r >> 3) & 1); }
// Byte offset of 16-byte chunk c of row r in a tile of 128-byte rows.
__device__ __forceinline__ int g_pos(int r, int c) { return r * 128 + ((c ^ g_swz(r)) << 4); }

template <int n>
__device__ __forceinline__ void g_wait_vm() {
  static_assert(n >= 0 && n < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ void g_wait_lgkm0() { __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4)); }

constexpr unsigned kOOB = 0x80000000u;  // a buffer offset past every range: the lane reads zeros

}  // namespace

template <typename TI, typename TO, int BM, int BN, bool BT, int NS, int WGM = 2, int WGN = 2, int KG = 1,
          bool GU = false>
__global__ __launch_bounds__(64 * WGM * WGN * KG) void gemm_dma_kernel(GemmArgs p) {
  // GU: gate and up weights as two tensors (B, B2: [Nc, K] each); tile columns
  // 64 j .. 64 j + 31 are rows 32 j .. of B, the next 32 those of B2, so that
  // the SwiGLU epilogue finds each pair in adjacent accumulator tiles.
  // TI: the operand format (bf16, fp16 or fp32); operands move as raw 16-byte
  // chunks, the format only picks the MFMA.
  // KG > 1: KG groups of WGM x WGN wavefronts share the tile; group g takes
  // K-steps g, g + KG, ... through its own part of each stage, and the groups'
  // accumulators are added in group order at the end.  Each SIMD then runs KG
  // wavefronts whose copy and fragment-read latencies hide each other's.
  constexpr bool H = std::is_same<TI, f16>::value;
  constexpr bool F32 = std::is_same<TI, float>::value;
  static_assert(H || F32 || std::is_same<TI, bf16>::value, "operand format");
  constexpr int E = VecE<TI>::value, SZ = sizeof(TI), BK = kBK<TI>;
  constexpr int NW = WGM * WGN;
  constexpr int A_BYTES = BM * 128;
  constexpr int B_BYTES = BN * 128;  // BN rows of 128 B (B^T) or BN / 64 sub-tiles of 64 x 128 B
  constexpr int STAGE = A_BYTES + B_BYTES;
  constexpr int A_PW = A_BYTES / 1024 / NW, B_PW = B_BYTES / 1024 / NW;  // DMA instructions per wavefront
  constexpr int LPT = A_PW + B_PW;
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
  static_assert(A_PW >= 1 && B_PW >= 1 && A_PW * NW * 1024 == A_BYTES && B_PW * NW * 1024 == B_BYTES,
                "tile too small");
  static_assert(TM >= 1 && TN >= 1 && TM * 32 * WGM == BM && TN * 32 * WGN == BN, "wavefront tiles");
  static_assert((NS - 2) * LPT < 64, "vmcnt range");
  static_assert(KG >= 1, "K groups");
  constexpr int SSET = KG * STAGE;  // one stage of every group
  __shared__ __align__(16) unsigned char lds[NS * SSET];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wall = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wall / NW, wid = wall % NW;  // K group, wavefront within it
  const int wm = wid / WGN, wn = wid % WGN;
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int bz = blockIdx.z;
  const TI* A = static_cast<const TI*>(p.A) + (long)bz * p.sA;
  const TI* B = static_cast<const TI*>(p.B) + (long)bz * p.sB;
  TO* C = static_cast<TO*>(p.C) + (long)bz * p.sC;
  const TO* R = p.R ? static_cast<const TO*>(p.R) + (long)bz * p.sR : nullptr;
  const int K = p.Kall ? min(p.K, p.Kall - bz * p.K) : p.K;
  const int Kr = (K + E - 1) / E * E;  // readable (K unless the rows are padded)

  // ---- DMA: instruction q of a 128-byte-row tile covers rows 8 q .. 8 q + 7;
  // lane l fills row 8 q + l / 8, physical chunk l % 8.
  const int dr = lane >> 3, dpc = lane & 7;
  // A rows m (B^T rows n): byte offset of the lane's chunk at K-step 0, or kOOB.
  const int rows_a = min(BM, p.M - m0);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A + (long)m0 * p.lda), (short)0, (int)min((long)SZ * ((rows_a - 1) * p.lda + Kr), 0x7fffffffL), 0x00020000);
  unsigned aoff[A_PW];
  int akc[A_PW];
#pragma unroll
  for (int u = 0; u < A_PW; ++u) {
    const int row = 8 * (wid * A_PW + u) + dr;
    const int lc = dpc ^ g_swz(row);
    akc[u] = E * lc;
    aoff[u] = row < rows_a ? (unsigned)(SZ * ((long)row * p.lda + E * lc)) : kOOB;
  }
  __amdgpu_buffer_rsrc_t rb;
  __amdgpu_buffer_rsrc_t rb2;  // GU: the up weight
  unsigned boff[B_PW];
  int bkc[B_PW], brow[B_PW], bq[B_PW];  // (bq: the instruction's 1024 bytes of the tile)
  if constexpr (GU) {
    // Even copies take gate rows, odd ones up rows: the resource is a
    // compile-time choice.  Instruction q covers 8 rows of one 32-row group.
    static_assert(BT && B_PW % 2 == 0 && TN % 2 == 0, "gate/up pairs");
    const int w0 = n0 / 2, rows_b = min(BN / 2, p.Nc - w0);
    rb = __builtin_amdgcn_make_buffer_rsrc((void*)(B + (long)w0 * p.ldb), (short)0,
                                           (int)min((long)SZ * ((rows_b - 1) * p.ldb + Kr), 0x7fffffffL), 0x00020000);
    rb2 = __builtin_amdgcn_make_buffer_rsrc((void*)(static_cast<const TI*>(p.B2) + (long)w0 * p.ldb2), (short)0,
                                            (int)min((long)SZ * ((rows_b - 1) * p.ldb2 + Kr), 0x7fffffffL), 0x00020000);
#pragma unroll
    for (int u = 0; u < B_PW; ++u) {
      const int i = wid * (B_PW / 2) + u / 2;  // eighth rows of the weight this copy takes
      const int q = (i / 4) * 8 + i % 4 + 4 * (u & 1);
      const int row = 8 * q + dr, wrow = 8 * i + dr;
      const int lc = dpc ^ g_swz(row);
      bq[u] = q;
      bkc[u] = E * lc;
      brow[u] = 0;
      boff[u] = wrow < rows_b ? (unsigned)(SZ * ((long)wrow * (u & 1 ? p.ldb2 : p.ldb) + E * lc)) : kOOB;
    }
  } else if constexpr (BT) {
    const int rows_b = min(BN, p.N - n0);
    rb = __builtin_amdgcn_make_buffer_rsrc((void*)(B + (long)n0 * p.ldb), (short)0,
                                           (int)min((long)SZ * ((rows_b - 1) * p.ldb + Kr), 0x7fffffffL), 0x00020000);
#pragma unroll
    for (int u = 0; u < B_PW; ++u) {
      const int row = 8 * (wid * B_PW + u) + dr;
      const int lc = dpc ^ g_swz(row);
      bq[u] = wid * B_PW + u;
      bkc[u] = E * lc;
      brow[u] = 0;
      boff[u] = row < rows_b ? (unsigned)(SZ * ((long)row * p.ldb + E * lc)) : kOOB;
    }
  } else {
    // [K, N]: 16-bit instruction q -> sub-tile q / 8 (64 columns), k rows
    // 8 (q % 8) + dr; fp32: 1024 bytes of the row-major [BK][BN] tile.
    const int cols_b = min(BN, p.N - n0);
    rb = __builtin_amdgcn_make_buffer_rsrc((void*)(B + n0), (short)0,
                                           (int)min((long)SZ * ((long)(K - 1) * p.ldb + cols_b), 0x7fffffffL), 0x00020000);
#pragma unroll
    for (int u = 0; u < B_PW; ++u) {
      const int q = wid * B_PW + u;
      const int sub = q / 8, row = F32 ? (256 * q + 4 * lane) / BN : 8 * (q % 8) + dr;
      const int col = F32 ? (256 * q + 4 * lane) % BN : 64 * sub + 8 * (dpc ^ g_swz(row));
      bq[u] = q;
      brow[u] = row;
      bkc[u] = 0;
      boff[u] = col < cols_b ? (unsigned)(SZ * ((long)row * p.ldb + col)) : kOOB;
    }
  }
  // Copy instruction u (A for u < A_PW, then B) of K-step s into stage st
  // (K-steps past K copy zeros).
  auto dma1 = [&](int s, int st, int u) __attribute__((always_inline)) {
    const int k0 = (KG * s + kg) * BK;
    unsigned char* sb = lds + st * SSET + kg * STAGE;
    if (u < A_PW) {
      const unsigned off = (aoff[u] != kOOB && k0 + akc[u] < K) ? aoff[u] + (unsigned)SZ * k0 : kOOB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(sb + (wid * A_PW + u) * 1024),
                                               16, (int)off, 0, 0, 0);
    } else {
      const int w = u - A_PW;
      unsigned off;
      if constexpr (BT)
        off = (boff[w] != kOOB && k0 + bkc[w] < K) ? boff[w] + (unsigned)SZ * k0 : kOOB;
      else
        off = (boff[w] != kOOB && k0 + brow[w] < K) ? boff[w] + (unsigned)((long)SZ * k0 * p.ldb) : kOOB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          GU && (w & 1) ? rb2 : rb, (__attribute__((address_space(3))) void*)(sb + A_BYTES + bq[w] * 1024), 16,
          (int)off, 0, 0, 0);
    }
  };
  auto dma = [&](int s, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < LPT; ++u) dma1(s, st, u);
  };

  // ---- fragment offsets within a stage (K-step sub-step ks = 0..3)
  const int lr = lane & 31, lg = lane >> 5;
  // The swizzle depends on row bits 1..3 only, so the 32-row tiles of a
  // wavefront sit 4096 bytes apart: one offset per sub-step, plus 4096 i.
  int afo[4], bto[4], bfo[TN][4][2];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    afo[ks] = g_pos(wm * WM + lr, 2 * ks + lg);
    bto[ks] = A_BYTES + g_pos(wn * WN + lr, 2 * ks + lg);
  }
  // fp32 B as [K, N]: element e of sub-step ks is row 8 ks + 4 lg + e.
  const int bf32 = A_BYTES + 16 * lg * BN + 4 * (wn * WN + lr);
  if constexpr (!BT && !F32) {
    const int i16 = lane & 15, g2 = (lane >> 4) & 1;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        // lane i of a 16-lane group reads row k (4 per read) at columns n .. n + 3
        const int n = wn * WN + j * 32 + 16 * g2 + 4 * (i16 & 3);
        const int sub = n / 64, nc = n % 64;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int krow = 16 * ks + 8 * lg + 4 * h + (i16 >> 2);
          bfo[j][ks][h] = A_BYTES + sub * 8192 + g_pos(krow, nc / 8) + (nc % 8) * 2;
        }
      }
  }

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // Fragments of sub-step ks (32 bytes of K) of the stage at sb.
  auto frags = [&](const unsigned char* sb, int ks, bf16x8 (&af)[TM], bf16x8 (&bfr)[TN])
                   __attribute__((always_inline)) {
    // With 16-bit B as [K, N] every fragment read is untracked (see
    // ds_read_tr16_b64_async); lds_wait_tie on the B fragments orders them all.
#pragma unroll
    for (int i = 0; i < TM; ++i)
      af[i] = BT || F32 ? *reinterpret_cast<const bf16x8*>(sb + afo[ks] + 4096 * i)
                        : ds_read_b128_async(sb + afo[ks] + 4096 * i);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (BT) {
        bfr[j] = *reinterpret_cast<const bf16x8*>(sb + bto[ks] + 4096 * j);
      } else if constexpr (F32) {
        floatx4 t;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          t[e] = *reinterpret_cast<const float*>(sb + bf32 + 4 * ((8 * ks + e) * BN + 32 * j));
        bfr[j] = __builtin_bit_cast(bf16x8, t);
      } else {
        // (untracked reads: tied by lds_wait_tie before the MFMAs use them)
        const shortx4 x = ds_read_tr16_b64_async(sb + bfo[j][ks][0]);
        const shortx4 y = ds_read_tr16_b64_async(sb + bfo[j][ks][1]);
        bfr[j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
  };
  // MFMA k of a sub-step: one per tile in 16 bits; four per tile in fp32, the
  // tiles in turn so that consecutive ones are independent.
  constexpr int NMMA = TM * TN * (F32 ? 4 : 1);
  auto mma1 = [&](const bf16x8 (&af)[TM], const bf16x8 (&bfr)[TN], int k) __attribute__((always_inline)) {
    const int t = k % (TM * TN), i = t / TN, j = t % TN;
    if constexpr (F32)
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(floatx4, af[i])[k / (TM * TN)],
                                                       __builtin_bit_cast(floatx4, bfr[j])[k / (TM * TN)], acc[i][j],
                                                       0, 0, 0);
    else
      acc[i][j] = mma32_16b<H>(af[i], bfr[j], acc[i][j]);
  };
  // Every wavefront's copies of a stage have landed once each waited for its
  // own (vmcnt) and all passed the barrier.  A bare s_barrier, not
  // __syncthreads(): the latter's fence makes the compiler wait for every
  // outstanding copy (vmcnt(0)), which would leave one stage in flight
  // instead of NS - 1.  The signal fences keep the compiler from moving LDS
  // accesses across the barrier; they emit no instruction.
  auto barrier = [&]() __attribute__((always_inline)) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };

  // Software pipeline: the fragments of sub-step ks + 1 are read while the
  // MFMAs of sub-step ks run; the stage hand-over (wait, barrier) sits between
  // the reads and the MFMAs of the last sub-step, so the barrier wait overlaps
  // MFMAs already issued.  The copies go out interleaved with MFMAs, never in
  // a burst (each holds the wavefront's issue while the address unit drains
  // it, ~35 cycles).  With three or more stages, the copies of K-step s+NS-1
  // (into the stage freed at the end of step s-1) are spread over the four
  // sub-steps of step s, NS-2 steps ahead of use; with two stages, the copies
  // of K-step s+NS go out in two parts, the first H2 with the last sub-step,
  // right after the barrier that frees their stage, the rest with the first
  // sub-step of step s+1, and must land by the end of step s+1.
  constexpr bool SPREAD = NS >= 3;
  constexpr int Q = (LPT + 3) / 4;  // copies per sub-step when spread
  constexpr int H2 = (LPT + 1) / 2;  // two stages: copies issued right after the barrier
  // Copies issued after K-step s+1's last one when step s waits for it: with
  // SPREAD, K-steps s+2 .. s+NS-2 and the first 3 Q copies of K-step s+NS-1
  // (its last ones go out after the wait); with two stages, none (the wait
  // takes every copy in flight).
  constexpr int WAITN = SPREAD ? (NS - 3) * LPT + 3 * Q : (NS - 2) * LPT;
  static_assert(!SPREAD || 3 * Q <= LPT, "the last sub-step's share of the copies is not negative");
  bf16x8 fa[2][TM], fb[2][TN];
  // The fragment reads of sub-step nks of the stage at nsb, then the MFMAs of
  // the current one with copies u0 .. u1-1 of K-step sd between them.
  auto sub_step = [&](int cur, const unsigned char* nsb, int nks, int sd, int u0, int u1)
                      __attribute__((always_inline)) {
    frags(nsb, nks, fa[cur ^ 1], fb[cur ^ 1]);
    __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the MFMAs
    const int nc = u1 - u0, per = (nc + NMMA - 1) / NMMA;
#pragma unroll
    for (int k = 0; k < NMMA; ++k) {
      mma1(fa[cur], fb[cur], k);
#pragma unroll
      for (int u = u0 + k * per; u < u0 + (k + 1) * per && u < u1; ++u) dma1(sd, sd % NS, u);
      if (nc > 0) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Steps of the loop: KG K-steps each (a group's K-steps past K copy zeros).
  const int nk = ((K + BK - 1) / BK + KG - 1) / KG;
  const unsigned char* const glds = lds + kg * STAGE;  // this group's part of stage 0
  // K-steps 0 .. NS-2, and with two stages the first H2 copies of K-step
  // NS-1 (step 0 issues the rest, as every step does for the K-step after it).
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) dma(s, s);
  if constexpr (!SPREAD) {
#pragma unroll
    for (int u = 0; u < H2; ++u) dma1(NS - 1, NS - 1, u);
  }
  g_wait_vm<(NS - 2) * LPT + (SPREAD ? 0 : H2)>();  // K-step 0 has landed
  barrier();
  frags(glds, 0, fa[0], fb[0]);
#pragma unroll 1
  for (int s = 0; s < nk; ++s) {
    const unsigned char* sb = glds + (s % NS) * SSET;
#pragma unroll
    for (int ks = 0; ks < 3; ++ks) {
      if constexpr (!BT && !F32) {  // B^T fragments of sub-step ks have landed (read one sub-step ago)
#pragma unroll
        for (int j = 0; j < TN; ++j) lds_wait_tie(fb[ks & 1][j]);
      }
      if constexpr (SPREAD)
        sub_step(ks & 1, sb, ks + 1, s + NS - 1, ks * Q, min((ks + 1) * Q, LPT));
      else
        sub_step(ks & 1, sb, ks + 1, s + NS - 1, H2, ks == 0 ? LPT : H2);  // the rest of K-step s+1
    }
    g_wait_vm<WAITN>();  // K-step s+1 has landed
    g_wait_lgkm0();      // this wavefront's reads of K-step s are done
    if constexpr (!BT && !F32) {
#pragma unroll
      for (int j = 0; j < TN; ++j) lds_wait_tie(fb[1][j]);
    }
    barrier();                    // ... for every wavefront
    // The last sub-step's MFMAs (fragments in registers), with the next
    // K-step's first fragment reads.
    const unsigned char* nsb = glds + ((s + 1) % NS) * SSET;
    if constexpr (SPREAD)
      sub_step(1, nsb, 0, s + NS - 1, 3 * Q, LPT);
    else
      sub_step(1, nsb, 0, s + NS, 0, H2);  // into K-step s's stage
  }
  __builtin_amdgcn_s_waitcnt(0);  // the copies of K-steps past K have landed

  // Epilogue staging (staged path): NW wavefronts x RP rows of PITCH floats.
  constexpr int OE = 16 / sizeof(TO);  // output elements per 16-byte store
  constexpr int WC_MAX = WN;           // staged columns per wavefront (SwiGLU: WN / 2)
  constexpr int PITCH = WC_MAX + 4;    // staged row pitch, floats
  constexpr int RED = (KG - 1) * NW * TM * TN * 4096;  // the K groups' partial sums, bytes
  constexpr int RP = NW * WM * PITCH * 4 + RED <= NS * SSET ? WM : 32;  // rows per pass
  constexpr int TP = RP / 32;                                      // tiles per pass
  static_assert(NW * RP * PITCH * 4 <= NS * SSET, "the staged rows fit the stages");
  if constexpr (KG > 1) {
    // Groups 1 .. KG-1 leave their accumulators in LDS past the staging
    // area (lane-major float4 chunks); group 0 adds them in group order and
    // writes the tile alone.  The second barrier is the last one any
    // wavefront takes part in.
    constexpr int NCH = TM * TN * 4;  // float4 chunks per lane
    constexpr int ROFF = (NW * RP * PITCH * 4 + 15) / 16 * 16;
    static_assert(ROFF + (KG - 1) * NW * NCH * 1024 <= NS * SSET, "the partial sums fit the stages");
    float4* red = reinterpret_cast<float4*>(lds + ROFF);
    __syncthreads();  // every wavefront is done with the stages
    if (kg > 0) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const floatx16& a = acc[c / 4 / TN][c / 4 % TN];
        red[(((kg - 1) * NW + wid) * NCH + c) * 64 + lane] =
            make_float4(a[4 * (c % 4)], a[4 * (c % 4) + 1], a[4 * (c % 4) + 2], a[4 * (c % 4) + 3]);
      }
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const float4 v = red[(((g - 1) * NW + wid) * NCH + c) * 64 + lane];
        floatx16& a = acc[c / 4 / TN][c / 4 % TN];
        a[4 * (c % 4)] += v.x;
        a[4 * (c % 4) + 1] += v.y;
        a[4 * (c % 4) + 2] += v.z;
        a[4 * (c % 4) + 3] += v.w;
      }
  }

  // Epilogue: accumulator element e of tile (i, j) is C[row][col] with
  // row = 8 * (e / 4) + 4 * (lane / 32) + e % 4, col = lane % 32.
  if (p.epi != kEpiElem) {
    // Staged: the wavefront writes RP rows of its WM x WC block (fp32) to its
    // own LDS rows, then each lane reads OE consecutive values of a row, adds
    // the residual in fp32 and stores them as one 16-byte vector; WM / RP
    // passes.  With the SwiGLU pairing, tiles 2k and 2k+1 of the wavefront
    // hold gate and up for the same 32 output columns (the weight rows are
    // interleaved in groups of 32), and the block written is
    // silu(TO(gate)) * TO(up): the values a gate and an up GEMM with TO
    // outputs would hand the SwiGLU kernel.
    if constexpr (KG == 1) __syncthreads();  // every wavefront is done with the stages (KG > 1: above)
    float* stg = reinterpret_cast<float*>(lds) + wid * (RP * PITCH);
    const bool sw = p.epi == kEpiSwiglu;
    const int wc = sw ? WN / 2 : WN;
    // Rows of the block go to rows m0 + wm WM ..; columns to c0 ...
    const int c0 = sw ? (n0 + wn * WN) / 2 : n0 + wn * WN;
    const int ncols = sw && !GU ? p.N / 2 : p.Nc;
    const int cpr = wc / OE;  // 16-byte chunks per staged row
#pragma unroll
    for (int ip = 0; ip < TM / TP; ++ip) {
      if (sw) {
        if constexpr (TN % 2 == 0) {  // gate/up tiles come in pairs (the host picks such a tile)
#pragma unroll
          for (int t = 0; t < TP; ++t)
#pragma unroll
            for (int k = 0; k < TN / 2; ++k)
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                const float g = to_f32<TO>(from_f32<TO>(acc[ip * TP + t][2 * k][e]));
                const float u = to_f32<TO>(from_f32<TO>(acc[ip * TP + t][2 * k + 1][e]));
                stg[(t * 32 + 8 * (e / 4) + 4 * lg + (e % 4)) * PITCH + k * 32 + lr] = silu(g) * u;
              }
        }
      } else {
#pragma unroll
        for (int t = 0; t < TP; ++t)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
              stg[(t * 32 + 8 * (e / 4) + 4 * lg + (e % 4)) * PITCH + j * 32 + lr] = acc[ip * TP + t][j][e];
      }
#pragma unroll 4
      for (int c = lane; c < RP * cpr; c += 64) {
        const int rl = c / cpr, cl = (c % cpr) * OE;
        const int row = m0 + wm * WM + ip * RP + rl, col = c0 + cl;
        if (row < p.M && col < ncols) {
          float v[OE];
#pragma unroll
          for (int e = 0; e < OE; e += 4) {
            const float4 x = *reinterpret_cast<const float4*>(stg + rl * PITCH + cl + e);
            v[e] = x.x;
            v[e + 1] = x.y;
            v[e + 2] = x.z;
            v[e + 3] = x.w;
          }
          if (R) {
            float r[OE];
            load16(R + (long)row * p.ldr + col, r);
#pragma unroll
            for (int e = 0; e < OE; ++e) v[e] += r[e];
          }
          store_vec<OE>(C + (long)row * p.ldc + col, v);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * WN + j * 32 + lr;
      if (col >= p.Nc) continue;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = m0 + wm * WM + i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
        if (row < p.M) {
          float vv = acc[i][j][e];
          if (R) vv += to_f32(R[(long)row * p.ldr + col]);
          C[(long)row * p.ldc + col] = from_f32<TO>(vv);
        }
      }
    }
}

// ----------------------------------------- register-staged GEMM, unaligned --
//
// Operands the buffer unit's copies cannot take (bases, K or leading dimensions
// off 16 bytes, N off 16 bytes with B as [K, N], 2 GiB or more).  Operand tiles
// go global -> registers -> LDS, PF K-steps ahead, with 16-byte loads at the
// element's own alignment (gfx950 takes them at any address); the last K-steps,
// and those with rows of a [K, N] B whose loads would end past it, are loaded
// with a check per chunk and the chunk that straddles K or N element by
// element.  Rows and columns past M and N repeat the last one (their products
// are never stored); K is padded with zeros in both operands.
//
// Bound by the K-step's chain (LDS reads, stores and a barrier, ~0.4 us with one
// workgroup on a CU) on small grids and by LDS traffic on large ones.  One
// wavefront per tile reading elements from global memory, as before, took 74 us
// at 1000 x 777 x 1301 bf16; this takes 13.6 on 64x64 tiles (rows at an odd
// address cost ~20%) and 10.5 on 64x128 with eight wavefronts, whose 176 tiles
// make one round where 336 make two.
//
// LDS tiles are the LDS-DMA kernel's: 128-byte rows (32 fp32 or 64 16-bit
// elements of K; B as [K, N] in 16 bits in sub-tiles of 64 columns), 16-byte
// chunks swizzled, and one b128 read per operand fragment: 8 elements of K for
// one 16-bit MFMA, or 4 for four fp32 MFMAs (32x32x2; lane group lg supplies
// k = 4 lg + j to MFMA j of the four, the same order in A and B).  fp32 B as
// [K, N] stays row-major and is read 4 bytes at a time, 32 columns a row.
//
// KG groups of WGM x WGN wavefronts share the tile as in the LDS-DMA kernel:
// group g takes K-steps g, g + KG, ... and the groups' accumulators are added
// in group order at the end, so that a GEMM of few tiles still has its K range
// spread over a CU's SIMDs.
__device__ __forceinline__ u32x4_t ld16_unaligned(const float* p) { return *reinterpret_cast<const u32x4_al4*>(p); }
template <typename T>
__device__ __forceinline__ u32x4_t ld16_unaligned(const T* p) {
  static_assert(sizeof(T) == 2, "16-bit elements");
  return *reinterpret_cast<const u32x4_al2*>(p);
}
// The first n elements at p, zeros after them.
template <typename T>
__device__ __forceinline__ u32x4_t ld16_first(const T* p, int n) {
  constexpr int E = VecE<T>::value;
  if (n >= E) return ld16_unaligned(p);
  u32x4_t r = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (e < n) {
      if constexpr (sizeof(T) == 4)
        r[e] = __float_as_uint(p[e]);
      else
        r[e / 2] |= (uint32_t)__builtin_bit_cast(uint16_t, p[e]) << (16 * (e & 1));
    }
  return r;
}

template <typename TI, typename TO, int BM, int BN, bool BT, int WGM, int WGN, int KG, int PF, int ACC = 1,
          bool SHORT = false>
__global__ __launch_bounds__(64 * WGM * WGN * KG) void gemm_reg_kernel(GemmArgs p) {
  // ACC = 2: even and odd K-steps are summed apart and added at the end, as two
  // K groups do.  SHORT: a K-step or two, loaded with checks and without the
  // sub-steps that hold zeros alone.
  constexpr bool F32 = sizeof(TI) == 4;
  constexpr bool H = std::is_same<TI, f16>::value;
  constexpr int E = VecE<TI>::value;  // elements per 16-byte chunk
  constexpr int BK = 128 / sizeof(TI);
  constexpr int NT = 64 * WGM * WGN;  // threads of a K group
  constexpr int A_BYTES = BM * 128, STAGE = A_BYTES + BN * 128, SSET = KG * STAGE;
  constexpr int A_CH = BM * 8 / NT, B_CH = BN * 8 / NT;  // chunks per thread and K-step
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
  static_assert(A_CH * NT == BM * 8 && B_CH * NT == BN * 8, "chunks split over the group");
  static_assert(F32 || BT || BN % 64 == 0, "16-bit [K, N] tiles are made of 64-column sub-tiles");
  __shared__ __align__(16) unsigned char lds[2 * SSET];

  const int tid = threadIdx.x % NT, lane = tid & 63;
  const int wall = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wall / (WGM * WGN), wid = wall % (WGM * WGN);
  const int wm = wid / WGN, wn = wid % WGN;
  const int lr = lane & 31, lg = lane >> 5;
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int bz = blockIdx.z;
  const TI* A = static_cast<const TI*>(p.A) + (long)bz * p.sA;
  const TI* B = static_cast<const TI*>(p.B) + (long)bz * p.sB;
  TO* C = static_cast<TO*>(p.C) + (long)bz * p.sC;
  const TO* R = p.R ? static_cast<const TO*>(p.R) + (long)bz * p.sR : nullptr;
  const int K = p.Kall ? min(p.K, p.Kall - bz * p.K) : p.K, N = p.N;

  // Chunk i of the thread: LDS byte, K offset within a K-step and address at
  // K-step 0.
  const TI* pa[A_CH];
  const TI* pb[B_CH];
  int la[A_CH], lb[B_CH], ka[A_CH], kb[B_CH], nb[B_CH];
#pragma unroll
  for (int i = 0; i < A_CH; ++i) {
    const int c = tid + NT * i, row = c / 8, pc = c % 8;
    la[i] = g_pos(row, pc);
    ka[i] = pc * E;
    pa[i] = A + (long)min(m0 + row, p.M - 1) * p.lda + ka[i];
  }
#pragma unroll
  for (int i = 0; i < B_CH; ++i) {
    const int c = tid + NT * i;
    if constexpr (BT) {
      const int row = c / 8, pc = c % 8;
      lb[i] = A_BYTES + g_pos(row, pc);
      kb[i] = pc * E;
      nb[i] = E;
      pb[i] = B + (long)min(n0 + row, N - 1) * p.ldb + kb[i];
    } else {
      constexpr int CPR = BN / E;  // chunks per K row
      const int kr = c / CPR, nc = c % CPR;
      const int n = min(n0 + nc * E, (N - 1) / E * E);  // columns past N repeat the last chunk
      lb[i] = A_BYTES + (F32 ? kr * BN * 4 + nc * 16 : nc / 8 * 8192 + g_pos(kr, nc % 8));
      kb[i] = kr;
      nb[i] = N - n;  // columns the chunk may read
      pb[i] = B + (long)kr * p.ldb + n;
    }
  }
  const long b_step = BT ? BK : (long)BK * p.ldb;
  // The leading K-steps whose loads all end within K and, with B as [K, N],
  // before B's last element.
  int kfast = K / BK;
  if constexpr (!BT) {
    const long end = (long)(K - 1) * p.ldb + N - min(n0 + BN, (N + E - 1) / E * E);  // last row a chunk fits in
    kfast = end < 0 ? 0 : (int)min((long)kfast, (end / p.ldb + 1) / BK);
  }

  // Registers of K-steps in flight: K-step s in slot s % PF.
  u32x4_t rra[PF][A_CH], rrb[PF][B_CH];
  auto gload = [&](int s, u32x4_t (&ra)[A_CH], u32x4_t (&rb)[B_CH])
                   __attribute__((always_inline)) {  // K-step s of this group, a leading one
    const int ks = KG * s + kg;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) ra[i] = ld16_unaligned(pa[i] + ks * BK);
#pragma unroll
    for (int i = 0; i < B_CH; ++i) rb[i] = ld16_unaligned(pb[i] + ks * b_step);
  };
  auto gload_checked = [&](int s, u32x4_t (&ra)[A_CH], u32x4_t (&rb)[B_CH]) __attribute__((always_inline)) {
    const int ks = KG * s + kg, k0 = ks * BK;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) ra[i] = ld16_first(pa[i] + k0, K - k0 - ka[i]);
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      if constexpr (BT)
        rb[i] = ld16_first(pb[i] + k0, K - k0 - kb[i]);
      else
        rb[i] = ld16_first(pb[i] + ks * b_step, k0 + kb[i] < K ? nb[i] : 0);
    }
  };
  auto lstore = [&](int st, const u32x4_t (&ra)[A_CH], const u32x4_t (&rb)[B_CH]) __attribute__((always_inline)) {
    unsigned char* sb = lds + st * SSET + kg * STAGE;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) *reinterpret_cast<u32x4_t*>(sb + la[i]) = ra[i];
#pragma unroll
    for (int i = 0; i < B_CH; ++i) *reinterpret_cast<u32x4_t*>(sb + lb[i]) = rb[i];
  };
  // The LDS stores and reads of every wavefront are done; the next K-step's
  // global loads stay in flight (__syncthreads() would wait for them).
  auto lds_barrier = [&]() __attribute__((always_inline)) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    g_wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };

  floatx16 accs[ACC][TM][TN];
#pragma unroll
  for (int x = 0; x < ACC; ++x)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) accs[x][i][j][e] = 0.f;

  const int nk = ((K + BK - 1) / BK + KG - 1) / KG;
  // Every fragment of the K-step in stage st (its first nks sub-steps) is read
  // in flight together, then `mid` runs behind the reads, then the MFMAs into
  // acc.
  auto compute = [&](int st, int nks, floatx16 (&acc)[TM][TN], auto mid) __attribute__((always_inline)) {
    const unsigned char* sb = lds + st * SSET + kg * STAGE;
    bf16x8 af[4][TM], bfr[4][TN];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks >= nks) break;
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[ks][i] = *reinterpret_cast<const bf16x8*>(sb + g_pos(wm * WM + lr, 2 * ks + lg) + 4096 * i);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (BT) {
          bfr[ks][j] = *reinterpret_cast<const bf16x8*>(sb + A_BYTES + g_pos(wn * WN + lr, 2 * ks + lg) + 4096 * j);
        } else if constexpr (F32) {
          const float* bp =
              reinterpret_cast<const float*>(sb + A_BYTES) + (8 * ks + 4 * lg) * BN + wn * WN + 32 * j + lr;
          bfr[ks][j] = __builtin_bit_cast(bf16x8, floatx4{bp[0], bp[BN], bp[2 * BN], bp[3 * BN]});
        } else {
          // Two transposed reads of 4 K rows: lane i of a 16-lane group
          // reads row i / 4, columns 4 (i % 4) .. + 3 of its 16.
          const int i16 = lane & 15, g2 = (lane >> 4) & 1;
          const int n = wn * WN + j * 32 + 16 * g2 + 4 * (i16 & 3), nc = n % 64;
          const unsigned char* bp = sb + A_BYTES + n / 64 * 8192 + (nc % 8) * 2;
          const shortx4 x = ds_read_tr16_b64_tracked(bp + g_pos(16 * ks + 8 * lg + (i16 >> 2), nc / 8));
          const shortx4 y = ds_read_tr16_b64_tracked(bp + g_pos(16 * ks + 8 * lg + 4 + (i16 >> 2), nc / 8));
          bfr[ks][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    mid();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks >= nks) break;
      if constexpr (F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(floatx4, af[ks][i])[e],
                                                               __builtin_bit_cast(floatx4, bfr[ks][j])[e], acc[i][j], 0,
                                                               0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = mma32_16b<H>(af[ks][i], bfr[ks][j], acc[i][j]);
      }
    }
  };
  // Leading steps (every group's K-step a leading one): no branch around a
  // load, so that each wait counts the loads issued after the one it waits
  // for.  The last steps' loads past nfast repeat the last leading step.
  const int nfast = SHORT ? 0 : kfast / KG;
  if (nfast > 0) {
#pragma unroll
    for (int u = 0; u < PF; ++u) gload(min(u, nfast - 1), rra[u], rrb[u]);
    lstore(0, rra[0], rrb[0]);
    gload(min(PF, nfast - 1), rra[0], rrb[0]);
    lds_barrier();
#pragma unroll 1
    for (int s0 = 0; s0 < nfast; s0 += max(PF, ACC))
#pragma unroll
      for (int u = 0; u < max(PF, ACC); ++u) {
        const int s = s0 + u;
        if (s >= nfast) break;
        compute(s & 1, 4, accs[u % ACC], [&]() __attribute__((always_inline)) {
          // The next K-step's LDS stores (its stage was read last in step
          // s - 1) and the global loads PF steps after it.
          lstore((s + 1) & 1, rra[(u + 1) % PF], rrb[(u + 1) % PF]);
          gload(min(s + 1 + PF, nfast - 1), rra[(u + 1) % PF], rrb[(u + 1) % PF]);
        });
        lds_barrier();
      }
  }
#pragma unroll 1
  for (int s = nfast; s < nk; ++s) {
    gload_checked(s, rra[0], rrb[0]);
    lstore(s & 1, rra[0], rrb[0]);
    lds_barrier();
    constexpr int SUB = BK / 4;  // K elements of a sub-step
    const int nks = SHORT ? (K - (KG * s + kg) * BK + SUB - 1) / SUB : 4;
    if (ACC == 1 || s % 2 == 0)
      compute(s & 1, nks, accs[0], []() {});
    else
      compute(s & 1, nks, accs[ACC - 1], []() {});
    lds_barrier();
  }
  floatx16(&acc)[TM][TN] = accs[0];
  if constexpr (ACC == 2) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += accs[1][i][j][e];
  }

  if constexpr (KG > 1) {
    // Groups 1 .. KG-1 leave their accumulators in LDS (lane-major float4
    // chunks); group 0 adds them in group order and writes the tile.
    constexpr int NCH = TM * TN * 4;
    static_assert((KG - 1) * WGM * WGN * NCH * 1024 <= 2 * SSET, "the partial sums fit the stages");
    floatx4* red = reinterpret_cast<floatx4*>(lds);
    if (kg > 0) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const floatx16& a = acc[c / 4 / TN][c / 4 % TN];
        red[(((kg - 1) * WGM * WGN + wid) * NCH + c) * 64 + lane] =
            floatx4{a[4 * (c % 4)], a[4 * (c % 4) + 1], a[4 * (c % 4) + 2], a[4 * (c % 4) + 3]};
      }
    }
    lds_barrier();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const floatx4 v = red[(((g - 1) * WGM * WGN + wid) * NCH + c) * 64 + lane];
        floatx16& a = acc[c / 4 / TN][c / 4 % TN];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[4 * (c % 4) + e] += v[e];
      }
  }

  // Accumulator element e of tile (i, j) is C[row][col] with
  // row = 8 * (e / 4) + 4 * (lane / 32) + e % 4, col = lane % 32.
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * WN + j * 32 + lr;
      if (col >= p.Nc) continue;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = m0 + wm * WM + i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
        if (row < p.M) {
          float vv = acc[i][j][e];
          if (R) vv += to_f32(R[(long)row * p.ldr + col]);
          C[(long)row * p.ldc + col] = from_f32<TO>(vv);
        }
      }
    }
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// The staged epilogue stores 16-byte vectors: C (and R) rows, batch strides
// and N must keep every vector 16-byte aligned.
template <typename TO>
static bool staged_ok(const GemmArgs& a) {
  constexpr long OE = 16 / sizeof(TO);
  const bool c_ok = aligned16(a.C) && a.ldc % OE == 0 && a.sC % OE == 0 && a.Nc % OE == 0;
  const bool r_ok = !a.R || (aligned16(a.R) && a.ldr % OE == 0 && a.sR % OE == 0);
  return c_ok && r_ok;
}

// Tiles of the LDS-DMA kernel.
// K2: two K groups of four wavefronts per tile.
enum DmaTile { kT64x64, kT64x128, kT128x128, kT128x256, kT256x128, kT256x192, kT256x256, kT64x64K2, kT64x128K2,
               kTileCount };

template <typename TI, typename TO, bool BT>
static void launch_dma(DmaTile t, const GemmArgs& g, int batch, hipStream_t st) {
  auto grid = [&](int bm, int bn) {
    return dim3((unsigned)((long)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn)), 1, (unsigned)batch);
  };
  switch (t) {
    case kT256x256: gemm_dma_kernel<TI, TO, 256, 256, BT, 2, 2, 4><<<grid(256, 256), dim3(512), 0, st>>>(g); break;
    case kT256x192: gemm_dma_kernel<TI, TO, 256, 192, BT, 2, 4, 2><<<grid(256, 192), dim3(512), 0, st>>>(g); break;
    case kT256x128: gemm_dma_kernel<TI, TO, 256, 128, BT, 3, 4, 2><<<grid(256, 128), dim3(512), 0, st>>>(g); break;
    case kT128x256: gemm_dma_kernel<TI, TO, 128, 256, BT, 3, 2, 4><<<grid(128, 256), dim3(512), 0, st>>>(g); break;
    case kT128x128: gemm_dma_kernel<TI, TO, 128, 128, BT, 4><<<grid(128, 128), dim3(256), 0, st>>>(g); break;
    case kT64x128: gemm_dma_kernel<TI, TO, 64, 128, BT, 6><<<grid(64, 128), dim3(256), 0, st>>>(g); break;
    case kT64x128K2: gemm_dma_kernel<TI, TO, 64, 128, BT, 3, 2, 2, 2><<<grid(64, 128), dim3(512), 0, st>>>(g); break;
    case kT64x64K2: gemm_dma_kernel<TI, TO, 64, 64, BT, 4, 2, 2, 2><<<grid(64, 64), dim3(512), 0, st>>>(g); break;
    default: gemm_dma_kernel<TI, TO, 64, 64, BT, 8><<<grid(64, 64), dim3(256), 0, st>>>(g); break;
  }
}

// NKL_GEMM_TILE=64x64|64x128|128x128|128x256|256x128|256x192|256x256|64x64k2|64x128k2
// forces a tile (for measurements); -1 when unset or unknown.
static int forced_tile() {
  static const int forced = [] {
    const char* f = getenv("NKL_GEMM_TILE");
    if (!f) return -1;
    static const char* names[kTileCount] = {"64x64",   "64x128",   "128x128",  "128x256", "256x128",
                                            "256x192", "256x256", "64x64k2", "64x128k2"};
    for (int i = 0; i < kTileCount; ++i)
      if (!strcmp(f, names[i])) return i;
    return -1;
  }();
  return forced;
}

static long tiles_of(const GemmArgs& a, int bm, int bn, int batch) {
  return (((long)a.M + bm - 1) / bm) * (((long)a.N + bn - 1) / bn) * batch;
}

// Tile choice.  With a 128x128 tile or larger for every CU, the tile whose
// rounds of 256 workgroups (one per CU) cost least, at the time per K-step
// of a round measured on MI355X (bf16, K-contiguous B): 256x256 1.9 us,
// 256x192 1.75 us, 256x128 1.25 us, 128x128 0.8 us.  256x192 fills the CUs
// where 256x256 leaves a quarter idle (2048 x 6144: 256 tiles against 192).
// Smaller GEMMs: the largest tile that still gives every CU a workgroup, with
// two K groups (64x64: 1024^3 9.0 -> 8.4 us; 64x128: 2-6% on 1024-2048-row
// shapes).
static DmaTile choose_tile(const GemmArgs& a, int batch) {
  if (forced_tile() >= 0) return (DmaTile)forced_tile();
  const long t128 = tiles_of(a, 128, 128, batch);
  if (t128 >= 256) {
    auto rounds = [](long t) { return (double)((t + 255) / 256); };
    const struct { DmaTile t; double c; } cand[] = {
        {kT256x256, 1.9 * rounds(tiles_of(a, 256, 256, batch))},
        {kT256x192, 1.75 * rounds(tiles_of(a, 256, 192, batch))},
        {kT256x128, 1.25 * rounds(tiles_of(a, 256, 128, batch))},
        {kT128x128, 0.8 * rounds(t128)}};
    DmaTile best = kT256x256;
    double cb = 1e30;
    for (const auto& c : cand)
      if (c.c < cb) cb = c.c, best = c.t;
    return best;
  }
  if (tiles_of(a, 64, 128, batch) >= 256) return kT64x128K2;
  return kT64x64K2;
}

// Rows and columns of a tile.
static void tile_dims(DmaTile t, int& bm, int& bn) {
  switch (t) {
    case kT256x256: bm = 256, bn = 256; break;
    case kT256x192: bm = 256, bn = 192; break;
    case kT256x128: bm = 256, bn = 128; break;
    case kT128x256: bm = 128, bn = 256; break;
    case kT128x128: bm = 128, bn = 128; break;
    case kT64x128:
    case kT64x128K2: bm = 64, bn = 128; break;
    default: bm = 64, bn = 64; break;
  }
}

// Time per K-step of a round of one-per-CU workgroups (the tile choice's
// figures), 0 for the tiles it does not price.
static double round_step_us(DmaTile t) {
  return t == kT256x256 ? 1.9 : t == kT256x192 ? 1.75 : t == kT256x128 ? 1.25 : t == kT128x128 ? 0.8 : 0.0;
}

// Column split of a launch whose 256-row tiles leave a partial last round:
// the columns of the whole rounds go to a first launch, the rest to a second
// launch with the tile chosen for them alone (2048 x 11264: 352 tiles of
// 256 x 256 make a round and then 96 -- instead, 256 such tiles over the first
// 8192 columns and 192 tiles of 256 x 128 over the last 3072).  The plan is
// the cheapest, at the round times above plus 2 us for a second launch, of
// the chosen tile over all columns and the column splits of the 256-row
// tiles.  n1 = 0: one launch with t1.  swiglu: the gate/up GEMM, whose
// wavefronts own 64 columns (no 256 x 192 tile).
struct TilePlan {
  DmaTile t1;
  int n1;
  DmaTile t2;
};
static TilePlan plan_tiles(const GemmArgs& a, DmaTile t, int batch, bool swiglu) {
  TilePlan best{t, 0, t};
  if (batch != 1 || forced_tile() >= 0 || round_step_us(t) == 0.0) return best;
  const long cus = cu_count();
  const double nk = (a.K + 63) / 64;
  auto cost = [&](DmaTile x, int n) {
    int bm, bn;
    tile_dims(x, bm, bn);
    const long tiles = (long)((a.M + bm - 1) / bm) * ((n + bn - 1) / bn);
    return round_step_us(x) * (double)((tiles + cus - 1) / cus) * nk;
  };
  double cb = cost(t, a.N);
  for (DmaTile x : {kT256x256, kT256x192, kT256x128}) {
    if (swiglu && x == kT256x192) continue;
    int bm, bn;
    tile_dims(x, bm, bn);
    const long tm = (a.M + 255) / 256, tiles = tm * ((a.N + bn - 1) / bn);
    if (tiles <= cus || tiles % cus == 0 || tm > cus) continue;
    const long n1 = (tiles / cus) * cus / tm * bn;  // the columns of the whole rounds
    if (n1 <= 0 || n1 >= a.N) continue;
    GemmArgs rest = a;
    rest.N = (int)(a.N - n1);
    DmaTile t2 = choose_tile(rest, 1);
    if (swiglu && t2 == kT256x192) t2 = kT256x256;
    if (round_step_us(t2) == 0.0) continue;
    const double c = cost(x, (int)n1) + cost(t2, rest.N) + 2.0;
    if (c < cb) cb = c, best = TilePlan{x, (int)n1, t2};
  }
  return best;
}

// launch_dma after plan_tiles: one launch, or two over a column split.
template <typename TI, typename TO, bool BT>
static void launch_dma_cols(DmaTile t, const GemmArgs& g, int batch, bool swiglu, hipStream_t st) {
  const TilePlan pl = plan_tiles(g, t, batch, swiglu);
  if (pl.n1 == 0) {
    launch_dma<TI, TO, BT>(pl.t1, g, batch, st);
    return;
  }
  GemmArgs g1 = g, g2 = g;
  g1.N = g1.Nc = pl.n1;
  g2.N = g.N - pl.n1;
  g2.Nc = g.Nc - pl.n1;
  const TI* B = static_cast<const TI*>(g.B);
  g2.B = BT ? B + (long)pl.n1 * g.ldb : B + pl.n1;
  const long coff = swiglu ? pl.n1 / 2 : pl.n1;
  g2.C = static_cast<TO*>(g.C) + coff;
  if (g.R) g2.R = static_cast<const TO*>(g.R) + coff;
  launch_dma<TI, TO, BT>(pl.t1, g1, 1, st);
  launch_dma<TI, TO, BT>(pl.t2, g2, 1, st);
}

// One launch, unless its threads pass HIP's limit (a column of 1.1G rows is
// 16.8M tiles of 256 threads): then over ranges of rows and columns.
template <typename T, typename TO, bool BT, int BM, int BN, int WGM, int WGN, int KG, int PF, int ACC = 1,
          bool SHORT = false>
static void launch_reg(const GemmArgs& a, int batch, hipStream_t st) {
  constexpr int NT = 64 * WGM * WGN * KG;
  const long fit = kMaxGridThreads / NT, cols = min(tiles_of(a, a.M, BN, 1), fit) * BN, rows = fit / (cols / BN) * BM;
  for (long m = 0; m < a.M; m += rows)
    for (long n = 0; n < a.N; n += cols) {
      GemmArgs g = a;
      g.M = (int)min(rows, a.M - m);
      g.N = (int)min(cols, a.N - n);
      g.Nc = (int)min((long)g.N, a.Nc - n);
      g.A = static_cast<const T*>(a.A) + m * a.lda;
      g.B = static_cast<const T*>(a.B) + (BT ? n * a.ldb : n);
      g.C = static_cast<TO*>(a.C) + m * a.ldc + n;
      if (a.R) g.R = static_cast<const TO*>(a.R) + m * a.ldr + n;
      const dim3 grid((unsigned)tiles_of(g, BM, BN, 1), 1, (unsigned)batch);
      gemm_reg_kernel<T, TO, BM, BN, BT, WGM, WGN, KG, PF, ACC, SHORT><<<grid, dim3(NT), 0, st>>>(g);
    }
}

// fp32 tiles of the LDS-DMA kernel (two or four K groups each).
enum F32Tile { kF128x128, kF64x128, kF64x64, kF32x64, kF32x32 };

template <typename TO, bool BT>
static void launch_f32(int t, const GemmArgs& g, int batch, hipStream_t st) {
  auto grid = [&](int bm, int bn) { return dim3((unsigned)tiles_of(g, bm, bn, 1), 1, (unsigned)batch); };
  switch (t) {
    case kF128x128: gemm_dma_kernel<float, TO, 128, 128, BT, 2, 2, 2, 2><<<grid(128, 128), dim3(512), 0, st>>>(g); break;
    case kF64x128: gemm_dma_kernel<float, TO, 64, 128, BT, 3, 2, 2, 2><<<grid(64, 128), dim3(512), 0, st>>>(g); break;
    case kF64x64: gemm_dma_kernel<float, TO, 64, 64, BT, 4, 2, 2, 2><<<grid(64, 64), dim3(512), 0, st>>>(g); break;
    case kF32x64: gemm_dma_kernel<float, TO, 32, 64, BT, 3, 1, 2, 4><<<grid(32, 64), dim3(512), 0, st>>>(g); break;
    default: gemm_dma_kernel<float, TO, 32, 32, BT, 4, 1, 1, 4><<<grid(32, 32), dim3(256), 0, st>>>(g); break;
  }
}

// The gate/up GEMM with SwiGLU in fp32 (nkl_gemm_gate_up): the tiles whose
// wavefronts own 64 columns, by the rule of choose_f32_tile over both weights'
// columns.  Bound by the fp32 MFMAs as the plain fp32 GEMM is; it saves two
// launches and the passes over gate and up: two GEMMs and the SwiGLU kernel took
// 17.1 us at 300 x 1024 x K 256, this 9.0; 16 x 768 x 256 16.6 -> 6.7, 1000 x
// 2048 x 512 52 -> 37, 2048 x 3072 x 1024 235 -> 199, 2048 x 6144 x 2048 793 ->
// 764.  The error against 64 bits is the same.
static void launch_f32_gate_up(const GemmArgs& g, hipStream_t st) {
  auto grid = [&](int bm, int bn) { return dim3((unsigned)tiles_of(g, bm, bn, 1)); };
  auto rounds = [&](int bm, int bn) { return (double)((tiles_of(g, bm, bn, 1) + 255) / 256); };
  if (tiles_of(g, 32, 64, 1) <= 256) {
    gemm_dma_kernel<float, float, 32, 64, true, 3, 1, 1, 4, true><<<grid(32, 64), dim3(256), 0, st>>>(g);
    return;
  }
  const double c64 = 0.69 * rounds(64, 64), c64x128 = 1.2 * rounds(64, 128), c128 = 2.0 * rounds(128, 128);
  if (c128 <= c64x128 && c128 <= c64)
    gemm_dma_kernel<float, float, 128, 128, true, 2, 2, 2, 2, true><<<grid(128, 128), dim3(512), 0, st>>>(g);
  else if (c64x128 < c64)
    gemm_dma_kernel<float, float, 64, 128, true, 3, 2, 2, 2, true><<<grid(64, 128), dim3(512), 0, st>>>(g);
  else
    gemm_dma_kernel<float, float, 64, 64, true, 2, 2, 1, 4, true><<<grid(64, 64), dim3(512), 0, st>>>(g);
}

// The LDS-DMA kernel takes 16-byte chunks at 32-bit buffer offsets, and K >= 1:
// at K = 0 the bytes of a [K, N] B, (K - 1) ldb + N elements, are negative, a
// range that no copy's offset is past.
template <typename T, bool BT>
static bool dma_ok(const GemmArgs& a) {
  constexpr int E = VecE<T>::value;
  constexpr long SZ = sizeof(T);
  const int K = a.Kall ? a.Kall : a.K;
  const long a_bytes = SZ * ((long)(a.M - 1) * a.lda + K),
             b_bytes = SZ * (BT ? (long)(a.N - 1) * a.ldb + K : (long)(K - 1) * a.ldb + a.N);
  return K > 0 && aligned16(a.A) && aligned16(a.B) && (K % E == 0 || a.padded) && a.lda % E == 0 && a.ldb % E == 0 && a.sA % E == 0 &&
         a.sB % E == 0 && (BT || a.N % E == 0) && a_bytes < (1L << 31) && b_bytes < (1L << 31);
}

// The smallest tile that needs one round of workgroups (us: 512^3 7.2 with
// 32x32, 9.4 32x64, 13.5 64x64; 300 x 1024 x K 256 5.6 / 6.9 / 8.6 at N 768,
// 9.5 / 7.0 / 8.6 at N 1024, whose 320 tiles of 32x32 make two rounds;
// 1000^3 39 / 30 / 25.7), else the least of rounds times the time per 32
// elements of K of a round.
static F32Tile choose_f32_tile(const GemmArgs& a, int batch) {
  if (tiles_of(a, 32, 32, batch) <= 256) return kF32x32;
  if (tiles_of(a, 32, 64, batch) <= 256) return kF32x64;
  auto rounds = [&](int bm, int bn) { return (double)((tiles_of(a, bm, bn, batch) + 255) / 256); };
  const double c64 = 0.69 * rounds(64, 64), c64x128 = 1.2 * rounds(64, 128), c128 = 2.0 * rounds(128, 128);
  return c128 <= c64x128 && c128 <= c64 ? kF128x128 : c64x128 < c64 ? kF64x128 : kF64x64;
}

template <typename T, typename TO, bool BT>
static void launch_naive(const GemmArgs& a, int batch, hipStream_t st) {
  gemm_naive_kernel<T, TO, BT><<<dim3((unsigned)((tiles_of(a, 32, 32, 1) + 3) / 4), 1, batch), dim3(256), 0, st>>>(a);
}

// Unaligned products with next to no K, which writing C bounds: one wavefront
// per tile and nothing staged (us, this / the best staged form below, copies
// of the operands included; 8192 x 3001, B as [K, N] and as [N, K]: bf16 K = 3
// 17.1 / 23.5 and 15.7 / 23.4, K = 15 18.3 / 24.0 and 23.7 / 23.7; fp32 K = 3 20.6 /
// 25, K = 15 26 / 30.6 and 30 / 32.6).  With a K of whole 32-byte sectors its
// strided loads collide (fp32 K = 16 36 / 27.4).  Within a round of tiles the
// staged kernels are level.
template <typename T, bool BT>
static bool unstaged(const GemmArgs& a, int batch) {
  const int lim = BT ? (sizeof(T) == 4 ? 17 : 12) : 20;
  return a.K <= lim && a.K > 0 && (a.K % 8 || (!BT && sizeof(T) == 2 && a.K == 8)) && !dma_ok<T, BT>(a) &&
         tiles_of(a, sizeof(T) == 4 ? 32 : 64, 64, batch) > 256 && tiles_of(a, 32, 32, 1) * 64 < kMaxGridThreads - 256;
}

// One product (or a batch of them) into C, by the kernel its operands allow.
template <typename T, typename TO, bool BT>
static void gemm_launch(const GemmArgs& a, int batch, hipStream_t st) {
  if (unstaged<T, BT>(a, batch)) return launch_naive<T, TO, BT>(a, batch, st);
  const bool dma = dma_ok<T, BT>(a);
  if constexpr (sizeof(T) == 4) {
    // fp32 with a short K and more than a round of tiles: the LDS-DMA kernel's
    // one workgroup a CU leaves its prologue and stores bare, where up to five
    // of the register-staged kernel's share one (us, DMA / this; B as [K, N]
    // and [N, K], 8192 x 4096: K = 4 72 / 30 and 72 / 31, K = 16 73 / 34 and 72 /
    // 34, K = 32 73 / 41 and 73 / 40, K = 48 74 / 66 and 73 / 63, K = 128 105 / 90
    // and 104 / 88, K = 384 230 / 209 and 229 / 208; past 32 with more than a round
    // of the larger tiles only, 777 x 300 x 1024 10.2 / 15.1).  Aligned products
    // past 32 keep the LDS-DMA kernel's sums over even and odd K-steps.
    if (tiles_of(a, 32, 64, batch) > 256 && a.K > 0 && (dma ? a.K <= 32 : a.K < 64 && (a.K - 1) % 32 < 24))
      return launch_reg<T, TO, BT, 64, 64, 2, 2, 1, 1, 1, true>(a, batch, st);
    if (dma && a.K > 32 && a.K <= 384 && tiles_of(a, 64, a.N <= 64 ? 64 : 128, batch) > 256) {
      if (a.N <= 64)
        launch_reg<T, TO, BT, 64, 64, 2, 2, 1, 1, 2>(a, batch, st);
      else
        launch_reg<T, TO, BT, 64, 128, 2, 4, 1, 2, 2>(a, batch, st);
      return;
    }
  }
  if (dma) {
    GemmArgs g = a;
    g.epi = staged_ok<TO>(a) ? kEpiStaged : kEpiElem;
    if constexpr (sizeof(T) == 4)
      launch_f32<TO, BT>(choose_f32_tile(a, batch), g, batch, st);
    else
      launch_dma_cols<T, TO, BT>(choose_tile(a, batch), g, batch, false, st);
    return;
  }
  // The tile with the least rounds of workgroups (one per CU) times the
  // measured time of a round.  16 bits, relative to a K-step: 64x64 0.36, 64x128
  // with eight wavefronts 0.55, 128x128 with sixteen 0.75 (us, bf16: 1000 x 777 x
  // 1301 13.6 / 10.5 / 12.9; 700 x 777 x 1301 9.1 / 10.2 / 13.4; 1001 x 4097 x
  // 1999 44.7 / 35.5 / 43.5; 1500 x 2049 x 2047 38.2 / 35.4 / 25.9; 4001 x 129 x
  // 1001 10.6 / 9.2 / 8.1; four wavefronts on 128x128 take 20.5 to 66 there).
  // fp32: 32x64 in four K groups where it makes one round (300 x 256 x 1024 7.2,
  // 64x64 8.9); 64x128, two K-steps ahead, costs 1.87 rounds of 64x64 (1000 x
  // 777 x 1301 31.4 with 64x64, 29.6 with 64x128; 1500 x 2049 x 2047 109 / 130;
  // 4001 x 2001 x 2003 271 / 254); 128x128 takes 142 at 2047 x 1023 x 2049, 64x64 92.
  auto rounds = [&](int bm, int bn) { return (double)((tiles_of(a, bm, bn, batch) + 255) / 256); };
  if constexpr (sizeof(T) == 4) {
    if (tiles_of(a, 32, 64, batch) <= 256)
      launch_reg<T, TO, BT, 32, 64, 1, 2, 4, 2>(a, batch, st);
    else if (1.87 * rounds(64, 128) < rounds(64, 64))
      launch_reg<T, TO, BT, 64, 128, 2, 4, 1, 2>(a, batch, st);
    else
      launch_reg<T, TO, BT, 64, 64, 2, 2, 1, 1>(a, batch, st);
  } else {
    const double c64 = 0.36 * rounds(64, 64), c64x128 = 0.55 * rounds(64, 128), c128 = 0.75 * rounds(128, 128);
    if (c128 < c64x128 && c128 < c64)
      launch_reg<T, TO, BT, 128, 128, 4, 4, 1, 1>(a, batch, st);
    else if (c64x128 < c64)
      launch_reg<T, TO, BT, 64, 128, 2, 4, 1, 1>(a, batch, st);
    else
      launch_reg<T, TO, BT, 64, 64, 2, 2, 1, 1>(a, batch, st);
  }
}

// -------------------------------------- workspace: packed operands, split K --
// Copies rows of `cols` elements (source stride ld) to rows of ldp elements (a
// multiple of 16 bytes, zeros past cols): one 16-byte chunk per thread, A's
// chunks first, then B's.
struct PackArgs {
  const void* src[2];
  void* dst[2];
  long ld[2], ldp[2];
  int cols[2];
  long chunks[2];  // 16-byte chunks of each destination (0: not packed)
};
template <typename T>
__global__ __launch_bounds__(256) void gemm_pack_kernel(PackArgs p) {
  constexpr int E = VecE<T>::value;
  long c = (long)blockIdx.x * 256 + threadIdx.x;
  const int w = c >= p.chunks[0];
  if (w) c -= p.chunks[0];
  if (c >= p.chunks[w]) return;
  const long cpr = p.ldp[w] / E;
  const long r = c / cpr;
  const int k = (int)(c - r * cpr) * E;
  const u32x4_t v = ld16_first(static_cast<const T*>(p.src[w]) + r * p.ld[w] + k, p.cols[w] - k);
  *reinterpret_cast<u32x4_t*>(static_cast<T*>(p.dst[w]) + r * p.ldp[w] + k) = v;
}

// C = sum over z < splits of P[z] (+ R), in the order of z; P: [splits][M][N] fp32.
template <typename TO>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ P, int splits, GemmArgs p) {
  const long mn = (long)p.M * p.Nc;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= mn) return;
  const long r = i / p.Nc, c = i - r * p.Nc;
  float v = 0.f;
#pragma unroll 8
  for (int z = 0; z < splits; ++z) v += P[z * mn + i];
  if (p.R) v += to_f32(static_cast<const TO*>(p.R)[r * p.ldr + c]);
  static_cast<TO*>(p.C)[r * p.ldc + c] = from_f32<TO>(v);
}

// What one product does beyond a plain launch, and the workspace it takes.
struct WsPlan {
  bool pack;           // copy the operands the LDS-DMA kernel cannot take into aligned rows
  bool pack_a, pack_b;
  long kp, np;         // packed K (A, B^T) and N (B as [K, N])
  int splits, kc;      // parts of K, and K elements of a part
  size_t a_off, b_off, p_off, bytes;
};
template <typename T, bool BT>
static WsPlan plan_ws(const GemmArgs& a) {
  constexpr int E = VecE<T>::value;
  constexpr int BK = 128 / (int)sizeof(T);
  WsPlan w{};
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  w.kp = a.K;
  w.np = a.N;
  // Packing pays from two rounds of 128x128 tiles on (bf16 4001 x 4099 x 3999
  // 202 -> 146 us, 3001 x 1001 x 3003 45 -> 40; below that it depends on K: 4001 x
  // 129 x 1001, 256 tiles, 9 -> 13, 2047 x 1023 x 2049, 272 tiles, 31 -> 28); the
  // fp32 kernels are close enough to each other that it does not.  Nor does it
  // where the copies would still not suit the LDS-DMA kernel (2 GiB or more), or
  // where one row or column of tiles reads each copy once (65536 x 65 x 33 20.4
  // with copies, 8.8 without; x 129 23.9 / 20.5, x 513 42.5 / 54.1).
  if (sizeof(T) == 2 && !dma_ok<T, BT>(a) && tiles_of(a, 128, 128, 1) >= 512 && min(a.M, a.N) > 128 &&
      !unstaged<T, BT>(a, 1)) {
    const bool pa = !aligned16(a.A) || a.K % E || a.lda % E;  // (K off a vector: zeros in A, and in B^T)
    const bool pb = !aligned16(a.B) || a.ldb % E || (BT ? a.K % E : a.N % E);
    const int kp = (int)(((long)a.K + E - 1) / E * E), np = BT ? a.N : (int)(((long)a.N + E - 1) / E * E);
    GemmArgs g = a;  // the product over the packed operands (null: an aligned base)
    if (pa) g.A = nullptr, g.lda = kp;
    if (pb) g.B = nullptr, g.ldb = BT ? kp : np;
    g.N = np, g.padded = 1;
    if ((pa || pb) && dma_ok<T, BT>(g)) {
      w.pack = true, w.pack_a = pa, w.pack_b = pb;
      w.kp = kp, w.np = np;
      if (pa) w.a_off = w.bytes, w.bytes += up(sizeof(T) * (size_t)a.M * kp);
      if (pb) w.b_off = w.bytes, w.bytes += up(sizeof(T) * (BT ? (size_t)a.N : (size_t)a.K) * (BT ? kp : np));
    }
  }
  // K is split over workgroups when their tiles leave half the CUs idle and K
  // is long: parts of at least 8 K-steps, up to one workgroup per CU (bf16
  // 8 x 8064 x 64 23.9 -> 7.2 us, 16 x 4096 x 4096 15.3 -> 12.4, 1 x 8192 x
  // 8192 39 -> 31; 304 x 1024 x 256 6.4 -> 7.9, so not below 48 K-steps).
  const bool dma = w.pack || dma_ok<T, BT>(a);
  const long tiles = sizeof(T) == 2 ? tiles_of(a, 64, 64, 1) : dma ? tiles_of(a, 32, 32, 1) : tiles_of(a, 32, 64, 1);
  const int steps = (a.K + BK - 1) / BK;
  w.splits = 1;
  if (tiles <= 128 && steps >= 48) {
    const int want = (int)min(256 / tiles, (long)steps / 8), per = (steps + want - 1) / want;
    w.kc = per * BK;
    w.splits = (steps + per - 1) / per;
    if (w.splits > 1) w.p_off = w.bytes, w.bytes += up(4 * (size_t)w.splits * a.M * a.Nc);
  }
  return w;
}

// A call's workspace: whether it may use one, and `need` to ask for its size
// instead of launching.
struct Workspace {
  bool use;
  void* p;
  size_t bytes;
  size_t* need;
};

template <typename T, typename TO, bool BT>
static int gemm_dispatch(const GemmArgs& a, int batch, int variant, Workspace ws, hipStream_t st) {
  if (variant == NKL_GEMM_NAIVE) {
    launch_naive<T, TO, BT>(a, batch, st);
    return check_launch("nkl_gemm(naive)");
  }
  if (ws.use) {  // (batch 1)
    const WsPlan w = plan_ws<T, BT>(a);
    if (ws.need) return *ws.need = w.bytes, NKL_OK;
    if (w.bytes > 0) {
      if (!ws.p || ws.bytes < w.bytes)
        return set_error(NKL_EWORKSPACE, "nkl_gemm_ws: workspace of %zu bytes needed, %zu given", w.bytes, ws.bytes);
      GemmArgs g = a;
      char* base = static_cast<char*>(ws.p);
      if (w.pack) {
        constexpr int E = VecE<T>::value;
        PackArgs k{};
        if (w.pack_a) {
          k.src[0] = a.A, k.dst[0] = base + w.a_off, k.ld[0] = a.lda, k.ldp[0] = w.kp, k.cols[0] = a.K;
          k.chunks[0] = (long)a.M * (w.kp / E);
          g.A = k.dst[0], g.lda = w.kp;
        }
        if (w.pack_b) {
          k.src[1] = a.B, k.dst[1] = base + w.b_off, k.ld[1] = a.ldb, k.ldp[1] = BT ? w.kp : w.np;
          k.cols[1] = BT ? a.K : a.N;
          k.chunks[1] = BT ? (long)a.N * (w.kp / E) : (long)a.K * (w.np / E);
          g.B = k.dst[1], g.ldb = k.ldp[1];
        }
        gemm_pack_kernel<T><<<dim3((unsigned)((k.chunks[0] + k.chunks[1] + 255) / 256)), dim3(256), 0, st>>>(k);
        g.N = (int)w.np, g.padded = 1;
      }
      if (w.splits > 1) {
        GemmArgs part = g;
        part.Kall = g.K;
        part.K = w.kc;
        part.sA = w.kc;
        part.sB = BT ? w.kc : w.kc * g.ldb;
        part.C = base + w.p_off;
        part.ldc = a.Nc;
        part.sC = (long)a.M * a.Nc;
        part.R = nullptr;
        gemm_launch<T, float, BT>(part, w.splits, st);
        const long mn = (long)a.M * a.Nc;
        gemm_reduce_kernel<TO><<<dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, st>>>(
            reinterpret_cast<const float*>(base + w.p_off), w.splits, a);
      } else {
        gemm_launch<T, TO, BT>(g, 1, st);
      }
      return check_launch("nkl_gemm_ws");
    }
  }
  gemm_launch<T, TO, BT>(a, batch, st);
  return check_launch("nkl_gemm(blocked)");
}

template <typename T, typename TO>
static int gemm_layout(const GemmArgs& a, int b_trans, int batch, int variant, Workspace ws,
                       hipStream_t st) {
  return b_trans ? gemm_dispatch<T, TO, true>(a, batch, variant, ws, st)
                 : gemm_dispatch<T, TO, false>(a, batch, variant, ws, st);
}

// Checks the arguments, then launches (need null) or asks for the workspace.
static int gemm_entry(const char* fn, const void* A, const void* B, void* C, const void* R, int M, int N, int K,
                      long lda, long ldb, long ldc, long ldr, int b_trans, int batch, long strideA, long strideB,
                      long strideC, long strideR, int dtype_in, int dtype_out, int variant, Workspace ws,
                      void* stream) {
  if (M < 0 || N < 0 || K < 0 || batch < 0)
    return set_error(NKL_EINVAL, "%s: negative shape M=%d N=%d K=%d batch=%d", fn, M, N, K, batch);
  if (variant != NKL_GEMM_BLOCKED && variant != NKL_GEMM_NAIVE)
    return set_error(NKL_EINVAL, "%s: unknown variant %d", fn, variant);
  if (M == 0 || N == 0 || batch == 0) return NKL_OK;
  if (lda < K || ldc < N || (R && ldr < N) || (b_trans ? ldb < K : ldb < N))
    return set_error(NKL_EINVAL, "%s: leading dimension too small (lda=%ld ldb=%ld ldc=%ld)", fn, lda, ldb, ldc);
  if (!A || !B || (!C && !ws.need)) return set_error(NKL_EINVAL, "%s: null operand pointer", fn);
  GemmArgs a{A, B, C, R, M, N, K, lda, ldb, ldc, ldr, strideA, strideB, strideC, strideR, kEpiElem, N, 0, 0};
  hipStream_t st = (hipStream_t)stream;
#define NKL_GEMM_TYPES(ti, TI, to, TO)  \
  if (dtype_in == ti && dtype_out == to) \
  return gemm_layout<TI, TO>(a, b_trans, batch, variant, ws, st)
  NKL_GEMM_TYPES(NKL_F32, float, NKL_F32, float);
  NKL_GEMM_TYPES(NKL_BF16, bf16, NKL_BF16, bf16);
  NKL_GEMM_TYPES(NKL_BF16, bf16, NKL_F32, float);
  NKL_GEMM_TYPES(NKL_F16, f16, NKL_F16, f16);
  NKL_GEMM_TYPES(NKL_F16, f16, NKL_F32, float);
#undef NKL_GEMM_TYPES
  return set_error(NKL_EDTYPE, "%s: unsupported dtype pair (%d -> %d)", fn, dtype_in, dtype_out);
}

}  // namespace nkl

using namespace nkl;

extern "C" int nkl_gemm(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda,
                        long ldb, long ldc, long ldr, int b_trans, int batch, long strideA, long strideB,
                        long strideC, long strideR, int dtype_in, int dtype_out, int variant, void* stream) {
  return gemm_entry("nkl_gemm", A, B, C, R, M, N, K, lda, ldb, ldc, ldr, b_trans, batch, strideA, strideB, strideC,
                    strideR, dtype_in, dtype_out, variant, Workspace{}, stream);
}

extern "C" size_t nkl_gemm_workspace_bytes(const void* A, const void* B, int M, int N, int K, long lda, long ldb,
                                           int b_trans, int dtype_in, int dtype_out) {
  size_t need = 0;
  const int rc = gemm_entry("nkl_gemm_workspace_bytes", A, B, nullptr, nullptr, M, N, K, lda, ldb, N, 0, b_trans, 1, 0,
                            0, 0, 0, dtype_in, dtype_out, NKL_GEMM_BLOCKED, Workspace{true, nullptr, 0, &need},
                            nullptr);
  return rc == NKL_OK ? need : 0;
}

extern "C" int nkl_gemm_ws(const void* A, const void* B, void* C, const void* R, void* workspace,
                           size_t workspace_bytes, int M, int N, int K, long lda, long ldb, long ldc, long ldr,
                           int b_trans, int dtype_in, int dtype_out, void* stream) {
  return gemm_entry("nkl_gemm_ws", A, B, C, R, M, N, K, lda, ldb, ldc, ldr, b_trans, 1, 0, 0, 0, 0, dtype_in, dtype_out,
                    NKL_GEMM_BLOCKED, Workspace{true, workspace, workspace_bytes, nullptr}, stream);
}

extern "C" int nkl_gemm_swiglu(const void* A, const void* Bgu, void* C, int M, int N, int K, long lda, long ldb,
                               long ldc, int dtype, void* stream) {
  if (M < 0 || N < 0 || K < 0)
    return set_error(NKL_EINVAL, "nkl_gemm_swiglu: negative shape M=%d N=%d K=%d", M, N, K);
  if (dtype != NKL_BF16 && dtype != NKL_F16)
    return set_error(NKL_EDTYPE, "nkl_gemm_swiglu: only bf16 and fp16 are supported (dtype %d)", dtype);
  if (M == 0 || N == 0) return NKL_OK;
  if (N % 32 != 0) return set_error(NKL_EINVAL, "nkl_gemm_swiglu: N=%d must be a multiple of 32", N);
  if (!A || !Bgu || !C) return set_error(NKL_EINVAL, "nkl_gemm_swiglu: null operand pointer");
  if (lda < K || ldb < K || ldc < N)
    return set_error(NKL_EINVAL, "nkl_gemm_swiglu: leading dimension too small (lda=%ld ldb=%ld ldc=%ld)", lda, ldb,
                     ldc);
  if (!aligned16(A) || !aligned16(Bgu) || !aligned16(C) || K % 8 != 0 || lda % 8 != 0 || ldb % 8 != 0 ||
      ldc % 8 != 0)
    return set_error(NKL_EINVAL, "nkl_gemm_swiglu: operands must be 16-byte aligned with K and leading dimensions "
                     "multiples of 8");
  const long a_bytes = 2L * ((long)(M - 1) * lda + K), b_bytes = 2L * ((long)(2L * N - 1) * ldb + K);
  if (a_bytes >= (1L << 31) || b_bytes >= (1L << 31))
    return set_error(NKL_EINVAL, "nkl_gemm_swiglu: operands must be under 2 GiB");
  GemmArgs a{A, Bgu, C, nullptr, M, 2 * N, K, lda, ldb, ldc, 0, 0, 0, 0, 0, kEpiSwiglu, 2 * N, 0, 0};
  hipStream_t st = (hipStream_t)stream;
  // A tile whose wavefronts own 64 columns (one gate/up pair), summing the
  // K-steps in the order the separate M x N gate and up GEMMs would: in two
  // K groups where their tile has them.
  GemmArgs half = a;
  half.N = N;
  const DmaTile th = choose_tile(half, 1);
  DmaTile t = th == kT64x64K2 || th == kT64x128K2 ? kT64x128K2 : choose_tile(a, 1);
  if (t == kT64x64) t = kT64x128;
  if (t == kT64x64K2) t = kT64x128K2;
  if (t == kT256x192) t = kT256x256;
  if (dtype == NKL_F16)
    launch_dma_cols<f16, f16, true>(t, a, 1, true, st);
  else
    launch_dma_cols<bf16, bf16, true>(t, a, 1, true, st);
  return check_launch("nkl_gemm_swiglu");
}

extern "C" int nkl_gemm_gate_up(const void* A, const void* Wg, const void* Wu, void* C, int M, int N, int K, long lda,
                                long ldg, long ldu, long ldc, int dtype, void* stream) {
  if (M < 0 || N < 0 || K < 0)
    return set_error(NKL_EINVAL, "nkl_gemm_gate_up: negative shape M=%d N=%d K=%d", M, N, K);
  if (dtype != NKL_F32) return set_error(NKL_EDTYPE, "nkl_gemm_gate_up: only fp32 is supported (dtype %d)", dtype);
  if (M == 0 || N == 0) return NKL_OK;
  if (!A || !Wg || !Wu || !C) return set_error(NKL_EINVAL, "nkl_gemm_gate_up: null operand pointer");
  if (lda < K || ldg < K || ldu < K || ldc < N)
    return set_error(NKL_EINVAL, "nkl_gemm_gate_up: leading dimension too small (lda=%ld ldg=%ld ldu=%ld ldc=%ld)", lda,
                     ldg, ldu, ldc);
  if (!aligned16(A) || !aligned16(Wg) || !aligned16(Wu) || !aligned16(C) || N % 4 || K % 4 || lda % 4 || ldg % 4 ||
      ldu % 4 || ldc % 4)
    return set_error(NKL_EINVAL, "nkl_gemm_gate_up: operands must be 16-byte aligned with N, K and leading dimensions "
                     "multiples of 4");
  const long lim = (1L << 31) / 4;
  if ((M - 1) * lda + K >= lim || (N - 1) * ldg + K >= lim || (N - 1) * ldu + K >= lim || N > (1 << 29))
    return set_error(NKL_EINVAL, "nkl_gemm_gate_up: operands must be under 2 GiB");
  GemmArgs a{A, Wg, C, nullptr, M, 2 * ((N + 31) / 32 * 32), K, lda, ldg, ldc, 0, 0, 0, 0, 0, kEpiSwiglu, N, 0, 0, Wu, ldu};
  launch_f32_gate_up(a, (hipStream_t)stream);
  return check_launch("nkl_gemm_gate_up");
}

extern "C" int nkl_check_blocks(int BM, int BN) {
  if (BM < 1 || BN < 1) return set_error(NKL_EINVAL, "nkl_check_blocks: BM=%d BN=%d must be positive", BM, BN);
  if (BM * BN > 8)
    return set_error(NKL_ELIMIT,
                     "BM*BN = %d fp32 [128,512] accumulators exceed the 8 PSUM banks the blocked matmul may hold",
                     BM * BN);
  return NKL_OK;
}
