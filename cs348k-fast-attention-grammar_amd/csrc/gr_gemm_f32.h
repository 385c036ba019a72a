// gr_gemm_f32.h -- batched fp32 GEMM with a fused epilogue on the fp32 matrix
// cores of gfx950 (v_mfma_f32_32x32x2_f32), for the grammar's fp32 programs.
//
//   C[z] = act(alpha * A[z] @ B[z]) [+ R[z]]   A [M, K], B [K, N] or K-major [N, K],
//                                              C, R [M, N]
//
// The reference's programs are fp32 end to end; without this their matmul
// stages would run on the generic LDS lowering's scalar FMAs.
//
// Design (one workgroup = WGM x WGN waves = a BM x BN tile of C):
//  * Transposed form C^T = B^T A^T, as in gr_gemm.h: the MFMA "A" operand is
//    a 32-column block of B (one n per lane), the "B" operand a 32-row block
//    of A (one m per lane); the accumulators give each lane one row m of C
//    with runs of 4 consecutive n, stored as 16-byte writes.
//  * A 32x32x2 MFMA contracts two k, one per half-wave. A lane reads 4
//    consecutive k of its row of A in one 16-byte LDS read and feeds them to 4
//    MFMAs; half-wave g takes k = kb + 4g + t in MFMA t. The B operand pairs
//    the same k: 16-byte reads of a K-major B, else four 4-byte reads down a
//    column of the [BK][BN] tile.
//  * Tiles go global -> registers -> LDS (16-byte accesses), two LDS stages,
//    the next tile's loads issued before the current tile's MFMAs and one
//    barrier per k tile. Rows are padded (A and K-major B by 4 floats, a
//    [BK][BN] B by 8) so the fragment reads of the 16 or 32 lanes that the
//    LDS serves together fall on distinct banks.
//  * M, N multiples of the tile, K of BK; row strides multiples of 4 floats.
//
// Grids of few tiles (gr_gemm_f32_groups_body). An fp32 32x32x2 MFMA takes 64
// cycles, so a wave that owns a 32 x 32 block of C and all of K = 1024 is a
// serial chain of 14 us, and 32 tiles of 64 x 64 leave seven of eight CUs
// idle. There a workgroup takes one 32 x 32 block instead and its four waves a
// quarter of K each, merged through LDS. One wave per SIMD and no operand
// shared between waves, so nothing is staged: fragments come straight from
// global memory into registers, two k tiles ahead. 256 x 512, K = 1024: 25.1 us
// on 32 workgroups of 64 x 64, 7.1 us on 128 of 32 x 32; 256 x 1024, K = 512:
// 14.1 -> 5.2; 512 x 1024, K = 1024: 25.6 -> 17; 1024 x 1024 (256 tiles of 64 x
// 64) 26 -> 33, so full grids keep their tile.
#pragma once
#include "gr_gemm.h"

template <int BM, int BN, int BK, int WGM, int WGN, bool B_KMAJOR>
struct gr_gemm_f32_cfg {
  static constexpr int NT = WGM * WGN * 64;
  static constexpr int WM = BM / WGM, WN = BN / WGN;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int A_LD = BK + 4;                          // floats per LDS row of A
  static constexpr int B_LD = B_KMAJOR ? BK + 4 : BN + 8;      // of B^T [BN][BK] or B [BK][BN]
  static constexpr int A_FLOATS = BM * A_LD;
  static constexpr int B_FLOATS = (B_KMAJOR ? BN : BK) * B_LD;
  static constexpr int STAGE = (A_FLOATS + B_FLOATS) * 4;
  static constexpr int LDS = 2 * STAGE;
  static constexpr int A_VEC = BM * BK / 4;                    // 16-byte pieces per tile
  static constexpr int B_VEC = BN * BK / 4;
  static constexpr int A_PER = (A_VEC + NT - 1) / NT;
  static constexpr int B_PER = (B_VEC + NT - 1) / NT;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "each wave owns whole 32x32 blocks");
  static_assert(BK % 8 == 0, "k tile: whole groups of 8 (4 MFMAs of 2)");
};

template <int BM, int BN, int BK, int WGM, int WGN, bool B_KMAJOR, int EPI>
__device__ __forceinline__ void gr_gemm_f32_tile_body(const gr_gemm_args& a, char* lds) {
  typedef gr_gemm_f32_cfg<BM, BN, BK, WGM, WGN, B_KMAJOR> G;
  constexpr int NT = G::NT, TM = G::TM, TN = G::TN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, g = lane >> 5;
  const int wm = wave / WGN, wn = wave % WGN;
  const int tiles_n = a.N / BN;
  const int bid = gr_xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int tm = bid / tiles_n, tn = bid % tiles_n;
  const long long z = blockIdx.y;
  // split K (ksplit > 1): this workgroup's part of the contraction, its
  // partial product written to its own C slice (gr_gemm_f32_reduce_body sums them)
  const int kpart = a.K / a.ksplit, k0 = (int)blockIdx.z * kpart;
  const float* A = static_cast<const float*>(a.a) + z * a.a_sb + (long long)tm * BM * a.a_sm + k0;
  const float* B = static_cast<const float*>(a.b) + z * a.b_sb +
                   (B_KMAJOR ? (long long)tn * BN * a.b_s + k0 : (long long)tn * BN + (long long)k0 * a.b_s);
  float* C = static_cast<float*>(a.c) + blockIdx.z * a.c_sz + z * a.c_sb + (long long)tm * BM * a.c_sm +
             (long long)tn * BN;

  gr_f32x16 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = (gr_f32x16)(0.f);

  // global -> register staging of one k tile, then register -> LDS
  gr_f32x4 ra[G::A_PER], rb[G::B_PER];
  auto gload = [&](int kt) {
#pragma unroll
    for (int i = 0; i < G::A_PER; ++i) {
      const int v = tid + i * NT;
      if (G::A_VEC % NT == 0 || v < G::A_VEC) {
        const int row = v / (BK / 4), c4 = v % (BK / 4);
        ra[i] = *reinterpret_cast<const gr_f32x4*>(A + (long long)row * a.a_sm + (long long)kt * BK + c4 * 4);
      }
    }
#pragma unroll
    for (int i = 0; i < G::B_PER; ++i) {
      const int v = tid + i * NT;
      if (G::B_VEC % NT == 0 || v < G::B_VEC) {
        if constexpr (B_KMAJOR) {
          const int row = v / (BK / 4), c4 = v % (BK / 4);          // row = n
          rb[i] = *reinterpret_cast<const gr_f32x4*>(B + (long long)row * a.b_s + (long long)kt * BK + c4 * 4);
        } else {
          const int row = v / (BN / 4), c4 = v % (BN / 4);          // row = k
          rb[i] = *reinterpret_cast<const gr_f32x4*>(B + ((long long)kt * BK + row) * a.b_s + c4 * 4);
        }
      }
    }
  };
  auto sstore = [&](char* st) {
    float* la = reinterpret_cast<float*>(st);
    float* lb = la + G::A_FLOATS;
#pragma unroll
    for (int i = 0; i < G::A_PER; ++i) {
      const int v = tid + i * NT;
      if (G::A_VEC % NT == 0 || v < G::A_VEC)
        *reinterpret_cast<gr_f32x4*>(la + (v / (BK / 4)) * G::A_LD + (v % (BK / 4)) * 4) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < G::B_PER; ++i) {
      const int v = tid + i * NT;
      if (G::B_VEC % NT == 0 || v < G::B_VEC) {
        constexpr int CPR = B_KMAJOR ? BK / 4 : BN / 4;
        *reinterpret_cast<gr_f32x4*>(lb + (v / CPR) * G::B_LD + (v % CPR) * 4) = rb[i];
      }
    }
  };
  auto mma_tile = [&](const char* st) {
    const float* la = reinterpret_cast<const float*>(st);
    const float* lb = la + G::A_FLOATS;
#pragma unroll
    for (int kb = 0; kb < BK; kb += 8) {
      gr_f32x4 af[TM], bf[TN];
#pragma unroll
      for (int j = 0; j < TM; ++j)
        af[j] = *reinterpret_cast<const gr_f32x4*>(la + (wm * G::WM + j * 32 + l32) * G::A_LD + kb + 4 * g);
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int n = wn * G::WN + i * 32 + l32;
        if constexpr (B_KMAJOR) {
          bf[i] = *reinterpret_cast<const gr_f32x4*>(lb + n * G::B_LD + kb + 4 * g);
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) bf[i][t] = lb[(kb + 4 * g + t) * G::B_LD + n];
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[i][t], af[j][t], acc[i][j], 0, 0, 0);
    }
  };

  const int nk = kpart / BK;
  gload(0);
  sstore(lds);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk) gload(kt + 1);
    mma_tile(lds + (kt & 1) * G::STAGE);
    if (kt + 1 < nk) sstore(lds + ((kt + 1) & 1) * G::STAGE);
    __syncthreads();
  }

  // lane (l32, g) of block (i, j): row m = wm*WM + 32j + l32, columns
  // n = wn*WN + 32i + 8q + 4g + (0..3) in accumulators 4q..4q+3
  // (a null residual adds nothing: a split stage whose sum is taken by its
  // consumer adds R in its first K part only)
  const float* R = ((EPI & GR_EPI_RES) && a.r) ? static_cast<const float*>(a.r) + z * a.r_sb +
                                                     (long long)tm * BM * a.r_sm + (long long)tn * BN
                                               : nullptr;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int row = wm * G::WM + j * 32 + l32;
    float* crow = C + (long long)row * a.c_sm;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = wn * G::WN + i * 32 + 8 * q + 4 * g;
        gr_f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = gr_epilogue<EPI>(a.alpha * acc[i][j][4 * q + e]);
        if constexpr ((EPI & GR_EPI_RES) != 0) {
          if (R) w += *reinterpret_cast<const gr_f32x4*>(R + (long long)row * a.r_sm + col);
        }
        *reinterpret_cast<gr_f32x4*>(crow + col) = w;
      }
  }
}

// LDS bytes of the k-group body: the four waves' 32 x 32 sums.
constexpr int GR_GEMM_F32_GROUPS_LDS = 4 * 32 * 32 * 4;

// One 32 x 32 block of C per workgroup of four waves; wave kg takes k tiles kg,
// kg + 4, ... of 16 (8 where KT is). K a multiple of KT; the grid covers
// (M / 32) (N / 32) blocks; no K split.
template <int KT, bool B_KMAJOR, int EPI>
__device__ __forceinline__ void gr_gemm_f32_groups_body(const gr_gemm_args& a, char* lds) {
  constexpr int BK = KT > 16 ? 16 : KT;
  constexpr int KB = BK / 8;                   // 8-deep steps per k tile
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_n = a.N / 32;
  const int bid = gr_xcd_remap_any((int)blockIdx.x, (int)gridDim.x);
  const int tm = bid / tiles_n, tn = bid % tiles_n;
  const long long z = blockIdx.y;
  // lane (l32, g): row l32 of A's block, column l32 of B's, k = 8 kb + 4 g + t.
  // A wave-uniform base per k tile and 32-bit lane offsets kept for the whole
  // loop: the 64-bit products of per-load addresses cost as much issue time
  // as the MFMAs (105 cycles per MFMA instead of 64).
  const char* A = reinterpret_cast<const char*>(static_cast<const float*>(a.a) + z * a.a_sb + (long long)tm * 32 * a.a_sm);
  const char* B = reinterpret_cast<const char*>(
      static_cast<const float*>(a.b) + z * a.b_sb + (B_KMAJOR ? (long long)tn * 32 * a.b_s : (long long)tn * 32));
  const long long b_tile = (B_KMAJOR ? 1LL : a.b_s) * BK * 4;        // bytes
  const unsigned int a_off = (unsigned int)((l32 * a.a_sm + 4 * g) * 4);
  unsigned int b_off[B_KMAJOR ? 1 : KB * 4];
  if constexpr (B_KMAJOR) {
    b_off[0] = (unsigned int)((l32 * a.b_s + 4 * g) * 4);
  } else {
#pragma unroll
    for (int i = 0; i < KB * 4; ++i) b_off[i] = (unsigned int)(((8 * (i / 4) + 4 * g + i % 4) * a.b_s + l32) * 4);
  }
  gr_f32x16 acc[2] = {(gr_f32x16)(0.f), (gr_f32x16)(0.f)};   // two chains: consecutive MFMAs are independent

  auto load = [&](int kt, gr_f32x4 (&fa)[KB], gr_f32x4 (&fb)[KB]) {
    const char* at = A + (long long)kt * (BK * 4);
    const char* bt = B + kt * b_tile;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      fa[kb] = *reinterpret_cast<const gr_f32x4*>(at + a_off + kb * 32);
      if constexpr (B_KMAJOR) {
        fb[kb] = *reinterpret_cast<const gr_f32x4*>(bt + b_off[0] + kb * 32);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) fb[kb][t] = *reinterpret_cast<const float*>(bt + b_off[kb * 4 + t]);
      }
    }
  };
  auto mma = [&](const gr_f32x4 (&fa)[KB], const gr_f32x4 (&fb)[KB]) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc[t & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[kb][t], fa[kb][t], acc[t & 1], 0, 0, 0);
  };
  // A ring of NB register buffers, NB - 1 tiles in flight. The loop over whole
  // turns of the ring has no branch (loads past the wave's last tile repeat
  // it) and its loads stay ahead of the MFMAs they precede, so that the wait
  // for a buffer is a count of the later loads. 16-deep tiles in three buffers:
  // 256 x 512 x 1024 in 7.1 us, against 7.9 / 8.1 / 9.1 for 32-deep ones in
  // two, three, four and 7.2 / 7.5 for 16-deep ones in two, four.
  constexpr int NB = 3;
  const int nk = a.K / BK, n = (nk - kg + 3) / 4, last = kg + (n - 1) * 4;   // this wave's tiles: n
  gr_f32x4 fa[NB][KB], fb[NB][KB];
  if (n > 0) {
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) load(gr_imin(kg + 4 * i, last), fa[i], fb[i]);
    int kt = kg;
    for (int turn = n / NB; turn > 0; --turn, kt += 4 * NB) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        load(gr_imin(kt + 4 * (i + NB - 1), last), fa[(i + NB - 1) % NB], fb[(i + NB - 1) % NB]);
        __builtin_amdgcn_sched_barrier(0);
        mma(fa[i], fb[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int i = 0; i < NB - 1; ++i)
      if (i < n % NB) mma(fa[i], fb[i]);
  }

  // wave q finishes quad q (columns 8q + 4g + 0..3 of the lane's row): the
  // groups' sums in order
  gr_f32x4* x = reinterpret_cast<gr_f32x4*>(lds);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    gr_f32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = acc[0][4 * q + e] + acc[1][4 * q + e];
    x[(kg * 4 + q) * 64 + lane] = w;
  }
  __syncthreads();
  gr_f32x4 sum = x[kg * 64 + lane];
#pragma unroll
  for (int k = 1; k < 4; ++k) sum += x[(k * 4 + kg) * 64 + lane];
  const long long row = tm * 32 + l32, col = tn * 32 + 8 * kg + 4 * g;
  gr_f32x4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = gr_epilogue<EPI>(a.alpha * sum[e]);
  if constexpr ((EPI & GR_EPI_RES) != 0)
    w += *reinterpret_cast<const gr_f32x4*>(static_cast<const float*>(a.r) + z * a.r_sb + row * a.r_sm + col);
  *reinterpret_cast<gr_f32x4*>(static_cast<float*>(a.c) + z * a.c_sb + row * a.c_sm + col) = w;
}

// A rendered stage: the program's tile, or (a.kgroups, a constant there) its
// 32 x 32 blocks on the k-group body, one workgroup of 256 threads each.
template <int BM, int BN, int BK, int WGM, int WGN, bool B_KMAJOR, int EPI>
__device__ __forceinline__ void gr_gemm_f32_body(const gr_gemm_args& a, char* lds) {
  if (a.kgroups == 4) gr_gemm_f32_groups_body<BK, B_KMAJOR, EPI>(a, lds);
  else gr_gemm_f32_tile_body<BM, BN, BK, WGM, WGN, B_KMAJOR, EPI>(a, lds);
}

// The second launch of a split-K GEMM: C = act(alpha * sum_s P_s) [+ R] over
// the ksplit partial products P_s (at ws + s * ws_sz, laid out as C with
// row stride N, batch stride M N). One thread per 4 consecutive columns of
// one row; the grid covers batch * M * N / 4 threads in workgroups of 256.
template <int EPI>
__device__ __forceinline__ void gr_gemm_f32_reduce_body(const gr_gemm_args& a, const float* ws, int ksplit,
                                                        long long ws_sz, int batch) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = (long long)a.M * a.N / 4;
  if (idx >= per * batch) return;
  const long long z = idx / per, e4 = (idx % per) * 4;
  const int row = (int)(e4 / a.N), col = (int)(e4 % a.N);
  gr_f32x4 sum = (gr_f32x4)(0.f);
  for (int s = 0; s < ksplit; ++s)
    sum += *reinterpret_cast<const gr_f32x4*>(ws + s * ws_sz + z * a.M * (long long)a.N + e4);
  gr_f32x4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = gr_epilogue<EPI>(a.alpha * sum[e]);
  if constexpr ((EPI & GR_EPI_RES) != 0)
    w += *reinterpret_cast<const gr_f32x4*>(static_cast<const float*>(a.r) + z * a.r_sb + (long long)row * a.r_sm + col);
  *reinterpret_cast<gr_f32x4*>(static_cast<float*>(a.c) + z * a.c_sb + (long long)row * a.c_sm + col) = w;
}

template <int BM, int BN, int BK, int WGM, int WGN, bool B_KMAJOR, int EPI>
__global__ __launch_bounds__(WGM * WGN * 64) void gr_gemm_f32_kernel(gr_gemm_args a) {
  extern __shared__ __attribute__((aligned(16))) char gr_lds[];
  gr_gemm_f32_tile_body<BM, BN, BK, WGM, WGN, B_KMAJOR, EPI>(a, gr_lds);
}

template <int BK, bool B_KMAJOR, int EPI>
__global__ __launch_bounds__(256) void gr_gemm_f32_groups_kernel(gr_gemm_args a) {
  extern __shared__ __attribute__((aligned(16))) char gr_lds[];
  gr_gemm_f32_groups_body<BK, B_KMAJOR, EPI>(a, gr_lds);
}
