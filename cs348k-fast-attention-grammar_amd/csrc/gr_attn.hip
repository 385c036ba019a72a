// gr_attn.hip -- prebuilt instances of the hand-written CDNA4 attention
// forward (gr_flash_fwd.h) behind gr_attn_fwd(), plus the MFMA layout self-test.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>

#include "gr_attn_groups.h"
#include "gr_flash_decode.h"
#include "gr_flash_w2.h"
#include "gr_flash_w2h.h"
#include "gr_host.h"
#include "grammar_rt.h"

namespace {

// ragged: the last query tile of a head may be part-filled (N a multiple of BN
// still), as picked plans launch it.
template <class T, int D, int BN, int NW, int QB, bool CAUSAL, bool KT, bool PIPE = false>
int launch_flash(const gr_attn_args& a, hipStream_t st, bool ragged = false) {
  constexpr int BM = NW * QB * 32;
  constexpr int LDS = gr_flash_lds<D, BN>::BYTES;
  // K/V tiles go straight into LDS when they give every thread the same
  // number of 16-byte chunks (D * BN / 8 per tile), else through registers.
  constexpr bool DIRECT = (D * BN / 8) % (NW * 64) == 0;
  if ((!ragged && a.N % BM != 0) || a.N % BN != 0)
    return gr::fail(GR_E_ARG, "gr_attn_fwd: N=%d must be a multiple of block_m=%d and block_n=%d", a.N, BM, BN);
  const long long nblk = (long long)a.B * a.H * ((a.N + BM - 1) / BM);
  if (nblk <= 0 || nblk > 0x7fffffffLL) return gr::fail(GR_E_ARG, "gr_attn_fwd: grid size %lld out of range", nblk);
  hipLaunchKernelGGL((gr_flash_fwd_kernel<T, D, BN, NW, QB, CAUSAL, KT, PIPE, true, DIRECT>), dim3((unsigned)nblk),
                     dim3(NW * 64), LDS, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd launch");
}

// fp16, D = 64, non-causal, 256 x 64 tiles (with or without the training
// forward's log-sum-exp): two waves per SIMD with the hand-ordered main loop
// (gr_flash_w2.h); N a multiple of 256.
template <bool KT>
int launch_w2(const gr_attn_args& a, hipStream_t st) {
  const long long nblk = (long long)a.B * a.H * (a.N / 256);
  if (nblk <= 0 || nblk > 0x7fffffffLL) return gr::fail(GR_E_ARG, "gr_attn_fwd: grid size %lld out of range", nblk);
  hipLaunchKernelGGL((gr_flash_w2_kernel<KT>), dim3((unsigned)nblk), dim3(512), GR_FLASH_W2_LDS, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd launch");
}

// fp16 or bf16, D = 128, K transposed, causal or not, 256 x 64 tiles without
// the training forward's log-sum-exp: two waves per SIMD with the
// hand-ordered main loop (gr_flash_w2h.h); N a multiple of 256.
template <class T, bool CAUSAL>
int launch_w2h(const gr_attn_args& a, hipStream_t st) {
  const long long nblk = (long long)a.B * a.H * (a.N / 256);
  if (nblk <= 0 || nblk > 0x7fffffffLL) return gr::fail(GR_E_ARG, "gr_attn_fwd: grid size %lld out of range", nblk);
  hipLaunchKernelGGL((gr_flash_w2h_kernel<T, CAUSAL>), dim3((unsigned)nblk), dim3(512), GR_FLASH_W2H_LDS, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd launch");
}

// The shape of a workgroup for a call that names no tile: nw waves of 32
// queries x kg key groups (gr_attn_groups.h), bn keys per tile.
//
// Modelled time of a launch: t0 + max(lat x iterations of the longest
// workgroup, thr x iterations per CU) + t1 x workgroups per CU, with `thr` the
// us per iteration that a CU sustains and `lat` the us that one workgroup
// alone takes. The constants are fitted to 2,300 launches (B H 1-64, N 64-4096,
// both head dims, fp16 and bf16, causal or not); the pick is within 0.9 % of
// the fastest shape (geometric mean, 19 % at worst of those) and takes 0.77x
// the time of the largest tile that divides N, which ran before. The 256-query
// tile that divides N is preferred within the model's error (5 %).
struct AttnShape {
  int nw, kg, bn;
  double lat, thr, t0, t1;
};
constexpr AttnShape kShapes64[] = {
    {1, 4, 32, 0.608, 0.432, 3.07, 1.13}, {1, 8, 32, 0.903, 1.027, 3.41, 1.77}, {2, 2, 64, 0.842, 0.621, 2.79, 1.23},
    {4, 2, 64, 1.175, 1.204, 3.05, 0.81}, {2, 1, 64, 0.735, 0.297, 2.12, 1.35}, {4, 1, 64, 0.772, 0.560, 2.78, 0.62},
    {8, 1, 64, 1.044, 1.081, 2.76, 0.83},
};
constexpr AttnShape kShapes128[] = {
    {2, 4, 32, 1.297, 1.333, 3.92, 1.37}, {4, 2, 64, 1.989, 1.990, 2.50, 1.81}, {2, 1, 64, 1.287, 0.704, 3.50, 0.67},
    {4, 1, 64, 1.129, 1.000, 3.05, 0.83}, {8, 1, 64, 1.665, 1.733, 3.73, 0.27},
};
// 128 x 128 at D = 64 (compiled for whole query tiles), non-causal: 17 heads at
// N 2432 43.2 us, 45.1 on 128 x 64 and 46.4 on 64 x 64
constexpr AttnShape kShape128x128 = {4, 1, 128, 1.26, 1.03, 3.1, 0.75};
// the two-wave bodies at 256 x 64 (gr_flash_w2.h, gr_flash_w2h.h)
constexpr AttnShape kShapeW2 = {8, 1, 64, 0.653, 0.961, 0.46, 1.19};
constexpr AttnShape kShapeW2h = {8, 1, 64, 1.080, 1.585, 2.61, 0.71};

// two_wave: a two-wave body takes the 256 x 64 tile of this call.
AttnShape pick_shape(int D, bool causal, bool two_wave, long long heads, int N) {
  const int cus = gr::cu_count() > 0 ? gr::cu_count() : 256;
  AttnShape best = {0, 0, 0, 0, 0, 0, 0};
  double best_t = 1e30;
  auto consider = [&](AttnShape s) {
    const int bm = 32 * s.nw;
    const double w = (double)heads * ((N + bm - 1) / bm), iters = ((N + s.bn - 1) / s.bn + s.kg - 1) / s.kg;
    double mean = iters, rounds = (double)(long long)((w + cus - 1) / cus);
    // 64 x 64 at D = 64, non-causal: a CU's first two workgroups of two waves
    // share SIMDs (9 heads, N 2432: 44.9 us for 342 workgroups), and a fifth
    // waits for LDS (26 heads, N 2944: 91 us for 1,196)
    if (!causal && D == 64 && s.nw == 2 && s.kg == 1) {
      if (w > cus) s.lat = 1.08;
      if (w > 4. * cus) s.thr = 0.36;
    }
    if (causal) {              // longest first, so a part round costs about a quarter
      mean *= 0.5 + 0.5 * bm / (N > bm ? N : bm);
      rounds = w <= cus ? 1. : w / cus + 0.25;
    }
    const double alone = iters * s.lat, shared = rounds * mean * s.thr;
    double t = s.t0 + (alone > shared ? alone : shared) + s.t1 * rounds;
    if (s.nw == 8 && N % 256 == 0) t *= 0.95;
    // Many short workgroups of 64 x 64: up to five are resident on a CU and
    // hide each other's start and end, which t0 and t1 count in full, while a
    // larger tile that does not divide N is part empty (200 heads, N 320, bf16:
    // 10.1 us, 13.1 on 128 x 64; 300 heads, N 192, causal 8.4 and 10.8).
    if (D == 64 && s.nw == 2 && s.kg == 1 && w > 3. * cus && iters <= 7 && N % 128 == 64) t *= 0.8;
    // 64 queries x 2 groups take 64 KiB of LDS, so from two workgroups per CU on
    // the rest wait (12 heads, N 4096, bf16: 75 us, 66 on 256 x 128)
    if (!causal && D == 64 && s.nw == 2 && s.kg == 2 && w > 2. * cus) t *= 1.1;
    if (t < best_t) {
      best_t = t;
      best = s;
    }
  };
  if (D == 64)
    for (const AttnShape& s : kShapes64)
      if (!(two_wave && s.nw == 8)) consider(s);
  if (D == 64 && !causal && N % 256 == 128) consider(kShape128x128);
  if (D == 128)
    for (const AttnShape& s : kShapes128)
      if (!(two_wave && s.nw == 8)) consider(s);
  if (two_wave) consider(D == 64 ? kShapeW2 : kShapeW2h);
  return best;
}

// The picked shape of a call (N a multiple of 64).
AttnShape pick_call(int dtype, int D, bool causal, bool kt, bool train, long long heads, int N) {
  const bool w2 = dtype == GR_F16 && D == 64 && !causal, w2h = D == 128 && kt && !train;
  return pick_shape(D, causal, N % 256 == 0 && (w2 || w2h), heads, N);
}

// Tile configurations compiled into the library: (block_m, block_n) ->
// (waves, query blocks per wave, key tile). One wave per 32 queries.
// block_m = block_n = 0 runs the picked shape (N a multiple of 64); where that
// is the 256-query tile and it divides N, and where only one of the two is 0,
// the zero ones are the largest tiles that divide N (256 x 128 at D = 64, 256
// x 64 at D = 128), except 256 x 64 where the two-wave body of gr_flash_w2.h
// applies (fp16, D = 64, non-causal, N a multiple of 256).
template <class T, int D, bool CAUSAL, bool KT>
int dispatch_tiles(const gr_attn_args& a, int bm, int bn, hipStream_t st) {
  constexpr bool W2 = gr_is_same<T, _Float16>::value && D == 64 && !CAUSAL;
  if (bm == 0 && bn == 0 && a.N % 64 == 0) {
    constexpr int DT = gr_is_same<T, _Float16>::value ? GR_F16 : GR_BF16;
    const AttnShape s = pick_call(DT, D, CAUSAL, KT, a.lse != nullptr, (long long)a.B * a.H, a.N);
    if (s.kg > 1) return gr::launch_flash_groups(a, DT, D, CAUSAL, KT, s.nw, s.kg, st);
    if constexpr (D == 64 && !CAUSAL)
      if (s.bn == 128) return launch_flash<T, D, 128, 4, 1, CAUSAL, KT>(a, st);
    if (s.nw == 2) return launch_flash<T, D, 64, 2, 1, CAUSAL, KT>(a, st, true);
    if (s.nw == 4) return launch_flash<T, D, 64, 4, 1, CAUSAL, KT>(a, st, true);
    if (a.N % 256 != 0) return launch_flash<T, D, 64, 8, 1, CAUSAL, KT>(a, st, true);
  }
  if (bm == 0) bm = a.N % 256 == 0 ? 256 : a.N % 128 == 0 ? 128 : 64;
  if (bn == 0) bn = (W2 && bm == 256 && a.N % 256 == 0) ? 64 : (D == 64 && a.N % 128 == 0) ? 128 : a.N % 64 == 0 ? 64 : 32;
  if constexpr (W2)
    if (bm == 256 && bn == 64 && a.N % 256 == 0 && a.Nq == a.N) return launch_w2<KT>(a, st);
  if constexpr (D == 128 && KT)
    if (bm == 256 && bn == 64 && a.lse == nullptr && a.N % 256 == 0 && a.Nq == a.N) return launch_w2h<T, CAUSAL>(a, st);
  if (bm == 256 && bn == 64) return launch_flash<T, D, 64, 8, 1, CAUSAL, KT>(a, st);
  if (bm == 256 && bn == 32) return launch_flash<T, D, 32, 8, 1, CAUSAL, KT>(a, st);
  if (bm == 128 && bn == 64) return launch_flash<T, D, 64, 4, 1, CAUSAL, KT>(a, st);
  if (bm == 128 && bn == 32) return launch_flash<T, D, 32, 4, 1, CAUSAL, KT>(a, st);
  if (bm == 64 && bn == 64) return launch_flash<T, D, 64, 2, 1, CAUSAL, KT>(a, st);
  if (bm == 64 && bn == 32) return launch_flash<T, D, 32, 2, 1, CAUSAL, KT>(a, st);
  // block_m = 129 / 257 select the software-pipelined schedule (128 / 256 queries).
  if (bm == 129 && bn == 64) return launch_flash<T, D, 64, 4, 1, CAUSAL, KT, true>(a, st);
  if (bm == 129 && bn == 32) return launch_flash<T, D, 32, 4, 1, CAUSAL, KT, true>(a, st);
  if (bm == 257 && bn == 64) return launch_flash<T, D, 64, 8, 1, CAUSAL, KT, true>(a, st);
  if (bm == 257 && bn == 32) return launch_flash<T, D, 32, 8, 1, CAUSAL, KT, true>(a, st);
  if constexpr (D == 64) {
    if (bm == 256 && bn == 128) return launch_flash<T, D, 128, 8, 1, CAUSAL, KT>(a, st);
    if (bm == 128 && bn == 128) return launch_flash<T, D, 128, 4, 1, CAUSAL, KT>(a, st);
    if (bm == 129 && bn == 128) return launch_flash<T, D, 128, 4, 1, CAUSAL, KT, true>(a, st);
  }
  return gr::fail(GR_E_ARG, "gr_attn_fwd: unsupported tile (block_m=%d, block_n=%d) for D=%d", bm, bn, D);
}

// fp16 with scale log2(e) > 1 (Q as given, every score scaled on the VALU):
// one tile, 64 queries x 32 keys (two waves).
template <int D, bool CAUSAL, bool KT>
int launch_unscaled_q(const gr_attn_args& a, hipStream_t st) {
  constexpr int BM = 64, BN = 32, NW = 2;
  constexpr bool DIRECT = (D * BN / 8) % (NW * 64) == 0;
  constexpr int LDS = gr_flash_lds<D, BN>::BYTES;
  if (a.N % BM != 0)
    return gr::fail(GR_E_ARG, "gr_attn_fwd: fp16 with scale * log2(e) > 1 needs N=%d a multiple of 64", a.N);
  const long long nblk = (long long)a.B * a.H * (a.N / BM);
  if (nblk <= 0 || nblk > 0x7fffffffLL) return gr::fail(GR_E_ARG, "gr_attn_fwd: grid size %lld out of range", nblk);
  hipLaunchKernelGGL((gr_flash_fwd_kernel<_Float16, D, BN, NW, 1, CAUSAL, KT, false, true, DIRECT, false, false>),
                     dim3((unsigned)nblk), dim3(NW * 64), LDS, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd launch");
}

int dispatch_unscaled_q(const gr_attn_args& a, int D, bool causal, bool kt, int bm, int bn, hipStream_t st) {
  if ((bm != 0 && bm != 64) || (bn != 0 && bn != 32))
    return gr::fail(GR_E_ARG, "gr_attn_fwd: fp16 with scale * log2(e) > 1 runs the 64 x 32 tile only (asked for %d x %d)",
                    bm, bn);
#define GR_CASE(DD, C, K) \
  if (D == DD && causal == C && kt == K) return launch_unscaled_q<DD, C, K>(a, st);
  GR_CASE(64, false, false)
  GR_CASE(64, false, true)
  GR_CASE(64, true, false)
  GR_CASE(64, true, true)
  GR_CASE(128, false, false)
  GR_CASE(128, false, true)
  GR_CASE(128, true, false)
  GR_CASE(128, true, true)
#undef GR_CASE
  return gr::fail(GR_E_ARG, "gr_attn_fwd: head dim D=%d unsupported (64 or 128)", D);
}

template <class T>
int dispatch_shape(const gr_attn_args& a, int D, bool causal, bool kt, int bm, int bn, hipStream_t st) {
#define GR_CASE(DD, C, K)                                                          \
  if (D == DD && causal == C && kt == K) return dispatch_tiles<T, DD, C, K>(a, bm, bn, st);
  GR_CASE(64, false, false)
  GR_CASE(64, false, true)
  GR_CASE(64, true, false)
  GR_CASE(64, true, true)
  GR_CASE(128, false, false)
  GR_CASE(128, false, true)
  GR_CASE(128, true, false)
  GR_CASE(128, true, true)
#undef GR_CASE
  return gr::fail(GR_E_ARG, "gr_attn_fwd: head dim D=%d unsupported (64 or 128)", D);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Merge of the key-split partials: one wave per (head, query) row.
// m_s are the parts' reference maxima (score units), l_s their row sums:
// O = sum_s w_s O_s / sum_s w_s l_s with w_s = 2^((m_s - max_s m_s) c).
// Bound by latency. SPREAD (many parts): a wave per row; lane s holds part s's
// (m, l), so the weights of 64 parts take one load, and its 64 / (D / 4) groups
// of lanes take every such part of O, 16 bytes per lane. Else: a group of
// lanes per row, looping over the few parts. One thread per 8 columns looping
// over all parts took 7.5 us for 640 rows of 11 parts at D = 64 (here 3.4) and
// 16 us for 40 rows of 32.
template <class T, int D, bool SPREAD>
__global__ __launch_bounds__(256) void gr_attn_combine_kernel(const float* __restrict__ po, const float* __restrict__ pml,
                                                              T* o, long long o_sb, long long o_sh, long long o_sn,
                                                              int B, int H, int Nq, int S, float c) {
  constexpr int CH = D / 4, GRP = 64 / CH;
  const int lane = threadIdx.x & 63, ch = lane % CH, grp = lane / CH;
  const long long rows = (long long)B * H * Nq;                 // rows per part
  const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const long long row = SPREAD ? wave : wave * GRP + grp;       // (b*H + h) * Nq + q
  if (row >= rows) return;
  auto part_ml = [&](int s) {
    return s < S ? *reinterpret_cast<const gr_f32x2*>(pml + (s * rows + row) * 2) : (gr_f32x2){-GR_INF, 0.f};
  };
  float mx = -GR_INF, L = 0.f;
  gr_f32x4 acc = (gr_f32x4)(0.f);
  if constexpr (SPREAD) {
    for (int s0 = 0; s0 < S; s0 += 64) mx = fmaxf(mx, part_ml(s0 + lane)[0]);
    mx = gr_wave_max(mx);
    const float base = mx == -GR_INF ? 0.f : mx;
    for (int s0 = 0; s0 < S; s0 += 64) {
      const gr_f32x2 ml = part_ml(s0 + lane);
      const float w = gr_exp2((ml[0] - base) * c);
      L += w * ml[1];
      const int n = gr_imin(S - s0, 64);
#pragma unroll 4
      for (int s = 0; s < n; s += GRP) {
        const int p = gr_imin(s + grp, n - 1);                  // past the last: its copy, not added
        const float wp = __shfl(w, p, 64);
        const gr_f32x4 v = *reinterpret_cast<const gr_f32x4*>(po + ((s0 + p) * rows + row) * D + ch * 4);
        if (s + grp < n) acc += wp * v;
      }
    }
    L = gr_wave_sum(L);
#pragma unroll
    for (int off = CH; off < 64; off <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
    if (grp != 0) return;
  } else {
    gr_f32x2 ml[4];            // at most four parts, all loads ahead of the first use
    gr_f32x4 v[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ml[s] = part_ml(s);
      v[s] = *reinterpret_cast<const gr_f32x4*>(po + (gr_imin(s, S - 1) * rows + row) * D + ch * 4);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) mx = fmaxf(mx, ml[s][0]);
    const float base = mx == -GR_INF ? 0.f : mx;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float w = gr_exp2((ml[s][0] - base) * c);
      if (s < S) {
        L += w * ml[s][1];
        acc += w * v[s];
      }
    }
  }
  const float inv = 1.0f / L;
  const int q = (int)(row % Nq), bh = (int)(row / Nq), b = bh / H, h = bh % H;
  *reinterpret_cast<gr_u32x2*>(o + b * o_sb + h * o_sh + (long long)q * o_sn + ch * 4) =
      (gr_u32x2){gr_pack2f<T>(acc[0] * inv, acc[1] * inv), gr_pack2f<T>(acc[2] * inv, acc[3] * inv)};
}

template <class T, int D>
int launch_combine(const gr_attn_args& a, int S, hipStream_t st) {
  const long long rows = (long long)a.B * a.H * a.Nq;
  const long long waves = S > 4 ? rows : (rows * (D / 4) + 63) / 64;
  const dim3 grid((unsigned)((waves + 3) / 4));
  if (S > 4)
    hipLaunchKernelGGL((gr_attn_combine_kernel<T, D, true>), grid, dim3(256), 0, st, a.part_o, a.part_ml,
                       static_cast<T*>(a.o), a.o_sb, a.o_sh, a.o_sn, a.B, a.H, a.Nq, S, a.scale_log2);
  else
    hipLaunchKernelGGL((gr_attn_combine_kernel<T, D, false>), grid, dim3(256), 0, st, a.part_o, a.part_ml,
                       static_cast<T*>(a.o), a.o_sb, a.o_sh, a.o_sn, a.B, a.H, a.Nq, S, a.scale_log2);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_decode combine launch");
}

template <class T, int D, int BN, int NW, bool SPLIT, bool PRESCALE = true, int KG = 1>
void decode_kernel(const gr_attn_args& a, dim3 grid, hipStream_t st) {
  constexpr int LDS = KG * gr_flash_lds<D, BN>::BYTES;
  hipLaunchKernelGGL((gr_flash_fwd_kernel<T, D, BN, NW, 1, false, false, false, true, true, SPLIT, PRESCALE, KG>), grid,
                     dim3(NW * KG * 64), LDS, st, a);
}

// nw 1 or 2: four key groups of 32-key tiles (a part's keys over 4 or 8 waves);
// 4, and one_group (D = 128 in one part): one group of 64-key tiles, or 32 when
// N is not a multiple of 64.
template <class T, int D, bool SPLIT>
void decode_nw(const gr_attn_args& a, int nw, bool one_group, bool bn64, dim3 grid, hipStream_t st) {
  if constexpr (D == 128 && !SPLIT)
    if (one_group) {
      if (nw == 1 && bn64) return decode_kernel<T, D, 64, 1, false>(a, grid, st);
      if (nw == 1) return decode_kernel<T, D, 32, 1, false>(a, grid, st);
      if (bn64) return decode_kernel<T, D, 64, 2, false>(a, grid, st);
      return decode_kernel<T, D, 32, 2, false>(a, grid, st);
    }
  if (nw == 1) decode_kernel<T, D, 32, 1, SPLIT, true, 4>(a, grid, st);
  else if (nw == 2) decode_kernel<T, D, 32, 2, SPLIT, true, 4>(a, grid, st);
  else if (bn64) decode_kernel<T, D, 64, 4, SPLIT>(a, grid, st);
  else decode_kernel<T, D, 32, 4, SPLIT>(a, grid, st);
}

template <class T, int D, int NQ>
void decode_stream(const gr_attn_args& a, int S, hipStream_t st) {
  constexpr int U = NQ == 1 ? 8 : 4;   // key-row loads of K and of V per lane and iteration
  hipLaunchKernelGGL((gr_attn_decode_stream_kernel<T, D, NQ, U>), dim3((unsigned)(a.B * a.H), (unsigned)S),
                     dim3(256), 0, st, a);
}

// Decode-shape launch: Nq queries (any count) against N keys, non-causal, K in
// [B, H, N, D]. Up to 4 queries: the streaming kernel (gr_flash_decode.h),
// one workgroup per head and key part. More: the flash body with 32 queries
// per wave: up to 64 queries, four key groups per workgroup and 32-key tiles
// (launch_decode has the exception); above, four waves and 64-key tiles (32 when
// N is not a multiple of 64).
// S > 1 splits the keys over S workgroups per head (or query tile) and merges
// their partials through the workspace.
// Message for a workspace smaller than the key split needs: the caller's
// buffer (gr_attn_decode) or the library's fixed scratch array
// (gr_attn_decode_noalloc).
int workspace_short(bool fixed, size_t need, int S, size_t have) {
  if (fixed)
    return gr::fail(GR_E_ARG, "gr_attn_decode_noalloc: %d key parts need %zu bytes of scratch, more than the "
                    "%zu-byte maximum (ask for fewer splits or use gr_attn_decode with a workspace)", S, need, have);
  return gr::fail(GR_E_ARG, "gr_attn_decode: workspace of %zu bytes needed for %d key parts", need, S);
}

template <class T, int D>
int launch_decode(gr_attn_args a, int S, void* ws, size_t ws_bytes, bool fixed_ws, hipStream_t st) {
  if (a.Nq <= 4) {
    if (S < 1) S = 1;
    if (S > a.N / 32) S = a.N / 32;
    a.kchunk = ((a.N / 32 + S - 1) / S) * 32;
    S = (a.N + a.kchunk - 1) / a.kchunk;         // every part gets keys
    if ((long long)a.B * a.H > 0x7fffffffLL || S > 65535) return gr::fail(GR_E_ARG, "gr_attn_decode: grid out of range");
    if (S > 1) {
      const size_t need = gr_attn_decode_workspace(a.B, a.H, a.Nq, D, S);
      if (!ws || ws_bytes < need) return workspace_short(fixed_ws, need, S, ws_bytes);
      a.part_o = static_cast<float*>(ws);
      a.part_ml = a.part_o + (size_t)S * a.B * a.H * a.Nq * D;
    }
    if (a.Nq == 1) decode_stream<T, D, 1>(a, S, st);
    else if (a.Nq == 2) decode_stream<T, D, 2>(a, S, st);
    else decode_stream<T, D, 4>(a, S, st);
    int rc = gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_decode launch");
    if (rc != 0 || S == 1) return rc;
    return launch_combine<T, D>(a, S, st);
  }
  // fp16 with scale log2(e) > 1: Q as given (one wave per query tile, 32-key tiles)
  const bool unscaled = gr_is_same<T, _Float16>::value && a.scale_log2 > 1.0f;
  const int nw = unscaled ? 1 : a.Nq <= 32 ? 1 : a.Nq <= 64 ? 2 : 4;
  const long long nqt = (a.Nq + 32 * nw - 1) / (32 * nw);
  const long long nblk = (long long)a.B * a.H * nqt;
  if (S < 1) S = 1;
  // D = 128 with key groups fills a CU's LDS (128 KiB): grids of more than one
  // workgroup per CU run in rounds, which few keys do not repay (300 heads, 32
  // queries: N 256 18.2 us, with one group 11.2; N 512 24.9 and 26.8). D = 64
  // has two per CU and no such line.
  const bool one_group = D == 128 && nw < 4 && !unscaled && S == 1 && a.N < 512 && nblk > gr::cu_count();
  const bool bn64 = (nw == 4 || one_group) && a.N % 64 == 0;
  const int bn = bn64 ? 64 : 32;
  const int tiles = a.N / bn;
  if (S > tiles) S = tiles;
  a.kchunk = ((tiles + S - 1) / S) * bn;
  S = (a.N + a.kchunk - 1) / a.kchunk;         // every part gets keys
  if (nblk > 0x7fffffffLL || S > 65535) return gr::fail(GR_E_ARG, "gr_attn_decode: grid out of range");
  if (S > 1) {
    const size_t need = gr_attn_decode_workspace(a.B, a.H, a.Nq, D, S);
    if (!ws || ws_bytes < need) return workspace_short(fixed_ws, need, S, ws_bytes);
    a.part_o = static_cast<float*>(ws);
    a.part_ml = a.part_o + (size_t)S * a.B * a.H * a.Nq * D;
  }
  const dim3 grid((unsigned)nblk, (unsigned)S);
  if (unscaled) {
    if constexpr (gr_is_same<T, _Float16>::value) {
      if (S > 1) decode_kernel<T, D, 32, 1, true, false>(a, grid, st);
      else decode_kernel<T, D, 32, 1, false, false>(a, grid, st);
    }
  } else if (S > 1) {
    decode_nw<T, D, true>(a, nw, false, bn64, grid, st);
  } else {
    decode_nw<T, D, false>(a, nw, one_group, bn64, grid, st);
  }
  int rc = gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_decode launch");
  if (rc != 0 || S == 1) return rc;
  return launch_combine<T, D>(a, S, st);
}

__global__ void gr_selftest_mfma32_kernel(const _Float16* A, const _Float16* B, float* Dm) {
  const int l = threadIdx.x, l32 = l & 31, g = l >> 5;
  gr_f16x8 a, b;
  for (int e = 0; e < 8; ++e) {
    a[e] = A[l32 * 16 + 8 * g + e];       // A[m][k], m = l % 32, k in group l / 32
    b[e] = B[(8 * g + e) * 32 + l32];     // B[k][n], n = l % 32
  }
  gr_f32x16 acc = (gr_f32x16)(0.f);
  acc = gr_mfma<_Float16>::mma32(a, b, acc);
  for (int r = 0; r < 16; ++r) {
    const int m = 8 * (r / 4) + 4 * g + (r % 4);
    Dm[m * 32 + l32] = acc[r];
  }
}

}  // namespace

namespace {

int attn_fwd(const void* q, const void* k, const void* v, void* o, float* lse, int dtype, int B, int H, int N, int D,
             const long long* qs, const long long* ks, const long long* vs, const long long* os, int k_transposed,
             int causal, float scale, int block_m, int block_n, void* stream) {
  if (!q || !k || !v || !o || !qs || !ks || !vs || !os) return gr::fail(GR_E_ARG, "gr_attn_fwd: null argument");
  if (B <= 0 || H <= 0 || N <= 0) return gr::fail(GR_E_ARG, "gr_attn_fwd: B, H, N must be positive");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o))
    return gr::fail(GR_E_ARG, "gr_attn_fwd: base pointers must be 16-byte aligned");
  const long long* all[4] = {qs, ks, vs, os};
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 3; ++i)
      if (all[t][i] < 0 || (all[t][i] % 8) != 0)
        return gr::fail(GR_E_ARG, "gr_attn_fwd: strides must be non-negative multiples of 8 elements");
  if (!(scale > 0.f)) return gr::fail(GR_E_ARG, "gr_attn_fwd: scale must be positive");
  gr_attn_args a;
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.q_sb = qs[0]; a.q_sh = qs[1]; a.q_sn = qs[2];
  a.k_sb = ks[0]; a.k_sh = ks[1]; a.k_sn = ks[2];
  a.v_sb = vs[0]; a.v_sh = vs[1]; a.v_sn = vs[2];
  a.o_sb = os[0]; a.o_sh = os[1]; a.o_sn = os[2];
  a.B = B;
  a.H = H;
  a.N = N;
  a.Nq = N;
  a.kchunk = N;
  a.part_o = nullptr;
  a.part_ml = nullptr;
  a.lse = lse;
  a.scale_log2 = scale * 1.4426950408889634f;
  hipStream_t st = (hipStream_t)stream;
  // fp16 pre-scales Q by scale * log2(e) in fp16; above 1 a finite q could
  // overflow, so such calls take the kernels that keep Q as given
  if (dtype == GR_F16 && a.scale_log2 > 1.0f)
    return dispatch_unscaled_q(a, D, causal != 0, k_transposed != 0, block_m, block_n, st);
  if (dtype == GR_F16) return dispatch_shape<_Float16>(a, D, causal != 0, k_transposed != 0, block_m, block_n, st);
  if (dtype == GR_BF16) return dispatch_shape<__bf16>(a, D, causal != 0, k_transposed != 0, block_m, block_n, st);
  if (dtype == GR_F32) return gr::attn_fwd_f32(a, D, causal != 0, k_transposed != 0, lse != nullptr, st);
  return gr::fail(GR_E_ARG, "gr_attn_fwd: dtype %d unsupported (GR_F16, GR_BF16 or GR_F32)", dtype);
}

}  // namespace

extern "C" int gr_attn_fwd(const void* q, const void* k, const void* v, void* o, int dtype, int B, int H, int N,
                           int D, const long long* qs, const long long* ks, const long long* vs, const long long* os,
                           int k_transposed, int causal, float scale, int block_m, int block_n, void* stream) {
  return attn_fwd(q, k, v, o, nullptr, dtype, B, H, N, D, qs, ks, vs, os, k_transposed, causal, scale, block_m,
                  block_n, stream);
}

extern "C" int gr_attn_fwd_shape(int dtype, int B, int H, int N, int D, int k_transposed, int causal, int train,
                                 int* out3) {
  if (!out3) return gr::fail(GR_E_ARG, "gr_attn_fwd_shape: null output");
  if ((dtype != GR_F16 && dtype != GR_BF16) || (D != 64 && D != 128) || B <= 0 || H <= 0 || N <= 0 || N % 64)
    return gr::fail(GR_E_ARG, "gr_attn_fwd_shape: no pick for dtype %d, D=%d, N=%d (fp16 or bf16, D 64 or 128, N a multiple of 64)",
                    dtype, D, N);
  const AttnShape s = pick_call(dtype, D, causal != 0, k_transposed != 0, train != 0, (long long)B * H, N);
  out3[0] = 32 * s.nw;
  out3[1] = s.kg;
  out3[2] = s.bn;
  return GR_OK;
}

extern "C" int gr_attn_fwd_train(const void* q, const void* k, const void* v, void* o, float* lse, int dtype, int B,
                                 int H, int N, int D, const long long* qs, const long long* ks, const long long* vs,
                                 const long long* os, int k_transposed, int causal, float scale, int block_m,
                                 int block_n, void* stream) {
  if (!lse || ((uintptr_t)lse & 3)) return gr::fail(GR_E_ARG, "gr_attn_fwd_train: lse must be a 4-byte aligned buffer");
  return attn_fwd(q, k, v, o, lse, dtype, B, H, N, D, qs, ks, vs, os, k_transposed, causal, scale, block_m, block_n,
                  stream);
}

extern "C" int gr_selftest_mfma32(const void* a, const void* b, float* d, void* stream) {
  if (!a || !b || !d) return gr::fail(GR_E_ARG, "gr_selftest_mfma32: null argument");
  hipLaunchKernelGGL(gr_selftest_mfma32_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, (const _Float16*)a,
                     (const _Float16*)b, d);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_selftest_mfma32 launch");
}

extern "C" size_t gr_attn_decode_workspace(int B, int H, int Nq, int D, int splits) {
  if (B <= 0 || H <= 0 || Nq <= 0 || D <= 0 || splits <= 1) return 0;
  return (size_t)splits * B * H * Nq * (D + 2) * sizeof(float);
}

namespace {

int attn_decode(const char* who, const void* q, const void* k, const void* v, void* o, int dtype, int B, int H,
                int Nq, int N, int D, const long long* qs, const long long* ks, const long long* vs,
                const long long* os, float scale, int splits, void* workspace, size_t workspace_bytes, bool fixed_ws,
                void* stream) {
  if (!q || !k || !v || !o || !qs || !ks || !vs || !os) return gr::fail(GR_E_ARG, "%s: null argument", who);
  if (B <= 0 || H <= 0 || Nq <= 0 || N <= 0) return gr::fail(GR_E_ARG, "%s: B, H, Nq, N must be positive", who);
  if (N % 32 != 0) return gr::fail(GR_E_ARG, "%s: N=%d keys must be a multiple of 32", who, N);
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o) || ((uintptr_t)workspace & 15))
    return gr::fail(GR_E_ARG, "%s: base pointers must be 16-byte aligned", who);
  const long long* all[4] = {qs, ks, vs, os};
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 3; ++i)
      if (all[t][i] < 0 || (all[t][i] % 8) != 0)
        return gr::fail(GR_E_ARG, "%s: strides must be non-negative multiples of 8 elements", who);
  if (!(scale > 0.f)) return gr::fail(GR_E_ARG, "%s: scale must be positive", who);
  gr_attn_args a;
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.q_sb = qs[0]; a.q_sh = qs[1]; a.q_sn = qs[2];
  a.k_sb = ks[0]; a.k_sh = ks[1]; a.k_sn = ks[2];
  a.v_sb = vs[0]; a.v_sh = vs[1]; a.v_sn = vs[2];
  a.o_sb = os[0]; a.o_sh = os[1]; a.o_sn = os[2];
  a.B = B;
  a.H = H;
  a.N = N;
  a.Nq = Nq;
  a.kchunk = N;
  a.part_o = nullptr;
  a.part_ml = nullptr;
  a.scale_log2 = scale * 1.4426950408889634f;
  hipStream_t st = (hipStream_t)stream;
#define GR_DT(TT)                                                                                  \
  if (D == 64) return launch_decode<TT, 64>(a, splits, workspace, workspace_bytes, fixed_ws, st);  \
  if (D == 128) return launch_decode<TT, 128>(a, splits, workspace, workspace_bytes, fixed_ws, st); \
  return gr::fail(GR_E_ARG, "%s: head dim D=%d unsupported (64 or 128)", who, D);
  if (dtype == GR_F16) { GR_DT(_Float16) }
  if (dtype == GR_BF16) { GR_DT(__bf16) }
#undef GR_DT
  return gr::fail(GR_E_ARG, "%s: dtype %d unsupported (GR_F16 or GR_BF16)", who, dtype);
}

// The key-split partials of gr_attn_decode_noalloc live in this array, one
// copy per device, held until the process ends. The kernels only ever see
// its device address (g_scratch), which hipGetSymbolAddress returns for the
// device current at the first call on it; the array's name is a host-side
// stand-in and never goes to a kernel.
constexpr size_t kDecodeScratch = (size_t)GR_DECODE_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kDecodeScratch];
constexpr int kMaxDevices = 64;
void* g_scratch[kMaxDevices] = {};
std::mutex g_scratch_lock;

int scratch_address(void** out) {
  int dev = 0;
  int rc = gr::hip_check(hipGetDevice(&dev), GR_E_RUNTIME, "gr_attn_decode_noalloc: hipGetDevice");
  if (rc) return rc;
  if (dev < 0 || dev >= kMaxDevices) return gr::fail(GR_E_ARG, "gr_attn_decode_noalloc: device %d out of range", dev);
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    rc = gr::hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), GR_E_RUNTIME,
                       "gr_attn_decode_noalloc: hipGetSymbolAddress(scratch)");
    if (rc) return rc;
    if (!p) return gr::fail(GR_E_RUNTIME, "gr_attn_decode_noalloc: no device address for the scratch array");
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return GR_OK;
}

}  // namespace

extern "C" int gr_attn_decode(const void* q, const void* k, const void* v, void* o, int dtype, int B, int H, int Nq,
                              int N, int D, const long long* qs, const long long* ks, const long long* vs,
                              const long long* os, float scale, int splits, void* workspace, size_t workspace_bytes,
                              void* stream) {
  return attn_decode("gr_attn_decode", q, k, v, o, dtype, B, H, Nq, N, D, qs, ks, vs, os, scale, splits, workspace,
                     workspace_bytes, false, stream);
}

extern "C" int gr_attn_decode_noalloc(const void* q, const void* k, const void* v, void* o, int dtype, int B, int H,
                                      int Nq, int N, int D, const long long* qs, const long long* ks,
                                      const long long* vs, const long long* os, float scale, int splits,
                                      void* stream) {
  void* ws = nullptr;
  const int rc = scratch_address(&ws);
  if (rc) return rc;
  return attn_decode("gr_attn_decode_noalloc", q, k, v, o, dtype, B, H, Nq, N, D, qs, ks, vs, os, scale, splits, ws,
                     kDecodeScratch, true, stream);
}
