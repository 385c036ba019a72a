// gr_gemm.hip -- prebuilt instances of the MFMA GEMM with fused epilogue
// (gr_gemm.h) behind gr_gemm(), and the two-GEMM MLP block gr_mlp_fwd().
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gr_gemm.h"
#include "gr_gemm_f32.h"
#include "gr_gemm_plan.h"
#include "gr_host.h"
#include "grammar_rt.h"

namespace {

template <class T, int BM, int BN, int BK, int WGM, int WGN, bool KM, int EPI>
int launch_gemm(const gr_gemm_args& a, int batch, hipStream_t st) {
  typedef gr_gemm_cfg<BM, BN, BK, WGM, WGN> G;
  if (a.K % BK)
    return gr::fail(GR_E_ARG, "gr_gemm: K=%d must be a multiple of the k tile %d", a.K, BK);
  const long long nblk = (long long)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  if (nblk <= 0 || nblk > 0x7fffffffLL || batch > 65535)
    return gr::fail(GR_E_ARG, "gr_gemm: grid (%lld tiles, batch %d) out of range", nblk, batch);
  hipLaunchKernelGGL((gr_gemm_kernel<T, BM, BN, BK, WGM, WGN, KM, EPI>), dim3((unsigned)nblk, (unsigned)batch),
                     dim3(G::NT), G::LDS, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
}

// The 256 x 256 tile: four waves (one per SIMD) of 128 x 128, the
// hand-ordered main loop of gr_gemm_w4_body, one workgroup per CU. When the
// last round of workgroups would leave more than half of the CUs idle (X W1
// of the C4 MLP: 1,376 tiles on 256 CUs, a sixth round of 96), the columns
// past the whole rounds go to a second launch of the same body on 256 x 128
// tiles (waves of 128 x 64), if those fit in one round: 1,280 + 192 there.
template <class T, bool KM, int EPI, int BK>
int launch_gemm_w4(const gr_gemm_args& a, int batch, hipStream_t st) {
  if (a.K % BK)
    return gr::fail(GR_E_ARG, "gr_gemm: K=%d must be a multiple of the k tile %d", a.K, BK);
  const int mt = (a.M + 255) / 256, nt = (a.N + 255) / 256;
  const long long nblk = (long long)mt * nt;
  if (nblk <= 0 || nblk > 0x7fffffffLL || batch > 65535)
    return gr::fail(GR_E_ARG, "gr_gemm: grid (%lld tiles, batch %d) out of range", nblk, batch);
  const int cus = gr::cu_count();
  if (batch == 1 && cus > 0 && nblk > cus) {
    const long long rounds = (nblk + cus - 1) / cus;
    const long long last = nblk - (rounds - 1) * cus;            // workgroups of the last round
    const int nt_main = (int)((rounds - 1) * cus / mt);          // column tiles of the whole rounds
    const int col0 = nt_main * 256;
    const long long rest = (long long)mt * ((a.N - col0 + 127) / 128);
    if (2 * last <= cus && nt_main > 0 && nt_main < nt && rest <= cus) {
      gr_gemm_args m = a, r = a;
      m.N = col0;
      r.N = a.N - col0;
      r.b = static_cast<const T*>(a.b) + (KM ? (long long)col0 * a.b_s : (long long)col0);
      r.c = static_cast<T*>(a.c) + col0;
      if (a.r) r.r = static_cast<const T*>(a.r) + col0;
      hipLaunchKernelGGL((gr_gemm_w4_kernel<T, KM, EPI, BK>), dim3((unsigned)((long long)mt * nt_main)), dim3(256),
                         gr_gemm_w4_lds<BK>::value, st, m);
      const int rc = gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
      if (rc) return rc;
      hipLaunchKernelGGL((gr_gemm_w4_kernel<T, KM, EPI, BK, 128>), dim3((unsigned)rest), dim3(256),
                         (gr_gemm_w4_lds<BK, 128>::value), st, r);
      return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
    }
  }
  hipLaunchKernelGGL((gr_gemm_w4_kernel<T, KM, EPI, BK>), dim3((unsigned)nblk, (unsigned)batch), dim3(256),
                     gr_gemm_w4_lds<BK>::value, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
}

// A 256 x 128 tile of the one-wave body on its own (picked plans only).
template <class T, bool KM, int EPI, int BK>
int launch_gemm_w4h(const gr_gemm_args& a, int batch, hipStream_t st) {
  const long long nblk = (long long)((a.M + 255) / 256) * ((a.N + 127) / 128);
  if (nblk > 0x7fffffffLL || batch > 65535)
    return gr::fail(GR_E_ARG, "gr_gemm: grid (%lld tiles, batch %d) out of range", nblk, batch);
  hipLaunchKernelGGL((gr_gemm_w4_kernel<T, KM, EPI, BK, 128>), dim3((unsigned)nblk, (unsigned)batch), dim3(256),
                     (gr_gemm_w4_lds<BK, 128>::value), st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
}

// The tile and K split for a shape, when the caller names neither: the one a
// model of the launch gives the least time.
//
// A workgroup takes t0 + tau us per 64-deep k tile, where tau grows from
// tau_idle to tau_full as the workgroups resident on the chip grow from few
// to `slots` per CU (they share HBM, L2 and the matrix cores); a launch is
// its rounds of resident workgroups, bounded below by reading B at the copy
// rate (less with too few workgroups to cover the latency). A split adds the
// merge launch (2 us) and the partial sums' round trip at 6 MB/us. The
// constants are a least-squares fit to 11,600 launches over M 24-4096, N
// 512-11008, K 512-11008 and up to 16 parts; the pick is within 4 % of the
// fastest of those (geometric mean over 504 shapes, 42 % at worst), the
// 256 x 256 tile that every shape took before at 1.94x of it.
struct TileModel {
  int bm, bn, slots;
  double tau_idle, tau_full, t0;
  bool whole, split;           // compiled without / with a K split
};
constexpr TileModel kTiles64[] = {          // 64-deep k tiles
    {32, 128, 2, 0.20, 0.66, 1.7, true, true},   {64, 128, 2, 0.35, 0.64, 1.6, true, true},
    {128, 128, 2, 0.54, 1.00, 1.8, true, true},  {256, 128, 1, 0.67, 0.95, 1.3, true, false},
    {256, 256, 1, 1.10, 1.40, 3.1, true, true},
};
constexpr TileModel kTiles32[] = {          // K not a multiple of 64: 32-deep k tiles from 128 rows on
    {32, 128, 2, 0.20, 0.66, 1.7, true, true},   {64, 128, 2, 0.35, 0.64, 1.6, true, true},
    {128, 128, 2, 0.96, 1.12, 0.8, true, true},  {256, 128, 1, 0.58, 0.91, 2.1, true, false},
    {256, 256, 1, 1.05, 1.39, 3.4, true, true},
};

gr::GemmPlan pick_plan(int batch, int M, int N, int K, size_t ws_max) {
  gr::GemmPlan best = {256, 256, 1, 0};
  const int cus = gr::cu_count();
  if (cus <= 0) return best;
  // Few k tiles and a C of more than half a round of 256 x 256 tiles: bound by
  // its store, which the model does not count (K 64: M 1024, N 11008 10.7 us,
  // 13.1 on 256 x 128; M 4096, N 4096 12.0 and 14.0 on 128 x 128)
  if (K < 256 && 2LL * batch * ((M + 255) / 256) * ((N + 255) / 256) > cus) return best;
  double best_t = 1e30;
  for (const TileModel& m : K % 64 == 0 ? kTiles64 : kTiles32) {
    // The 32-row tile reads B once per 32 rows: up to 32, or 64 while a short K
    // leaves the launch bound by its start (M 48, K 1024: 7.1 us against 10.3
    // on 64 rows; K 4096 x N 11008: 32 against 24). The larger tiles start
    // at more than half a tile of rows.
    if (m.bm == 32 ? M > (K <= 1024 ? 64 : 32) : m.bm > 64 && 2 * M <= m.bm) continue;
    if (m.bm < 128 && K < 64) continue;        // one 64-deep k tile at least
    const double tiles = (double)batch * ((M + m.bm - 1) / m.bm) * ((N + m.bn - 1) / m.bn);
    for (int ks = 1; ks <= 16; ks *= 2) {
      if (ks == 1 ? !m.whole : !m.split || K / ks < 256 || tiles * ks > 2 * cus) continue;
      const size_t ws = ks == 1 ? 0 : (size_t)ks * (size_t)tiles * m.bm * m.bn * sizeof(float);
      if (ws > ws_max) continue;
      const double nk = K / 64.0 / ks, w = tiles * ks, per = (double)cus * m.slots;
      auto round = [&](double r) { return nk * (m.tau_idle + (m.tau_full - m.tau_idle) * r / per) + m.t0; };
      const double full = (double)(long long)(w / per), rem = w - full * per;
      double t = full * round(per) + (rem > 0 ? round(rem) : 0.);
      const double rate = w * 0.033 < 4.7 ? w * 0.033 : 4.7;           // MB per us
      const double read = 2e-6 * batch * N * (double)K / rate;
      if (t < read) t = read;
      if (ks > 1) t += 2.0 + 2e-6 * (double)ws / 6.0;
      if (t < best_t) {
        best_t = t;
        best = {m.bm, m.bn, ks, ws};
      }
    }
  }
  return best;
}

// (block_m, block_n) -> (k tile, wave grid) compiled into the library; the
// 128x128 and 256x256 tiles take 64-deep k tiles when K allows, else 32.
template <class T, bool KM, int EPI>
int dispatch_tile(const gr_gemm_args& a, int batch, int bm, int bn, hipStream_t st) {
  if (bm == 0) bm = 256;
  if (bn == 0) bn = 256;
  const bool k64 = a.K % 64 == 0;
  if (bm == 128 && bn == 128)
    return k64 ? launch_gemm<T, 128, 128, 64, 2, 2, KM, EPI>(a, batch, st)
               : launch_gemm<T, 128, 128, 32, 2, 2, KM, EPI>(a, batch, st);
  if (bm == 256 && bn == 128) return launch_gemm<T, 256, 128, 32, 2, 2, KM, EPI>(a, batch, st);
  if (bm == 128 && bn == 256) return launch_gemm<T, 128, 256, 32, 2, 2, KM, EPI>(a, batch, st);
  if (bm == 256 && bn == 256)
    return k64 ? launch_gemm_w4<T, KM, EPI, 64>(a, batch, st) : launch_gemm_w4<T, KM, EPI, 32>(a, batch, st);
  return gr::fail(GR_E_ARG, "gr_gemm: unsupported tile (block_m=%d, block_n=%d)", bm, bn);
}

// plan: a picked one (bm, bn are its tile), or null for the caller's tile.
template <class T, bool KM, int EPI>
int dispatch_plan(const gr_gemm_args& a, int batch, int bm, int bn, const gr::GemmPlan* plan, hipStream_t st) {
  if (plan && bm == 256 && bn == 128)
    return a.K % 64 == 0 ? launch_gemm_w4h<T, KM, EPI, 64>(a, batch, st) : launch_gemm_w4h<T, KM, EPI, 32>(a, batch, st);
  return dispatch_tile<T, KM, EPI>(a, batch, bm, bn, st);
}

template <class T>
int dispatch(const gr_gemm_args& a, int batch, bool km, int epi, int bm, int bn, const gr::GemmPlan* plan,
             hipStream_t st) {
#define GR_CASE(K, E) \
  if (km == K && epi == E) return dispatch_plan<T, K, E>(a, batch, bm, bn, plan, st);
  GR_CASE(false, GR_EPI_NONE)
  GR_CASE(false, GR_EPI_RELU)
  GR_CASE(false, GR_EPI_SILU)
  GR_CASE(true, GR_EPI_NONE)
  GR_CASE(true, GR_EPI_RELU)
  GR_CASE(true, GR_EPI_SILU)
#undef GR_CASE
  return gr::fail(GR_E_ARG, "gr_gemm: epilogue %d unsupported", epi);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// fp32 on the fp32 matrix cores (gr_gemm_f32.h): (block_m, block_n) in
// {32, 64, 128}^2, one wave per 32 rows / columns up to 2 x 2 waves; k tile 32
// when K allows, else 16 or 8. M and N must be multiples of the tile.
template <int BM, int BN, bool KM, int EPI>
int launch_gemm_f32(const gr_gemm_args& a, int batch, hipStream_t st) {
  constexpr int WGM = BM >= 64 ? 2 : 1, WGN = BN >= 64 ? 2 : 1;
  if (a.M % BM || a.N % BN)
    return gr::fail(GR_E_ARG, "gr_gemm: fp32 needs M=%d, N=%d multiples of the tile %dx%d", a.M, a.N, BM, BN);
  const long long nblk = (long long)(a.M / BM) * (a.N / BN);
  if (nblk > 0x7fffffffLL || batch > 65535) return gr::fail(GR_E_ARG, "gr_gemm: grid out of range");
#define GR_F32K(BK)                                                                                        \
  hipLaunchKernelGGL((gr_gemm_f32_kernel<BM, BN, BK, WGM, WGN, KM, EPI>), dim3((unsigned)nblk, (unsigned)batch), \
                     dim3(WGM * WGN * 64), (gr_gemm_f32_cfg<BM, BN, BK, WGM, WGN, KM>::LDS), st, a)
  if (a.K % 32 == 0) GR_F32K(32);
  else if (a.K % 16 == 0) GR_F32K(16);
  else if (a.K % 8 == 0) GR_F32K(8);
  else return gr::fail(GR_E_ARG, "gr_gemm: fp32 needs K=%d a multiple of 8", a.K);
#undef GR_F32K
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
}

// 32 x 32 blocks with K over the four waves of a workgroup.
template <bool KM, int EPI>
int launch_gemm_f32_groups(const gr_gemm_args& a, int batch, hipStream_t st) {
  const long long nblk = (long long)(a.M / 32) * (a.N / 32);
  if (nblk > 0x7fffffffLL || batch > 65535) return gr::fail(GR_E_ARG, "gr_gemm: grid out of range");
#define GR_F32G(BK)                                                                                              \
  hipLaunchKernelGGL((gr_gemm_f32_groups_kernel<BK, KM, EPI>), dim3((unsigned)nblk, (unsigned)batch), dim3(256), \
                     GR_GEMM_F32_GROUPS_LDS, st, a)
  if (a.K % 16 == 0) GR_F32G(16);
  else if (a.K % 8 == 0) GR_F32G(8);
  else return gr::fail(GR_E_ARG, "gr_gemm: fp32 needs K=%d a multiple of 8", a.K);
#undef GR_F32G
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
}

// Whether the k-group body takes a call whose tile is bm x bn (gr_gemm_f32_groups
// is the rule).
bool f32_groups(const gr_gemm_args& a, int batch, bool km, int bm, int bn) {
  if (a.M % 32 || a.N % 32) return false;
  const int cus = gr::cu_count();
  return cus > 0 && gr_gemm_f32_groups(batch, a.M, a.N, a.K / (a.K % 16 == 0 ? 16 : 8), km, bm, bn, cus) == 1;
}

template <bool KM, int EPI>
int dispatch_f32_tile(const gr_gemm_args& a, int batch, int bm, int bn, hipStream_t st) {
  const bool pick = bm == 0 && bn == 0;
  if (bm == 0) bm = a.M % 128 == 0 ? 128 : a.M % 64 == 0 ? 64 : 32;
  if (bn == 0) bn = a.N % 128 == 0 ? 128 : a.N % 64 == 0 ? 64 : 32;
  if (pick && f32_groups(a, batch, KM, bm, bn)) return launch_gemm_f32_groups<KM, EPI>(a, batch, st);
#define GR_T(M_, N_) \
  if (bm == M_ && bn == N_) return launch_gemm_f32<M_, N_, KM, EPI>(a, batch, st);
  GR_T(32, 32) GR_T(32, 64) GR_T(32, 128) GR_T(64, 32) GR_T(64, 64) GR_T(64, 128)
  GR_T(128, 32) GR_T(128, 64) GR_T(128, 128)
#undef GR_T
  return gr::fail(GR_E_ARG, "gr_gemm: unsupported fp32 tile (block_m=%d, block_n=%d)", bm, bn);
}

int dispatch_f32(const gr_gemm_args& a, int batch, bool km, int epi, int bm, int bn, hipStream_t st) {
#define GR_CASE(K, E) \
  if (km == K && epi == E) return dispatch_f32_tile<K, E>(a, batch, bm, bn, st);
  GR_CASE(false, GR_EPI_NONE)
  GR_CASE(false, GR_EPI_RELU)
  GR_CASE(false, GR_EPI_SILU)
  GR_CASE(true, GR_EPI_NONE)
  GR_CASE(true, GR_EPI_RELU)
  GR_CASE(true, GR_EPI_SILU)
#undef GR_CASE
  return gr::fail(GR_E_ARG, "gr_gemm: epilogue %d unsupported", epi);
}

}  // namespace

namespace {

int gemm(const void* a, const void* b, void* c, int dtype, int batch, int M, int N, int K, const long long* a_strides,
         const long long* b_strides, const long long* c_strides, int b_kmajor, int epilogue, float alpha, int block_m,
         int block_n, void* workspace, size_t workspace_bytes, void* stream) {
  if (!a || !b || !c || !a_strides || !b_strides || !c_strides) return gr::fail(GR_E_ARG, "gr_gemm: null argument");
  if (batch <= 0 || M <= 0 || N <= 0 || K <= 0) return gr::fail(GR_E_ARG, "gr_gemm: sizes must be positive");
  if (dtype != GR_F32 && (N % 8 != 0 || K % 32 != 0))
    return gr::fail(GR_E_ARG, "gr_gemm: N=%d must be a multiple of 8 and K=%d a multiple of 32", N, K);
  if (!aligned16(a) || !aligned16(b) || !aligned16(c))
    return gr::fail(GR_E_ARG, "gr_gemm: base pointers must be 16-byte aligned");
  const long long* all[3] = {a_strides, b_strides, c_strides};
  const int sq = dtype == GR_F32 ? 4 : 8;    // elements per 16 bytes
  for (int t = 0; t < 3; ++t)
    for (int i = 0; i < 2; ++i)
      if (all[t][i] < 0 || (all[t][i] % sq) != 0)
        return gr::fail(GR_E_ARG, "gr_gemm: strides must be non-negative multiples of 16 bytes");
  // 32-bit per-thread offsets inside one tile walk: the rows a tile spans
  if (a_strides[1] > 0x3fffffffLL / 256 || b_strides[1] > 0x3fffffffLL / 256)
    return gr::fail(GR_E_ARG, "gr_gemm: row strides too large");
  gr_gemm_args g;
  g.a = a;
  g.b = b;
  g.c = c;
  g.a_sb = a_strides[0]; g.a_sm = a_strides[1];
  g.b_sb = b_strides[0]; g.b_s = b_strides[1];
  g.c_sb = c_strides[0]; g.c_sm = c_strides[1];
  g.M = M;
  g.N = N;
  g.K = K;
  g.alpha = alpha;
  hipStream_t st = (hipStream_t)stream;
  const bool km = b_kmajor != 0;
  if ((dtype == GR_F16 || dtype == GR_BF16) && block_m == 0 && block_n == 0 && epilogue >= GR_EPI_NONE &&
      epilogue <= GR_EPI_SILU) {
    const size_t have = workspace ? workspace_bytes : 0;
    const gr::GemmPlan p = pick_plan(batch, M, N, K, have < gr::kGemmWorkspaceMax ? have : gr::kGemmWorkspaceMax);
    g.ws = static_cast<float*>(workspace);
    if (p.bm < 128 || p.ks > 1) return gr::launch_gemm_planned(g, dtype, batch, km, epilogue, p, st);
    if (dtype == GR_F16) return dispatch<_Float16>(g, batch, km, epilogue, p.bm, p.bn, &p, st);
    return dispatch<__bf16>(g, batch, km, epilogue, p.bm, p.bn, &p, st);
  }
  if (dtype == GR_F16) return dispatch<_Float16>(g, batch, km, epilogue, block_m, block_n, nullptr, st);
  if (dtype == GR_BF16) return dispatch<__bf16>(g, batch, km, epilogue, block_m, block_n, nullptr, st);
  if (dtype == GR_F32) return dispatch_f32(g, batch, b_kmajor != 0, epilogue, block_m, block_n, st);
  return gr::fail(GR_E_ARG, "gr_gemm: dtype %d unsupported (GR_F32, GR_F16 or GR_BF16)", dtype);
}

int mlp_fwd(const void* x, const void* w1, const void* w2, void* h, void* y, int dtype, int M, int D, int F,
            int block_m, int block_n, void* workspace, size_t workspace_bytes, void* stream) {
  const long long xs[2] = {0, D}, w1s[2] = {0, F}, hs[2] = {0, F}, w2s[2] = {0, D}, ys[2] = {0, D};
  const int rc = gemm(x, w1, h, dtype, 1, M, F, D, xs, w1s, hs, 0, GR_EPI_SILU, 1.0f, block_m, block_n, workspace,
                      workspace_bytes, stream);
  if (rc != 0) return rc;
  return gemm(h, w2, y, dtype, 1, M, D, F, hs, w2s, ys, 0, GR_EPI_NONE, 1.0f, block_m, block_n, workspace,
              workspace_bytes, stream);
}

}  // namespace

// Two lines. Matrix-core time per SIMD of the launch's rounds, in 32 x 32 blocks x
// k tiles, below 0.8 of the tile's; and few rounds, since blocks read their
// operands without sharing them: up to two per 32 x 32 block that a wave of the
// tile owns (a third where it owns one and B is not K-major), four where the tile
// has two waves, which leave half of a CU's SIMDs idle; from 32 k tiles on also
// 2.5 per block of the tile's rounds of four waves per CU, the last of them
// part-filled (960 x 1152, K 704 on 64 x 64 tiles: five rounds 29.5 us, the tile's
// two 31.9). Over 11,054 pairs of shape and tile (M, N 64-4096, K 32-2048; tiles
// of 32, 64, 128 a side) the choice is within 0.4 % of the faster body (geometric
// mean; 2.3 % with the first line alone, which took M 768, N 4096, K 1024 from 79
// us on 128 x 128 to 98 and 4096 x 512, K 64 K-major on 32 x 32 from 7.0 to 11.8).
extern "C" int gr_gemm_f32_groups(int batch, int M, int N, int ktiles, int b_kmajor, int block_m, int block_n, int cus) {
  if (batch <= 0 || M <= 0 || N <= 0 || ktiles <= 0 || block_m < 32 || block_n < 32 || cus <= 0) return 0;
  const int waves = (block_m >= 64 ? 2 : 1) * (block_n >= 64 ? 2 : 1);
  const long long tiles = (long long)batch * ((M + block_m - 1) / block_m) * ((N + block_n - 1) / block_n);
  const long long blocks = (long long)batch * (M / 32) * (N / 32);
  const long long chain = (long long)(block_m / 32) * (block_n / 32) / waves;       // 32 x 32 blocks per wave
  const long long rounds = (blocks + cus - 1) / cus, full = (tiles * waves + 4LL * cus - 1) / (4LL * cus);
  const long long few = waves == 2 ? 4 * chain : 2 * chain + (chain == 1 && !b_kmajor);
  if (rounds > few && (ktiles < 32 || 2 * rounds > 5 * chain * full)) return 0;
  return 10 * rounds * ((ktiles + 3) / 4) < 8 * ((tiles + cus - 1) / cus) * chain * ktiles;
}

extern "C" int gr_gemm(const void* a, const void* b, void* c, int dtype, int batch, int M, int N, int K,
                       const long long* a_strides, const long long* b_strides, const long long* c_strides,
                       int b_kmajor, int epilogue, float alpha, int block_m, int block_n, void* stream) {
  return gemm(a, b, c, dtype, batch, M, N, K, a_strides, b_strides, c_strides, b_kmajor, epilogue, alpha, block_m,
              block_n, nullptr, 0, stream);
}

extern "C" size_t gr_gemm_workspace(int dtype, int batch, int M, int N, int K) {
  if ((dtype != GR_F16 && dtype != GR_BF16) || batch <= 0 || M <= 0 || N <= 0 || K <= 0) return 0;
  return pick_plan(batch, M, N, K, gr::kGemmWorkspaceMax).ws;
}

extern "C" int gr_gemm_ws(const void* a, const void* b, void* c, int dtype, int batch, int M, int N, int K,
                          const long long* a_strides, const long long* b_strides, const long long* c_strides,
                          int b_kmajor, int epilogue, float alpha, void* workspace, size_t workspace_bytes,
                          void* stream) {
  if ((uintptr_t)workspace & 15) return gr::fail(GR_E_ARG, "gr_gemm_ws: workspace must be 16-byte aligned");
  return gemm(a, b, c, dtype, batch, M, N, K, a_strides, b_strides, c_strides, b_kmajor, epilogue, alpha, 0, 0,
              workspace, workspace_bytes, stream);
}

extern "C" int gr_mlp_fwd(const void* x, const void* w1, const void* w2, void* h, void* y, int dtype, int M,
                          int D, int F, int block_m, int block_n, void* stream) {
  return mlp_fwd(x, w1, w2, h, y, dtype, M, D, F, block_m, block_n, nullptr, 0, stream);
}

extern "C" size_t gr_mlp_fwd_workspace(int dtype, int M, int D, int F) {
  const size_t up = gr_gemm_workspace(dtype, 1, M, F, D), down = gr_gemm_workspace(dtype, 1, M, D, F);
  return up > down ? up : down;
}

extern "C" int gr_mlp_fwd_ws(const void* x, const void* w1, const void* w2, void* h, void* y, int dtype, int M,
                             int D, int F, void* workspace, size_t workspace_bytes, void* stream) {
  if ((uintptr_t)workspace & 15) return gr::fail(GR_E_ARG, "gr_mlp_fwd_ws: workspace must be 16-byte aligned");
  return mlp_fwd(x, w1, w2, h, y, dtype, M, D, F, 0, 0, workspace, workspace_bytes, stream);
}
