// gr_gemm_split.hip -- the GEMM launches for shapes that leave CUs idle on
// whole-K 128- and 256-row tiles: 32- and 64-row tiles for few rows, and K
// split over workgroups with a merge launch (gr_gemm_merge_kernel).
//
// Few rows are bound by reading B once from HBM, i.e. by bytes in flight: the
// 32- and 64-row tiles keep 3 and 2 k tiles of 20 and 24 KiB in flight per
// workgroup, two workgroups per CU. M 24 against B 4096 x 11008 (90 MB) went
// from 77 us on 43 workgroups of 256 x 256 to 21 us (4.2 TB/s) on 86 x 2 of
// 32 x 128, B 11008 x 4096 from 188 to 23 us (32 x 8). A stream of B straight
// into registers (no LDS, the waves splitting K) measured 23.6 and 24.2 us.
#include <hip/hip_runtime.h>

#include "gr_gemm_plan.h"
#include "gr_host.h"
#include "grammar_rt.h"

namespace {

// Merge launch: 8 columns of one row per thread.
template <class T, int BM, int BN, int WGM, int WGN, int EPI>
int launch_merge(const gr_gemm_args& a, long long ntile, int tiles_n, int tiles_per_batch, hipStream_t st) {
  typedef gr_gemm_cfg<BM, BN, 32, WGM, WGN> G;
  const long long threads = ntile * G::TN * G::TM * 4 * (G::NT / 2);
  hipLaunchKernelGGL((gr_gemm_merge_kernel<T, BM, BN, WGM, WGN, EPI>), dim3((unsigned)((threads + 255) / 256)),
                     dim3(256), 0, st, a, ntile, tiles_n, tiles_per_batch);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm merge launch");
}

template <class T, int BM, int BN, int WGM, int WGN>
int launch_merge_epi(const gr_gemm_args& a, int epi, long long ntile, int tiles_n, int per_batch, hipStream_t st) {
  if (epi == GR_EPI_RELU) return launch_merge<T, BM, BN, WGM, WGN, GR_EPI_RELU>(a, ntile, tiles_n, per_batch, st);
  if (epi == GR_EPI_SILU) return launch_merge<T, BM, BN, WGM, WGN, GR_EPI_SILU>(a, ntile, tiles_n, per_batch, st);
  return launch_merge<T, BM, BN, WGM, WGN, GR_EPI_NONE>(a, ntile, tiles_n, per_batch, st);
}

// 32- and 64-row tiles: four waves across 128 columns, 64-deep k tiles (K a
// multiple of 32, at least 64) in a ring of STAGES.
template <class T, int BM, int STAGES, bool KM>
int launch_rows(const gr_gemm_args& a, int batch, int epi, int tiles, int tiles_n, hipStream_t st) {
  typedef gr_gemm_cfg<BM, 128, 64, 1, 4, STAGES> G;
  if (a.ksplit > 1) {
    hipLaunchKernelGGL((gr_gemm_kernel<T, BM, 128, 64, 1, 4, KM, GR_EPI_NONE, STAGES, true, true>),
                       dim3((unsigned)(tiles * a.ksplit), (unsigned)batch), dim3(G::NT), G::LDS, st, a);
    const int rc = gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
    return rc ? rc : launch_merge_epi<T, BM, 128, 1, 4>(a, epi, (long long)tiles * batch, tiles_n, tiles, st);
  }
#define GR_E(E)                                                                                                  \
  if (epi == E)                                                                                                  \
    hipLaunchKernelGGL((gr_gemm_kernel<T, BM, 128, 64, 1, 4, KM, E, STAGES, false, true>),                       \
                       dim3((unsigned)tiles, (unsigned)batch), dim3(G::NT), G::LDS, st, a);
  GR_E(GR_EPI_NONE) GR_E(GR_EPI_RELU) GR_E(GR_EPI_SILU)
#undef GR_E
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
}

// K-split launches of the 128 x 128 and 256 x 256 tiles.
template <class T, int BK, bool KM>
int launch_split128(const gr_gemm_args& a, int batch, int epi, int tiles, int tiles_n, hipStream_t st) {
  typedef gr_gemm_cfg<128, 128, BK, 2, 2> G;
  hipLaunchKernelGGL((gr_gemm_kernel<T, 128, 128, BK, 2, 2, KM, GR_EPI_NONE, 2, true>),
                     dim3((unsigned)(tiles * a.ksplit), (unsigned)batch), dim3(G::NT), G::LDS, st, a);
  const int rc = gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
  return rc ? rc : launch_merge_epi<T, 128, 128, 2, 2>(a, epi, (long long)tiles * batch, tiles_n, tiles, st);
}

template <class T, int BK, bool KM>
int launch_split256(const gr_gemm_args& a, int batch, int epi, int tiles, int tiles_n, hipStream_t st) {
  hipLaunchKernelGGL((gr_gemm_w4_kernel<T, KM, GR_EPI_NONE, BK, 256, true>),
                     dim3((unsigned)(tiles * a.ksplit), (unsigned)batch), dim3(256), gr_gemm_w4_lds<BK>::value, st, a);
  const int rc = gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_gemm launch");
  return rc ? rc : launch_merge_epi<T, 256, 256, 2, 2>(a, epi, (long long)tiles * batch, tiles_n, tiles, st);
}

template <class T, bool KM>
int launch(const gr_gemm_args& a, int batch, int epi, const gr::GemmPlan& p, hipStream_t st) {
  const int tiles_n = (a.N + p.bn - 1) / p.bn;
  const long long tiles = (long long)((a.M + p.bm - 1) / p.bm) * tiles_n;
  if (tiles * p.ks > 0x7fffffffLL || batch > 65535)
    return gr::fail(GR_E_ARG, "gr_gemm: grid (%lld tiles, batch %d) out of range", tiles, batch);
  const bool k64 = a.K % 64 == 0;
  if (p.bm == 32) return launch_rows<T, 32, 4, KM>(a, batch, epi, (int)tiles, tiles_n, st);
  if (p.bm == 64) return launch_rows<T, 64, 3, KM>(a, batch, epi, (int)tiles, tiles_n, st);
  if (p.bm == 128)
    return k64 ? launch_split128<T, 64, KM>(a, batch, epi, (int)tiles, tiles_n, st)
               : launch_split128<T, 32, KM>(a, batch, epi, (int)tiles, tiles_n, st);
  return k64 ? launch_split256<T, 64, KM>(a, batch, epi, (int)tiles, tiles_n, st)
             : launch_split256<T, 32, KM>(a, batch, epi, (int)tiles, tiles_n, st);
}

}  // namespace

int gr::launch_gemm_planned(gr_gemm_args a, int dtype, int batch, bool km, int epi, const GemmPlan& plan,
                            hipStream_t st) {
  a.ksplit = plan.ks;
  if (dtype == GR_F16)
    return km ? launch<_Float16, true>(a, batch, epi, plan, st) : launch<_Float16, false>(a, batch, epi, plan, st);
  return km ? launch<__bf16, true>(a, batch, epi, plan, st) : launch<__bf16, false>(a, batch, epi, plan, st);
}
