// gr_attn_groups.hip -- instances of the flash body with key groups (KG > 1)
// for grids of few query tiles; gr_attn.hip picks among them and the one-group
// tiles.
//
// A grid below one 256-query workgroup per CU leaves CUs idle, and smaller
// query tiles alone leave SIMDs idle (64 queries are two waves). Here 32 to
// 128 queries get 4 to 8 waves, each group with its own K/V ring: B1 H12 N1344
// d128 bf16 (252 workgroups of 64 queries) 31.3 -> 19.9 us, B1 H4 N1024 d64
// fp16 14.3 -> 9.0 us, N4096 44.7 -> 30.8 us. The price is K/V read from L2
// once per 32-128 queries instead of 256, so full grids stay on one group.
#include <hip/hip_runtime.h>

#include "gr_attn_groups.h"
#include "gr_host.h"
#include "grammar_rt.h"

namespace {

template <class T, int D, int BN, int NW, int KG, bool CAUSAL, bool KT>
int launch(const gr_attn_args& a, hipStream_t st) {
  constexpr int BM = NW * 32, LDS = KG * gr_flash_lds<D, BN>::BYTES;
  static_assert((D * BN / 8) % (NW * 64) == 0, "direct loads: whole chunks per thread");
  const long long nblk = (long long)a.B * a.H * ((a.N + BM - 1) / BM);
  if (nblk <= 0 || nblk > 0x7fffffffLL) return gr::fail(GR_E_ARG, "gr_attn_fwd: grid size %lld out of range", nblk);
  hipLaunchKernelGGL((gr_flash_fwd_kernel<T, D, BN, NW, 1, CAUSAL, KT, false, true, true, false, true, KG>),
                     dim3((unsigned)nblk), dim3(NW * KG * 64), LDS, st, a);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd launch");
}

template <class T, bool CAUSAL, bool KT>
int dispatch(const gr_attn_args& a, int D, int nw, int kg, hipStream_t st) {
  if (D == 64 && nw == 1 && kg == 4) return launch<T, 64, 32, 1, 4, CAUSAL, KT>(a, st);
  if (D == 64 && nw == 1 && kg == 8) return launch<T, 64, 32, 1, 8, CAUSAL, KT>(a, st);
  if (D == 64 && nw == 2 && kg == 2) return launch<T, 64, 64, 2, 2, CAUSAL, KT>(a, st);
  if (D == 64 && nw == 4 && kg == 2) return launch<T, 64, 64, 4, 2, CAUSAL, KT>(a, st);
  if (D == 128 && nw == 2 && kg == 4) return launch<T, 128, 32, 2, 4, CAUSAL, KT>(a, st);
  if (D == 128 && nw == 4 && kg == 2) return launch<T, 128, 64, 4, 2, CAUSAL, KT>(a, st);
  return gr::fail(GR_E_ARG, "gr_attn_fwd: no instance of %d waves x %d key groups at D=%d", nw, kg, D);
}

}  // namespace

int gr::launch_flash_groups(const gr_attn_args& a, int dtype, int D, bool causal, bool kt, int nw, int kg,
                            hipStream_t st) {
#define GR_CASE(C, K)                                                                 \
  if (causal == C && kt == K)                                                         \
    return dtype == GR_F16 ? dispatch<_Float16, C, K>(a, D, nw, kg, st) : dispatch<__bf16, C, K>(a, D, nw, kg, st);
  GR_CASE(false, false)
  GR_CASE(false, true)
  GR_CASE(true, false)
  GR_CASE(true, true)
#undef GR_CASE
  return GR_E_ARG;
}
