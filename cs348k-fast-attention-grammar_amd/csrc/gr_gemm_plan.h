// gr_gemm_plan.h -- the tile and K split that gr_gemm picks for a shape (host
// side), and the launches that only a picked plan reaches (gr_gemm_split.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "gr_gemm.h"

namespace gr {

// A tile of C, the parts its K is split into (1: none) and the workspace the
// split's fp32 partial sums take (0 without one).
struct GemmPlan {
  int bm, bn, ks;
  size_t ws;
};

// Largest workspace a picked split may ask for. The splits measured fastest
// over M 24-4096, N 512-11008, K 512-11008 on 256 CUs stay below it.
constexpr size_t kGemmWorkspaceMax = (size_t)64 << 20;

// 32- and 64-row tiles (ks >= 1) and K-split launches of every tile (ks > 1);
// plan.ks parts, partial sums in a.ws.
int launch_gemm_planned(gr_gemm_args a, int dtype, int batch, bool km, int epi, const GemmPlan& plan, hipStream_t st);

}  // namespace gr
