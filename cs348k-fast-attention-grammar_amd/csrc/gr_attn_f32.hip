// gr_attn_f32.hip -- the fp32 attention forward (gr_flash_f32.h) behind
// gr_attn_fwd(). Compiled with MFMAs in VGPR form (build_native.py): left to
// its heuristics the backend keeps the score accumulators in AGPRs and copies
// them to VGPRs and back for the softmax of every key block.
#include <hip/hip_runtime.h>

#include <mutex>
#include <thread>
#include <vector>

#include "gr_attn_groups.h"
#include "gr_flash_f32.h"
#include "gr_host.h"
#include "grammar_rt.h"

namespace {

// A workgroup owns 32 queries and shares its keys out over its four waves
// (merged through LDS); with PARTS > 1 the keys of a query block are also
// shared out over PARTS workgroups. d = 64 fits two waves per SIMD, whose
// softmax and MFMAs then overlap (192 VGPRs); d = 128 takes one. Bound by the
// fp32 matrix cores (155 TFLOP/s at most) once they are filled: 16 heads,
// N 2048, D 128 278 us (124 TFLOP/s; with equal power-of-two shares of the
// keys, K and V double-buffered and 64-bit row products per load it was 406),
// 8 heads D 64 72 us (was 94); below that by the longest wave.
template <int D, int NW, bool KT, int PARTS, bool WIDE, int ONE>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1)))
void gr_flash32_kernel(gr_attn_args a, int blocks, float* ws_o, float* ws_ml) {
  extern __shared__ __attribute__((aligned(16))) char gr_lds[];
  gr_flash32_fwd_body<D, 32, NW, KT, PARTS, WIDE, ONE>(a, gr_lds, ws_o, ws_ml, blocks);
}

template <int D, int PARTS>
__global__ __launch_bounds__(256) void gr_flash32_merge_kernel(gr_attn_args a, const float* ws_o, const float* ws_ml) {
  gr_flash32_merge_body<D, PARTS>(a, ws_o, ws_ml);
}

// Workgroups a split launch may have: one per CU of an MI355X. It bounds the
// workspace.
constexpr long long kF32SplitTarget = 256;

// Workspace of the fp32 key split: one buffer per (device, stream), allocated
// by the first call that splits on it and kept until the process ends (queued
// work and captured graphs may still read it). Calls on one stream run in
// order, so they can share it. hipStreamPerThread names a different stream in
// every host thread, so its buffers are kept per thread as well. A split
// launch has at most kF32SplitTarget workgroups of 32 query rows (query
// blocks x parts), so one size holds every call's. It has two halves: the splits
// that captured calls may take (capture_parts) have the first to themselves, so
// that a graph replayed on another stream shares it with such calls only.
constexpr size_t kF32WorkspaceBytes = (size_t)kF32SplitTarget * 32 * (128 + 2) * sizeof(float);   // 4.3 MB a half

struct F32Workspace {
  int dev;
  hipStream_t st;
  std::thread::id thread;
  void* p;
};
std::mutex g_f32_ws_lock;
std::vector<F32Workspace> g_f32_ws;
thread_local int t_fail_workspaces = 0;   // gr_selftest_f32_no_workspace: lookups still to fail

// The caller holds g_f32_ws_lock, and keeps it over the launches that use the
// buffer: another thread's split call on the same stream then queues behind
// both of them.
int f32_workspace(hipStream_t st, void** out) {
  int dev = 0;
  int rc = gr::hip_check(hipGetDevice(&dev), GR_E_RUNTIME, "gr_attn_fwd: hipGetDevice");
  if (rc) return rc;
  const std::thread::id thread = st == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id();
  size_t bytes = 2 * kF32WorkspaceBytes;
  if (t_fail_workspaces > 0) {
    --t_fail_workspaces;
    bytes = (size_t)1 << 60;              // more than any device has
  } else {
    for (auto& e : g_f32_ws)
      if (e.dev == dev && e.st == st && e.thread == thread) {
        *out = e.p;
        return GR_OK;
      }
  }
  void* p = nullptr;
  rc = gr::hip_check(hipMalloc(&p, bytes), GR_E_RUNTIME, "gr_attn_fwd: fp32 key-split workspace");
  if (rc) return rc;
  g_f32_ws.push_back({dev, st, thread, p});
  *out = p;
  return GR_OK;
}

bool capturing(hipStream_t st) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const bool known = hipStreamIsCapturing(st, &cap) == hipSuccess;
  if (!known) (void)hipGetLastError();
  return !known || cap != hipStreamCaptureStatusNone;
}

template <int D, bool KT, int PARTS, bool WIDE = false>
int launch_parts(const gr_attn_args& a, long long nblk, float* ws_o, float* ws_ml, hipStream_t st) {
  const dim3 grid((unsigned)(nblk * PARTS));
  constexpr int LDS = gr_flash32_lds<D, 4>::BYTES;
  const int blocks = a.N / 32;
  // one and two blocks: as many waves (5 heads, N 32, D 128: 7.2 us, 7.8 with
  // three idle waves in the merge)
  if (!WIDE && PARTS == 1 && blocks == 1)
    hipLaunchKernelGGL((gr_flash32_kernel<D, 1, KT, 1, false, 1>), grid, dim3(64), (gr_flash32_lds<D, 1>::BYTES), st, a,
                       blocks, ws_o, ws_ml);
  else if (!WIDE && PARTS == 1 && blocks == 2)
    hipLaunchKernelGGL((gr_flash32_kernel<D, 2, KT, 1, false, 1>), grid, dim3(128), (gr_flash32_lds<D, 2>::BYTES), st, a,
                       blocks, ws_o, ws_ml);
  else if (!WIDE && blocks == 4 * PARTS)
    hipLaunchKernelGGL((gr_flash32_kernel<D, 4, KT, PARTS, false, 1>), grid, dim3(256), LDS, st, a, blocks, ws_o, ws_ml);
  else if (!WIDE && blocks < 4 * PARTS)
    hipLaunchKernelGGL((gr_flash32_kernel<D, 4, KT, PARTS, false, 2>), grid, dim3(256), LDS, st, a, blocks, ws_o, ws_ml);
  else
    hipLaunchKernelGGL((gr_flash32_kernel<D, 4, KT, PARTS, WIDE, 0>), grid, dim3(256), LDS, st, a, blocks, ws_o, ws_ml);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd fp32 launch");
}

template <int D, bool KT, int PARTS>
int launch_split(const gr_attn_args& a, long long nblk, int fixed, hipStream_t st) {
  const long long rows = (long long)a.B * a.H * a.N;
  const size_t o_floats = (size_t)PARTS * rows * D;
  std::lock_guard<std::mutex> hold(g_f32_ws_lock);
  void* ws = nullptr;
  int rc = f32_workspace(st, &ws);
  if (rc && !capturing(st)) return launch_parts<D, KT, 1>(a, nblk, nullptr, nullptr, st);   // no memory for it
  if (rc) return rc;
  float* ws_o = static_cast<float*>(ws) + (PARTS == fixed ? 0 : kF32WorkspaceBytes / sizeof(float));
  float* ws_ml = ws_o + o_floats;
  rc = launch_parts<D, KT, PARTS>(a, nblk, ws_o, ws_ml, st);
  if (rc) return rc;
  const long long threads = rows * (D / 8);
  hipLaunchKernelGGL((gr_flash32_merge_kernel<D, PARTS>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st,
                     a, (const float*)ws_o, (const float*)ws_ml);
  return gr::hip_check(hipGetLastError(), GR_E_LAUNCH, "gr_attn_fwd fp32 merge launch");
}

// Key parts of a call: the number that a model of the launch gives the least
// time. A wave takes `block` us per 32-key block; CUs run their workgroups'
// waves together at d = 64 (two per SIMD) and one after another at d = 128;
// more than one part adds the merge launch. The blocks need not divide: 3
// heads at N 1184, D 128 take two parts of four and five blocks a wave, 31 us
// (one wave per query block, as N not a multiple of 64 had it, 178 us); 4 heads
// at N 320, D 64 two of one and two, 9 us (one workgroup of two waves 15.7).
int pick_parts(int D, long long nblk, int blocks) {
  const double block = D == 64 ? 2.1 : 4.1, shared = D == 64 ? 1.85 : 4.1;
  const int cus = gr::cu_count() > 0 ? gr::cu_count() : 256;
  int best = 1;
  double best_t = 1e30;
  for (int p = 1; p <= 8; p *= 2) {
    if (p > 1 && (nblk * p > kF32SplitTarget || 4 * (p / 2) >= blocks)) break;
    const int run = (blocks + 4 * p - 1) / (4 * p);
    const double per_cu = (double)((nblk * p + cus - 1) / cus) * run * shared;
    const double t = (per_cu > run * block ? per_cu : run * block) + (p > 1 ? 3.0 : 0.0);
    if (t < best_t) {
      best_t = t;
      best = p;
    }
  }
  return best;
}

// The key parts that a captured call may use: the workspace of a split must
// be there already and not be shared with other work, so under capture only
// the shapes split that are documented to (N a multiple of 256 ...).
int capture_parts(long long nblk, int N) {
  const int run = N % 128 == 0 ? N / 128 : 0;
  for (int p = 8; p > 1; p /= 2)
    if (run > 0 && run % p == 0 && nblk * p <= kF32SplitTarget) return p;
  return 1;
}

template <int D, bool KT>
int launch_flash32(const gr_attn_args& a, hipStream_t st) {
  const long long nblk = (long long)a.B * a.H * (a.N / 32);
  if (nblk <= 0 || nblk > 0x7fffffffLL) return gr::fail(GR_E_ARG, "gr_attn_fwd: grid size %lld out of range", nblk);
  constexpr long long kWide = 1LL << 27;
  if (a.v_sn >= kWide || (KT && a.k_sn >= kWide)) return launch_parts<D, KT, 1, true>(a, nblk, nullptr, nullptr, st);
  int parts = pick_parts(D, nblk, a.N / 32);
  const int fixed = capture_parts(nblk, a.N);
  if (parts > 1 && parts != fixed && capturing(st)) parts = fixed;
  if (parts == 8) return launch_split<D, KT, 8>(a, nblk, fixed, st);
  if (parts == 4) return launch_split<D, KT, 4>(a, nblk, fixed, st);
  if (parts == 2) return launch_split<D, KT, 2>(a, nblk, fixed, st);
  return launch_parts<D, KT, 1>(a, nblk, nullptr, nullptr, st);
}

}  // namespace

int gr::attn_fwd_f32(const gr_attn_args& a, int D, bool causal, bool k_transposed, bool train, hipStream_t st) {
  if (causal) return gr::fail(GR_E_ARG, "gr_attn_fwd: fp32 is non-causal only (the reference's fp32 workload)");
  if (train) return gr::fail(GR_E_ARG, "gr_attn_fwd_train: fp32 has no training path (GR_F16 or GR_BF16)");
  if (a.N % 32) return gr::fail(GR_E_ARG, "gr_attn_fwd: fp32 needs N a multiple of 32 (got %d)", a.N);
  if (D == 64) return k_transposed ? launch_flash32<64, true>(a, st) : launch_flash32<64, false>(a, st);
  if (D == 128) return k_transposed ? launch_flash32<128, true>(a, st) : launch_flash32<128, false>(a, st);
  return gr::fail(GR_E_ARG, "gr_attn_fwd: head dim %d unsupported (64 or 128)", D);
}

extern "C" int gr_selftest_f32_no_workspace(int lookups) {
  if (lookups < 0) return gr::fail(GR_E_ARG, "gr_selftest_f32_no_workspace: negative count");
  t_fail_workspaces = lookups;
  return GR_OK;
}
