// gr_flash_f32.h -- fp32 attention forward on the fp32 matrix cores of gfx950
// (v_mfma_f32_32x32x2_f32), for the grammar's fp32 programs: keys split over
// the waves of a workgroup (merged in LDS) and, optionally, over workgroups
// (merged by a second launch).
//
//   O = softmax(scale * Q K^T) V      Q, V, O [B, H, N, D], K natural or K^T
//
// The reference's own attention workload is fp32 and small (one head,
// N = 512, d = 64: 67 MFLOP). At the fp32 matrix cores' rate one wave takes
// about 2 us per 32 x 32 block of queries x keys, so the work is spread as
// wide as the problem allows. A workgroup owns one 32-query block and NW
// consecutive runs of 32-key blocks, one per wave; a wave runs the online softmax
// over its run with its operands read straight from global memory into registers
// (the next block's K in flight during this block's MFMAs). The runs are BN / 32
// blocks each in rendered stages (there PARTS = N / (NW BN)); behind gr_attn_fwd
// the call's N / 32 blocks are shared out over the NW PARTS waves in runs that
// differ by at most one. The NW partials (O, m, l) are merged through LDS, each
// wave merging a D / NW slice. With PARTS > 1 workgroups per query block, each
// leaves its merged partial in a workspace and a second launch
// (gr_flash32_merge_body) combines them,
//   O = sum_s 2^((m_s - M) c) O_s / sum_s 2^((m_s - M) c) l_s,  M = max_s m_s.
// The workspace is module-scope device arrays the renderer sizes for the
// stage (two launches of one module must not overlap), or, behind
// gr_attn_fwd, a buffer the library keeps per (device, stream).
//
//  * Transposed form as in gr_flash_fwd_body: S^T = K Q^T, O^T = V^T P^T. A
//    32x32x2 MFMA contracts one index per half-wave: for d the lane of half g
//    takes d = 8 dg + 4 g + t in MFMA t of group dg (one 16-byte load of Q and
//    of a natural K row per group); for the keys the score accumulators are
//    the P operand as they stand (accumulator r is key 8 (r / 4) + 4 g + r % 4,
//    MFMA t takes r = t), and V's row of that key is read at d = lane % 32.
//  * Lane-local softmax (each lane owns one query and half the block's keys):
//    one exchange with the other half-wave per block for the max.
#pragma once
#include "gr_flash_fwd.h"

template <int D, int NW>
struct gr_flash32_lds {
  static constexpr int LD = D + 4;                       // padded row of a wave's O partial (floats)
  static constexpr int O_FLOATS = NW * 32 * LD;
  static constexpr int BYTES = (O_FLOATS + NW * 32 * 2) * 4;
};

// blocks: the call's 32-key blocks, N / 32, shared out over the NW PARTS waves
// in consecutive runs that differ by at most one (the library launches; a wave
// may get none); 0: BN / 32 blocks each (rendered stages).
// ONE: 1: every wave has exactly one block (no branch, loop or rescale: 6.3 ->
// 5.9 us at D 64, N 512, one head); 2: at most one.
// WIDE: 64-bit lane addresses for V and K^T (row strides of 2^27 elements and
// more), else a wave-uniform row pointer plus a 32-bit lane offset.
template <int D, int BN, int NW, bool KT_LAYOUT, int PARTS, bool WIDE = false, int ONE = 0>
__device__ __forceinline__ void gr_flash32_fwd_body(const gr_attn_args& a, char* lds, float* ws_o, float* ws_ml,
                                                    int blocks = 0) {
  constexpr int DB = D / 32;       // 32-wide head-dim blocks of O^T
  constexpr int DG = D / 8;        // groups of 8 d (4 MFMAs of 2)
  constexpr int SL = D / NW;       // head dims each wave merges
  typedef gr_flash32_lds<D, NW> L;
  static_assert(D % 32 == 0 && BN % 32 == 0 && SL % 16 == 0, "tile shape: D / NW a multiple of 16");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5, l32 = lane & 31;
  const int lead = a.B * a.H;
  const int nqb = a.N / 32;
  const int wg = gr_xcd_remap_any((int)blockIdx.x, (int)gridDim.x);
  const int bh = wg / (nqb * PARTS);
  const int rem = wg % (nqb * PARTS);
  const int part = rem / nqb, qblk = rem % nqb;        // an XCD's workgroups share a part's keys
  const int b = bh / a.H, h = bh % a.H;
  const float* Qp = (const float*)a.q + b * a.q_sb + h * a.q_sh;
  const float* Kp = (const float*)a.k + b * a.k_sb + h * a.k_sh;
  const float* Vp = (const float*)a.v + b * a.v_sb + h * a.v_sh;
  float* Op = (float*)a.o + b * a.o_sb + h * a.o_sh;
  const int q0 = qblk * 32;
  const int chunk = part * NW + __builtin_amdgcn_readfirstlane(wave);
  const int b0 = blocks > 0 ? blocks * chunk / (NW * PARTS) : chunk * (BN / 32);                 // first key block
  const int nb = blocks > 0 ? blocks * (chunk + 1) / (NW * PARTS) - b0 : BN / 32;                // their count
  const float c = a.scale_log2;

  gr_f32x4 qf[DG];
#pragma unroll
  for (int dg = 0; dg < DG; ++dg)
    qf[dg] = *reinterpret_cast<const gr_f32x4*>(Qp + (long long)(q0 + l32) * a.q_sn + 8 * dg + 4 * g);

  // Operands of one 32-key block: K (MFMA A of the scores) and V (MFMA A of P
  // V). V and K^T are read down a column of the tile, one row per load: a
  // wave-uniform row pointer stepped by the stride (two scalar adds) plus the
  // lane's 32-bit offset, made opaque per block so that it stays 32 bits wide
  // (as hoisted 64-bit lane addresses the loads cost a vector add each, as
  // products by run-time strides more scalar time than the MFMAs).
  const unsigned int v_off = (unsigned int)(4 * g * a.v_sn + l32) * 4u, k_off = (unsigned int)(4 * g * a.k_sn + l32) * 4u;
  const float* const k_lane = Kp + (long long)l32 * a.k_sn + 4 * g;          // natural K: the lane's key row
  auto column = [&](const float* base, unsigned int off, long long g_elems) {   // base + off, as the load wants it
    struct ptr {
      const char* row;
      unsigned int off;
      __device__ __forceinline__ float at(int bytes) const {
        return *reinterpret_cast<const float*>(row + off + bytes);
      }
    };
    if constexpr (WIDE) return ptr{reinterpret_cast<const char*>(base + g_elems), 0u};
    asm volatile("" : "+v"(off));
    return ptr{reinterpret_cast<const char*>(base), off};
  };
  // a block's K, group dg of 8 d at a time, from p (K^T, stepped) or kp
  auto k_column = [&](int kr) { return column(Kp + kr, k_off, 4 * g * a.k_sn + l32); };
  auto load_k = [&](auto& p, int kr, int dg, gr_f32x4 (&kf)[DG]) {
    if constexpr (KT_LAYOUT) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        kf[dg][t] = p.at(0);
        p.row += a.k_sn * 4 * (t == 3 ? 5 : 1);
      }
    } else {
      kf[dg] = *reinterpret_cast<const gr_f32x4*>(k_lane + (long long)kr * a.k_sn + 8 * dg);
    }
  };
  // its V, row t at a time
  auto load_v = [&](auto& p, int t, float (&vf)[DB][16]) {
#pragma unroll
    for (int db = 0; db < DB; ++db) vf[db][t] = p.at(128 * db);
    p.row += a.v_sn * 4 * ((t & 3) == 3 ? 5 : 1);
  };

  gr_f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = (gr_f32x16)(0.f);
  float m = -GR_INF, l = 0.f;
  gr_f32x4 kf[DG];
  float vf[DB][16];
  gr_f32x16 s;
  // One 32-key block, its K in kf: S^T = K Q^T (s[r]: key 8 (r / 4) + 4 g + r
  // % 4, query q0 + l32), the online softmax, O^T += V^T P^T. One buffer each
  // for K and V: V's rows are loaded between the score MFMAs and (NEXT) the
  // K of block `next` between the P V MFMAs, in the order of their use, so
  // that every load has 2,048 (d = 64) or 4,096 cycles of MFMAs to land behind
  // and its address arithmetic issues under them (all loads ahead of the MFMAs
  // took D 128, one block per wave, from 8.8 to 9.5 us). HOLD pins that order;
  // the compiler's own is the better one only for a single block of natural K
  // at D 128 (9.8 -> 9.5 us; at D 64 5.9 -> 7.4).
  constexpr bool HOLD = !(ONE && D == 128 && !KT_LAYOUT);
  auto block = [&](int kr, int next, auto next_tag) {
    constexpr bool NEXT = decltype(next_tag)::value;
    auto vp = column(Vp + (long long)kr * a.v_sn, v_off, 4 * g * a.v_sn + l32);
    s = (gr_f32x16)(0.f);
#pragma unroll
    for (int dg = 0; dg < DG; ++dg) {
#pragma unroll
      for (int t = dg * 16 / DG; t < (dg + 1) * 16 / DG; ++t) load_v(vp, t, vf);
#pragma unroll
      for (int t = 0; t < 4; ++t) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[dg][t], qf[dg][t], s, 0, 0, 0);
      if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);
    }
    float mt = -GR_INF;
#pragma unroll
    for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[r]);
    mt = fmaxf(mt, gr_xor32(mt));
    const float mn = fmaxf(m, mt);
    if constexpr (ONE) {                           // nothing before it
      m = mt;
    } else if (gr_any(mn > m)) {                   // else every factor is 1
      const float alpha = gr_exp2((m - mn) * c);   // m = -inf -> 0
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
      m = mn;
    }
    const float mc = m * c;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = gr_exp2(fmaf(s[r], c, -mc));
      l += s[r];
    }
    auto kp = k_column(next);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      if constexpr (NEXT) {
#pragma unroll
        for (int dg = t * DG / 16; dg < (t + 1) * DG / 16; ++dg) load_k(kp, next, dg, kf);
      }
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[db][t], s[t], o[db], 0, 0, 0);
      if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (ONE == 1 || nb > 0) {
    {
      auto kp = k_column(32 * b0);
#pragma unroll
      for (int dg = 0; dg < DG; ++dg) load_k(kp, 32 * b0, dg, kf);
    }
    // The last block: from K^T it loads its own K again, from natural K it is a
    // copy of the body without that load (16-byte loads that are not wanted cost
    // more than the copy's join, which waits for K).
    if (ONE || (blocks == 0 && BN == 32)) {
      block(32 * b0, 0, gr_ic<0>{});
    } else {
      constexpr int COPY = KT_LAYOUT ? 0 : 1;
#pragma unroll 1
      for (int i = 0; i < nb - COPY; ++i)
        block(32 * (b0 + i), 32 * (b0 + gr_imin(i + 1, nb - 1)), gr_ic<1>{});
      if constexpr (COPY == 1) block(32 * (b0 + nb - 1), 0, gr_ic<0>{});
    }
  }
  l += gr_xor32(l);

  // the NW wave partials -> LDS: O^T lane (query l32, half g) holds d =
  // 32 db + 8 (r / 4) + 4 g + r % 4; rows padded so the 16-byte writes of 16
  // consecutive queries fall on distinct banks
  float* lo = reinterpret_cast<float*>(lds);
  float* lml = lo + L::O_FLOATS;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      *reinterpret_cast<gr_f32x4*>(lo + (wave * 32 + l32) * L::LD + 32 * db + 8 * rr + 4 * g) =
          (gr_f32x4){o[db][4 * rr], o[db][4 * rr + 1], o[db][4 * rr + 2], o[db][4 * rr + 3]};
  if (g == 0) *reinterpret_cast<gr_f32x2*>(lml + (wave * 32 + l32) * 2) = (gr_f32x2){m, l};
  __syncthreads();

  // merge of the workgroup's chunks: wave w, lane (query l32, half g) takes
  // head dims SL w + 16 p + 8 g + 0..7 of its slice
  const int d0 = SL * wave + 8 * g;
  float mx = -GR_INF;
#pragma unroll
  for (int w = 0; w < NW; ++w) mx = fmaxf(mx, lml[(w * 32 + l32) * 2]);
  constexpr int PER = SL / 16;                         // 8-wide pieces per lane
  float acc[PER][8];
#pragma unroll
  for (int p = 0; p < PER; ++p)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[p][e] = 0.f;
  float L_ = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const gr_f32x2 ml = *reinterpret_cast<const gr_f32x2*>(lml + (w * 32 + l32) * 2);
    const float e = gr_exp2((ml[0] - mx) * c);
    L_ = fmaf(e, ml[1], L_);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const float* src = lo + (w * 32 + l32) * L::LD + d0 + 16 * p;
      const gr_f32x4 v0 = *reinterpret_cast<const gr_f32x4*>(src);
      const gr_f32x4 v1 = *reinterpret_cast<const gr_f32x4*>(src + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[p][i] = fmaf(e, v0[i], acc[p][i]);
        acc[p][4 + i] = fmaf(e, v1[i], acc[p][4 + i]);
      }
    }
  }
  auto store_o = [&](float Lv) {
    const float inv = 1.0f / Lv;
    float* dst = Op + (long long)(q0 + l32) * a.o_sn + d0;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      *reinterpret_cast<gr_f32x4*>(dst + 16 * p) =
          (gr_f32x4){acc[p][0] * inv, acc[p][1] * inv, acc[p][2] * inv, acc[p][3] * inv};
      *reinterpret_cast<gr_f32x4*>(dst + 16 * p + 4) =
          (gr_f32x4){acc[p][4] * inv, acc[p][5] * inv, acc[p][6] * inv, acc[p][7] * inv};
    }
  };
  if constexpr (PARTS == 1) {
    store_o(L_);
  } else {
    // this workgroup's merged partial -> workspace, for gr_flash32_merge_body
    const long long row = (long long)(part * lead + bh) * a.N + q0 + l32;
    float* wo = ws_o + row * D + d0;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      *reinterpret_cast<gr_f32x4*>(wo + 16 * p) = (gr_f32x4){acc[p][0], acc[p][1], acc[p][2], acc[p][3]};
      *reinterpret_cast<gr_f32x4*>(wo + 16 * p + 4) = (gr_f32x4){acc[p][4], acc[p][5], acc[p][6], acc[p][7]};
    }
    if (wave == 0 && g == 0) *reinterpret_cast<gr_f32x2*>(ws_ml + row * 2) = (gr_f32x2){mx, L_};
  }
}

// The second launch of a split stage: O from the PARTS partials of every
// query, O = sum_s 2^((m_s - M) c) O_s / sum_s 2^((m_s - M) c) l_s with
// M = max_s m_s. One thread per (query row, 8 head dims); the grid covers
// lead * N * D / 8 threads in workgroups of 256.
template <int D, int PARTS>
__device__ __forceinline__ void gr_flash32_merge_body(const gr_attn_args& a, const float* ws_o, const float* ws_ml) {
  constexpr int CH = D / 8;
  const int lead = a.B * a.H;
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long rows = (long long)lead * a.N;
  if (idx >= rows * CH) return;
  const int ch = (int)(idx % CH);
  const long long r = idx / CH;                     // bh * N + q
  const int bh = (int)(r / a.N), q = (int)(r % a.N);
  const float c = a.scale_log2;
  float mx = -GR_INF;
#pragma unroll
  for (int s = 0; s < PARTS; ++s) mx = fmaxf(mx, ws_ml[((long long)s * rows + r) * 2]);
  float L = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < PARTS; ++s) {
    const gr_f32x2 ml = *reinterpret_cast<const gr_f32x2*>(ws_ml + ((long long)s * rows + r) * 2);
    const float w = gr_exp2((ml[0] - mx) * c);
    L = fmaf(w, ml[1], L);
    const float* src = ws_o + ((long long)s * rows + r) * D + ch * 8;
    const gr_f32x4 v0 = *reinterpret_cast<const gr_f32x4*>(src);
    const gr_f32x4 v1 = *reinterpret_cast<const gr_f32x4*>(src + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[e] = fmaf(w, v0[e], acc[e]);
      acc[4 + e] = fmaf(w, v1[e], acc[4 + e]);
    }
  }
  const float inv = 1.0f / L;
  const int b = bh / a.H, h = bh % a.H;
  float* dst = (float*)a.o + b * a.o_sb + h * a.o_sh + (long long)q * a.o_sn + ch * 8;
  *reinterpret_cast<gr_f32x4*>(dst) = (gr_f32x4){acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
  *reinterpret_cast<gr_f32x4*>(dst + 4) = (gr_f32x4){acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv};
}
