// gr_attn_groups.h -- attention forward launches compiled outside gr_attn.hip:
// workgroups that split the keys over groups of waves (gr_flash_fwd_body's KG,
// gr_attn_groups.hip) and the fp32 forward (gr_attn_f32.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "gr_flash_fwd.h"

namespace gr {

// nw waves of 32 queries x kg key groups; N a multiple of 64, any remainder of
// the query tile. (nw, kg) in {(1, 4), (1, 8), (2, 2), (4, 2)} at D = 64,
// {(2, 4), (4, 2)} at D = 128; dtype GR_F16 (Q pre-scaled) or GR_BF16.
int launch_flash_groups(const gr_attn_args& a, int dtype, int D, bool causal, bool kt, int nw, int kg, hipStream_t st);

// fp32 attention forward (gr_attn_f32.hip).
int attn_fwd_f32(const gr_attn_args& a, int D, bool causal, bool k_transposed, bool train, hipStream_t st);

}  // namespace gr
