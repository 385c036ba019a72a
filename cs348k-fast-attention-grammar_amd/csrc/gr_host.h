// gr_host.h -- host-side helpers shared by the HIP translation units of
// libgrammar_rt.so: the error slot and HIP status mapping.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdarg>
#include <cstdio>

#include "gr_err.h"

namespace gr {

// Map a HIP status to GR_OK / `code` with a message naming `what`. A failure is
// taken out of the thread's last-error slot, which keeps it across later
// successful calls: a caller that recovers from it must not meet it again.
int hip_check(hipError_t e, int code, const char* what);

// Compute units of the current device (0 if unknown), read once per device.
int cu_count();

}  // namespace gr
