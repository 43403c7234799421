#pragma once

#include "svdq_common.h"

namespace svdq {

// The kernel with 256-row tiles (gemm_w4a4_wide.hip).  `a` has wgt_planes and has passed svdq_gemm_w4a4's checks.
bool wide_runs(const svdq_gemm_args &a);             // whether it can run this launch: blocked fp6 codes and scales
bool wide_takes(const svdq_gemm_args &a, int cus);  // whether it then is the faster one on a device of `cus` compute units

// The launch; `a` has rows to write.
void launch_gemm_wide(const svdq_gemm_args &a, int cus, hipStream_t s);

}  // namespace svdq
