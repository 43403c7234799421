#pragma once

#include "svdq_common.h"

namespace svdq {

// The split-K kernel for launches with few rows (gemm_w4a4_split.hip) on a device of `cus` compute units; returns false, and
// launches nothing, where the kernels with 128 x 128 tiles are the better ones.  `a` has passed svdq_gemm_w4a4's checks and
// has wgt_planes, unsigned activations or act_blocked == 2, and rows to write.
bool launch_gemm_split(const svdq_gemm_args &a, int cus, hipStream_t s);

}  // namespace svdq
