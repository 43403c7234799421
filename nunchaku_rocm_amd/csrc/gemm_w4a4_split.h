#pragma once

#include "svdq_common.h"

namespace svdq {

// Wavefronts of a workgroup of the split-K kernel for launches with few rows (gemm_w4a4_split.hip) on a device of `cus`
// compute units, 0 where the kernels with 128 x 128 tiles are the better ones.  `a` has wgt_planes, and unsigned activations or
// act_blocked == 2.
int split_wavefronts(const svdq_gemm_args &a, int cus);

// The launch on a device of `cus` compute units, for `wavefronts` = 4 or 8; `a` has passed svdq_gemm_w4a4's checks and has rows to write.
void launch_gemm_split(const svdq_gemm_args &a, int wavefronts, int cus, hipStream_t s);

}  // namespace svdq
