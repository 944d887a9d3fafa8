// float32 x by bfloat16 w on the bfloat16 matrix instruction (gemm_split.hip), for the general product's entry (gemm_generic.hip).
#pragma once

#include "common.h"

namespace lc {

bool gemm_split_takes(int K);
// part == nullptr: out.  Else the sums of every chunk of 256 k go to part[chunk][M][N], `shares` workgroups a tile with `per` chunks each.
void launch_gemm_split(const float* x, const bf16* w, float* out, int M, int N, int K, float* part, int per, int shares, hipStream_t stream);

}  // namespace lc
