// The bfloat16 product of a few rows with the norm ahead of it (gemm_norm.hip).
#pragma once
#include "common.h"

#define NORMED_MAX_M 8
#define NORMED_MAX_K 1024  // a float4 for each of 256 threads
// waves and units as the skinny kernel's shape has them: 8 and 1, 16 and 2 or 3; -1 where there is no such kernel
int lev_normed_launch(int waves, int units, const float* x, const float* nw, const float* nb, float eps, int rms, const bf16_t* w, const float* bias,
                      bf16_t* out, long ldo, int M, int N, int K, int act, hipStream_t stream);
