// The bfloat16 product of some dozen to about a thousand rows (gemm_ring.hip): its launch's shape and its launch.
#pragma once
#include "common.h"

#define RING_MAX_K (1 << 24)  // 128 rows of w within 2^32 bytes
struct RingPlan {
  int shape;   // place in the kernel's list of tiles
  int splits;  // ranges of K (1: none)
  double us;   // the estimate, in microseconds
};
RingPlan lev_ring_plan(int M, int N, int K, bool left);  // left: the sums of ranges are left to whoever reads the product next, no kernel of this product's own adds them
// plan.splits > 1: the sums of the ranges go to partial [splits][M][N], without bias, activation and residual
int lev_ring_launch(const RingPlan& plan, const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr, void* out, long ldo,
                    float* partial, int M, int N, int K, int act, int out_dtype, hipStream_t stream);
