// What the kernels of the experts' products share.
#pragma once
#include "common.h"

#define MOE_BIG 128  // rows of a tile of the list in steps of more than a few tokens

struct MoeLinearArgs {
  const bf16_t* a;
  long a_stride;
  const bf16_t* w;
  void* out;
  long o_stride;
  const int *tiles, *meta, *sorted;
  int top, gather, K, N, F, act;
  float limit, up_shift;
  int n_cols, vec;
  bool spread;  // tiles of 128 rows: their columns begin at places of their own along K
};

__device__ __forceinline__ float moe_act(float gate, float up, int act, float limit, float up_shift) {
  if (limit > 0.f) gate = fminf(gate, limit), up = fminf(fmaxf(up, -limit), limit);
  return lev_activate(gate, act) * (up + up_shift);
}

// The products of tiles of 128 rows by workgroups that stay (moe_ring.hip). 1: not for these sizes, nothing has been launched.
int lev_moe_ring(const MoeLinearArgs& args, long a_rows, int out_dtype, int glu, int max_tiles, hipStream_t stream);
