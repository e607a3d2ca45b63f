// Sums over the lanes of a wave of several values at once (gemm_norm.hip, gemm_f32_norm.hip).
#pragma once
#include "common.h"

// The sums over a wave's lanes of up to four values, as wave_sum has them: where the halves (and the rows of 16) change places, one register
// takes two values along, so that four cost ten instructions instead of forty.
template <int RP, int WAVES>
__device__ __forceinline__ void store_wave_sums(const float (&part)[RP], float (&to)[RP][WAVES], int wave, int lane) {
  typedef __attribute__((ext_vector_type(2))) uint32_t pair_t;
  auto halves = [](float a, float b) __attribute__((always_inline)) {
    const pair_t h = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);  // {a's lower half, b's lower}, {a's upper, b's upper}
    return __uint_as_float(h[0]) + __uint_as_float(h[1]);
  };
  const float ab = halves(part[0], part[RP > 1 ? 1 : 0]), cd = RP > 2 ? halves(part[RP > 2 ? 2 : 0], part[RP > 3 ? 3 : 0]) : ab;
  const pair_t q = __builtin_amdgcn_permlane16_swap(__float_as_uint(ab), __float_as_uint(cd), false, false);  // {rows ab 0, cd 0, ab 2, cd 2}, {1, 1, 3, 3}
  float v = __uint_as_float(q[0]) + __uint_as_float(q[1]);
#define LEV_ROW_ROTATED(N) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, false))
  v += LEV_ROW_ROTATED(8);
  v += LEV_ROW_ROTATED(4);
  v += LEV_ROW_ROTATED(2);
  v += LEV_ROW_ROTATED(1);
#undef LEV_ROW_ROTATED
  const int j = (lane >> 5) + (lane >> 4 & 1) * 2;  // rows of 16: values 0, 2, 1, 3
  if ((lane & 15) == 0 && j < RP) to[j][wave] = v;
}
