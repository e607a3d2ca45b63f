// What the kernels of the 32-bit products share (gemm_f32.hip, gemm_f32_split.hip).
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float gf_f32x4;

// gemm_f32_split.hip: its tiles, and a product with one of them (inputs and lda up to GEMM_F32_SPLIT_MOST: offsets within a tile are 32-bit numbers of bytes)
#define GEMM_F32_SPLIT_MOST (1 << 22)
struct GemmF32SplitTile {
  int rows, outputs, groups;   // groups of waves that share the steps of 32 inputs
  float start, alone, among;   // microseconds: before and behind the products, of a step of the one workgroup on a CU, and of one among several,
  float odd, single;           // what a step takes longer where the last of several is left alone, and a tile whose outputs are stored one by one (N no multiple of 4)
};
static const GemmF32SplitTile GEMM_F32_SPLIT_TILES[] = {{128, 128, 1, 5.093f, 1.048f, 1.257f, 0.125f, 2.561f}, {64, 128, 1, 2.216f, 0.768f, 0.689f, 0.256f, 1.586f},
                                                        {64, 64, 2, 5.049f, 0.651f, 1.132f, 0.052f, 1.553f}};
#define GEMM_F32_N_SPLIT_TILES (int)(sizeof(GEMM_F32_SPLIT_TILES) / sizeof(GEMM_F32_SPLIT_TILES[0]))
extern "C" int lev_linear_f32_choice(int M, int N, int K);
extern "C" int lev_linear_f32_split(int M, int N, int K);
int lev_gemm_f32_split(int tile, const float* a, long lda, const float* w, const float* bias, const float* residual, long ldr, float* out, long ldo, int M, int N, int K,
                       int act, int vec, hipStream_t stream);

// four neighbouring outputs of a row
__device__ __forceinline__ void gemm_f32_store(gf_f32x4 v, const float* bias, const float* residual, long ldr, float* out, long ldo, int m, int o, int N, int act, int vec) {
  if (vec && o + 4 <= N) {
    if (bias) v += *reinterpret_cast<const gf_f32x4*>(bias + o);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = lev_activate(v[r], act);
    if (residual) v += *reinterpret_cast<const gf_f32x4*>(residual + (size_t)m * ldr + o);
    *reinterpret_cast<gf_f32x4*>(out + (size_t)m * ldo + o) = v;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (o + r >= N) break;
      float x = v[r];
      if (bias) x += bias[o + r];
      x = lev_activate(x, act);
      if (residual) x += residual[(size_t)m * ldr + o + r];
      out[(size_t)m * ldo + o + r] = x;
    }
  }
}
