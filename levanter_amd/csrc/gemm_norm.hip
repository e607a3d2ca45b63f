// out = act(norm(x) . w^T + bias) for up to 8 rows of up to 1,024 numbers: LayerNorm or RMSNorm of float32 rows x [M][K] and the bfloat16 product behind it in one
// launch. The skinny kernel (gemm_mfma.hip) with every workgroup normalising the rows for itself.
// What bounds the two kernels apart is waiting: the norm of a few rows computes for a fraction of a microsecond, the rest of its 2 to 5 is its launch and the
// trip to memory for scale and shift (a model's weights have passed through the caches since they were read last); then the product begins its own trip. Here
// both trips are one: a wave requests its rows, then scale and shift (loads come back in order, and the statistics wait for the rows alone), then ALL its weights, and
// the statistics pass while the weights are on their way. A barrier without a wait keeps the weights of the first waves behind the rows of the last.
// The norm is worked out as norm_reg_kernel works it out with 256 threads a row (groups of four waves, a vector a thread, the same order of sums), and the
// product as gemm_skinny_kernel does: the same bits as the two kernels one after the other. The rows stay in LDS in bfloat16, an odd number of 16-byte chunks
// apart, so that the operand's 16 rows are read without a conflict.
// Measured in graphs over distinct weights and norms, microseconds, two kernels / here: 2304 x 768 at 1 / 4 / 8 rows 5.1 / 3.5, 5.7 / 4.4, 5.9 / 5.0; 4096 x 1024
// 6.0 / 3.6, 6.4 / 4.5, 6.6 / 5.1; 8192 x 1024 8.0 / 6.0, 8.6 / 6.7, 8.6 / 7.4. A session of GPT-2 small, one request: 7.50 -> 6.66 ms. Not beyond 8 rows or 1,024 numbers: the work that
// every workgroup repeats then costs what the launch did (12 rows of 768 6.0 / 8.2; 4800 x 1600 at 4 / 6 / 8 rows 8.6 / 8.1, 8.8 / 8.9, 9.0 / 9.0).
#include "gemm_norm.h"
#include "wave_sums.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}

#define STAGE_SLOTS 72  // 8 rows x (8 chunks + 1 of padding)

// WAVES, NT: as in the skinny kernel, a wave's pairs of k-steps beside them (1,024 / 64 over the waves). RP: rows a group of four waves normalises.
template <int WAVES, int NT, int RP>
__global__ void __launch_bounds__(WAVES * 64, 1)
gemm_norm_kernel(const bf16_t* __restrict__ w, const float* __restrict__ x, int K, int N, int M, float eps, const float* __restrict__ nw,
                 const float* __restrict__ nb, const float* __restrict__ bias, int rms, bf16_t* __restrict__ out, long ldo, int act) {
  constexpr int GROUPS = WAVES / 4, SUMS = WAVES >= 16 ? 1 : 2, PP = NORMED_MAX_K / 64 / WAVES;
  extern __shared__ u32x4 rows[];  // [M][K / 8 | 1]
  __shared__ f32x4 red[WAVES][NT][64];
  __shared__ u32x4 stage[WAVES][2][STAGE_SLOTS];
  __shared__ float sums[2][RP][WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave >> 2, t256 = tid & 255;
  const int n0 = blockIdx.x * 16 * NT;
  const int row_chunks = (K / 8) | 1;

  // all from clamped addresses
  const int d = t256 * 4, dc = min(d, K - 4);
  float4 v[RP];
#pragma unroll
  for (int j = 0; j < RP; ++j) v[j] = *reinterpret_cast<const float4*>(x + (size_t)min(group + j * GROUPS, M - 1) * K + dc);
  __builtin_amdgcn_sched_barrier(0);
  const float4 g = *reinterpret_cast<const float4*>(nw + dc);
  float4 b = *reinterpret_cast<const float4*>((nb ? nb : nw) + dc);  // nw stands in for a missing one
  const int fr = lane & 15, kg = lane >> 4, lr = lane >> 3, lc = lane & 7;
  const int bn = min(n0 + 16 * min(wave, NT - 1) + fr, N - 1);
  float pre_bias = *(bias ? bias + bn : nw);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  // the weights: whole lines, eight rows an instruction; for a pair beyond the last, which counts for nothing, a
  // line that the wave has asked for anyway
  const int npairs = (K + 63) / 64;
  const int rot = (int)((blockIdx.x * 2654435761u) % (unsigned)npairs);
  uint32_t row_at[NT][2];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) row_at[j][i] = (uint32_t)(min(n0 + 16 * j + 8 * i + lr, N - 1) * K);
  auto pair = [&](int p) __attribute__((always_inline)) {  // the same for all lanes; beyond the last the wave's first once more
    int pr = wave + (wave + p * WAVES < npairs ? p * WAVES : 0);
    pr = min(pr, npairs - 1) + rot;
    return pr >= npairs ? pr - npairs : pr;
  };
  u32x4 wv[PP][NT][2];
#pragma unroll
  for (int p = 0; p < PP; ++p) {
    const uint32_t kc = min(pair(p) * 64 + lc * 8, K - 8);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) wv[p][j][i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(w) + (row_at[j][i] + kc) * 2);
  }
  __builtin_amdgcn_sched_barrier(0);

  if (d >= K) {
#pragma unroll
    for (int j = 0; j < RP; ++j) v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float mean[RP], rstd[RP], part[RP];
#pragma unroll
  for (int j = 0; j < RP; ++j) mean[j] = 0.f;
  if (!rms) {
#pragma unroll
    for (int j = 0; j < RP; ++j) part[j] = (v[j].x + v[j].y) + (v[j].z + v[j].w);
    store_wave_sums<RP, WAVES>(part, sums[0], wave, lane);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) t += sums[0][j][group * 4 + q];
      mean[j] = t / (float)K;
    }
  }
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const float c0 = v[j].x - mean[j], c1 = v[j].y - mean[j], c2 = v[j].z - mean[j], c3 = v[j].w - mean[j];
    part[j] = d < K ? (c0 * c0 + c1 * c1) + (c2 * c2 + c3 * c3) : 0.f;
  }
  store_wave_sums<RP, WAVES>(part, sums[1], wave, lane);
  lds_barrier();
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) t += sums[1][j][group * 4 + q];
    rstd[j] = 1.0f / sqrtf(t / (float)K + eps);
  }
  if (!nb) b = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const int r = group + j * GROUPS;
    if (r < M && d < K) {
      uint2 o;
      o.x = float2_to_bf16x2((v[j].x - mean[j]) * rstd[j] * g.x + b.x, (v[j].y - mean[j]) * rstd[j] * g.y + b.y);
      o.y = float2_to_bf16x2((v[j].z - mean[j]) * rstd[j] * g.z + b.z, (v[j].w - mean[j]) * rstd[j] * g.w + b.w);
      *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(rows + r * row_chunks) + d) = o;
    }
  }
  lds_barrier();

  const u32x4* arow = rows + min(fr, M - 1) * row_chunks;
  u32x4* my_stage = &stage[wave][0][0];
  const int st_slot = lr * 9 + lc, ld_slot = (fr >> 3) * STAGE_SLOTS + (fr & 7) * 9 + kg;
  f32x4 acc[SUMS][NT];
#pragma unroll
  for (int s = 0; s < SUMS; ++s)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[s][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < PP; ++p) {
    const bool ok = wave + p * WAVES < npairs;
    const int k0 = pair(p) * 64;
    const uint32_t keep = ok && k0 + lc * 8 < K ? 0xffffffffu : 0u;
    const uint32_t keep_lo = ok && k0 + kg * 8 < K ? 0xffffffffu : 0u, keep_hi = ok && k0 + 32 + kg * 8 < K ? 0xffffffffu : 0u;
    const u32x4 a_lo = arow[min(k0 + kg * 8, K - 8) >> 3] & u32x4{keep_lo, keep_lo, keep_lo, keep_lo};
    const u32x4 a_hi = arow[min(k0 + 32 + kg * 8, K - 8) >> 3] & u32x4{keep_hi, keep_hi, keep_hi, keep_hi};
    const u32x4 mk = u32x4{keep, keep, keep, keep};
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      // LDS executes a wave's instructions in order: the area is used again and again without a barrier
      lds_wave_order();
      my_stage[st_slot] = wv[p][j][0] & mk;
      my_stage[STAGE_SLOTS + st_slot] = wv[p][j][1] & mk;
      lds_wave_order();
      const u32x4 w_lo = my_stage[ld_slot], w_hi = my_stage[ld_slot + 4];
      acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a_lo), as_bf16x8(w_lo), acc[0][j], 0, 0, 0);
      acc[1 % SUMS][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a_hi), as_bf16x8(w_hi), acc[1 % SUMS][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
#pragma unroll
    for (int s = 1; s < SUMS; ++s) acc[0][j] += acc[s][j];
    red[wave][j][lane] = acc[0][j];
  }
  lds_barrier();
  if (!bias) pre_bias = 0.f;
  // 16x16 accumulator: register r of lane l is row 4*(l/16) + r, column l%16. Partial sums are added in wave order.
  if (wave >= NT) return;
  f32x4 s = red[0][wave][lane];
#pragma unroll
  for (int u = 1; u < WAVES; ++u) {
    const f32x4 o = red[u][wave][lane];
    s[0] += o[0]; s[1] += o[1]; s[2] += o[2]; s[3] += o[3];
  }
  const int nn = n0 + 16 * wave + fr;
  if (nn >= N) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = kg * 4 + r;
    if (m < M) out[(size_t)m * ldo + nn] = from_float<bf16_t>(lev_activate(s[r] + pre_bias, act));
  }
}

int lev_normed_launch(int waves, int units, const float* x, const float* nw, const float* nb, float eps, int rms, const bf16_t* w, const float* bias,
                      bf16_t* out, long ldo, int M, int N, int K, int act, hipStream_t stream) {
  if (M < 1 || M > NORMED_MAX_M || K < 8 || K > NORMED_MAX_K || K % 8 || (size_t)N * K >= (1ull << 31)) return -1;
  const int lds = M * ((K / 8) | 1) * 16, columns = (N + 16 * units - 1) / (16 * units);  // 16.5 KB of rows at most
  const int per_group = (M + waves / 4 - 1) / (waves / 4);
#define LEV_NORMED(W_, NT_, RP_)                                                                                          \
  if (waves == W_ && units == NT_ && per_group == RP_) {                                                                  \
    gemm_norm_kernel<W_, NT_, RP_><<<columns, W_ * 64, lds, stream>>>(w, x, K, N, M, eps, nw, nb, bias, rms, out, ldo, act); \
    return lev_check_launch("norm_linear");                                                                               \
  }
  LEV_NORMED(8, 1, 1)
  LEV_NORMED(8, 1, 2)
  LEV_NORMED(8, 1, 3)
  LEV_NORMED(8, 1, 4)
  LEV_NORMED(16, 2, 1)
  LEV_NORMED(16, 2, 2)
  LEV_NORMED(16, 3, 1)
  LEV_NORMED(16, 3, 2)
#undef LEV_NORMED
  return -1;
}
