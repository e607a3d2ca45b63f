// out = act(norm(x) . w^T + bias) in 32 bits for up to 8 rows of up to 1,024 numbers: LayerNorm or RMSNorm of float32 rows x [M][K] and the product behind it in one launch, as
// gemm_norm.hip has it in bfloat16: what the two kernels apart take is their launches and their trips to memory, one behind the other, and here a wave requests its
// rows, then scale and shift, then all its weights, and the statistics pass while the weights are on their way.
// The norm is worked out as norm_reg_kernel works it out with 256 threads a row, and the product as gemm_f32_kernel<1, 1, 8> does (16 outputs a workgroup, K dealt to eight waves
// in stretches): the same bits as the two kernels one after the other.
// Measured in graphs over weights and norms that no cache holds, microseconds, two kernels / here: 2304 x 768 at 3 / 8 rows 7.6 / 5.9, 8.0 / 6.8; 3072 x 768 at 4 rows 7.7 / 6.3; 4096 x 1024 at 2 / 8 rows
// 8.6 / 6.4, 8.8 / 7.6; 1024 x 256 at 4 rows 5.7 / 4.2. A session of GPT-2 small in 32 bits, 4 requests: 10.00 -> 9.29 ms.
#include "gemm_f32.h"
#include "wave_sums.h"

#define GN_MAX_M 8
#define GN_MAX_K 1024  // a float4 for each of 256 threads

// RP: rows a group of four waves normalises
template <int RP>
__global__ void __launch_bounds__(512)
gemm_f32_norm_kernel(const float* __restrict__ w, const float* __restrict__ x, int K, int N, int M, float eps, const float* __restrict__ nw, const float* __restrict__ nb,
                     int n_cols, int rms, const float* __restrict__ bias, float* __restrict__ out, long ldo, int vec, int act) {  // up to bias in registers when the waves start
  constexpr int W = 8, STEPS = GN_MAX_K / (16 * W);
  extern __shared__ __attribute__((aligned(16))) float gn_rows[];  // [M][K + 4]
  __shared__ __attribute__((aligned(16))) gf_f32x4 part[W][64];
  __shared__ float sums[2][RP][W];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, g = lane >> 4;
  const int per = (n_cols + 7) / 8, tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // neighbouring outputs on a chiplet, as in gemm_f32.hip
  if ((blockIdx.x >> 3) >= per || tile >= n_cols) return;  // the whole workgroup
  const int group = wave >> 2, d = (tid & 255) * 4, dc = min(d, K - 4), o0 = tile * 16;

  // all from clamped addresses
  gf_f32x4 v[RP];
#pragma unroll
  for (int j = 0; j < RP; ++j) v[j] = *reinterpret_cast<const gf_f32x4*>(x + (size_t)min(group + 2 * j, M - 1) * K + dc);
  __builtin_amdgcn_sched_barrier(0);
  const gf_f32x4 scale = *reinterpret_cast<const gf_f32x4*>(nw + dc);
  gf_f32x4 shift = *reinterpret_cast<const gf_f32x4*>((nb ? nb : nw) + dc);  // nw stands in for a missing one
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();  // without a wait: the weights of the first waves stay behind the rows of the last
  // the wave's stretch of K; steps beyond it are read again and multiply zeros
  const int share = (K + 16 * W - 1) / (16 * W) * 16, k_lo = min(K, wave * share), k_hi = min(K, k_lo + share);
  const float* wr = w + (size_t)min(o0 + col, N - 1) * K;
  gf_f32x4 wv[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) wv[s] = *reinterpret_cast<const gf_f32x4*>(wr + min(k_lo + (16 * s < share ? 16 * s : 0) + 4 * g, K - 4));
  __builtin_amdgcn_sched_barrier(0);

  if (d >= K)
#pragma unroll
    for (int j = 0; j < RP; ++j) v[j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
  float mean[RP], rstd[RP], sum[RP];
#pragma unroll
  for (int j = 0; j < RP; ++j) mean[j] = 0.f;
  auto whole = [&](int which, int j) __attribute__((always_inline)) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) t += sums[which][j][group * 4 + q];
    return t;
  };
  if (!rms) {
#pragma unroll
    for (int j = 0; j < RP; ++j) sum[j] = (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
    store_wave_sums<RP, W>(sum, sums[0], wave, lane);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < RP; ++j) mean[j] = whole(0, j) / (float)K;
  }
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const float c0 = v[j][0] - mean[j], c1 = v[j][1] - mean[j], c2 = v[j][2] - mean[j], c3 = v[j][3] - mean[j];
    sum[j] = d < K ? (c0 * c0 + c1 * c1) + (c2 * c2 + c3 * c3) : 0.f;
  }
  store_wave_sums<RP, W>(sum, sums[1], wave, lane);
  lds_barrier();
#pragma unroll
  for (int j = 0; j < RP; ++j) rstd[j] = 1.0f / sqrtf(whole(1, j) / (float)K + eps);
  if (!nb) shift = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const int r = group + 2 * j;
    if (r < M && d < K) {
      gf_f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (v[j][e] - mean[j]) * rstd[j] * scale[e] + shift[e];
      *reinterpret_cast<gf_f32x4*>(gn_rows + r * (K + 4) + d) = o;
    }
  }
  lds_barrier();

  const float* ar = gn_rows + min(col, M - 1) * (K + 4);
  gf_f32x4 acc = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int k = k_lo + 16 * s;
    if (k >= k_hi) break;  // the whole wave
    gf_f32x4 a = *reinterpret_cast<const gf_f32x4*>(ar + min(k + 4 * g, K - 4));
    if (k + 4 * g >= K) a = wv[s] = gf_f32x4{0.f, 0.f, 0.f, 0.f};  // chunks beyond K count as zeros
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s][e], a[e], acc, 0, 0, 0);
  }
  part[wave][lane] = acc;
  lds_barrier();
  if (wave != 0) return;
  gf_f32x4 total = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < W; ++q) total += part[q][lane];
  const int o = o0 + 4 * g;
  if (col < M && o < N) gemm_f32_store(total, bias, nullptr, 0, out, ldo, col, o, N, act, vec);
}

// Where the product alone is gemm_f32_kernel<1, 1, 8>'s, up to the outputs from which on the work that every workgroup repeats costs what the launch did: two rounds of workgroups, one of
// more than four rows (6400 x 512 at 4 / 6 rows 8.1 / 7.5, 8.2 / 8.2; 8192 x 1024 at 4 / 8 rows 12.1 / 10.9, 12.1 / 12.1) or short sums (12288 x 256 at 1 row 7.8 / 8.6).
extern "C" int lev_linear_f32_normed_takes(int M, int N, int K) {
  return M >= 1 && M <= GN_MAX_M && K >= 64 && K <= GN_MAX_K && K % 4 == 0 && (N <= 4096 || (N <= 8192 && M <= 4 && K >= 512)) && lev_linear_f32_choice(M, N, K) == 0;
}

extern "C" int lev_linear_f32_normed(const float* x, const float* norm_w, const float* norm_b, float eps, int rms, const float* w, const float* bias, float* out, long ldo,
                                     int M, int N, int K, int act, hipStream_t stream) {
  LEV_REQUIRE(x && norm_w && w && out && lev_linear_f32_normed_takes(M, N, K), "norm and linear: no kernel for M=%d N=%d K=%d", M, N, K);
  LEV_REQUIRE((((uintptr_t)x | (uintptr_t)norm_w | (uintptr_t)norm_b | (uintptr_t)w) & 15) == 0, "norm and linear: operands must be 16-byte aligned");
  LEV_REQUIRE(ldo >= N && eps > 0.f && act >= LEV_ACT_NONE && act <= LEV_ACT_LAST, "norm and linear: bad ldo=%ld, eps=%g or activation %d", ldo, eps, act);
  const int vec = ldo % 4 == 0 && ((uintptr_t)out & 15) == 0 && (!bias || ((uintptr_t)bias & 15) == 0);
  const int n_cols = (N + 15) / 16, lds = M * (K + 4) * (int)sizeof(float);  // 33 KB at most
  const unsigned blocks = (n_cols + 7) / 8 * 8;
#define LEV_NORMED_F32(RP) \
  gemm_f32_norm_kernel<RP><<<blocks, 512, lds, stream>>>(w, x, K, N, M, eps, norm_w, norm_b, n_cols, rms, bias, out, ldo, vec, act)
  switch ((M + 1) / 2) {
    case 1: LEV_NORMED_F32(1); break;
    case 2: LEV_NORMED_F32(2); break;
    case 3: LEV_NORMED_F32(3); break;
    default: LEV_NORMED_F32(4);
  }
#undef LEV_NORMED_F32
  return lev_check_launch("norm and linear (32-bit)");
}
