// y = act(a . w^T + bias) + residual in 32 bits for some hundred rows and more, on the bfloat16 matrix instruction, which multiplies sixteen times as fast as the
// 32-bit one (splitting as in Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019). Every number is the sum of
// three bfloat16 numbers of 8 bits each, 24 in all, the products of bfloat16 numbers are exact in 32 bits and are added up in
// 32 bits, and six of the nine partial products are taken: the three left out are at most 2^-24 of a product, 2^-27.5 rms and of
// either sign (a sum of one product is off by up to 1.75 times 2^-24 instead of once; with eight partial products it is off by once, and they take 52.5 -> 60 us at 777 rows of 4096 x 1024). The products of the first parts
// have sums of their own, which join the total every 128 numbers (256 of long sums); the others, a hundredth as large, go to a second sum, so that a total of K numbers has
// K / 16 + K / 128 roundings of its size. Errors against 64 bits of 300 shapes of 32 .. 2,048 rows and 256 .. 16,384 numbers a sum, normal numbers and positive ones: 0.12 .. 0.99 of
// the kernels' that had these products, 0.53 in the middle (4096 x 1024 at 777 rows 2.1e-7 / 0.83e-7, 1024 x 4096 5.8e-7 / 1.0e-7).
// What bounds it: the vector instructions that split a number (27 for four, on their way into LDS) take slots of the matrix pipe: beside 32 of them 32-cycle products
// took 168 us, alone 115, the vector instructions alone 134. At 128 x 128 outputs a step of 32 numbers is 1,536 cycles of products, 2,500 in all. 32 x 32 products, which leave more room
// beside them than 16 x 16 ones, tiles of eight waves and reads of LDS spread between the products gave the most (777 rows, 4096 x 1024: four waves of 16 x 16 products 67 us, eight 50,
// eight of 32 x 32 49); a phase of splitting and one of products in turn for the halves of a workgroup 55, all of a step's reads at once 53. Before / now, microseconds: 4096 x 1024 at
// 777 rows 62 / 47, 1024 x 4096 72 / 63, 1024 x 1024 22 / 20, 4096 x 4096 at 2,048 rows 502 / 360 (191 TFLOP/s; the 32-bit instruction's peak is 157).
#include "gemm_f32.h"
#include <math.h>

typedef __attribute__((ext_vector_type(8))) __bf16 gs_bf16x8;
typedef __attribute__((ext_vector_type(4))) uint32_t gs_u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t gs_u32x2;

#define GS_K 32           // numbers of a row a step
#define GS_UP 0x1p24f     // on both operands: the last of the 24 bits of any number, the smallest ones' too, is one of a bfloat16 number's then
#define GS_DOWN 0x1p-48f

// four numbers into three times four
__device__ __forceinline__ void gs_split(gf_f32x4 v, gs_u32x2 (&p)[3]) {
  v *= GS_UP;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const uint32_t lo = float2_to_bf16x2(v[0], v[1]), hi = float2_to_bf16x2(v[2], v[3]);
    p[q] = gs_u32x2{lo, hi};
    if (q == 2) break;
    v[0] -= __uint_as_float(lo << 16), v[1] -= __uint_as_float(lo & 0xffff0000u);
    v[2] -= __uint_as_float(hi << 16), v[3] -= __uint_as_float(hi & 0xffff0000u);
  }
}
typedef __attribute__((ext_vector_type(16))) float gs_f32x16;
__device__ __forceinline__ gs_f32x16 gs_mfma(gs_u32x4 a, gs_u32x4 b, gs_f32x16 c) {
  union { gs_u32x4 u; gs_bf16x8 v; } x, y;
  x.u = a, y.u = b;
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.v, y.v, c, 0, 0, 0);
}

// RT x NT: tiles of 32 x 32 of a wave; WM x WN: waves of a group; KG: groups that share the steps.
template <int RT, int NT, int WM, int WN, int KG>
__global__ void __launch_bounds__(64 * WM * WN * KG, RT * NT * KG == 1 ? 4 : 2)
gemm_f32_split_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias, const float* residual, long ldr,
                      float* out, long ldo, int M, int N, int K, int act, int n_rows, int n_cols, int vec) {
  constexpr int BM = 32 * RT * WM, BN = 32 * NT * WN, ROWS = BM + BN, TG = 64 * WM * WN, PASS = TG / 8, NR = ROWS / PASS;
  static_assert(ROWS % PASS == 0, "whole passes of loads");
  constexpr int AHEAD = RT * NT * KG == 1 ? 1 : 2;  // steps whose loads are on their way; two workgroups a CU have registers for one each
  constexpr int BUF = ROWS * GS_K * 3;
  extern __shared__ __attribute__((aligned(16))) uint16_t gs_lds[];  // [KG][2][ROWS / 16][3 parts][4 chunks of 8 numbers][16 rows][8]
  const int tid = threadIdx.x % TG, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kgroup = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / TG);
  const int col = lane & 31, g = lane >> 5, wm = wave / WN, wn = wave % WN;
  const int n_tiles = n_rows * n_cols, per = (n_tiles + 7) / 8;  // neighbouring columns of tiles on a chiplet, as in gemm_f32.hip
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || tile >= n_tiles) return;  // the whole workgroup
  const int m0 = (tile % n_rows) * BM, o0 = (tile / n_rows) * BN;
  const int row = tid >> 3, kc = (tid & 7) * 4;
  // A pass of loads: eight rows a wave, of a or of w, the same for all its lanes. Bytes from the tile's first row on; rows beyond the matrix: read again, never stored
  const char* a0 = reinterpret_cast<const char*>(a + (size_t)m0 * lda);
  const char* w0 = reinterpret_cast<const char*>(w + (size_t)o0 * K);
  const char* base[NR];
  uint32_t at[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const bool of_a = PASS * i + 8 * wave < BM;
    const int r = PASS * i + row;
    base[i] = of_a ? a0 : w0;
    at[i] = of_a ? (uint32_t)(min(r, M - 1 - m0) * (int)lda + kc) * 4u : (uint32_t)(min(r - BM, N - 1 - o0) * K + kc) * 4u;
  }
  uint16_t* mine = gs_lds + (size_t)kgroup * 2 * BUF;
  // a chunk's rows lie 16 bytes apart, turned by twice the chunk's number: what neighbouring lanes write and read falls on all banks
  uint16_t* put = mine + (row >> 4) * 3 * 512 + (kc >> 3) * 128 + ((row & 15) ^ (kc >> 3) * 2) * 8 + (kc & 4);
  const uint16_t* get[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) get[ks] = mine + (col >> 4) * 3 * 512 + (2 * ks + g) * 128 + ((col & 15) ^ (2 * ks + g) * 2) * 8;

  // Steps in the order they are taken: what is missing to a whole number of steps for every group, then a partial one (K % 32 != 0), then whole ones, so
  // that only the first needs masks.
  const int tail = K % GS_K, all = (K + GS_K - 1) / GS_K, steps = (all + KG - 1) / KG, skip = steps * KG - all;
  gf_f32x4 ahead[AHEAD][NR];
  auto fetch = [&](gf_f32x4 (&to)[NR], int t) __attribute__((always_inline)) {  // t >= 1; beyond the end: loaded again, not used
    const size_t k = max(min(t, steps - 1) * KG + kgroup - skip - (tail ? 1 : 0), 0) * GS_K;  // K >= 32
#pragma unroll
    for (int i = 0; i < NR; ++i) to[i] = *reinterpret_cast<const gf_f32x4*>(base[i] + k * 4 + at[i]);
  };
  auto stage = [&](gf_f32x4 v, int i, int buf) __attribute__((always_inline)) {
    gs_u32x2 p[3];
    gs_split(v, p);
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<gs_u32x2*>(put + buf * BUF + i * (PASS / 16) * 3 * 512 + q * 512) = p[q];
  };
  gs_f32x16 sum[RT][NT], acc[RT][NT], low[RT][NT];  // products of the first parts, of them the last steps', all others
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[i][j][r] = acc[i][j][r] = low[i][j][r] = 0.f;
  auto settle = [&](bool with_low) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          if (with_low) acc[i][j][r] += low[i][j][r], low[i][j][r] = 0.f;
          sum[i][j][r] += acc[i][j][r], acc[i][j][r] = 0.f;
        }
  };
  gs_u32x4 ops[2][RT + NT][3];
  auto read = [&](int buf, int ks, int i) __attribute__((always_inline)) {
    const int tile32 = i < NT ? BM / 32 + wn * NT + i : wm * RT + i - NT;
#pragma unroll
    for (int q = 0; q < 3; ++q) ops[ks][i][q] = *reinterpret_cast<const gs_u32x4*>(get[ks] + buf * BUF + (tile32 * 6 + q) * 512);
  };
  auto products = [&](int ks, int part, int parts) __attribute__((always_inline)) {  // the small ones first
    constexpr int PW[6] = {2, 0, 1, 1, 0, 0}, PA[6] = {0, 2, 1, 0, 1, 0}, TILES = RT * NT, ALL = 6 * TILES;
#pragma unroll
    for (int p = 0; p < ALL; ++p) {
      if (p < part * ALL / parts || p >= (part + 1) * ALL / parts) continue;
      const int q = p / TILES, j = p % TILES / RT, i = p % RT;
      gs_f32x16& c = q == 5 ? acc[i][j] : low[i][j];
      c = gs_mfma(ops[ks][j][PW[q]], ops[ks][NT + i][PA[q]], c);
    }
  };
  {
    const int s = kgroup - skip;  // the group's first step
    const int k = s < 0 ? K : s == 0 && tail ? K - tail : (s - (tail ? 1 : 0)) * GS_K;
#pragma unroll
    for (int i = 0; i < NR; ++i) ahead[0][i] = *reinterpret_cast<const gf_f32x4*>(base[i] + (ptrdiff_t)(min(k + kc, K - 4) - kc) * 4 + at[i]);
    if (AHEAD > 1) fetch(ahead[AHEAD - 1], 1);
    if (k + kc >= K)  // chunks beyond K count as zeros
#pragma unroll
      for (int i = 0; i < NR; ++i) ahead[0][i] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NR; ++i) stage(ahead[0][i], i, 0);
    fetch(ahead[0], AHEAD);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RT + NT; ++i) read(0, 0, i);
  }
  // Step t from buffer t % 2; step t + 1 (and t + 2) is on its way in registers. The products of 16 numbers while step t + 1 is split into the
  // other buffer, those of the other 16 while the first operands of step t + 1 are read.
  auto step = [&](int t, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
#pragma unroll
      for (int e = i * (RT + NT) / NR; e < (i + 1) * (RT + NT) / NR; ++e) read(buf, 1, e);
      products(0, i, NR);
      stage(ahead[AHEAD > 1 ? buf ^ 1 : 0][i], i, buf ^ 1);  // behind the last step: numbers that nobody uses
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
    fetch(ahead[AHEAD > 1 ? buf ^ 1 : 0], t + 1 + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RT + NT + 1; ++i) {
      if (i < RT + NT) read(buf ^ 1, 0, i);
      products(1, i, RT + NT + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int piece = K < 4096 ? 4 : 8;  // steps whose products are added up before they join the sum
  int t = 0;
  while (t + 1 < steps) {
    const int stop = min(t + piece, steps - 1);
    for (; t < stop; t += 2) {
      step(t, 0);
      step(t + 1, 1);
    }
    if (t % 16 == 0) settle(true);  // a hundredth as large, and so are their roundings
    else settle(false);
  }
  if (t < steps) step(t, 0);
  settle(true);
  if (KG > 1) {  // the groups' sums, in order
    float* part = reinterpret_cast<float*>(gs_lds);  // [KG - 1][RT NT 16][TG]
    __syncthreads();
    if (kgroup > 0)
#pragma unroll
      for (int i = 0; i < RT * NT * 16; ++i) part[((kgroup - 1) * RT * NT * 16 + i) * TG + tid] = sum[i / 16 / NT][i / 16 % NT][i % 16];
    __syncthreads();
    if (kgroup > 0) return;
#pragma unroll
    for (int q = 0; q < KG - 1; ++q)
#pragma unroll
      for (int i = 0; i < RT * NT * 16; ++i) sum[i / 16 / NT][i / 16 % NT][i % 16] += part[(q * RT * NT * 16 + i) * TG + tid];
  }
#pragma unroll
  for (int i = 0; i < RT * NT * 16; ++i) sum[i / 16 / NT][i / 16 % NT][i % 16] *= GS_DOWN;
  // An infinity or NaN has no parts: every sum that it meets comes out infinite or NaN, and so does no sum of finite numbers unless it is too large. A wave with
  // such a sum multiplies its tiles again, as they are, on the 32-bit instruction, from memory: slow, for what no working model has (4096 x 1024 at 777 rows 53 us, with one infinite input 112, with all sums
  // beyond 2^80, which the scaled parts cannot hold, 152; the 32-bit kernels 73 either way).
  bool finite = true;
#pragma unroll
  for (int i = 0; i < RT * NT * 16; ++i) finite &= fabsf(sum[i / 16 / NT][i / 16 % NT][i % 16]) < INFINITY;
  if (!__all(finite)) {
#pragma unroll
    for (int i = 0; i < RT * NT * 16; ++i) sum[i / 16 / NT][i / 16 % NT][i % 16] = 0.f;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 8) {
      if (k0 % 128 == 0) settle(false);
      const int k = k0 + 4 * g, kr = min(k, K - 4);
      gf_f32x4 x[RT + NT];
#pragma unroll
      for (int i = 0; i < RT + NT; ++i) {
        x[i] = i < NT ? *reinterpret_cast<const gf_f32x4*>(w + (size_t)min(o0 + 32 * (wn * NT + i) + col, N - 1) * K + kr)
                      : *reinterpret_cast<const gf_f32x4*>(a + (size_t)min(m0 + 32 * (wm * RT + i - NT) + col, M - 1) * lda + kr);
        if (k >= K) x[i] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[j][e], x[NT + i][e], acc[i][j], 0, 0, 0);
    }
    settle(false);
  }
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 32 * (wm * RT + i) + col, o = o0 + 32 * (wn * NT + j) + 8 * r + 4 * g;
        const gs_f32x16& v = sum[i][j];
        if (m < M && o < N) gemm_f32_store(gf_f32x4{v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]}, bias, residual, ldr, out, ldo, m, o, N, act, vec);
      }
}

template <int RT, int NT, int WM, int WN, int KG>
static int gemm_f32_split_launch(const float* a, long lda, const float* w, const float* bias, const float* residual, long ldr, float* out, long ldo, int M, int N, int K,
                                 int act, int vec, hipStream_t stream) {
  constexpr int BM = 32 * RT * WM, BN = 32 * NT * WN, lds = KG * 2 * (BM + BN) * GS_K * 6;
  static std::atomic<unsigned long long> reserved{0};
  if (lev_reserve_lds((const void*)gemm_f32_split_kernel<RT, NT, WM, WN, KG>, lds, reserved)) return -1;
  const int n_rows = (M + BM - 1) / BM, n_cols = (N + BN - 1) / BN;
  const long blocks = ((long)n_rows * n_cols + 7) / 8 * 8;
  LEV_REQUIRE(blocks <= 0x7fffffffL, "linear: too many tiles (%ld)", blocks);
  gemm_f32_split_kernel<RT, NT, WM, WN, KG><<<(unsigned)blocks, 64 * WM * WN * KG, lds, stream>>>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, n_rows, n_cols, vec);
  return lev_check_launch("linear (32-bit, split)");
}

int lev_gemm_f32_split(int tile, const float* a, long lda, const float* w, const float* bias, const float* residual, long ldr, float* out, long ldo, int M, int N, int K,
                       int act, int vec, hipStream_t stream) {
  if (tile == 0) return gemm_f32_split_launch<1, 2, 4, 2, 1>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, vec, stream);
  if (tile == 1) return gemm_f32_split_launch<1, 1, 2, 4, 1>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, vec, stream);
  return gemm_f32_split_launch<1, 1, 2, 2, 2>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, vec, stream);
}
