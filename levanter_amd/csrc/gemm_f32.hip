// y = act(a . w^T + bias) + residual in 32 bits on the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32: full 32-bit products and
// sums, no reduced mode). a [M, K] (row stride lda), w [N, K], y [M, N]. Some hundred rows and more go to gemm_f32_split.hip by the rule at this file's end.
#include "gemm_f32.h"
#include <math.h>

// A workgroup of W waves owns 16 RT rows and 16 NT outputs; its waves split K (steps of 16 dealt in stretches) and the partial sums are
// added through LDS in wave order. The product is transposed, out^T = w a^T, so that a lane ends with four neighbouring outputs of one
// row. Both operands come straight from global memory, 16 bytes a lane (row = lane % 16, k = 4 (lane / 16) + j for the j-th of the
// four products of a step): the 32-bit instruction takes 32 cycles for 1,024 multiply-adds, which hides much of what such loads cost
// the vector cache (a look-up for every lane).
// What bounds it: few rows, the read of the weights (4096 x 4096 at 4 rows 14.3 us, 4.7 TB/s; 768 x 768 at 16 rows 5.3 us, a launch and a chain of
// loads); some dozens, L2 at about 9.5 TB/s (1024 x 4096 at 203 rows 32 us) or the last round of tiles. The plain kernel of
// gemm_simple.hip (64 x 64 tiles, vector ALU, scalar loads) took 84 us for 768 x 768 at 4 rows, 378 us for 768 x 3072 (this one 4.8 and 10; with so few rows
// and outputs the few-row kernel below goes before it, 3.9 and 5.9).
template <int RT, int NT, int W>
__global__ void __launch_bounds__(64 * W)
gemm_f32_kernel(const float* __restrict__ w, const float* __restrict__ a, uint32_t lda4, int K, int N, int M, int n_rows, int n_cols, int vec, int act,
                const float* __restrict__ bias, const float* residual, float* out, long ldr, long ldo) {  // up to bias in registers when the waves start
  const size_t lda = (size_t)lda4 * 4;
  extern __shared__ __attribute__((aligned(16))) float gf_part[];  // [W][RT * NT][64][4]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
  // the chiplets (workgroups are dealt to the eight in turn) take neighbouring columns of tiles each, rows fastest: a weight is read by
  // one chiplet's L2 only
  const int n_tiles = n_rows * n_cols, per = (n_tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || tile >= n_tiles) return;  // the whole workgroup
  const int m0 = (tile % n_rows) * 16 * RT, o0 = (tile / n_rows) * 16 * NT;
  const float *ar[RT], *wr[NT];
#pragma unroll
  for (int i = 0; i < RT; ++i) ar[i] = a + (size_t)min(m0 + 16 * i + col, M - 1) * lda;  // rows beyond the matrix: read again, never stored
#pragma unroll
  for (int j = 0; j < NT; ++j) wr[j] = w + (size_t)min(o0 + 16 * j + col, N - 1) * K;
  gf_f32x4 acc[RT][NT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
  const int share = (K + 16 * W - 1) / (16 * W) * 16;
  const int k_lo = min(K, wave * share), k_hi = min(K, k_lo + share);
  const int k_full = k_lo + (k_hi - k_lo) / 16 * 16;
  auto load = [&](int k0, gf_f32x4 (&av)[RT], gf_f32x4 (&wv)[NT]) {
    const int kk = k0 + 4 * g;
#pragma unroll
    for (int j = 0; j < NT; ++j) wv[j] = *reinterpret_cast<const gf_f32x4*>(wr[j] + kk);
#pragma unroll
    for (int i = 0; i < RT; ++i) av[i] = *reinterpret_cast<const gf_f32x4*>(ar[i] + kk);
  };
  auto products = [&](const gf_f32x4 (&av)[RT], const gf_f32x4 (&wv)[NT]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][e], av[i][e], acc[i][j], 0, 0, 0);
  };
  // steps whose loads are on their way at a time; a wave with many products a step instead asks for the next step ahead of this one's products
  constexpr bool AHEAD = RT * NT >= 4;
  constexpr int U = AHEAD ? 2 : 4;
  gf_f32x4 av[U][RT], wv[U][NT];
  int k0 = k_lo;
  if (AHEAD) {
    if (k0 < k_full) load(k0, av[0], wv[0]);
    for (; k0 + 32 <= k_full; k0 += 32) {
      load(k0 + 16, av[1], wv[1]);
      __builtin_amdgcn_sched_barrier(0);
      products(av[0], wv[0]);
      load(min(k0 + 32, k_full - 16), av[0], wv[0]);  // at the end: read again, not used
      __builtin_amdgcn_sched_barrier(0);
      products(av[1], wv[1]);
    }
    if (k0 < k_full) products(av[0], wv[0]);
  } else {
    for (; k0 + 16 * U <= k_full; k0 += 16 * U) {
#pragma unroll
      for (int u = 0; u < U; ++u) load(k0 + 16 * u, av[u], wv[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) products(av[u], wv[u]);
    }
    for (; k0 < k_full; k0 += 16) {
      load(k0, av[0], wv[0]);
      products(av[0], wv[0]);
    }
  }
  if (k_full < k_hi) {  // the last step of a K that is no multiple of 16: chunks beyond it count as zeros
    const int kk = k_full + 4 * g, kc = min(kk, K - 4);
    const bool in = kk < K;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      wv[0][j] = *reinterpret_cast<const gf_f32x4*>(wr[j] + kc);
      if (!in) wv[0][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      av[0][i] = *reinterpret_cast<const gf_f32x4*>(ar[i] + kc);
      if (!in) av[0][i] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    products(av[0], wv[0]);
  }
  if (W > 1) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) *reinterpret_cast<gf_f32x4*>(gf_part + ((size_t)(wave * RT * NT + i * NT + j) * 64 + lane) * 4) = acc[i][j];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < RT; ++i) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int t = i * NT + j;
      if (W > 1 && t % W != wave) continue;  // the waves finish a tile each in turn
      gf_f32x4 v = acc[i][j];
      if (W > 1) {
        v = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < W; ++q) v += *reinterpret_cast<const gf_f32x4*>(gf_part + ((size_t)(q * RT * NT + t) * 64 + lane) * 4);
      }
      const int m = m0 + 16 * i + col, o = o0 + 16 * j + 4 * g;
      if (m < M && o < N) gemm_f32_store(v, bias, residual, ldr, out, ldo, m, o, N, act, vec);
    }
  }
}

// Some hundred rows and more: a workgroup of four waves (2 x 2) owns 32 RT rows and 32 NT outputs, a wave 16 RT x 16 NT of them over the whole
// of K. Both operands come as whole lines (32 numbers of a row a step, the step after next on its way in registers) and are turned into the
// instruction's operands by two buffers in LDS, rows of 36 numbers: 16 lanes' reads of 16 bytes fall on all banks. A load's four products of a tile
// go to SETS sums in turn (so many that none waits for the one before it), which join the tile's sum every 128 or 256 k, below GF_SHORT every 64: chains of
// 128, 128 and 64 numbers for 1, 2 and 4 sets, in short sums of 64, 32 and 16, no more than a quarter of K as in the kernel above (errors against
// 64 bits at 777 rows, that kernel's / this one's: K = 1,024 2.9e-7 / 2.1e-7; 4,096 5.7e-7 / 2.1e-7; 256 1.5e-7 / 1.1e-7 - 1.5e-7, with chains of 128 2.05e-7).
// What bounds it: the matrix pipe (4096 x 252 at 1,500 rows 34 us, 91 TFLOP/s; 1697 x 1060 at 743 35, 76), of some hundred rows the last round of
// tiles. Larger products, long sums into many outputs above all, go to gemm_f32_split.hip by the rule at this file's end; this kernel has those of less than 256 inputs, those whose few tiles or steps
// would leave the other one's larger tiles idle, and rows too far apart for it. A mask on the chunks in the loop cost it 15 %: it waited for loads that had just gone out.
#define GF_LD 36
#define GF_SHORT 512  // inputs: below, single chains of 128 would be less exact than the split of K
template <int RT, int NT, int SETS>
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias, const float* residual, long ldr,
                     float* out, long ldo, int M, int N, int K, int act, int n_rows, int n_cols, int vec) {
  constexpr int BM = 32 * RT, BN = 32 * NT;
  const int piece = K < GF_SHORT ? 2 : SETS == 1 ? 4 : 8;  // steps whose products are added up before they join the sum
  __shared__ __attribute__((aligned(16))) float sm[2][BM + BN][GF_LD];  // rows of a, then of w
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int n_tiles = n_rows * n_cols, per = (n_tiles + 7) / 8;  // neighbouring columns of tiles on a chiplet, as above
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || tile >= n_tiles) return;  // the whole workgroup
  const int m0 = (tile % n_rows) * BM, o0 = (tile / n_rows) * BN;
  const int row = tid >> 3, kc = (tid & 7) * 4;
  const float* src[RT + NT];
#pragma unroll
  for (int i = 0; i < RT; ++i) src[i] = a + (size_t)min(m0 + 32 * i + row, M - 1) * lda;  // rows beyond the matrix: read again, never stored
#pragma unroll
  for (int j = 0; j < NT; ++j) src[RT + j] = w + (size_t)min(o0 + 32 * j + row, N - 1) * K;
  gf_f32x4 ahead[2][RT + NT];
  // the steps in the order they are taken: a partial one (K % 32 != 0) first, so that the loop needs no masks (one there waits for its load)
  const int tail = K % 32, steps = (K + 31) / 32;
  auto fetch = [&](gf_f32x4 (&to)[RT + NT], int t) {  // t >= 1; beyond the end: loaded again, not used
    const int k = min(max(min(t, steps - 1) - (tail ? 1 : 0), 0) * 32 + kc, K - 4);
#pragma unroll
    for (int i = 0; i < RT + NT; ++i) to[i] = *reinterpret_cast<const gf_f32x4*>(src[i] + k);
  };
  auto stage = [&](gf_f32x4 (&from)[RT + NT], int buf) {
#pragma unroll
    for (int i = 0; i < RT + NT; ++i) *reinterpret_cast<gf_f32x4*>(&sm[buf][32 * i + row][kc]) = from[i];
  };
  gf_f32x4 sum[RT][NT], acc[SETS][RT][NT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      sum[i][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < SETS; ++e) acc[e][i][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    }
  auto settle = [&]() {
#pragma unroll
    for (int e = 0; e < SETS; ++e)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sum[i][j] += acc[e][i][j], acc[e][i][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
  };
  gf_f32x4 av[2][RT], wv[2][NT];
  auto read = [&](int set, int buf, int half) {
#pragma unroll
    for (int i = 0; i < RT; ++i) av[set][i] = *reinterpret_cast<const gf_f32x4*>(&sm[buf][16 * (wm * RT + i) + col][16 * half + 4 * g]);
#pragma unroll
    for (int j = 0; j < NT; ++j) wv[set][j] = *reinterpret_cast<const gf_f32x4*>(&sm[buf][BM + 16 * (wn * NT + j) + col][16 * half + 4 * g]);
  };
  auto products = [&](int half) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          gf_f32x4& c = acc[(4 * half + e) % SETS][i][j];
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[half][j][e], av[half][i][e], c, 0, 0, 0);
        }
  };
  const int k0 = (tail ? K - tail : 0) + kc;
#pragma unroll
  for (int i = 0; i < RT + NT; ++i) ahead[0][i] = *reinterpret_cast<const gf_f32x4*>(src[i] + min(k0, K - 4));
  fetch(ahead[1], 1);
  if (k0 >= K)  // chunks beyond K count as zeros
#pragma unroll
    for (int i = 0; i < RT + NT; ++i) ahead[0][i] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
  stage(ahead[0], 0);
  lds_barrier();
  read(0, 0, 0);
  // Step t: step t + 1 goes to the other buffer and step t + 2 is asked for between the first half's products, the operands of a half are read
  // while those of the half before are multiplied. The barrier in the middle: the other buffer is whole, this one has been read.
  auto step = [&](int t, int buf) {
    constexpr int NM = 4 * RT * NT, NR = RT + NT;
    read(1, buf, 1);
    products(0);
    stage(ahead[buf ^ 1], buf ^ 1);  // behind the last step: numbers that nobody uses
    fetch(ahead[buf], t + 2);
#pragma unroll
    for (int m = 0; m < NM; ++m) {  // the order of issue: a product, then at most a few of the others
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
      for (int o = m * 3 * NR / NM; o < (m + 1) * 3 * NR / NM; ++o) {
        if (o < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        else if (o < 2 * NR) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        else __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    lds_barrier();
    read(0, buf ^ 1, 0);
    products(1);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
      for (int o = m * NR / NM; o < (m + 1) * NR / NM; ++o) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  };
  int t = 0;
  while (t + 1 < steps) {
    const int stop = min(t + piece, steps - 1);
    for (; t < stop; t += 2) {
      step(t, 0);
      step(t + 1, 1);
    }
    settle();
  }
  if (t < steps) {
    step(t, 0);
    settle();
  }
#pragma unroll
  for (int i = 0; i < RT; ++i) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int m = m0 + 16 * (wm * RT + i) + col, o = o0 + 16 * (wn * NT + j) + 4 * g;
      if (m < M && o < N) gemm_f32_store(sum[i][j], bias, residual, ldr, out, ldo, m, o, N, act, vec);
    }
  }
}

// Up to eight rows and few outputs: 16 of them a workgroup would leave most CUs without one. A workgroup of eight waves owns four outputs; a thread
// multiplies 16 bytes of each weight row with every row of a, two stretches of 2,048 k on their way at once, and the partial sums go over the lanes
// and, through LDS, over the waves: chains of 4 ceil(K / 2048) + 13 roundings (errors 0.8e-7 .. 1.1e-7 up to K = 6,400; the 16-output tiles 1.9e-7 .. 5e-7).
// What bounds it: a launch, one read of the weights (768 x 3072 at 4 rows 5.9 us, 1.6 TB/s) and 4 sums over the lanes for every row.
#define GF_FEW_OUT 4
template <int MR>
__global__ void __launch_bounds__(512)
gemm_f32_few_kernel(const float* __restrict__ w, const float* __restrict__ a, uint32_t lda4, int K, int N, int M, const float* __restrict__ bias,
                    const float* residual, float* out, long ldr, long ldo, int act) {  // in registers when the waves start: all but the last three
  const size_t lda = (size_t)lda4 * 4;
  __shared__ float part[8][GF_FEW_OUT * MR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, o0 = blockIdx.x * GF_FEW_OUT;
  const float *ar[MR], *wr[GF_FEW_OUT];
#pragma unroll
  for (int m = 0; m < MR; ++m) ar[m] = a + (size_t)min(m, M - 1) * lda;  // rows and outputs beyond the matrices: read again, never stored
#pragma unroll
  for (int j = 0; j < GF_FEW_OUT; ++j) wr[j] = w + (size_t)min(o0 + j, N - 1) * K;
  float acc[GF_FEW_OUT][MR] = {};
  for (int k0 = 0; k0 < K; k0 += 4096) {
    gf_f32x4 av[2][MR], wv[2][GF_FEW_OUT];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int kc = min(k0 + 2048 * u + 4 * tid, K - 4);
#pragma unroll
      for (int j = 0; j < GF_FEW_OUT; ++j) wv[u][j] = *reinterpret_cast<const gf_f32x4*>(wr[j] + kc);
#pragma unroll
      for (int m = 0; m < MR; ++m) av[u][m] = *reinterpret_cast<const gf_f32x4*>(ar[m] + kc);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (k0 + 2048 * u + 4 * tid < K)
#pragma unroll
        for (int j = 0; j < GF_FEW_OUT; ++j)
#pragma unroll
          for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][m] = fmaf(wv[u][j][e], av[u][m][e], acc[j][m]);
  }
#pragma unroll
  for (int j = 0; j < GF_FEW_OUT; ++j)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float s = wave_sum(acc[j][m]);
      if (lane == 0) part[wave][j * MR + m] = s;
    }
  __syncthreads();
  const int m = tid % MR, o = o0 + tid / MR;
  if (tid >= GF_FEW_OUT * MR || m >= M || o >= N) return;
  float x = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) x += part[q][tid];
  if (bias) x += bias[o];
  x = lev_activate(x, act);
  if (residual) x += residual[(size_t)m * ldr + o];
  out[(size_t)m * ldo + o] = x;
}

// Which tile: the fewest microseconds by an estimate from what was measured over 14 weights and 17 .. 2,048 rows (all tiles of both lists).
// Of the first kernel: the longest of the weights' read from memory (5.2 TB/s), the operands that a CU pulls through its L2 (37 GB/s and CU) and
// the products of the CU with the most workgroups (waves that fewer than four SIMDs hold leave the others idle). Of the second: its steps on that
// CU (a lone workgroup of 32 x 96 at what it takes with weights that no cache holds; 0.44 us a step with weights in the last cache made it the choice where it is up to
// 15 % behind: 5120 x 6400 at 100 rows 129 us, 64 x 64 of the first 113). Checked over 1,386 shapes of 512 inputs and more, weights that no cache holds: 0.3 % behind the
// best tile on average, 18 by more than 5 %, and behind the first kernel's best alone by 4 - 7 % at six, where the second's shorter chains are taken (6400 x 3072 at 100 rows 65 us, the
// first 61). (Shapes that the kernel of split operands takes by the rule below are among them.) The ends: 16 x 16 for 16 rows of 768 x 768; 64 x 64 of the second for 2304 x 256 at 777 rows, 64 x 96 for 1697 x
// 1060 at 743. Below about 100 rows and for long sums into few outputs the first stays ahead of the second: its waves split K (1024 x 4096 at 203 rows 32 us, the second 61; 768 x 3072 at 606 35).
struct GemmF32Tile {
  int rt, nt, w;
  float pipe;   // share of the matrix pipe that the tile reaches
  float start;  // microseconds before and behind the products that smaller tiles do not have
};
static const GemmF32Tile GEMM_F32_TILES[] = {{1, 1, 8, 0.8f, 0.f}, {2, 1, 8, 0.8f, 0.f}, {1, 2, 8, 0.8f, 0.f}, {1, 4, 8, 0.8f, 0.f}, {2, 2, 4, 0.8f, 0.f}, {2, 4, 4, 0.8f, 0.f}, {4, 4, 4, 0.85f, 7.f}};
struct GemmF32LineTile {
  int rt, nt, sets;
  float alone, among;  // microseconds of a step: of the one workgroup on a CU, and of one among several
  float start;
};
static const GemmF32LineTile GEMM_F32_LINE_TILES[] = {{1, 1, 4, 0.32f, 0.155f, 0.f},  {1, 2, 2, 0.37f, 0.28f, 0.5f}, {1, 3, 2, 0.6f, 0.395f, 1.f},
                                                      {2, 2, 1, 0.6f, 0.5f, 1.f},     {2, 3, 1, 0.76f, 0.73f, 2.f}};
#define GEMM_F32_N_TILES (int)(sizeof(GEMM_F32_TILES) / sizeof(GEMM_F32_TILES[0]))

static int gemm_f32_choose(int M, int N, int K, double* estimate) {  // an index into the first list, or behind its end into the second
  int best = 0;
  double best_us = 1e30;
  const double memory = 4.0 * N * K / 5.2e6;
  for (int i = 0; i < GEMM_F32_N_TILES; ++i) {
    const GemmF32Tile& t = GEMM_F32_TILES[i];
    const double groups = (double)((M + 16 * t.rt - 1) / (16 * t.rt)) * ((N + 16 * t.nt - 1) / (16 * t.nt));
    const double n = ceil(groups / 256.0), waves = n * t.w < 4.0 ? n * t.w : 4.0;
    const double l2 = n * ((16 * t.rt < M ? 16 * t.rt : M) + 16 * t.nt) * 4.0 * K / 37e3;
    const double pipe = n * (K / 4.0) * t.rt * t.nt * 32.0 / waves / (2400.0 * t.pipe);
    const double us = t.start + fmax(memory, fmax(l2, pipe));
    if (us < best_us) best_us = us, best = i;
  }
  for (int i = 0; i < (int)(sizeof(GEMM_F32_LINE_TILES) / sizeof(GEMM_F32_LINE_TILES[0])); ++i) {
    const GemmF32LineTile& t = GEMM_F32_LINE_TILES[i];
    if (t.sets < (K < 128 ? 4 : K < 256 ? 2 : 1)) continue;  // chains longer than a quarter of K
    const double n = ceil((double)((M + 32 * t.rt - 1) / (32 * t.rt)) * ((N + 32 * t.nt - 1) / (32 * t.nt)) / 256.0);
    const double us = t.start + fmax(memory, (K + 31) / 32 * fmax(t.alone + 0.15 * (n - 1) * t.among, n * t.among));
    if (us < best_us) best_us = us, best = GEMM_F32_N_TILES + i;
  }
  *estimate = best_us;
  return best;
}

// Rows that the few-row kernel has room for, or 0 where it would be behind the tiles: it reads longer sums faster than their few workgroups, and pays for
// every row and output with sums over the lanes. The inputs from which on it is level, by its room (1, 2, 4, 8) and the outputs in rounds of 256 workgroups
// (the last: all further ones), from 317 weights of 16 .. 12,800 outputs and 64 .. 16,384 inputs at 1 .. 8 rows: 4 of the 2,536 shapes are 5 % behind the tiles, none
// further. Tiles / few, microseconds, 1 / 2 / 4 / 8 rows: 768 x 768 4.5, 4.6, 4.8, 5.0 / 2.8, 3.3, 3.9, 5.3; 768 x 3072 9.8, 10.0, 10.8, 11.7 / 4.2, 5.0, 5.9, 7.7; 1024 x 4096 12.0,
// 12.2, 13.3, 14.6 / 5.1, 5.6, 6.6, 8.7; 1600 x 1600 7.1, 7.1, 7.3, 7.8 / 4.9, 5.6, 6.6, 11.9; 1600 x 2048 at 8 rows 9.0 / 12.4, 1600 x 4096 14.8 / 14.9; 1200 x 256 at 4
// rows 3.4 / 4.6; 3072 x 1024 6.0, 6.1, 5.9, 6.3 / 5.3, 5.9, 8.0, 14.9; 4096 x 4096 15.6, 15.0, 14.9, 15.7 / 12.9, 13.1, 15.3, 27.3.
static const int GEMM_F32_FEW_INPUTS[4][5] = {{0, 0, 256, 256, 768}, {256, 384, 768, 1280, 2048}, {512, 768, 2560, 8192, 8192}, {1024, 4096, 4096, 4096, 4096}};
static int gemm_f32_few(int M, int N, int K) {
  if (M < 1 || M > 8 || N < 1) return 0;
  const int i = M > 4 ? 3 : M > 2 ? 2 : M - 1, rounds = (N - 1) / (256 * GF_FEW_OUT);
  if (((long)N << i) > (K >= 2048 ? 12800 : 6400)) return 0;
  return K >= GEMM_F32_FEW_INPUTS[i][rounds < 4 ? rounds : 4] ? 1 << i : 0;
}

// the kernel of a product on the 32-bit instruction: 0 less the few-row kernel's room, or the tile's place in the two lists, one behind the other
static int gemm_f32_choice(int M, int N, int K, double* us) {
  const int few = gemm_f32_few(M, N, K);
  return few > 0 ? -few : gemm_f32_choose(M, N, K, us);
}
extern "C" int lev_linear_f32_choice(int M, int N, int K) {
  double us;
  return gemm_f32_choice(M, N, K, &us);
}

// The tile of the kernel that splits its operands into bfloat16 numbers (gemm_f32_split.hip), or -1 where the kernels above, which take `us` by their estimate, are not behind by an estimate as theirs, fitted
// to 700 shapes of 17 .. 2,200 rows and 256 .. 6,800 inputs: it is taken at 263 of them, the kernels above are up to 2 % faster at five of these, and what is kept is 0.4 % behind the best on average. Outputs
// that are stored one by one and a last workgroup alone on a CU have their terms: without them 14 of 480 shapes lost 2 - 19 % (50257 x 576 at 92 rows 62 us above, 74 here; 3072 x 1192 at 1,451 91, 97). Below 256
// inputs the kernels above stay ahead of it, or level; and it knows no rows more than GEMM_F32_SPLIT_MOST apart. Kernels above / this one, microseconds: 4096 x 1024 at 777 rows 64 / 50, 1024 x 4096 74 / 64,
// 50257 x 768 at 300 rows 209 / 166, 4096 x 4096 at 2,048 502 / 366, 1600 x 1600 at 512 34 / 27; not taken: 768 x 3072 at 606 rows 36 / 46, 1024 x 1024 at 404 15 / 19.
static int gemm_f32_split_tile(int M, int N, int K, int choice, double us) {
  if (K % 4 != 0 || K < 256 || K > GEMM_F32_SPLIT_MOST || choice < 0) return -1;
  us *= 0.92;  // the estimates' own errors (0.964 would take 20 more of the shapes, two of them 2 - 4 % slower)
  int best = -1;
  for (int i = 0; i < GEMM_F32_N_SPLIT_TILES; ++i) {
    const GemmF32SplitTile& t = GEMM_F32_SPLIT_TILES[i];
    const double n = ceil((double)((M + t.rows - 1) / t.rows) * ((N + t.outputs - 1) / t.outputs) / 256.0);
    const double step = n <= 1.0 ? t.alone : n * t.among + fmod(n, 2.0) * t.odd;
    const double own = t.start + fmax(4.0 * N * K / 5.2e6, ((K + 31) / 32 + t.groups - 1) / t.groups * step) + (N % 4 != 0 ? n * t.single : 0.0);
    if (own < us) us = own, best = i;
  }
  return best;
}
extern "C" int lev_linear_f32_split(int M, int N, int K) {
  double us;
  const int choice = gemm_f32_choice(M, N, K, &us);
  return gemm_f32_split_tile(M, N, K, choice, us);
}

// 1: not for these operands (nothing has been launched): 16-byte loads need rows of a multiple of 4 numbers at 16-byte addresses
int lev_gemm_f32(const float* a, long lda, const float* w, const float* bias, const float* residual, long ldr, float* out, long ldo, int M, int N, int K,
                 int act, hipStream_t stream) {
  if (K % 4 != 0 || lda % 4 != 0 || ((uintptr_t)a & 15) != 0 || ((uintptr_t)w & 15) != 0) return 1;
  const int vec = ldo % 4 == 0 && ((uintptr_t)out & 15) == 0 && (!bias || ((uintptr_t)bias & 15) == 0) && (!residual || (ldr % 4 == 0 && ((uintptr_t)residual & 15) == 0));
  double us;
  const int choice = gemm_f32_choice(M, N, K, &us), split = lda <= GEMM_F32_SPLIT_MOST ? gemm_f32_split_tile(M, N, K, choice, us) : -1;
  if (split >= 0) return lev_gemm_f32_split(split, a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, vec, stream);
  const int few = -choice, line = choice - GEMM_F32_N_TILES;
  if (few > 0) {
#define GEMM_F32_FEW(MR) \
  if (few == MR) gemm_f32_few_kernel<MR><<<(N + GF_FEW_OUT - 1) / GF_FEW_OUT, 512, 0, stream>>>(w, a, (uint32_t)(lda / 4), K, N, M, bias, residual, out, ldr, ldo, act)
    GEMM_F32_FEW(1);
    else GEMM_F32_FEW(2);
    else GEMM_F32_FEW(4);
    else GEMM_F32_FEW(8);
#undef GEMM_F32_FEW
    return lev_check_launch("linear (32-bit, few rows)");
  }
  const int rt = line < 0 ? GEMM_F32_TILES[choice].rt : 2 * GEMM_F32_LINE_TILES[line].rt, nt = line < 0 ? GEMM_F32_TILES[choice].nt : 2 * GEMM_F32_LINE_TILES[line].nt;
  const int n_rows = (M + 16 * rt - 1) / (16 * rt), n_cols = (N + 16 * nt - 1) / (16 * nt);
  const long blocks = ((long)n_rows * n_cols + 7) / 8 * 8;
  LEV_REQUIRE(blocks <= 0x7fffffffL, "linear: too many tiles (%ld)", blocks);
#define GEMM_F32_CASE(RT, NT, W)                                                                                                                    \
  if (line < 0 && rt == RT && nt == NT)                                                                                                             \
    gemm_f32_kernel<RT, NT, W><<<(unsigned)blocks, 64 * W, W * RT * NT * 1024, stream>>>(w, a, (uint32_t)(lda / 4), K, N, M, n_rows, n_cols, vec, act, bias, residual, out, ldr, ldo)
#define GEMM_F32_LINE_CASE(RT, NT, SETS)                                                                                                            \
  if (rt == 2 * RT && nt == 2 * NT)                                                                                                                 \
    gemm_f32_tile_kernel<RT, NT, SETS><<<(unsigned)blocks, 256, 0, stream>>>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, n_rows, n_cols, vec)
  GEMM_F32_CASE(1, 1, 8);
  else GEMM_F32_CASE(2, 1, 8);
  else GEMM_F32_CASE(1, 2, 8);
  else GEMM_F32_CASE(1, 4, 8);
  else GEMM_F32_CASE(2, 2, 4);
  else GEMM_F32_CASE(2, 4, 4);
  else GEMM_F32_CASE(4, 4, 4);
  else GEMM_F32_LINE_CASE(1, 1, 4);
  else GEMM_F32_LINE_CASE(1, 2, 2);
  else GEMM_F32_LINE_CASE(1, 3, 2);
  else GEMM_F32_LINE_CASE(2, 2, 1);
  else GEMM_F32_LINE_CASE(2, 3, 1);
#undef GEMM_F32_LINE_CASE
#undef GEMM_F32_CASE
  return lev_check_launch("linear (32-bit)");
}
