// bfloat16 matrix products of some dozen to about a thousand rows: y = act(a . w^T + bias) (+ residual), a [M, K] (row stride lda), w [N, K],
// 32-bit accumulation, y bfloat16 or float32. K and lda multiples of 8, any M and N.
//
// What bounds such a product is neither memory nor the matrix pipe but what a CU fetches: tiles are small (the outputs have to be spread over
// 256 CUs), so every CU reads its rows of both operands line by line, half of them from memory the first time, and a CU has about 600
// lines of 128 bytes in flight at most, hits behind misses (lines fetched 1,280 a microsecond when all lie in L2, 600 when the weights come from memory:
// 264 rows of 4800 x 1600 spend 7.5 of 11.4 us on it). So the lines are kept in flight all the time: k-tiles of 64 (whole lines) go straight
// into LDS, into a ring of 4 to 6 of them, and wait there for nobody's registers; a wave's operands for the next k-tile are read from LDS while
// this one's products run; one barrier a k-tile. Small tiles leave room for two workgroups a CU, large ones have eight waves.
// In LDS a row's eight chunks of 16 bytes change places with the row, so that reads of one chunk of 16 rows meet no bank twice; a load puts 64 lanes'
// chunks one behind the other, so the lane's address does the swapping.
// Measured in graphs over distinct weights, microseconds, before (the library, the tile kernel through registers or row blocks) / here: 264 rows of 4800 x
// 1600 14.5 / 9.9, 6400 x 1600 19.3 / 13.9, 1600 x 1600 11.8 / 7.1, 1600 x 6400 22.3 / 18.7 (15.0 where the norm behind it adds the ranges); 128 rows of 4800 x 1600 9.5 / 8.1,
// 768 x 3072 12.8 / 8.1, 2048 x 5376 at 600 rows 31.2 / 26.1, 4096 x 16384 at 264 rows 73 / 56. Errors against 64 bits, before / here: 264 rows of 4800 x
// 1600 2.4e-7 / 1.2e-7, 1600 x 6400 1.95e-7 / 1.4e-7, 2048 x 5376 at 400 rows 4.6e-7 / 2.2e-7; of the row blocks and ranges of K (with one chain of K / 128 here they were
// exceeded, 1.3e-7 at 2,048 inputs: the joins are for these) 96 rows of 3072 x 2048 8.6e-8 / 8.2e-8, 256 of 1600 x 1600 8.3e-8 / 7.9e-8, 192 of 2560 x 1024 7.5e-8 / 7.4e-8, 128 of
// 4096 x 4096 1.24e-7 / 0.92e-7, 700 of 384 x 1536 9.9e-8 / 9.1e-8; of 856 sizes (45 weights, 17 to 2,020 rows), with
// the ranges left and not, none is further off. Taken back: k-tiles that begin at another place in every
// workgroup (up to 40 % slower where neighbours then no longer wait for the same line, 2 - 9 % faster at K = 16384 alone), a ring twice as deep (8 % slower), a
// CU for every workgroup where two fit (the same).
#include "gemm_ring.h"
#include "ring.h"
#include <math.h>
#include <algorithm>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}

// How many sums in turn a wave of so many 16 x 16 tiles has registers for, one of so many waves of a workgroup, and whether for a total beside them. (128 x 128 at 1,300
// rows of 2048 x 2048 21.8 us with four sums, 17.8 with two.)
constexpr int ring_sums(int tiles, int waves) { return tiles <= 6 ? 4 : waves == 8 ? 2 : 1; }
constexpr bool ring_joins(int tiles) { return tiles <= 6; }

// A workgroup of WGM x WGN waves computes BM x BN outputs, a wave BM / WGM x BN / WGN, in 16 x 16 x 32 products with w as the first operand: a lane then holds four
// neighbouring outputs of a row, and eight of a pair of tiles, whose rows of w are dealt out for that. R: k-tiles of the ring.
template <typename TO, int BM, int BN, int WGM, int WGN, int R>
__global__ void __launch_bounds__(WGM * WGN * 64, R * (BM + BN) * 128 <= 80 * 1024 ? WGM * WGN / 2 : WGM * WGN / 4)
gemm_ring_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, uint32_t lda, int K, int M, int N, int tiles_m, int tiles_n, int S, int act,
                 const float* __restrict__ bias, const float* residual, TO* out, float* __restrict__ partial, long ldr, long ldo, int vec_ok, int fold, size_t range) {  // range: numbers of a range's sums
  constexpr int W = WGM * WGN, WM = BM / WGM, WN = BN / WGN, TI = WM / 16, TJ = WN / 16;
  static_assert(TJ % 2 == 0 && WM % 16 == 0 && BM % (8 * W) == 0 && BN % (8 * W) == 0 && R >= 3, "pairs of column tiles; whole loads a wave");
  constexpr int LA = BM / 8 / W, LW = BN / 8 / W, L = LA + LW;  // a wave's loads a k-tile, 8 lines each
  constexpr int TILE = (BM + BN) * 128;
  extern __shared__ __attribute__((aligned(1024))) char lds_ring[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  // each chiplet takes a stretch of tiles: tiles of the same rows of w one behind the other, then the next, then the next range of K
  const int total = gridDim.x, q8 = total >> 3, r8 = total & 7, xcd = blockIdx.x & 7;
  const int id = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
  const int split = id / (tiles_m * tiles_n), tile = id - split * (tiles_m * tiles_n);
  const int tn = tile / tiles_m, m0 = (tile - tn * tiles_m) * BM, n0 = tn * BN;
  // The k-tiles in the order they are taken: tile 0 is the partial one (K % 64 != 0), if there is one, so that no other needs a mask; tile t starts at
  // k = 64 t - (64 - K % 64), or 64 t. This workgroup takes t0 .. t0 + nk - 1.
  const int tail = K & 63, nk_all = (K + 63) >> 6, per = (nk_all + S - 1) / S, t0 = split * per, nk = min(nk_all, t0 + per) - t0;

  // Rows beyond the matrix read the last one; their products are never stored. Offsets are within the tile, below 2^32 bytes (the launch sees to that).
  uint32_t off[L];
  const int lr = lane >> 3, lc = lane & 7;
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = (wave * LA + i) * 8 + lr;
    off[i] = (uint32_t)min(r, M - 1 - m0) * lda * 2 + (uint32_t)((lc ^ ring_swap_rows(r)) * 16);
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int r = (wave * LW + i) * 8 + lr;
    off[LA + i] = (uint32_t)min(r, N - 1 - n0) * (uint32_t)K * 2 + (uint32_t)((lc ^ ring_swap_columns(r)) * 16);
  }
  const uint32_t lds0 = lds_offset(lds_ring);
  const long first = tail ? (t0 == 0 ? 0 : (long)t0 * 64 - (64 - tail)) : (long)t0 * 64;
  const char *ab = reinterpret_cast<const char*>(a + (size_t)m0 * lda + first), *wb = reinterpret_cast<const char*>(w + (size_t)n0 * K + first);
  auto load_one = [&](uint32_t at, int i) {
    if (i < LA) lines_to_lds(at + (wave * LA + i) * 1024, off[i], ab);
    else lines_to_lds(at + BM * 128 + (wave * LW + i - LA) * 1024, off[i], wb);
  };
  int ahead = 0;  // k-tiles asked for
  if (tail && t0 == 0) {  // the partial tile: chunks beyond it repeat the row's last one inside it, and are cleared once they have landed
    const int chunks = tail >> 3;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int r = ((i < LA ? wave * LA + i : wave * LW + i - LA)) * 8 + lr;
      const int c = lc ^ (i < LA ? ring_swap_rows(r) : ring_swap_columns(r));
      const uint32_t o = off[i] - (uint32_t)((c - min(c, chunks - 1)) * 16);
      if (i < LA) lines_to_lds(lds0 + (wave * LA + i) * 1024, o, ab);
      else lines_to_lds(lds0 + BM * 128 + (wave * LW + i - LA) * 1024, o, wb);
    }
    ab += tail * 2, wb += tail * 2;
    ahead = 1;
  }
  const int most = min(R, nk);
#pragma unroll 1
  for (; ahead < most; ++ahead) {
#pragma unroll
    for (int i = 0; i < L; ++i) load_one(lds0 + ahead * TILE, i);
    ab += 128, wb += 128;
  }
  // Sums in turn, joined at the end and on the way: a chain of roundings is at most `fold` * 2 / SUMS products long (ring_fold says why).
  constexpr int SUMS = ring_sums(TI * TJ, W);
  constexpr bool JOINS = ring_joins(TI * TJ);
  f32x4 sums[SUMS][TI][TJ], joined[JOINS ? TI : 1][JOINS ? TJ : 1];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      if constexpr (JOINS) joined[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < SUMS; ++s) sums[s][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  auto join = [&](bool last) __attribute__((always_inline)) {  // last: what all outputs take is in sums[0]
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        if constexpr (SUMS == 4) sums[2][i][j] += sums[3][i][j];
        if constexpr (SUMS >= 2) sums[0][i][j] += sums[1][i][j];
        if constexpr (SUMS == 4) sums[0][i][j] += sums[2][i][j];
        if constexpr (JOINS) {
          if (last) {
            sums[0][i][j] += joined[i][j];
            continue;
          }
          joined[i][j] += sums[0][i][j];
#pragma unroll
          for (int s = 0; s < SUMS; ++s) sums[s][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
  };
  auto join_in_time = [&](int kt) __attribute__((always_inline)) {  // kt: k-tiles summed up
    if constexpr (JOINS)
      if (((kt + (fold >> 1)) & (fold - 1)) == 0) join(false);
  };
  auto& acc = sums[0];
  // operand (row l % 16, k-group l / 16) of a k-step of 32; column tile j = 2 p + h takes the rows 32 p + 8 (l % 16 / 4) + 4 h + l % 4 of w
  const int fr = lane & 15, kg = lane >> 4, wr = 8 * (fr >> 2) + (fr & 3);
  const int a_at = (wm * WM + fr) * 128 + ((kg ^ ring_swap_rows(fr)) * 16);
  const int w_at[2] = {(BM + wn * WN + wr) * 128 + ((kg ^ ring_swap_columns(wr)) * 16), (BM + wn * WN + wr + 4) * 128 + ((kg ^ ring_swap_columns(wr + 4)) * 16)};
  u32x4 af[2][2][TI], wf[2][2][TJ];
  constexpr int READS = 2 * (TI + TJ), PRODUCTS = 2 * TI * TJ;
  auto read_one = [&](auto set, const char* kt, int o) {  // the o-th of a k-tile's operands
    constexpr int c = decltype(set)::value;
    const int ks = o / (TI + TJ), q = o % (TI + TJ);
    if (q < TJ) wf[c][ks][q] = *reinterpret_cast<const u32x4*>(kt + (w_at[q & 1] ^ (ks * 64)) + (q >> 1) * 4096);
    else af[c][ks][q - TJ] = *reinterpret_cast<const u32x4*>(kt + (a_at ^ (ks * 64)) + (q - TJ) * 2048);
  };
  auto product = [&](auto set, int m) {
    constexpr int c = decltype(set)::value;
    const int ks = m / (TI * TJ), i = m % (TI * TJ) / TJ, j = m % TJ;
    f32x4& sum = sums[(2 * c + ks) % SUMS][i][j];
    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wf[c][ks][j]), as_bf16x8(af[c][ks][i]), sum, 0, 0, 0);
  };
  typedef std::integral_constant<int, 0> Zero;
  typedef std::integral_constant<int, 1> One;
  ring_wait_for<R, L>(most - 1);
  if (tail && t0 == 0) {
    const int chunks = tail >> 3;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int at = i < LA ? (wave * LA + i) * 1024 : BM * 128 + (wave * LW + i - LA) * 1024;
      const int r = ((i < LA ? wave * LA + i : wave * LW + i - LA)) * 8 + lr;
      if ((lc ^ (i < LA ? ring_swap_rows(r) : ring_swap_columns(r))) >= chunks) *reinterpret_cast<u32x4*>(lds_ring + at + lane * 16) = u32x4{0, 0, 0, 0};
    }
  }
  lds_barrier();
#pragma unroll
  for (int o = 0; o < READS; ++o) read_one(Zero(), lds_ring, o);

  // One k-tile: its products, between them the reads of the next one's operands (landed, and seen by all behind the barrier) and, into its own place of
  // the ring (every wave has read it), the loads of the one R further on. The order of issue is as written.
  int place = 0;
  auto step = [&](auto set, auto loads, int kt) {
    constexpr bool on = decltype(loads)::value;
    if constexpr (on) ring_wait<(R - 2) * L>(); else ring_wait_for<R, L>(min(R - 2, nk - 2 - kt));
    lds_barrier();
    const uint32_t into = lds0 + place * TILE;
    place = place + 1 == R ? 0 : place + 1;
    const char* next = lds_ring + place * TILE;
#pragma unroll
    for (int m = 0; m < PRODUCTS; ++m) {
#pragma unroll
      for (int o = m * READS / PRODUCTS; o < (m + 1) * READS / PRODUCTS; ++o) read_one(std::integral_constant<int, decltype(set)::value ^ 1>(), next, o);
      if constexpr (on) {
#pragma unroll
        for (int i = m * L / PRODUCTS; i < (m + 1) * L / PRODUCTS; ++i) load_one(into, i);
      }
      product(set, m);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (on) ab += 128, wb += 128;
  };
  auto last = [&](auto set) {
#pragma unroll
    for (int m = 0; m < PRODUCTS; ++m) product(set, m);
  };
  int kt = 0;
  for (; kt + 1 + R < nk; kt += 2) {
    step(Zero(), One(), kt);
    step(One(), One(), kt + 1);
    join_in_time(kt + 2);
  }
  bool odd = false;  // the next k-tile's operands are in the second set
  if (kt + R < nk) {
    step(Zero(), One(), kt++);
    odd = true;
    if (kt + 1 < nk) {
      step(One(), Zero(), kt++);
      odd = false;
      join_in_time(kt);
    }
  }
  for (; kt + 2 < nk; kt += 2) {
    step(Zero(), Zero(), kt);
    step(One(), Zero(), kt + 1);
    join_in_time(kt + 2);
  }
  if (kt + 1 < nk) {
    step(Zero(), Zero(), kt);
    odd = true;
  }
  if (odd) last(One()); else last(Zero());
  join(true);

  // register r of lane l: column 8 (l / 16) + 4 h + r of a pair of tiles, row l % 16
  if (S > 1) {
#pragma unroll
    for (int p = 0; p < TJ / 2; ++p) {
      const int n = n0 + wn * WN + p * 32 + kg * 8;
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int m = m0 + wm * WM + i * 16 + fr;
        if (m >= M) continue;
        float* o = partial + split * range + (size_t)m * N + n;
        if ((vec_ok & 2) && n + 7 < N) {
          reinterpret_cast<f32x4*>(o)[0] = acc[i][2 * p];
          reinterpret_cast<f32x4*>(o)[1] = acc[i][2 * p + 1];
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < N) o[e] = acc[i][2 * p + (e >> 2)][e & 3];
        }
      }
    }
    return;
  }
  auto store8 = [&](float (&v)[8], int m, int n) {
    TO* o = out + (size_t)m * ldo + n;
    if ((vec_ok & 1) && n + 7 < N) {
      if (residual) {
        const f32x4* rr = reinterpret_cast<const f32x4*>(residual + (size_t)m * ldr + n);
        const f32x4 r0 = rr[0], r1 = rr[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += r0[e], v[4 + e] += r1[e];
      }
      if constexpr (sizeof(TO) == 4) {
        reinterpret_cast<f32x4*>(o)[0] = f32x4{v[0], v[1], v[2], v[3]};
        reinterpret_cast<f32x4*>(o)[1] = f32x4{v[4], v[5], v[6], v[7]};
      } else {
        *reinterpret_cast<u32x4*>(o) = u32x4{float2_to_bf16x2(v[0], v[1]), float2_to_bf16x2(v[2], v[3]), float2_to_bf16x2(v[4], v[5]), float2_to_bf16x2(v[6], v[7])};
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < N) o[e] = from_float<TO>(residual ? v[e] + residual[(size_t)m * ldr + n + e] : v[e]);
    }
  };
  auto finish = [&](auto activation) {
    constexpr int ACT = decltype(activation)::value;
#pragma unroll
    for (int p = 0; p < TJ / 2; ++p) {
      const int n = n0 + wn * WN + p * 32 + kg * 8;
      if (n >= N) continue;
      float b[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = bias ? bias[min(n + e, N - 1)] : 0.f;
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int m = m0 + wm * WM + i * 16 + fr;
        if (m >= M) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = lev_activate_as<ACT>(acc[i][2 * p + (e >> 2)][e & 3] + b[e], 0);
        store8(v, m, n);
      }
    }
  };
  if (act == LEV_ACT_NONE) {
    finish(std::integral_constant<int, LEV_ACT_NONE>());
  } else if (act == LEV_ACT_GELU_TANH) {
    finish(std::integral_constant<int, LEV_ACT_GELU_TANH>());
  } else {
    // The other activations are long; one copy of them, in a loop over the wave's sums in LDS (an area of its own; the ring has been read by all).
    lds_barrier();
    constexpr int CS = WN + 4;
    float* mine = reinterpret_cast<float*>(lds_ring) + wave * 16 * CS;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
      for (int p = 0; p < TJ / 2; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<f32x4*>(mine + fr * CS + p * 32 + kg * 8 + h * 4) = acc[i][2 * p + h];
      lds_wave_order();
      const int m = m0 + wm * WM + i * 16 + fr;
#pragma unroll 1
      for (int p = 0; p < TJ / 2; ++p) {
        const int n = n0 + wn * WN + p * 32 + kg * 8;
        if (m >= M || n >= N) continue;
        float v[8];
#pragma unroll 1
        for (int e = 0; e < 8; ++e) {
          float* at = mine + fr * CS + p * 32 + kg * 8 + e;
          const float u = *at + (bias ? bias[min(n + e, N - 1)] : 0.f);
          *at = (act == LEV_ACT_GELU_ERF && sizeof(TO) == 2) ? lev_gelu_erf_coarse(u) : lev_activate(u, act);  // exact GELU of a bfloat16 output: the short erf
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = mine[fr * CS + p * 32 + kg * 8 + e];
        store8(v, m, n);
      }
      lds_wave_order();
    }
  }
}

// The tiles: whether two workgroups fit a CU, and microseconds of a k-tile, for one alone on its CU and for one of two, and of a round's ends.
struct RingShape {
  int bm, bn;
  bool two;
  double alone, beside, ends;
};
static const RingShape kRing[8] = {
    {32, 64, true, 0.142, 0.259, 1.24}, {64, 64, true, 0.174, 0.340, 1.42},
    {96, 64, true, 0.212, 0.430, 1.41}, {128, 64, false, 0.269, 0.269, 1.83},
    {64, 128, false, 0.291, 0.291, 1.92}, {96, 128, false, 0.363, 0.363, 2.19},
    {128, 128, false, 0.402, 0.402, 2.23}, {192, 128, false, 0.491, 0.491, 2.71},
};

// An estimate of every tile and number of ranges: rounds of the CUs times a workgroup's k-tiles, joined (exponent 1.27: neither hides the other wholly) with the time the
// weights take from memory, and what writing the sums costs; of ranges also the pass that adds them: a kernel of its own, or, where they are left, what
// the norm behind the product pays for them (64 rows of 1600: 2.5 us, with 2 / 4 / 8 ranges 3.2 / 3.4 / 4.1; 264 rows 2.8, 4.4 / 5.0 / 6.1), which gives a row a thousand threads then:
// beyond two rows a CU they take turns; activations that no L2 holds are read by each column of tiles (4,000 rows of 512 x 2048: 128 columns a tile 17.8 us, 64 24.5). One price for all sums of K >= 4 N, as if a norm always followed, put 2,020 rows of 128 x 2048 into two ranges and a pass (9.5 us; in one 8.7), 128 x 512 at
// 1,024 into four (6.6, 4.9), and with the norm 64 x 4096 at 4,000 into four (21.6, 20.2). It stands for longer sums with a pass of their own: in one range their small tiles take up to 30 % more
// than the estimate, about what the pass costs (700 rows of 1280 x 5120 28.7 us in one, 23.9 in three). The tiles' numbers are fitted to
// 13,000 launches (25 weights of 512 x 2048 to 16384 x 4096, 64 to 2,048 rows, up to five million outputs), off by 6 % on average; the prices of ranges to 16,000 more (34 weights of
// 16 x 2048 to 4096 x 16384 in no cache, 17 to 4,000 rows, each with its own pass and with the norm): the choice is 0.9 and 1.5 % behind the best on average, more than 8 % at 9 and 19 of
// 440 shapes (264 rows of 2048 x 5376 22.8 us for 20.4).
static RingPlan ring_choice(int M, int N, int K, bool left) {
  const int nk = (K + 63) >> 6;
  const double weights = 2e-6 * N * K * 0.140, outputs = 4e-6 * M * N;
  RingPlan best = {0, 1, 1e30};
  for (int i = 0; i < 8; ++i) {
    const RingShape& sh = kRing[i];
    const long tiles = (long)((M + sh.bm - 1) / sh.bm) * ((N + sh.bn - 1) / sh.bn);
    for (int s = 1; s <= 8; ++s) {
      const long wgs = tiles * s;
      const int per = (nk + s - 1) / s;
      if (s > 1 && (wgs > 520 || nk / s < 2)) break;
      if (per * (s - 1) >= nk) continue;  // a range would be empty
      if ((i == 7 && per > 96) || (i == 5 && per > 64) || (i > 4 && M <= 128)) continue;  // no registers for a total (96 x 128: for a second sum): chains would be longer than before
      const double beyond = 2e-6 * M * K / s / 4.2 - 1.0;  // activations of a range that an L2 does not hold
      double cus;
      if (sh.two) {
        const long rest = wgs % 512;
        cus = (double)(wgs / 512) * (per * sh.beside + sh.ends) + (rest > 256 ? per * sh.beside + sh.ends : rest > 0 ? per * sh.alone + sh.ends : 0.0);
      } else {
        cus = (double)((wgs + 255) / 256) * (per * sh.alone + sh.ends);
      }
      cus *= 1.0 + 0.110 * (beyond < 0.0 ? 0.0 : beyond > 1.0 ? 1.0 : beyond);
      const double rows = 2e-6 * M * K / s > 16.0 ? 0.028 * ((N + sh.bn - 1) / sh.bn) * 2e-6 * M * K : 0.0;  // every column of tiles reads them from beyond the caches of a chiplet
      double us = 1.63 + pow(pow(cus, 1.27) + pow(weights + rows, 1.27), 1.0 / 1.27) + 0.214 * s * outputs;
      if (s > 1) {
        const int more_rows = std::max(0, M - 512);
        if (left) us += 0.1 + s * outputs / 4.5 + 1.5e-3 * more_rows;
        else if (K >= 4L * N && (long)N * K >= (3L << 19)) us += 0.1 + s * outputs / 4.5;
        else us += 1.5 + 0.22 * (s + 1) * outputs + 0.8e-3 * more_rows;
      }
      if (us < best.us) best = {i, s, us};
    }
  }
  return best;
}

// The choice takes the host 3 us, a launch less: the last ones are kept, by the sizes and `left` alone.
RingPlan lev_ring_plan(int M, int N, int K, bool left) {
  static thread_local struct { int M, N, K; bool left; RingPlan plan; } kept[64];
  auto& slot = kept[((unsigned)M * 31u + (unsigned)N * 7u + (unsigned)K * 2u + left) * 2654435769u >> 26];
  if (slot.M != M || slot.N != N || slot.K != K || slot.left != left) slot = {M, N, K, left, ring_choice(M, N, K, left)};
  return slot.plan;
}

// Every how many k-tiles (a power of two; the first time after half as many) a wave's sums join its total: so that no chain of roundings is longer than in the kernels that
// had these products before. Those were row blocks up to 256 rows (2 to 4 products a chain), ranges of K up to 128 rows of larger weights (10 and more), up to 320 rows of
// small ones and of long sums of narrow outputs (700 rows of 384 x 1536: 9.9e-8 then, 1.14e-7 in one chain), and else above 256 rows the library's kernels and tiles of one chain. In 64 x 64 tiles a join every 8 k-tiles costs 2 - 3 %.
static int ring_fold(int BM, int BN, int M) {
  const int never = 1 << 20;
  if (BM * BN > 64 * 64) return M <= 128 ? 16 : never;
  return M <= 256 ? 8 : 16;
}

template <typename TO, int BM, int BN, int WGM, int WGN, int R>
static int launch_ring(const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr, TO* out, long ldo, float* partial, int M,
                       int N, int K, int act, int S, int vec_ok, hipStream_t stream) {
  constexpr int lds = R * (BM + BN) * 128;
  static std::atomic<unsigned long long> reserved{0};  // per instantiation
  if (int rc = lev_reserve_lds((const void*)gemm_ring_kernel<TO, BM, BN, WGM, WGN, R>, lds, reserved)) return rc;
  const int fold = ring_fold(BM, BN, M), tiles_n = (N + BN - 1) / BN;
  // as many rows a launch as a tile's offsets reach (rows of a tile are 70 MB and more apart, if that is fewer than a tile has: a column block of a very wide matrix)
  const long reach = ((1L << 32) - 256) / (2 * lda) + 1;
  const int rows = reach >= std::min(BM, M) ? M : (int)reach;
  for (int m = 0; m < M; m += rows) {
    const int here = std::min(rows, M - m), tiles_m = (here + BM - 1) / BM;
    gemm_ring_kernel<TO, BM, BN, WGM, WGN, R><<<tiles_m * tiles_n * S, WGM * WGN * 64, lds, stream>>>(
        a + m * lda, w, (uint32_t)(here > 1 ? lda : 0), K, here, N, tiles_m, tiles_n, S, act, bias, residual ? residual + m * ldr : nullptr, out + m * ldo,
        partial ? partial + (size_t)m * N : nullptr, ldr, ldo, vec_ok, fold, (size_t)M * N);
  }
  return lev_check_launch("linear_ring");
}

template <typename TO>
static int launch_ring_typed(const RingPlan& plan, const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr, TO* out, long ldo,
                             float* partial, int M, int N, int K, int act, hipStream_t stream) {
  if (K > RING_MAX_K) return lev_fail("linear: a sum of %d products is too long for the ring kernel", K);
  const int S = plan.splits;
  if (S > 1 && !partial) return lev_fail("linear: M=%d N=%d K=%d needs a workspace of lev_linear_mfma_workspace bytes", M, N, K);
  const int vec_out = ldo % (sizeof(TO) == 4 ? 4 : 8) == 0 && ((uintptr_t)out & 15) == 0 && (!residual || (ldr % 4 == 0 && ((uintptr_t)residual & 15) == 0));
  const int vec_ok = vec_out | (N % 4 == 0 && ((uintptr_t)partial & 15) == 0 ? 2 : 0);
#define LEV_RING(BM_, BN_, WGM_, WGN_, R_) \
  return launch_ring<TO, BM_, BN_, WGM_, WGN_, R_>(a, lda, w, bias, residual, ldr, out, ldo, partial, M, N, K, act, S, vec_ok, stream)
  switch (plan.shape) {
    case 0: LEV_RING(32, 64, 2, 2, 6);
    case 1: LEV_RING(64, 64, 2, 2, 5);
    case 2: LEV_RING(96, 64, 2, 2, 4);
    case 3: LEV_RING(128, 64, 4, 2, 6);
    case 4: LEV_RING(64, 128, 2, 4, 6);
    case 5: LEV_RING(96, 128, 2, 2, 5);
    case 6: LEV_RING(128, 128, 2, 4, 5);
    default: LEV_RING(192, 128, 4, 2, 4);
  }
#undef LEV_RING
}

int lev_ring_launch(const RingPlan& plan, const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr, void* out, long ldo,
                    float* partial, int M, int N, int K, int act, int out_dtype, hipStream_t stream) {
  if (out_dtype == LEV_F32) return launch_ring_typed<float>(plan, a, lda, w, bias, residual, ldr, (float*)out, ldo, partial, M, N, K, act, stream);
  return launch_ring_typed<bf16_t>(plan, a, lda, w, bias, residual, ldr, (bf16_t*)out, ldo, partial, M, N, K, act, stream);
}
