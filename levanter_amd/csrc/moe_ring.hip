// The experts' products over tiles of 128 rows, by workgroups that stay on their CU: out[pos] = act(w[expert] a[row(pos)]), bfloat16 operands, 32-bit sums.
//
// A workgroup of eight waves has a CU to itself and takes every 32nd of its chiplet's units (a tile of the list and 256 rows of w: 256 outputs, or with glu 128
// outputs' gate rows and up rows); their k-tiles of 64 form one stream through a ring of three in LDS, loaded straight from memory: while the last products of a
// unit run and its outputs leave, the first k-tiles of the next are on their way. A tile's and its neighbours' units follow each other on one chiplet, whose L2
// then has an expert's rows of w for all of its tiles. Waves whose 64 rows lie beyond a tile's rows skip the products (the other of their SIMD has them).
// Every unit walks K from a place of its own, given by its expert and columns: rows of w a power of two apart lie in the same channels of the memory, and units
// that walk together ask those alone. (By expert and columns, so that a token's sums have one order whatever the other tokens choose.)
// What bounds it: the products (1.0 - 1.1 PFLOP/s where experts have thousands of rows), the read of the weights (5 TB/s) with up to about 100 rows an expert; between
// them both, and the last round of units. Measured, microseconds of 2048 outputs of 2048 (bfloat16 / 32-bit / gated), tiles of 128 x 128 by four waves through registers, two
// workgroups a CU / here: 32 experts of 254 drawn rows 134, 133, 227 / 120, 117, 192; of 256 109, 115, 187 / 84, 86, 156; of 128 64, 66, 131 / 62, 63, 111; of 40 drawn 54,
// 56, 101 / 51, 53, 98; of 600 232, 244, 440 / 194, 209, 359; 4 of 2,048 75, 77, 148 / 63, 69, 129. Not kept: 128 rows of w a unit (each CU then fetches a third more: 130,
// 127, 223 of the first), places along K by the columns alone (32 of 256 91), the same place for all (118).
#include "moe.h"
#include "ring.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}

#define MOE_RING_BN 256    // rows of w a unit
#define MOE_RING_TILES 3   // k-tiles of the ring
#define MOE_RING_TILE ((MOE_BIG + MOE_RING_BN) * 128)
#define MOE_RING_LDS (MOE_RING_TILES * MOE_RING_TILE + 2 * MOE_BIG * (int)sizeof(int))
#define MOE_RING_CUS 32  // workgroups a chiplet

typedef const __attribute__((address_space(4))) int* scalar_ints;  // read by scalar loads, which do not queue up behind the ring's

// eight neighbouring outputs of a row; vec 2: as 16-byte stores, 1: (bfloat16) as 8-byte ones, `left`: so many are inside the row
__device__ __forceinline__ void moe_store8(float* to, const float (&v)[8], int left, int vec) {
  if (vec && left >= 8) {
    reinterpret_cast<f32x4*>(to)[0] = f32x4{v[0], v[1], v[2], v[3]};
    reinterpret_cast<f32x4*>(to)[1] = f32x4{v[4], v[5], v[6], v[7]};
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < left) to[e] = v[e];
  }
}
__device__ __forceinline__ void moe_store8(bf16_t* to, const float (&v)[8], int left, int vec) {
  const u32x4 b = u32x4{float2_to_bf16x2(v[0], v[1]), float2_to_bf16x2(v[2], v[3]), float2_to_bf16x2(v[4], v[5]), float2_to_bf16x2(v[6], v[7])};
  if (vec == 2 && left >= 8) {
    *reinterpret_cast<u32x4*>(to) = b;
  } else if (vec && left >= 8) {
    reinterpret_cast<uint2*>(to)[0] = make_uint2(b[0], b[1]);
    reinterpret_cast<uint2*>(to)[1] = make_uint2(b[2], b[3]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < left) to[e] = (bf16_t)(b[e / 2] >> (e % 2 * 16));
  }
}

template <typename TO, bool GLU>
__global__ void __launch_bounds__(512, 2)
moe_ring_kernel(const MoeLinearArgs p) {
  constexpr int R = MOE_RING_TILES, TILE = MOE_RING_TILE, BN = MOE_RING_BN, OUT = GLU ? BN / 2 : BN, WGN = BN / 64, WM = MOE_BIG / (8 / WGN);
  constexpr int TI = WM / 16, TJ = 4;  // a wave: 64 rows, 64 rows of w (glu: 32 gate rows, their up rows), in 16 x 16 x 32 products with w as the first operand
  constexpr int LA = 2, LW = BN / 64, L = LA + LW;  // its loads a k-tile
  extern __shared__ __attribute__((aligned(1024))) char lds_ring[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WGN, wn = wave % WGN;
  const scalar_ints tiles = (scalar_ints)p.tiles, meta = (scalar_ints)p.meta;
  const int K = p.K, F = p.F, steps = K >> 6;

  // this chiplet's tiles, and of their units this workgroup's: slot, slot + 32, ..; larger tiles first, in all columns: what runs last is short
  const int n_tiles = meta[0], per = (n_tiles + 7) / 8, lo = (blockIdx.x & 7) * per, n = min(per, n_tiles - lo), slot = blockIdx.x >> 3;
  const int units = n > 0 && slot < n * p.n_cols ? (n * p.n_cols - slot + MOE_RING_CUS - 1) / MOE_RING_CUS : 0;
  if (units == 0) return;
  unsigned long long larger = 0, smaller = 0;
  if (n <= 64) {
    const bool large = lane < n && p.tiles[3 * (lo + min(lane, n - 1)) + 2] > MOE_BIG / 2;
    larger = __ballot(large), smaller = __ballot(lane < n) & ~larger;
  }
  const int n_larger = __popcll(larger) * p.n_cols;
  struct Unit {
    int first, rows, o0, e, turn;
  };
  auto locate = [&](int u) __attribute__((always_inline)) {
    const int s = slot + u * MOE_RING_CUS;
    int tile, col;
    if (n <= 64) {
      const bool is_larger = s < n_larger;
      const unsigned long long of = is_larger ? larger : smaller;
      const int at = is_larger ? s : s - n_larger, kind = __popcll(of);
      col = at / kind;
      tile = lo + __ffsll(__ballot((of >> lane & 1) && __popcll(of & ((1ull << lane) - 1)) == at % kind)) - 1;
    } else {
      tile = lo + s % n, col = s / n;
    }
    tile = __builtin_amdgcn_readfirstlane(tile), col = __builtin_amdgcn_readfirstlane(col);
    const int e = tiles[3 * tile];
    return Unit{tiles[3 * tile + 1], tiles[3 * tile + 2], col * OUT, e, (col * 3 + e * 7) % steps};
  };

  // ---- the stream of loads
  const uint32_t lds0 = lds_offset(lds_ring), index0 = lds0 + R * TILE;
  int* index = reinterpret_cast<int*>(lds_ring + R * TILE);  // [2][128]: which pair a row is, of two units in turn
  const int lr = lane >> 3, lc = lane & 7;
  uint32_t off[L];
  const char *a_line, *w_line, *a_end;
  auto ask_rows = [&](const Unit& x, int u) __attribute__((always_inline)) {  // the unit's pairs, through LDS: nothing waits for them
    if (!p.gather || wave >= 2) return;
    const uint32_t at = (uint32_t)(x.first + min(wave * 64 + lane, x.rows - 1)) * 4;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(index0 + (u & 1) * MOE_BIG * 4 + wave * 256), "v"(at), "s"(p.sorted) : "memory");
  };
  auto aim = [&](const Unit& x, int u, bool at_start) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int r = (wave * LA + i) * 8 + lr, at = min(r, x.rows - 1);
      int row = x.first + at;
      if (p.gather) row = (at_start ? p.sorted[row] : index[(u & 1) * MOE_BIG + at]) / p.top;
      off[i] = (uint32_t)row * (uint32_t)p.a_stride * 2 + (uint32_t)((lc ^ ring_swap_rows(r)) * 16);
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      const int r = (wave * LW + i) * 8 + lr, q = r & 63;
      const int o = GLU ? min(x.o0 + (r >> 6) * 32 + (q & 31), F - 1) + (q >= 32 ? F : 0) : min(x.o0 + r, F - 1);
      off[LA + i] = (uint32_t)o * (uint32_t)K * 2 + (uint32_t)((lc ^ ring_swap_columns(r)) * 16);
    }
    a_line = reinterpret_cast<const char*>(p.a) + x.turn * 128;
    w_line = reinterpret_cast<const char*>(p.w + (size_t)x.e * p.N * K) + x.turn * 128;
    a_end = reinterpret_cast<const char*>(p.a) + (size_t)K * 2;
  };
  auto load_one = [&](uint32_t at, int i) __attribute__((always_inline)) {
    if (i < LA) lines_to_lds(at + (wave * LA + i) * 1024, off[i], a_line);
    else lines_to_lds(at + MOE_BIG * 128 + (wave * LW + i - LA) * 1024, off[i], w_line);
  };
  Unit now = locate(0), ahead = now;  // ahead: the unit behind the one that is being loaded
  aim(now, 0, true);
  if (units > 1) ask_rows(ahead = locate(1), 1);
  int asked = 0, asked_of = 0;  // k-tiles of unit asked_of asked for
  auto further = [&]() __attribute__((always_inline)) {
    a_line += 128, w_line += 128;
    if (a_line == a_end) a_line -= (size_t)K * 2, w_line -= (size_t)K * 2;
    if (++asked == steps && asked_of + 1 < units) {
      asked = 0, ++asked_of;
      aim(ahead, asked_of, false);
      if (asked_of + 1 < units) ask_rows(ahead = locate(asked_of + 1), asked_of + 1);
    }
  };
  const int total = units * steps;  // at least 2 R (the caller sees to that)
#pragma unroll 1
  for (int t = 0; t < R; ++t) {
#pragma unroll
    for (int i = 0; i < L; ++i) load_one(lds0 + t * TILE, i);
    further();
  }

  // ---- the products
  const int fr = lane & 15, kg = lane >> 4, wr = 8 * (fr >> 2) + (fr & 3);
  const int a_at = (wm * WM + fr) * 128 + ((kg ^ ring_swap_rows(fr)) * 16);
  const int w_at[2] = {(MOE_BIG + wn * 64 + wr) * 128 + ((kg ^ ring_swap_columns(wr)) * 16), (MOE_BIG + wn * 64 + wr + 4) * 128 + ((kg ^ ring_swap_columns(wr + 4)) * 16)};
  u32x4 af[2][2][TI], wf[2][2][TJ];
  f32x4 sums[TI][TJ];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) sums[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  constexpr int READS = 2 * (TI + TJ), PRODUCTS = 2 * TI * TJ;
  auto read_one = [&](auto set, const char* kt, int o) __attribute__((always_inline)) {
    constexpr int c = decltype(set)::value;
    const int ks = o / (TI + TJ), q = o % (TI + TJ);
    if (q < TJ) wf[c][ks][q] = *reinterpret_cast<const u32x4*>(kt + (w_at[q & 1] ^ (ks * 64)) + (q >> 1) * 4096);
    else af[c][ks][q - TJ] = *reinterpret_cast<const u32x4*>(kt + (a_at ^ (ks * 64)) + (q - TJ) * 2048);
  };
  typedef std::integral_constant<int, 0> Zero;
  typedef std::integral_constant<int, 1> One;
  ring_wait<(R - 1) * L>();
  lds_barrier();
#pragma unroll
  for (int o = 0; o < READS; ++o) read_one(Zero(), lds_ring, o);

  int place = 0, done = 0;  // done: k-tiles of the whole stream
  // one k-tile: its products, between them the reads of the next one's operands and the loads of the one R further on
  auto step = [&](auto set, auto loads, auto active) __attribute__((always_inline)) {
    constexpr int c = decltype(set)::value;
    if constexpr (decltype(loads)::value) ring_wait<(R - 2) * L>(); else ring_wait_for<R, L>(min(R - 2, total - 2 - done));
    lds_barrier();
    const uint32_t into = lds0 + place * TILE;
    place = place + 1 == R ? 0 : place + 1;
    const char* kt = lds_ring + place * TILE;
#pragma unroll
    for (int m = 0; m < PRODUCTS; ++m) {
#pragma unroll
      for (int o = m * READS / PRODUCTS; o < (m + 1) * READS / PRODUCTS; ++o) read_one(std::integral_constant<int, c ^ 1>(), kt, o);
      if constexpr (decltype(loads)::value) {
#pragma unroll
        for (int i = m * L / PRODUCTS; i < (m + 1) * L / PRODUCTS; ++i) load_one(into, i);
      }
      if constexpr (decltype(active)::value) {
        const int ks = m / (TI * TJ), i = m % (TI * TJ) / TJ, j = m % TJ;
        sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wf[c][ks][j]), as_bf16x8(af[c][ks][i]), sums[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (decltype(loads)::value) further();
    ++done;
  };
  auto finish = [&](auto activation) __attribute__((always_inline)) {  // register r of lane l: column 8 (l / 16) + 4 h + r of a pair of tiles, row l % 16
    constexpr int ACT = decltype(activation)::value;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int at = wm * WM + i * 16 + fr;
      if (at >= now.rows) continue;
      TO* row = static_cast<TO*>(p.out) + (size_t)(now.first + at) * p.o_stride;
#pragma unroll
      for (int q = 0; q < (GLU ? 1 : 2); ++q) {
        const int o = now.o0 + wn * (GLU ? 32 : 64) + q * 32 + kg * 8;
        if (o >= F) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float s = sums[i][2 * q + (e >> 2)][e & 3];
          v[e] = GLU ? moe_act(s, sums[i][2 + (e >> 2)][e & 3], ACT, p.limit, p.up_shift) : lev_activate(s, ACT);
        }
        moe_store8(row + o, v, F - o, p.vec);
      }
    }
  };
  for (int u = 0; u < units; ++u) {
    auto run = [&](auto active) __attribute__((always_inline)) {
      int t = 0;
      const int with_loads = min(steps, total - R - done);
      for (; t + 1 < with_loads; t += 2) {
        step(Zero(), One(), active);
        step(One(), One(), active);
      }
      if (t < with_loads) {
        step(Zero(), One(), active);
        step(One(), Zero(), active);
        t += 2;
      }
      for (; t < steps; t += 2) {
        step(Zero(), Zero(), active);
        step(One(), Zero(), active);
      }
    };
    if (wm * WM < now.rows) {
      run(One());
      switch (p.act) {  // one decision for all outputs
        case LEV_ACT_GELU_TANH: finish(std::integral_constant<int, LEV_ACT_GELU_TANH>()); break;
        case LEV_ACT_GELU_ERF: finish(std::integral_constant<int, LEV_ACT_GELU_ERF>()); break;
        case LEV_ACT_RELU: finish(std::integral_constant<int, LEV_ACT_RELU>()); break;
        case LEV_ACT_SILU: finish(std::integral_constant<int, LEV_ACT_SILU>()); break;
        case LEV_ACT_QUICK_GELU: finish(std::integral_constant<int, LEV_ACT_QUICK_GELU>()); break;
        case LEV_ACT_TANH: finish(std::integral_constant<int, LEV_ACT_TANH>()); break;
        case LEV_ACT_RELU_SQUARED: finish(std::integral_constant<int, LEV_ACT_RELU_SQUARED>()); break;
        default: finish(std::integral_constant<int, LEV_ACT_NONE>());
      }
      clear();
    } else {
      run(Zero());
    }
    if (u + 1 < units) now = locate(u + 1);
  }
}

template <typename TO, bool GLU>
static int launch_moe_ring(const MoeLinearArgs& args, hipStream_t stream) {
  hipError_t e = hipFuncSetAttribute((const void*)moe_ring_kernel<TO, GLU>, hipFuncAttributeMaxDynamicSharedMemorySize, MOE_RING_LDS);
  LEV_REQUIRE(e == hipSuccess, "experts: %d bytes of LDS a workgroup: %s", MOE_RING_LDS, hipGetErrorString(e));
  moe_ring_kernel<TO, GLU><<<8 * MOE_RING_CUS, 512, MOE_RING_LDS, stream>>>(args);
  return lev_check_launch("moe_linear (ring)");
}

// Which products: N rows of w an expert, K numbers each, as many tiles as the step's sizes allow. Below 0.6 full units a CU the CUs that have one walk it alone, and twice as many tiles of 128 x 128, two
// a CU, are ahead. Measured over 192 shapes (4 to 128 experts, 300 to 12,000 rows, 64 to 2,048 outputs of 384 to 2048; microseconds, tiles of 128 x 128 / here, at so many full units a CU): 0.12 8 experts, 1,000 rows, 384 outputs of
// 768 16.0 / 21.4; 0.23 1024 of 2048 34.3 / 44.0; 0.47 2048 of 1408 30.5 / 39.1; 0.59 12,000 rows, 384 of 768 23.3 / 23.5; 0.61 32 experts, 1,000 rows, 1024 of 2048 45.4 / 48.4; 0.64 8 experts, gated 1408 of 2048 56.3 / 47.9; 0.73 32
// experts, 12,000 rows, 384 of 768 28.8 / 26.3; 0.98 4,000 rows, 1024 of 2048 63.1 / 55.6; 1.95 12,000 rows 104 / 87.
extern "C" int lev_moe_ring_takes(int max_tiles, int K, int N) {
  return K % 128 == 0 && K >= 128 * MOE_RING_TILES && 5L * max_tiles * N >= 3L * 8 * MOE_RING_CUS * MOE_RING_BN;
}

int lev_moe_ring(const MoeLinearArgs& args, long a_rows, int out_dtype, int glu, int max_tiles, hipStream_t stream) {
  if (!lev_moe_ring_takes(max_tiles, args.K, args.N) || (size_t)a_rows * args.a_stride >= (1ull << 31) || (size_t)args.N * args.K >= (1ull << 31)) return 1;
  MoeLinearArgs p = args;
  const int out = glu ? MOE_RING_BN / 2 : MOE_RING_BN;
  p.n_cols = (p.F + out - 1) / out;
  LEV_REQUIRE((long)(max_tiles + 7) / 8 * p.n_cols <= 0x7fffffffL, "experts: too many tiles (%d)", max_tiles);
  if (out_dtype == LEV_F32) return glu ? launch_moe_ring<float, true>(p, stream) : launch_moe_ring<float, false>(p, stream);
  return glu ? launch_moe_ring<bf16_t, true>(p, stream) : launch_moe_ring<bf16_t, false>(p, stream);
}
