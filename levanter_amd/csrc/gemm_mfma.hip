// bfloat16 matrix products on the matrix cores (MFMA), 32-bit accumulation, fused epilogue:
//   y = act(a . w^T + bias) (+ residual),  a [M, K] (row stride lda), w [N, K], y [M, N] bf16 or f32.
// Three kernels here and one in gemm_ring.hip, chosen by the sizes:
//   ring kernel   (M > 64 and fewer than four million outputs, long sums from 17 rows: use_ring): in gemm_ring.hip;
//   tile kernel   (more outputs, M > 128): a 256x256, 256x192, 256x128 or 128x128 tile per workgroup of 4 waves, 32x32x16 MFMA,
//                 (K split into ranges, with a second kernel for the sums, where the tiles alone would leave CUs idle)
//                 operands staged through LDS (two buffers), the next k-tile's global loads in registers meanwhile;
//   stream kernel (M <= 64, and up to 128 rows of more than 32,768 outputs; where an estimate puts it ahead of the skinny kernel: long sums, many rows): the weights are the traffic; `a` is shared through LDS by the 4 to 16 waves of a
//                 workgroup, the weights go straight into MFMA operand registers, K is split over workgroups
//                 and a second kernel adds the partial sums in a fixed order;
//   skinny kernel (M <= 64, the smallest weights to 256 rows, see use_skinny): a workgroup owns 8 to 64 output columns; its waves split K, bring whole lines of w
//                 and a through an LDS area of their own into MFMA operand registers (16x16x32), and their partial sums are
//                 added through LDS in a fixed order.
// No atomics anywhere: results are deterministic. K and lda must be multiples of 8 (16-byte operand loads);
// any M and N.
#include "common.h"
#include "gemm_norm.h"
#include "gemm_ring.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}

__device__ __forceinline__ u32x4 load16(const bf16_t* p) { return *reinterpret_cast<const u32x4*>(p); }

template <typename TO>
__device__ __forceinline__ void epilogue_store(float v, int m, int n, const float* bias, const float* residual, long ldr,
                                               TO* out, long ldo, int act) {
  if (bias) v += bias[n];
  v = lev_activate(v, act);
  if (residual) v += residual[(size_t)m * ldr + n];
  out[(size_t)m * ldo + n] = from_float<TO>(v);
}

// ------------------------------------------------------------------------------------------------
// Tile kernel. A workgroup of 4 waves (2 x 2) computes a BM x BN tile; a wave computes (BM/2) x (BN/2)
// with 32x32x16 MFMA. The larger the wave's tile, the fewer LDS bytes per MFMA: 64 x 64 per wave needs
// the whole LDS bandwidth, 128 x 128 half of it. Operand tiles of BK = 64 go global -> registers -> LDS
// (two LDS buffers, one barrier per k-tile). With one wave per SIMD nothing else fills the matrix pipe
// while a wave issues loads and LDS traffic, so those are interleaved one by one between the products.
// Workgroups are numbered so that each XCD (id % 8) works on a contiguous band of tiles and shares
// operands in its own L2.
#define TK 64
#define LDS_STRIDE 72  // bf16 elements per LDS row: 64 + 8 of padding (144 bytes): 16-byte reads without bank conflicts

template <typename TO>
__device__ __forceinline__ void store_vec4(TO* p, const float v[4]);
template <>
__device__ __forceinline__ void store_vec4<float>(float* p, const float v[4]) {
  *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
}
template <>
__device__ __forceinline__ void store_vec4<bf16_t>(bf16_t* p, const float v[4]) {
  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
  *reinterpret_cast<u32x2*>(p) = u32x2{float2_to_bf16x2(v[0], v[1]), float2_to_bf16x2(v[2], v[3])};
}

// Output of a wave's (TI x 32) x (TJ x 32) accumulators through an LDS area of its own: 32 rows at a time are
// staged and written out as rows of 4 consecutive columns per lane, so that stores are wide and coalesced.
// No barrier: LDS executes a wave's instructions in order, and a barrier that also waited for the global
// stores (as __syncthreads() does) would expose their latency once per 32 rows.
// 32x32 accumulator: register r of lane l is row 8*(r/4) + 4*(l/32) + r%4, column l%32.
template <typename TO, int ACT, int TI, int TJ>
__device__ __forceinline__ void tile_epilogue(const f32x16 (&acc)[TI][TJ], float* Cs, int lane, int mw, int nw,
                                              const float* __restrict__ bias, const float* residual, long ldr, TO* out,
                                              long ldo, int M, int N, int act, int vec_ok) {
  constexpr int WN = TJ * 32, CS = WN + 4;
  constexpr int QUADS = WN / 4;           // groups of 4 columns in a staged row
  constexpr int TURNS = 32 * QUADS / 64;  // per lane and 32 rows
  constexpr int UNROLL_TURNS = ACT >= 0 ? 4 : 1;
#pragma unroll
  for (int i = 0; i < TI; ++i) {
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) Cs[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * CS + j * 32 + (lane & 31)] = acc[i][j][r];
#pragma unroll UNROLL_TURNS
    for (int q = 0; q < TURNS; ++q) {  // four LDS reads in flight where the activation's code is short
      const int idx = lane + 64 * q;
      const int row = idx / QUADS, c4 = idx % QUADS;
      const int m = mw + i * 32 + row;
      const int n = nw + c4 * 4;
      const f32x4 cv = *reinterpret_cast<const f32x4*>(&Cs[row * CS + c4 * 4]);
      if (m >= M || n >= N) continue;
      float v[4] = {cv[0], cv[1], cv[2], cv[3]};
      const bool whole = vec_ok && n + 3 < N;
      if (bias) {
        if (whole) {
          const f32x4 b = *reinterpret_cast<const f32x4*>(bias + n);
          v[0] += b[0]; v[1] += b[1]; v[2] += b[2]; v[3] += b[3];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bias[min(n + e, N - 1)];
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)  // the exact GELU of a bfloat16 output takes the short erf
        v[e] = (ACT == LEV_ACT_GELU_ERF && sizeof(TO) == 2) ? lev_gelu_erf_coarse(v[e]) : lev_activate_as<ACT>(v[e], act);
      if (residual) {
        const float* rrow = residual + (size_t)m * ldr;
        if (whole) {
          const f32x4 rr = *reinterpret_cast<const f32x4*>(rrow + n);
          v[0] += rr[0]; v[1] += rr[1]; v[2] += rr[2]; v[3] += rr[3];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += rrow[min(n + e, N - 1)];
        }
      }
      TO* orow = out + (size_t)m * ldo + n;
      if (whole) {
        store_vec4<TO>(orow, v);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) orow[e] = from_float<TO>(v[e]);
      }
    }
  }
}

template <typename TO, int BM, int BN>
__global__ void __launch_bounds__(256)
gemm_tile_kernel(const bf16_t* __restrict__ a, long lda, const bf16_t* __restrict__ w, const float* __restrict__ bias,
                 const float* residual, long ldr, TO* out, long ldo, int M, int N, int K, int act, int tiles_m, int tiles_n,
                 int vec_ok, int S, float* __restrict__ partial) {
  constexpr int WM = BM / 2, WN = BN / 2;    // the wave's tile
  constexpr int TI = WM / 32, TJ = WN / 32;  // in 32 x 32 MFMA tiles
  constexpr int CA = BM * (TK / 8) / 256;    // 16-byte chunks of the a tile per thread
  constexpr int CW = BN * (TK / 8) / 256;
  extern __shared__ __attribute__((aligned(16))) bf16_t smem[];
  bf16_t* As = smem;                               // [2][BM * LDS_STRIDE]
  bf16_t* Ws = smem + 2 * BM * LDS_STRIDE;         // [2][BN * LDS_STRIDE]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int n_tiles = tiles_m * tiles_n;
  int id = blockIdx.x;
  if (n_tiles % 8 == 0) id = (id % 8) * (n_tiles / 8) + id / 8;
  const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;

  // Rows beyond the matrix read the last row instead: their products land in output rows / columns that are
  // never stored. Only the k range needs zeros, and the partial k-tile (K % 64 != 0) is taken FIRST, in the
  // prologue, so that the main loop needs no masks at all.
  uint32_t pa[CA], pw[CW];
  const int kc = (tid & 7) * 8;
#pragma unroll
  for (int i = 0; i < CA; ++i) pa[i] = (uint32_t)((size_t)min(m0 + ((tid + 256 * i) >> 3), M - 1) * lda);
#pragma unroll
  for (int i = 0; i < CW; ++i) pw[i] = (uint32_t)((size_t)min(n0 + ((tid + 256 * i) >> 3), N - 1) * K);
  // The k-tiles in the order they are taken: tile 0 is the partial one (K % 64 != 0) or the first, tile t >= 1 starts at
  // (t - kshift) * 64. With S > 1 (few output tiles: the K range is split over blockIdx.y) this workgroup takes
  // tiles t0 .. t1 - 1 and leaves its sums, without epilogue, in partial[blockIdx.y].
  const int ktail = K % TK, nk_all = (K + TK - 1) / TK;
  const int per = (nk_all + S - 1) / S;
  const int t0 = blockIdx.y * per, t1 = min(nk_all, t0 + per);
  const int nk = t1 - t0;
  const int kshift = ktail ? 1 : 0;
  auto kpos = [&](int t) {  // for t >= 1 (tiles past this range repeat its last one; they are loaded but never used)
    return max(min(t, t1 - 1) - kshift, 0) * TK;
  };
  u32x4 ra[2][CA], rw[2][CW];
  auto gload_one = [&](int set, uint32_t koff, int i) {
    if (i < CA) ra[set][i] = load16(a + pa[i] + koff);
    else rw[set][i - CA] = load16(w + pw[i - CA] + koff);
  };
  bf16_t* a_st = As + (tid >> 3) * LDS_STRIDE + kc;
  bf16_t* w_st = Ws + (tid >> 3) * LDS_STRIDE + kc;
  auto lstore_one = [&](int set, int buf, int i) {
    if (i < CA) *reinterpret_cast<u32x4*>(a_st + buf * BM * LDS_STRIDE + i * 32 * LDS_STRIDE) = ra[set][i];
    else *reinterpret_cast<u32x4*>(w_st + buf * BN * LDS_STRIDE + (i - CA) * 32 * LDS_STRIDE) = rw[set][i - CA];
  };

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  {  // prologue: this range's first tile (masked in k if it is the partial one) to LDS buffer 0, the next into register set 1
    const int k0 = t0 == 0 ? (ktail ? K - ktail : 0) : kpos(t0);
    const bool ok = k0 + kc < K;
    const uint32_t koff = (uint32_t)min(k0 + kc, K - 8);
#pragma unroll
    for (int i = 0; i < CA + CW; ++i) gload_one(0, koff, i);
#pragma unroll
    for (int i = 0; i < CA; ++i) if (!ok) ra[0][i] = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < CW; ++i) if (!ok) rw[0][i] = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < CA + CW; ++i) lstore_one(0, 0, i);
    const uint32_t koff1 = (uint32_t)min(kpos(t0 + 1) + kc, K - 8);
#pragma unroll
    for (int i = 0; i < CA + CW; ++i) gload_one(1, koff1, i);
  }
  lds_barrier();
  const int fr = lane & 31, fk = (lane >> 5) * 8;
  constexpr int KS = TK / 16;
  constexpr int NM = TI * TJ, NR = TI + TJ;
  constexpr int PW = (CA + CW + KS - 2) / (KS - 1);  // LDS writes / global loads per k-step, in the first KS - 1 k-steps
  const bf16_t* a_rd = As + (wm * WM + fr) * LDS_STRIDE + fk;
  const bf16_t* w_rd = Ws + (wn * WN + fr) * LDS_STRIDE + fk;
  u32x4 af[2][TI], wf[2][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i) af[0][i] = *reinterpret_cast<const u32x4*>(a_rd + i * 32 * LDS_STRIDE);
#pragma unroll
  for (int j = 0; j < TJ; ++j) wf[0][j] = *reinterpret_cast<const u32x4*>(w_rd + j * 32 * LDS_STRIDE);

  // One k-tile. `cur` is the register set that holds tile kt + 1 (it goes to the other LDS buffer during the
  // first KS - 1 k-steps); the other set receives the loads of tile kt + 2. Then one barrier, and the last
  // k-step's products cover the LDS reads of tile kt + 1's first fragments. Every product is followed by at
  // most two other instructions so that the matrix pipe never waits for the wave to issue them in a block.
  auto ktile = [&](int kt, int cur) {
    const int buf = kt & 1;
    const uint32_t koff = (uint32_t)min(kpos(t0 + kt + 2) + kc, K - 8);
    const bf16_t* Ab = a_rd + buf * BM * LDS_STRIDE;
    const bf16_t* Wb = w_rd + buf * BN * LDS_STRIDE;
    const bf16_t* Abn = a_rd + (buf ^ 1) * BM * LDS_STRIDE;
    const bf16_t* Wbn = w_rd + (buf ^ 1) * BN * LDS_STRIDE;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int c = ks & 1, nx = c ^ 1;
      if (ks + 1 < KS) {
#pragma unroll
        for (int i = 0; i < TI; ++i) af[nx][i] = *reinterpret_cast<const u32x4*>(Ab + i * 32 * LDS_STRIDE + (ks + 1) * 16);
#pragma unroll
        for (int j = 0; j < TJ; ++j) wf[nx][j] = *reinterpret_cast<const u32x4*>(Wb + j * 32 * LDS_STRIDE + (ks + 1) * 16);
      } else {
        lds_barrier();
#pragma unroll
        for (int i = 0; i < TI; ++i) af[nx][i] = *reinterpret_cast<const u32x4*>(Abn + i * 32 * LDS_STRIDE);
#pragma unroll
        for (int j = 0; j < TJ; ++j) wf[nx][j] = *reinterpret_cast<const u32x4*>(Wbn + j * 32 * LDS_STRIDE);
      }
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(af[c][i]), as_bf16x8(wf[c][j]), acc[i][j], 0, 0, 0);
      if (ks + 1 < KS) {
#pragma unroll
        for (int q = 0; q < PW; ++q)
          if (ks * PW + q < CA + CW) lstore_one(cur, buf ^ 1, ks * PW + q);
#pragma unroll
        for (int q = 0; q < PW; ++q)
          if (ks * PW + q < CA + CW) gload_one(cur ^ 1, koff, ks * PW + q);
      }
      constexpr int others = NR + 2 * PW;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (ks + 1 < KS) {
          const int lo = m * others / NM, hi = (m + 1) * others / NM;
#pragma unroll
          for (int o = lo; o < hi; ++o) {
            if (o < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else if (o < NR + PW) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            else __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
          }
        } else {
          const int lo = m * NR / NM, hi = (m + 1) * NR / NM;
#pragma unroll
          for (int o = lo; o < hi; ++o) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      }
    }
  };
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    ktile(kt, 1);
    ktile(kt + 1, 0);
  }
  if (kt < nk) ktile(kt, 1);

  // Epilogue (the operand buffers are free now), specialised for no activation and the two GELUs so that the
  // loop over the outputs has no switch inside
  lds_barrier();
  float* Cs = reinterpret_cast<float*>(smem) + wave * 32 * (BN / 2 + 4);
  const int mw = m0 + wm * WM, nw = n0 + wn * WN;
  if (S > 1)  // vec_ok: bit 1 says whether the partial sums can be stored as vectors
    tile_epilogue<float, LEV_ACT_NONE, TI, TJ>(acc, Cs, lane, mw, nw, nullptr, nullptr, 0, partial + (size_t)blockIdx.y * M * N, N, M, N,
                                               LEV_ACT_NONE, (vec_ok >> 1) & 1);
  else if (act == LEV_ACT_NONE)
    tile_epilogue<TO, LEV_ACT_NONE, TI, TJ>(acc, Cs, lane, mw, nw, bias, residual, ldr, out, ldo, M, N, act, vec_ok & 1);
  else if (act == LEV_ACT_GELU_TANH)
    tile_epilogue<TO, LEV_ACT_GELU_TANH, TI, TJ>(acc, Cs, lane, mw, nw, bias, residual, ldr, out, ldo, M, N, act, vec_ok & 1);
  else if (act == LEV_ACT_GELU_ERF)
    tile_epilogue<TO, LEV_ACT_GELU_ERF, TI, TJ>(acc, Cs, lane, mw, nw, bias, residual, ldr, out, ldo, M, N, act, vec_ok & 1);
  else
    tile_epilogue<TO, -1, TI, TJ>(acc, Cs, lane, mw, nw, bias, residual, ldr, out, ldo, M, N, act, vec_ok & 1);
}

// out = act(sum_s partial[s] + bias) + residual (defined with the stream kernel below)
template <typename TO>
static int launch_splitk_reduce(const float* workspace, const float* bias, const float* residual, long ldr, TO* out, long ldo, int M,
                                int N, int S, int act, hipStream_t stream);

template <typename TO, int BM, int BN>
static int launch_tile(const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr, TO* out,
                       long ldo, float* workspace, int M, int N, int K, int act, int S, int defer, hipStream_t stream) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const size_t lds_ops = (size_t)2 * (BM + BN) * LDS_STRIDE * sizeof(bf16_t);
  const size_t lds_out = (size_t)4 * 32 * (BN / 2 + 4) * sizeof(float);
  const size_t lds = lds_ops > lds_out ? lds_ops : lds_out;
  static std::atomic<unsigned long long> reserved{0};  // per instantiation
  if (int rc = lev_reserve_lds((const void*)gemm_tile_kernel<TO, BM, BN>, (int)lds, reserved)) return rc;
  if (S > 1 && !workspace) return lev_fail("linear: M=%d N=%d K=%d needs a workspace of lev_linear_mfma_workspace bytes", M, N, K);
  // rows of 4 outputs are stored (and bias / residual read) as vectors when everything is aligned for it
  const int vec_out = (ldo % 4 == 0) && (((uintptr_t)out & 15) == 0) && (!residual || (ldr % 4 == 0 && ((uintptr_t)residual & 15) == 0)) &&
                      (!bias || ((uintptr_t)bias & 15) == 0);
  const int vec_partial = (N % 4 == 0) && (((uintptr_t)workspace & 15) == 0);
  gemm_tile_kernel<TO, BM, BN><<<dim3(tiles_m * tiles_n, S), 256, lds, stream>>>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act,
                                                                                   tiles_m, tiles_n, vec_out | (vec_partial << 1), S,
                                                                                   workspace);
  if (S > 1) {
    if (int rc = lev_check_launch("linear_tile")) return rc;
    if (defer) return 0;  // the caller folds the sum of the ranges into its next kernel
    return launch_splitk_reduce<TO>(workspace, bias, residual, ldr, out, ldo, M, N, S, act, stream);
  }
  return 0;
}

// ------------------------------------------------------------------------------------------------
// Skinny kernel (M <= 64: MT = 1 .. 4 tiles of 16 rows; small weights up to 256 rows, in blocks of rows). A workgroup owns NT units of 16 output columns (or, HALF, one of 8); its
// WAVES waves split K. A wave takes pairs of adjacent 32-wide k-steps (64 k = 128 bytes of a row), U pairs in flight. Weights and `a`
// alike are read as WHOLE 128-byte lines - lane (row l/8, 16-byte chunk l%8), one instruction for 8 rows - and turned into the operand
// layout (row l%16, k-group l/16) through a small LDS area of the wave's own. The vector cache looks lines up by neighbouring
// lanes: read in operand layout (16 rows, 64 bytes of each) an instruction costs one look-up for every lane, 16 bytes a cycle and CU, and
// weights and `a` together were bound by that and not by memory (of data in L2, 9.6 TB/s against 33 TB/s in whole lines).
// The loads stand under no condition, from clamped addresses (a condition is a branch, and at its join everything in flight is waited
// for); what lies beyond K is masked on its way into LDS, rows beyond M and columns beyond N are read again and never stored.
// Measured in graphs over distinct weights, before (weights straight into the operand, conditional loads) and now, microseconds: 4800 x
// 1600 at 6 / 24 rows 8.0 / 12.5 -> 6.4 / 8.9; 6400 x 1600 8.3 / 12.9 -> 7.0 / 9.2; 4608 x 2048 9.1 / 14.2 -> 6.8 / 9.0; 768 x 768 3.8 / 4.8 -> 3.5 /
// 4.0; 4096 x 4096 8.6 / 12.5 -> 8.4 / 10.2; 16384 x 4096 25.0 -> 24.2 at 6 rows (memory: 5.5 TB/s).
// The partial sums of the waves are added through LDS in wave order. Every workgroup starts at another
// place of the k range, so that they do not all read the same part of `a` and the same residue of the weight
// rows at the same time; the order of a sum depends on the column tile
// and, through the launch's shape (skinny_shape), on the number of rows, never on what other rows hold.
#define SKINNY_SLOTS 72  // 16-byte slots of one staged instruction: 8 rows x (8 chunks + 1 of padding)
#define SKINNY_MAX_M 256  // which of these row counts it takes: use_skinny(); blocks of more rows have not been measured

template <typename TO, int WAVES, int U, int MT, int NT, bool HALF, bool BLOCKS>
// at most 128 registers a lane for 2 x 2 tiles (130 cost 7 % at 2048 x 2048 and 96 rows); with four waves at most 256, so that the sums stay in
// registers that every instruction reads (where 512 are allowed the compiler moves them to and fro: 16384 x 4096 at 64 rows 34.2 us)
__global__ void __launch_bounds__(WAVES * 64, U == 2 && NT * MT == 4 ? 4 : WAVES == 4 ? 2 : 1)
gemm_skinny_kernel(const bf16_t* __restrict__ w, const bf16_t* __restrict__ a, uint32_t lda8, int K, int N, int M, const float* __restrict__ bias,
                   const float* residual, TO* out, long ldr, long ldo, int act) {  // in registers when the waves start: all but the last three
  const size_t lda = (size_t)lda8 * 8;
  static_assert(NT * MT <= WAVES * 4 && (!HALF || NT == 1), "a wave finishes a few tiles; half a unit stands alone");
  constexpr int AI = 2 * MT, WI = HALF ? 1 : 2;  // instructions per pair of k-steps and unit: 8 rows each
  constexpr int COLS = HALF ? 8 : 16;
  // Partial sums of a wave: 16 of them a workgroup, so that none is a longer chain of roundings than with 16 waves (the error against
  // 64 bits of a 4096-long sum is 1.15e-7 with 16 chains, 1.37e-7 with 8, 1.9e-7 with 4). Not where the registers would cost a workgroup
  // its place beside another: many rows times many columns.
  constexpr int SUMS = WAVES >= 16 || NT * MT >= 12 ? 1 : (WAVES == 4 && U >= 2 ? 4 : 2);
  __shared__ f32x4 red[WAVES][NT][MT][64];
  __shared__ u32x4 stage[WAVES][2][SKINNY_SLOTS];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n0 = blockIdx.x * COLS * NT;
  if constexpr (BLOCKS) {
    if (n0 >= N) return;  // the grid's columns are a multiple of 8
    const int m0 = blockIdx.y * 16 * MT;
    a += (size_t)m0 * lda;
    out += (size_t)m0 * ldo;
    if (residual) residual += (size_t)m0 * ldr;
    M = min(M - m0, 16 * MT);
  }
  const int fr = lane & 15, kg = lane >> 4;
  const int lr = lane >> 3, lc = lane & 7;  // loads: row (0..7, instruction i adds 8 i) and chunk of the line
  const bf16_t* wrow[NT][WI];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < WI; ++i) wrow[j][i] = w + (size_t)min(n0 + 16 * j + 8 * i + lr, N - 1) * K;
  const bf16_t* arow[AI];
#pragma unroll
  for (int i = 0; i < AI; ++i) arow[i] = a + (size_t)min(8 * i + lr, M - 1) * lda;
  u32x4* my_stage = &stage[wave][0][0];
  const int st_slot = lr * 9 + lc;                                   // where this lane's chunk is staged
  const int ld_slot = (fr >> 3) * SKINNY_SLOTS + (fr & 7) * 9 + kg;  // operand (row fr, k-group kg) of the pair's first step

  // The lanes that will finish the sum fetch their bias and residual values now, so that the end of the kernel
  // (which no other workgroup's streaming overlaps: all of them finish together) has no dependent loads left.
  // `w` stands in for a missing operand.
  constexpr int TURNS = (NT * MT + WAVES - 1) / WAVES;  // wave v finishes the tiles v, v + WAVES, ..
  float pre_bias[TURNS];
  f32x4 pre_res[TURNS];
#pragma unroll
  for (int q = 0; q < TURNS; ++q) {
    const int tile = min(wave + q * WAVES, NT * MT - 1), j = tile % NT, t = tile / NT;
    const int nn = min(n0 + 16 * j + fr, N - 1);
    const float* bp = bias ? bias + nn : reinterpret_cast<const float*>(w);
    pre_bias[q] = *bp;
    if (!bias) pre_bias[q] = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = min(t * 16 + kg * 4 + r, M - 1);
      const float* rp = residual ? residual + (size_t)m * ldr + nn : reinterpret_cast<const float*>(w);
      pre_res[q][r] = *rp;
    }
  }

  f32x4 acc[SUMS][NT][MT];
#pragma unroll
  for (int s = 0; s < SUMS; ++s)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[s][j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int npairs = (K + 63) / 64;
  const int rot = (int)((blockIdx.x * 2654435761u) % (unsigned)npairs);
  auto take = [&](auto pairs, int p0) {
    constexpr int UU = decltype(pairs)::value;
    u32x4 wv[UU][NT][WI], av[UU][AI];
    uint32_t keep[UU];
#pragma unroll
    for (int u = 0; u < UU; ++u) {
      int pr = p0 + u * WAVES;
      const bool p_ok = pr < npairs;
      pr = min(pr, npairs - 1) + rot;
      pr = pr >= npairs ? pr - npairs : pr;
      const int k = pr * 64 + lc * 8, kc = min(k, K - 8);
      keep[u] = p_ok && k < K ? 0xffffffffu : 0u;
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < WI; ++i) wv[u][j][i] = load16(wrow[j][i] + kc);
#pragma unroll
      for (int i = 0; i < AI; ++i) av[u][i] = load16(arow[i] + kc);
    }
    __builtin_amdgcn_sched_barrier(0);  // all of them are on their way before the first is waited for
#pragma unroll
    for (int u = 0; u < UU; ++u) {
      // LDS executes a wave's instructions in order: the area is used again and again without a barrier
      const u32x4 mk = u32x4{keep[u], keep[u], keep[u], keep[u]};
      u32x4 wf[NT][2];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int i = 0; i < WI; ++i) my_stage[i * SKINNY_SLOTS + st_slot] = wv[u][j][i] & mk;
        const int at = HALF ? (fr & 7) * 9 + kg : ld_slot;  // half a unit: columns 8 .. 15 repeat 0 .. 7
        wf[j][0] = my_stage[at], wf[j][1] = my_stage[at + 4];
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        my_stage[st_slot] = av[u][2 * t] & mk;
        my_stage[SKINNY_SLOTS + st_slot] = av[u][2 * t + 1] & mk;
        const u32x4 a_lo = my_stage[ld_slot], a_hi = my_stage[ld_slot + 4];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          f32x4 &lo = acc[2 * u % SUMS][j][t], &hi = acc[(2 * u + 1) % SUMS][j][t];
          lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a_lo), as_bf16x8(wf[j][0]), lo, 0, 0, 0);
          hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a_hi), as_bf16x8(wf[j][1]), hi, 0, 0, 0);
        }
      }
    }
  };
  // U pairs at a time; of the few that are left a half or a quarter as many, so that short sums do not read their last pairs twice or more
  // (34768 x 320 at 13 rows 10.7 -> 7.9 us, 55128 x 576 at one row 15.6 -> 13.5)
  int p0 = U > 1 ? __builtin_amdgcn_readfirstlane(wave) : wave;
  for (; p0 + WAVES * (U / 2) < npairs; p0 += WAVES * U) take(std::integral_constant<int, U>(), p0);
  if constexpr (U == 4) {
    if (p0 + WAVES < npairs) {
      take(std::integral_constant<int, 2>(), p0);
      p0 = npairs;
    }
  }
  if constexpr (U > 1) {
    if (p0 < npairs) take(std::integral_constant<int, 1>(), p0);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
      for (int s = 1; s < SUMS; ++s) acc[0][j][t] += acc[s][j][t];
      red[wave][j][t][lane] = acc[0][j][t];
    }
  __syncthreads();
  // 16x16 accumulator: register r of lane l is row 4*(l/16) + r, column l%16. Partial sums are added in wave order.
#pragma unroll
  for (int q = 0; q < TURNS; ++q) {
    const int tile = wave + q * WAVES, j = tile % NT, t = tile / NT;
    if (tile >= NT * MT) break;
    const int nn = n0 + 16 * j + fr;
    f32x4 s = red[0][j][t][lane];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) {
      const f32x4 o = red[v][j][t][lane];
      s[0] += o[0]; s[1] += o[1]; s[2] += o[2]; s[3] += o[3];
    }
    if (nn < N && fr < COLS) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = t * 16 + kg * 4 + r;
        if (m >= M) continue;
        float v = lev_activate(s[r] + pre_bias[q], act);
        if (residual) v += pre_res[q][r];
        out[(size_t)m * ldo + nn] = from_float<TO>(v);
      }
    }
  }
}

// Choices measured on MI355X (graphs over distinct weights, 1 to 64 rows, weights of 768 x 768 to 6144 x 24576). What decides is how many
// columns the busiest CU streams, and that every `a` fragment feeds several of weights where the rows are many:
//   up to 2,048 columns (256 workgroups of 8 columns): half units up to 32 rows: 1600 x 6400 at 6 rows 9.3 -> 7.7 us, at 24 rows 13.3 -> 11.6,
//     2048 x 8192 11.0 -> 9.1; 16 waves with two pairs each for long rows and up to 8 rows of `a` (8.9 -> 7.7, 10.7 -> 9.1), else 8 waves;
//   else as many units a workgroup as make one round of the CUs: two up to 512 units (4800 x 1600 at 6 rows 7.5 -> 6.4, 4608 x 2048 7.8 -> 6.8, 6144 x
//     6144 18.0 -> 15.7), three up to 768 (12288 x 4096 at 24 rows 24.3 -> 21.2, 10752 x 2048 13.7 -> 10.6), four with 4 waves up to 1,024 (16384 x
//     4096 at 24 rows 31.0 -> 26.4, at 48 rows 40.7 -> 28.4); above that three up to 32 rows (18432 x 6144 at 24 rows 55.8 -> 49.5), else four
//     (32000 x 2048 at 48 rows 28.3 against 35.1 for the stream kernel, 50257 x 4096 89.5 against 105 with three);
//   but up to 16 rows above 720 units one unit and 4 waves with four pairs in flight: 12288 x 4096 at 6 rows 20.7 -> 18.9, 16384 x 4096 29 -> 24.3.
// Beside the lines, at 6 rows: 16 / 8 waves of two units, 7600 outputs, sums of 1,664 / 1,920: 7.5 / 7.4, 8.6 / 8.0; three units / one with 4 waves, sums of
// 2,048: 10752 outputs 10.6 / 11.1, 12288 11.4 / 11.7, 14336 17.1 / 13.5, sums of 4,096: 18.8 / 18.7, 20.9 / 19.6, 30.6 / 23.6; 16 / 8 waves of half a unit, 2048
// outputs, sums of 4,096 / 5,120 / 8,192: 5.9 / 6.1, 7.3 / 7.9, 9.2 / 10.7.
struct SkinnyShape {
  int waves, in_flight, row_tiles, units;  // the kernel's WAVES, U, MT, NT
  bool half;
  int cols() const { return half ? 8 : 16 * units; }
};
// Above 64 rows the rows are cut into blocks of 32 (the grid's y; its x a multiple of 8, so that the blocks of a column tile share a chiplet's L2) where 32 x 32
// outputs a workgroup make one round of the CUs: waves that split K need no barrier, and all their loads are out at once. Measured in graphs over
// distinct weights, microseconds, here / the ring kernel: 768 x 768 at 96 / 256 rows 4.5 / 5.0, 5.1 / 5.5; 1024 x 1024 at 256 rows 5.8 / 6.4; 2048 x 2048 at 96 /
// 128 rows 6.5 / 7.1, 7.3 / 7.5; 2304 x 768 at 96 rows 5.0 / 5.2. Beyond one round the ring kernel is ahead (2304 x 768 at 128 rows 5.7 / 5.2, 2048 x 2048 at 160 rows
// 8.5 / 7.6, 4800 x 1600 at 96 rows in blocks of 64 x 48 9.6 / 6.9), and for long sums.
static bool skinny_in_blocks(int M, int N, int K) {
  return M > 64 && M <= SKINNY_MAX_M && K <= 2048 && (long)((M + 31) / 32) * (((N + 31) / 32 + 7) / 8 * 8) <= 256;
}
static SkinnyShape skinny_shape(int M, int N, int K) {
  if (M > 64) return {8, 2, 2, 2, false};
  const int tiles = (N + 15) / 16;
  if (M <= 16) {
    if (N <= 2048) return K > 4096 && M <= 8 ? SkinnyShape{16, 2, 1, 1, true} : SkinnyShape{8, 2, 1, 1, true};
    if (tiles <= 256) return {8, 2, 1, 1, false};
    if (tiles <= 512) return K < 1792 ? SkinnyShape{16, 1, 1, 2, false} : SkinnyShape{8, 2, 1, 2, false};
    if (tiles <= 720) return {16, 1, 1, 3, false};
    if (K <= 256 && tiles >= 1024) return {4, 1, 1, 2, false};  // a pair a wave at most: two units share `a`
    return {4, 4, 1, 1, false};
  }
  if (M <= 32) {
    if (N <= 2048) return {8, 2, 2, 1, true};
    if (tiles <= 256) return {8, 2, 2, 1, false};
    if (tiles <= 512) return {8, 2, 2, 2, false};
    return tiles > 768 && tiles <= 1024 ? SkinnyShape{4, 1, 2, 4, false} : SkinnyShape{8, 1, 2, 3, false};
  }
  const int mt = M <= 48 ? 3 : 4;
  if (tiles <= 768) return {8, 1, mt, tiles <= 256 ? 1 : tiles <= 512 ? 2 : 3, false};
  return {4, 1, mt, 4, false};
}

template <typename TO>
static void launch_skinny(const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr,
                          TO* out, long ldo, int M, int N, int K, int act, hipStream_t stream) {
  const SkinnyShape sh = skinny_shape(M, N, K);
  const int cols = sh.cols(), columns = (N + cols - 1) / cols;
#define LEV_SKINNY(W_, U_, MT_, NT_, H_)                                                                                          \
  if (sh.waves == W_ && sh.in_flight == U_ && sh.row_tiles == MT_ && sh.units == NT_ && sh.half == H_)                             \
    gemm_skinny_kernel<TO, W_, U_, MT_, NT_, H_, false><<<columns, W_ * 64, 0, stream>>>(w, a, (uint32_t)(lda / 8), K, N, M, bias, residual, out, ldr, ldo, act)
  if (M > 64) {  // row blocks are a variant of their own: what finds them costs the small steps' kernels 0.2 - 0.4 us
    const dim3 grid((columns + 7) / 8 * 8, (M + 31) / 32);
    gemm_skinny_kernel<TO, 8, 2, 2, 2, false, true><<<grid, 8 * 64, 0, stream>>>(w, a, (uint32_t)(lda / 8), K, N, M, bias, residual, out, ldr, ldo, act);
    return;
  }
  LEV_SKINNY(16, 2, 1, 1, true);
  LEV_SKINNY(8, 2, 1, 1, true);
  LEV_SKINNY(8, 2, 1, 1, false);
  LEV_SKINNY(16, 1, 1, 2, false);
  LEV_SKINNY(8, 2, 1, 2, false);
  LEV_SKINNY(16, 1, 1, 3, false);
  LEV_SKINNY(4, 4, 1, 1, false);
  LEV_SKINNY(4, 1, 1, 2, false);
  LEV_SKINNY(8, 2, 2, 1, true);
  LEV_SKINNY(8, 2, 2, 1, false);
  LEV_SKINNY(8, 2, 2, 2, false);
  LEV_SKINNY(8, 1, 2, 3, false);
  LEV_SKINNY(4, 1, 2, 4, false);
  LEV_SKINNY(8, 1, 3, 1, false);
  LEV_SKINNY(8, 1, 4, 1, false);
  LEV_SKINNY(8, 1, 3, 2, false);
  LEV_SKINNY(8, 1, 4, 2, false);
  LEV_SKINNY(8, 1, 3, 3, false);
  LEV_SKINNY(8, 1, 4, 3, false);
  LEV_SKINNY(4, 1, 3, 4, false);
  LEV_SKINNY(4, 1, 4, 4, false);
#undef LEV_SKINNY
}

// ------------------------------------------------------------------------------------------------
// Stream kernel, for M <= 128 where the skinny kernel is not ahead: the weights are still the traffic that matters, but fetching the `a`
// fragments from L2 once per wave (as the skinny kernel does) would cost more than the weights. Here a
// workgroup of NW waves (4, 8, 12 or 16) owns NW x 16 output columns and all M rows; `a` goes through LDS in chunks
// of 64 k and is shared by the waves, each wave loads its own 16 weight rows straight into MFMA operand
// registers. To fill the chip the K range is split over `S` workgroups (blockIdx.y); with S > 1 the partial
// sums go to a float32 workspace [S][M][N] and a second kernel adds them in order and applies the epilogue.
#define SK_CHUNK 64
#define SK_LDS_STRIDE (SK_CHUNK + 8)

template <typename TO, int MT, int NW>
__global__ void __launch_bounds__(NW * 64, NW == 4 ? 2 : 1)
gemm_stream_kernel(const bf16_t* __restrict__ w, const bf16_t* __restrict__ a, uint32_t lda8, int K, int N, int M, int S, float* __restrict__ partial,
                   const float* __restrict__ bias, const float* residual, TO* out, long ldr, long ldo, int act) {
  const size_t lda = (size_t)lda8 * 8;
  constexpr int BM = MT * 16;
  constexpr int NT = NW * 64;
  constexpr int A_CHUNKS = BM * (SK_CHUNK / 8);       // 16-byte chunks of the a tile
  constexpr int XCH = (A_CHUNKS + NT - 1) / NT;       // per thread (threads beyond the tile repeat its last chunk)
  __shared__ __attribute__((aligned(16))) bf16_t Xs[2][BM * SK_LDS_STRIDE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  const int n0 = blockIdx.x * (NW * 16) + wave * 16;
  const int split = blockIdx.y;
  const int n_chunks = (K + SK_CHUNK - 1) / SK_CHUNK;
  const int per = (n_chunks + S - 1) / S;
  const int c_begin = split * per, c_end = min(n_chunks, c_begin + per);
  const int n = n0 + fr;
  const bf16_t* wrow = w + (size_t)min(n, N - 1) * K;  // a row beyond N reads the last one; its column is never stored
  // this thread's chunks of the a tile
  uint32_t xoff[XCH];
  int xk[XCH], xlds[XCH];
#pragma unroll
  for (int i = 0; i < XCH; ++i) {
    const int c = min(tid + NT * i, A_CHUNKS - 1);
    const int row = c / (SK_CHUNK / 8);
    xk[i] = (c % (SK_CHUNK / 8)) * 8;
    xoff[i] = (uint32_t)((size_t)min(row, M - 1) * lda);
    xlds[i] = row * SK_LDS_STRIDE + xk[i];
  }
  // two register sets for the a tile as for the weights: a chunk's loads are issued two iterations before it is
  // stored to LDS. With one set an iteration could not be shorter than the L2 latency of the a loads of the
  // iteration before (about a microsecond, where its own work is a few hundred cycles).
  u32x4 xr[2][XCH];
  constexpr int KS = SK_CHUNK / 32;  // k-steps per chunk
  u32x4 wr[2][KS];
  auto load_x = [&](int set, int c) {
    const int k0 = min(c, n_chunks - 1) * SK_CHUNK;
#pragma unroll
    for (int i = 0; i < XCH; ++i) {
      const int k = k0 + xk[i];
      xr[set][i] = load16(a + xoff[i] + (k < K ? k : K - 8));
    }
  };
  auto store_x = [&](int buf, int set, int c) {
    const int k0 = c * SK_CHUNK;
#pragma unroll
    for (int i = 0; i < XCH; ++i)
      *reinterpret_cast<u32x4*>(&Xs[buf][xlds[i]]) = (k0 + xk[i] < K) ? xr[set][i] : u32x4{0, 0, 0, 0};
  };
  auto load_w = [&](int set, int c) {
    const int k0 = min(c, n_chunks - 1) * SK_CHUNK;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = k0 + s * 32 + fk;
      wr[set][s] = load16(wrow + (k < K ? k : K - 8));  // beyond K the a fragment is zero, whatever this holds
    }
  };
  // up to 32 rows four sums in turn (a k-step's, of even and of odd chunks): a short chain of roundings each, as the skinny kernel's; more
  // rows have no registers for that
  constexpr int SUMS = MT <= 2 ? 4 : 1;
  f32x4 acc[SUMS][MT];
#pragma unroll
  for (int s = 0; s < SUMS; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (c_begin < c_end) {
    load_x(0, c_begin);
    load_w(0, c_begin);
    load_x(1, c_begin + 1);
    load_w(1, c_begin + 1);
    store_x(0, 0, c_begin);
    load_x(0, c_begin + 2);
    lds_barrier();
    // chunk c (weights in set `set`, a tile in LDS buffer `set`): the a tile of chunk c + 1, in registers since the
    // iteration before last, goes to the other buffer; its registers are refilled three chunks ahead, this chunk's
    // weight registers two chunks ahead
    auto chunk = [&](int c, int set) {
      store_x(set ^ 1, set ^ 1, c + 1);  // past this split's last chunk it fills the buffer nobody reads
      load_x(set ^ 1, c + 3);
      const bf16_t* xb = &Xs[set][fr * SK_LDS_STRIDE + fk];
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const u32x4 af = *reinterpret_cast<const u32x4*>(xb + t * 16 * SK_LDS_STRIDE + s * 32);
          f32x4& sum = acc[(set * KS + s) % SUMS][t];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(af), as_bf16x8(wr[set][s]), sum, 0, 0, 0);
        }
      // the weight registers are refilled behind the products that read them: refilled ahead of them (from a copy),
      // the new values landed in other registers and were moved into place at the end of the loop, which waits for
      // loads issued a moment before
      load_w(set, c + 2);
      lds_barrier();
      // Nothing moves across the end of a chunk: the compiler had lifted the next chunk's masking of its a registers
      // (a select per register) to the top of the loop, where it waited for every load in flight, the weights
      // requested a moment before among them, and each pair of chunks cost a whole memory latency.
      __builtin_amdgcn_sched_barrier(0);
    };
    int c = c_begin;
    for (; c + 1 < c_end; c += 2) {
      chunk(c, 0);
      chunk(c + 1, 1);
    }
    if (c < c_end) chunk(c, 0);
  }
#pragma unroll
  for (int s = 1; s < SUMS; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[0][t] += acc[s][t];
  // 16x16 accumulator: register r of lane l is row 4*(l/16) + r, column l%16
  if (n < N) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = t * 16 + (lane >> 4) * 4 + r;
        if (m < M) {
          if (S == 1)
            epilogue_store<TO>(acc[0][t][r], m, n, bias, residual, ldr, out, ldo, act);
          else
            partial[((size_t)split * M + m) * N + n] = acc[0][t][r];
        }
      }
  }
}

// out = act(sum_s partial[s] + bias) + residual, the partial sums added in the order of s.
// VEC: four consecutive columns per thread (N a multiple of 4 and every pointer and row stride aligned for it).
template <typename TO, int VEC>
__global__ void __launch_bounds__(256)
splitk_reduce_kernel(const float* __restrict__ partial, const float* __restrict__ bias, const float* residual, long ldr, TO* out,
                     long ldo, int M, int N, int S, int act) {
  const size_t total = (size_t)M * N;
  const size_t idx = ((size_t)blockIdx.x * 256 + threadIdx.x) * (VEC ? 4 : 1);
  if (idx >= total) return;
  const int m = (int)(idx / N), n = (int)(idx % N);
  if (VEC) {
    // four ranges are requested at once and added in their order: a loop of load - add - load paid the latency of
    // every range in turn (the partial sums come from other CUs, out of L2 at best)
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* src = partial + idx;
    int s = 0;
    for (; s + 4 <= S; s += 4) {
      f32x4 p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = *reinterpret_cast<const f32x4*>(src + (size_t)(s + j) * total);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[0] += p[j][0]; v[1] += p[j][1]; v[2] += p[j][2]; v[3] += p[j][3];
      }
    }
    {
      f32x4 p[3];
#pragma unroll
      for (int j = 0; j < 3; ++j)  // the last ranges, unconditionally from a valid place
        p[j] = *reinterpret_cast<const f32x4*>(src + (size_t)min(s + j, S - 1) * total);
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (s + j < S) {
          v[0] += p[j][0]; v[1] += p[j][1]; v[2] += p[j][2]; v[3] += p[j][3];
        }
    }
    float o[4] = {v[0], v[1], v[2], v[3]};
    if (bias) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(bias + n);
      o[0] += b[0]; o[1] += b[1]; o[2] += b[2]; o[3] += b[3];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = lev_activate(o[e], act);
    if (residual) {
      const f32x4 r = *reinterpret_cast<const f32x4*>(residual + (size_t)m * ldr + n);
      o[0] += r[0]; o[1] += r[1]; o[2] += r[2]; o[3] += r[3];
    }
    store_vec4<TO>(out + (size_t)m * ldo + n, o);
  } else {
    float v = 0.f;
    for (int s = 0; s < S; ++s) v += partial[(size_t)s * total + idx];
    epilogue_store<TO>(v, m, n, bias, residual, ldr, out, ldo, act);
  }
}

template <typename TO>
static int launch_splitk_reduce(const float* workspace, const float* bias, const float* residual, long ldr, TO* out, long ldo, int M,
                                int N, int S, int act, hipStream_t stream) {
  const size_t total = (size_t)M * N;
  const bool vec = (N % 4 == 0) && (ldo % 4 == 0) && (((uintptr_t)out & 15) == 0) && (((uintptr_t)workspace & 15) == 0) &&
                   (!residual || (ldr % 4 == 0 && ((uintptr_t)residual & 15) == 0)) && (!bias || ((uintptr_t)bias & 15) == 0);
  if (vec)
    splitk_reduce_kernel<TO, 1><<<(unsigned)((total / 4 + 255) / 256), 256, 0, stream>>>(workspace, bias, residual, ldr, out, ldo, M, N, S,
                                                                                          act);
  else
    splitk_reduce_kernel<TO, 0><<<(unsigned)((total + 255) / 256), 256, 0, stream>>>(workspace, bias, residual, ldr, out, ldo, M, N, S, act);
  return lev_check_launch("linear_reduce");
}

// The shape of the stream kernel's launch: how many waves a workgroup has (16 columns each) and into how many k ranges
// K is split. An estimate in microseconds of every combination, fitted to measurements on MI355X of weights from
// 5 MB to 400 MB at 32 to 128 rows.
//   What the CUs fetch is the weights once and the activations once per column tile: a wider workgroup shares its a
//     tile among more columns (at 64 rows and 64 columns the a tiles are as many bytes as the weights). Together
//     the CUs get about 7.5 TB/s out of L2.
//   A CU holds 16 waves of this kernel. The slowest CU has r = ceil(workgroups / 256) workgroups and takes r times a
//     workgroup's share of that time, plus about a microsecond each. With 4 or 8 waves on a CU the loads in flight do
//     not cover the memory latency (x 1.45, x 1.12); 12 or 16 do.
//   More than one range: the second kernel's launch (3 us) and the partial sums, M x N floats per range that are
//     written and read again (4 S M / K of the weights' bytes, mostly out of the caches: weighted half).
//   Measured at the 7B sizes, 64 rows (qkv / proj / fc / mproj, second kernel included): 4 waves 33 / 18 / 42 / 43 us,
//     the shapes chosen here (12 x 4 ranges, 12 x 11, 16 x 4, 16 x 16) 29 / 17 / 40 / 38 us; at 128 rows 47 / 20 / 58 / 55
//     against 37 / 22 / 46 / 45 us.
struct StreamPlan {
  int waves;   // waves of a workgroup (16 columns each): 4, 8, 12 or 16
  int splits;  // k ranges
  double cost; // the estimate, in the model's microseconds
};
static StreamPlan plan_stream(int M, int N, int K) {
  static const int nw[4] = {4, 8, 12, 16};
  const int chunks = (K + SK_CHUNK - 1) / SK_CHUNK;
  const int s_max = chunks / 2 < 16 ? (chunks / 2 < 1 ? 1 : chunks / 2) : 16;  // at least two chunks each
  const double w_bytes = (double)N * K * 2.0;
  StreamPlan best = {4, 1, 1e30};
  double best_cost = 1e30;
  const int n_widths = w_bytes < 24e6 ? 1 : 4;  // weights of a few MB: the narrow workgroup measured best throughout
  for (int i = 0; i < n_widths; ++i) {
    const int tiles = (N + nw[i] * 16 - 1) / (nw[i] * 16);
    const int per_cu = 16 / nw[i];  // workgroups that stay on a CU at once
    const double a_bytes = (double)tiles * M * K * 2.0;  // every column tile reads all of a, once over its ranges
    for (int s = 1; s <= s_max; ++s) {
      const long wgs = (long)tiles * s;
      const long r = (wgs + 255) / 256;  // workgroups of the slowest CU
      if (r > per_cu && wgs > 256L * per_cu) continue;
      const int waves_cu = (int)r * nw[i];
      const double latency = waves_cu <= 4 ? 1.45 : (waves_cu <= 8 ? 1.12 : 1.0);
      const double t = (w_bytes + a_bytes) / 7.5e6;  // microseconds at what the CUs get out of L2 together
      double cost = (double)r * (1.0 + t * 256.0 / wgs * latency);
      if (s > 1) cost += 3.0 + 2.0 * s * M / K * (w_bytes / 4.5e6);
      if (cost < best_cost - 1e-9) {
        best_cost = cost;
        best = {nw[i], s, cost};
      }
    }
  }
  return best;
}

// Tile shape and number of k ranges of the tile kernel. Estimated time of each tile shape: rounds of workgroups over the 256
// CUs times (k-tiles x the shape's time per k-tile + a fixed cost for a tile's first loads and its epilogue). Two
// 128 x 128 workgroups fit a CU and then share it; up to 256 of them have a CU each. Where the output has so few
// tiles that most CUs would idle (a few hundred rows times a narrow weight), K is split into ranges, as in the
// stream kernel: the second kernel then costs its launch and the traffic of the partial sums. The constants are
// microseconds measured on MI355X.
struct TilePlan {
  int shape;   // 0: 256 x 256, 1: 256 x 192, 2: 256 x 128, 3: 128 x 128
  int splits;  // k ranges (1: none)
};
static TilePlan plan_tiles(int M, int N, int K) {
  static const int bm[4] = {256, 256, 256, 128}, bn[4] = {256, 192, 128, 128};
  static const double us_per_ktile[4] = {1.72, 1.36, 0.97, 0.6}, fixed[4] = {13.0, 11.0, 9.0, 7.0};
  const long nk = (K + TK - 1) / TK;
  TilePlan best = {0, 1};
  double best_cost = 1e30;
  for (int i = 0; i < 4; ++i) {
    const long tiles = (long)((M + bm[i] - 1) / bm[i]) * ((N + bn[i] - 1) / bn[i]);
    double cost;
    if (i == 3 && tiles > 256)
      cost = (double)((tiles + 511) / 512) * (nk * 1.05 + 9.0);
    else
      cost = (double)((tiles + 255) / 256) * (nk * us_per_ktile[i] + fixed[i]);
    if (cost < best_cost) {
      best_cost = cost;
      best = {i, 1};
    }
    for (int s = 2; s <= 16 && tiles * s <= 256 && nk / s >= 4; ++s) {
      const long per = (nk + s - 1) / s;
      if (per * (s - 1) >= nk) continue;  // a range would be empty
      const double reduce = 4.0 + (double)(s + 1) * M * N * 4.0 / 3.0e6;
      const double c = per * us_per_ktile[i] + fixed[i] + reduce;
      if (c < best_cost) {
        best_cost = c;
        best = {i, s};
      }
    }
  }
  return best;
}

// Which kernel takes M <= 64 rows (above: skinny_in_blocks). An estimate of the skinny kernel in microseconds: a launch and its ramp, and
// the longest of the weights' read from memory, the share of it that falls to the busiest CU, and what that CU pulls through its caches
// (its columns and most of `a`, for each of its workgroups: the rate depends on how much of that is waited for at once). The stream
// kernel's time hardly grows with the rows, but it pays for its K ranges: plan_stream's cost and a launch; unsplit, its workgroups all
// start at their rows' beginnings, and rows a multiple of 4 KB apart (K = 2,048 n) then meet on the same memory channels.
// The constants are those that choose best over 2,400 cases (weights of 0.15 M to 206 M numbers, sums of 64 to 24,576, 1 to 64 rows; 400 weights
// drawn, 32 of layers), under the condition that weights of 17 MB and more at 64 rows, which the norm behind them adds up, stay split. The choice
// is 0.3 % behind the better kernel on average, and more than 5 % at 2 % of the cases; the estimate of the one that is chosen is 15 % off on average. The
// fit before it, to 154 cases of layers, took no account of the stream kernel's own launch and of long sums of few outputs and was 3.2 %
// behind: 65024 x 2048 at 25 rows 73 us (stream) for 53, 464 x 16384 at 22 rows 17.2 (skinny) for 12.0, 3118 x 128 at 64 rows 7.0 (stream)
// for 3.7. Measured, skinny / stream: 16384 x 4096 at 8 / 64 rows 24.9 / 32.6, 30.6 / 37.6; 4096 x 16384 at 8 / 24 / 64 rows 24.5 / 33.0,
// 28.9 / 34.1, 44.8 / 36.7; 1600 x 6400 at 16 / 64 rows 9.2 / 11.5, 19.4 / 13.6; 6144 x 24576 at 4 / 24 rows 55.4 / 60.0, 68.1 / 61.2.
static double skinny_estimate(int M, int N, int K) {
  const SkinnyShape sh = skinny_shape(M, N, K);
  const long wgs = (N + sh.cols() - 1) / sh.cols(), r = (wgs + 255) / 256;  // r: workgroups of the busiest CU
  const double memory = 2.0 * N * K / 7.3e6, own = r * (double)sh.cols() * K * 2.0 / 34e3;
  double rate = (long)N * K <= (1L << 23) ? 66e3 : sh.waves == 4 ? 34.7e3 : sh.units > 1 ? 45e3 : 39e3;  // small weights stay in the caches' reach
  const double most = sh.units > 1 ? 34e3 : 38.4e3;
  if (K >= 8192 && rate > most) rate = most;  // long sums: a chain of round trips a workgroup
  const double caches = r * (sh.cols() + (M > 32 ? 0.93 : 0.74) * M) * K * 2.0 / rate;
  double cost = memory > own ? memory : own;
  if (caches > cost) cost = caches;
  return 2.4 + cost + (sh.row_tiles > 1 ? 0.75 * (r - 1) : 0.0);
}
// 0: the estimate decides; 1 / 2: the skinny / the stream kernel wherever it takes the row count (up to 64 rows and where use_skinny has blocks / to 128 rows), the tile kernel above. For measurements of the
// choice itself (a test times both candidates at widths the estimates were not fitted to); not used by the engine.
static int g_force_kernel = 0;
extern "C" int lev_linear_mfma_force(int kind) {
  LEV_REQUIRE(kind >= 0 && kind <= 2, "linear: unknown kernel choice %d (0: by estimate, 1: skinny, 2: stream)", kind);
  g_force_kernel = kind;
  return 0;
}
static bool use_skinny(int M, int N, int K) {
  if (M > 64) return skinny_in_blocks(M, N, K) && g_force_kernel != 2;
  if (g_force_kernel) return g_force_kernel == 1;
  const StreamPlan plan = plan_stream(M, N, K);
  return skinny_estimate(M, N, K) <= 2.3 + 1.17 * plan.cost * (plan.splits == 1 && K % 2048 == 0 ? 1.2 : 1.0);
}

// Where the ring kernel is ahead of the library and of the kernels here, measured at 25 weights of 512 x 2048 to 16384 x 4096 and 65 to 2,048 rows (microseconds, before /
// ring; the library's kernels are chosen by timing): below 2^22 outputs 0.9 to 1.9 times as fast; above, 12288 x 4096 at 400 / 512 rows 54.7 / 59, 55.8 / 77, 6400 x 1600
// at 1,000 28.9 / 37, 4096 x 2048 at 2,048 34 / 45. Heads of more outputs than a layer has stay where they were: 50257 x 768 at 65 rows 23.4 / 29.8.
// Of 17 to 64 rows it takes long sums up to 48 million weights, and from 41 rows other large ones: the kernels for them have few outputs a CU or a range too
// many. Microseconds with what adds the ranges, before / ring. By the norm behind the product (left): 1600 x 6400 at 24 / 64 rows 13.2 / 10.5, 14.2 / 12.0; 768 x 3072 8.0 / 7.4, 11.0 / 7.9; 32 x 4096 at 24
// 7.9 / 6.6; from 41 rows 4096 x 4096 at 64 18.1 / 13.7, 3072 x 6144 at 48 / 64 18.4 / 14.6, 19.3 / 15.6, 5120 x 5120 23.4 / 18.6, 22.6 / 19.5, 3584 x 4864 17.7 / 14.1, 18.7 / 14.7, 4096 x 11008 30.1 / 25.4, 30.9 / 26.3.
// By a pass of its own, which is all that up to 24 rows of the smaller weights gain: 768 x 3072 at 24 rows 5.6 / 7.1, 32 x 4096 5.8 / 6.3, 1024 x 4096 at 17 8.3 / 8.9, but at 28 9.7 / 8.9, and
// 1280 x 5120 at 17 / 24 8.9 / 8.4, 9.8 / 8.9; 768 x 3072 at 64 8.7 / 7.5. Not 1600 x 1600 at 24 rows (5.1 / 4.3, less than the norm then pays for the ranges) nor gated inner sizes (2048 x 5376 at
// 32 rows 11.0 / 7.4, but a session of Lelatar 33.1 -> 33.8 ms: a kernel of its own adds the ranges there). A forced kernel is not this one.
static bool use_ring(int M, int N, int K, bool left) {
  if (g_force_kernel || K > RING_MAX_K) return false;
  const long weights = (long)N * K;
  if (M > 16 && M <= 64) return N <= K && weights < 48000000L && ((K >= 4L * N && K >= 3072 && (left || M > 24 || weights > (1L << 22))) || (M > 40 && weights >= (1L << 24)));
  return M > 64 && N <= 32768 && (long)M * N < (1L << 22) && !use_skinny(M, N, K);
}

// The tile and the ranges of the ring kernel, 16 x tile + ranges; -1 where another kernel takes the product.
extern "C" int lev_linear_mfma_ring_of(int M, int N, int K, int left) {
  if (!use_ring(M, N, K, left != 0)) return -1;
  const RingPlan plan = lev_ring_plan(M, N, K, left != 0);
  return 16 * plan.shape + plan.splits;
}

// the same of a product whose ranges may be left
extern "C" int lev_linear_mfma_ring(int M, int N, int K) { return lev_linear_mfma_ring_of(M, N, K, 1); }

// Into how many ranges the sum over K is split (1: the kernel finishes its outputs itself).
extern "C" int lev_linear_mfma_ranges_of(int M, int N, int K, int left) {
  if (use_ring(M, N, K, left != 0)) return lev_ring_plan(M, N, K, left != 0).splits;
  if (use_skinny(M, N, K)) return 1;
  return M <= 128 ? plan_stream(M, N, K).splits : plan_tiles(M, N, K).splits;
}

// the same of a product that adds them itself
extern "C" int lev_linear_mfma_ranges(int M, int N, int K) { return lev_linear_mfma_ranges_of(M, N, K, 0); }

extern "C" long lev_linear_mfma_workspace(int M, int N, int K, int left) {
  const int S = lev_linear_mfma_ranges_of(M, N, K, left);
  return S > 1 ? (long)S * M * N * (long)sizeof(float) : 0;
}

// out = act(sum of the S ranges in workspace [S][M][N] + bias) + residual: what lev_linear_mfma runs itself unless it was
// asked to leave the ranges to the caller.
extern "C" int lev_linear_mfma_finish(const float* workspace, const float* bias, const float* residual, long ldr, void* out, long ldo,
                                      int M, int N, int S, int act, int out_dtype, hipStream_t stream) {
  LEV_REQUIRE(workspace && M > 0 && N > 0 && S > 1, "linear: nothing to finish (M=%d N=%d ranges=%d)", M, N, S);
  if (out_dtype == LEV_F32) return launch_splitk_reduce<float>(workspace, bias, residual, ldr, (float*)out, ldo, M, N, S, act, stream);
  if (out_dtype == LEV_BF16) return launch_splitk_reduce<bf16_t>(workspace, bias, residual, ldr, (bf16_t*)out, ldo, M, N, S, act, stream);
  return lev_fail("linear: unknown output dtype %d", out_dtype);
}

template <typename TO>
static int launch_stream(const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr, TO* out,
                         long ldo, float* workspace, int M, int N, int K, int act, int defer, hipStream_t stream) {
  if ((size_t)M * lda >= (1ull << 32)) return lev_fail("linear: the activation matrix is too large (M=%d lda=%ld)", M, lda);
  const StreamPlan plan = plan_stream(M, N, K);
  const int S = plan.splits;
  if (S > 1 && !workspace) return lev_fail("linear: M=%d N=%d K=%d needs a workspace of lev_linear_mfma_workspace bytes", M, N, K);
  dim3 grid((N + plan.waves * 16 - 1) / (plan.waves * 16), S);
#define LEV_STREAM(MT_, NW_) \
  gemm_stream_kernel<TO, MT_, NW_><<<grid, NW_ * 64, 0, stream>>>(w, a, (uint32_t)(lda / 8), K, N, M, S, workspace, bias, residual, out, ldr, ldo, act)
#define LEV_STREAM_MT(MT_)                 \
  switch (plan.waves) {                    \
    case 4: LEV_STREAM(MT_, 4); break;     \
    case 8: LEV_STREAM(MT_, 8); break;     \
    case 12: LEV_STREAM(MT_, 12); break;   \
    default: LEV_STREAM(MT_, 16); break;   \
  }
  if (M <= 32) {
    LEV_STREAM_MT(2)
  } else if (M <= 64) {
    LEV_STREAM_MT(4)
  } else {
    LEV_STREAM_MT(8)
  }
#undef LEV_STREAM_MT
#undef LEV_STREAM
  if (int rc = lev_check_launch("linear_stream")) return rc;
  if (S > 1 && !defer) return launch_splitk_reduce<TO>(workspace, bias, residual, ldr, out, ldo, M, N, S, act, stream);
  return 0;
}

template <typename TO>
static int linear_mfma_typed(const bf16_t* a, long lda, const bf16_t* w, const float* bias, const float* residual, long ldr,
                             TO* out, long ldo, float* workspace, int M, int N, int K, int act, int defer, hipStream_t stream) {
  if (use_ring(M, N, K, defer != 0)) {
    const RingPlan plan = lev_ring_plan(M, N, K, defer != 0);
    const int rc = lev_ring_launch(plan, a, lda, w, bias, residual, ldr, out, ldo, workspace, M, N, K, act, sizeof(TO) == 4 ? LEV_F32 : LEV_BF16, stream);
    if (rc || plan.splits == 1 || defer) return rc;
    return launch_splitk_reduce<TO>(workspace, bias, residual, ldr, out, ldo, M, N, plan.splits, act, stream);
  } else if (use_skinny(M, N, K)) {
    launch_skinny<TO>(a, lda, w, bias, residual, ldr, out, ldo, M, N, K, act, stream);
  } else if (M <= 128) {
    return launch_stream<TO>(a, lda, w, bias, residual, ldr, out, ldo, workspace, M, N, K, act, defer, stream);
  } else {
    if ((size_t)M * lda >= (1ull << 31) || (size_t)N * K >= (1ull << 31))
      return lev_fail("linear: operands of more than 2^31 elements are not supported (M=%d lda=%ld N=%d K=%d)", M, lda, N, K);
    const TilePlan plan = plan_tiles(M, N, K);
    int rc;
    if (plan.shape == 0)
      rc = launch_tile<TO, 256, 256>(a, lda, w, bias, residual, ldr, out, ldo, workspace, M, N, K, act, plan.splits, defer, stream);
    else if (plan.shape == 1)
      rc = launch_tile<TO, 256, 192>(a, lda, w, bias, residual, ldr, out, ldo, workspace, M, N, K, act, plan.splits, defer, stream);
    else if (plan.shape == 2)
      rc = launch_tile<TO, 256, 128>(a, lda, w, bias, residual, ldr, out, ldo, workspace, M, N, K, act, plan.splits, defer, stream);
    else
      rc = launch_tile<TO, 128, 128>(a, lda, w, bias, residual, ldr, out, ldo, workspace, M, N, K, act, plan.splits, defer, stream);
    if (rc) return rc;
  }
  return lev_check_launch("linear_mfma");
}

// leave_ranges: where the sum over K is split into ranges (lev_linear_mfma_ranges > 1) the kernel stops after writing
// them to workspace [S][M][N]; bias, activation and residual are then the caller's to apply (lev_linear_mfma_finish, or
// a kernel of its own that reads the ranges).
extern "C" int lev_linear_mfma(const void* a, long lda, const void* w, const float* bias, const float* residual, long ldr,
                               void* out, long ldo, void* workspace, int M, int N, int K, int act, int out_dtype,
                               int leave_ranges, hipStream_t stream) {
  LEV_REQUIRE(M >= 0 && N > 0 && K > 0, "linear: bad sizes M=%d N=%d K=%d", M, N, K);
  LEV_REQUIRE(K % 8 == 0 && lda % 8 == 0, "linear (bfloat16): K=%d and the row stride %ld must be multiples of 8", K, lda);
  LEV_REQUIRE(((uintptr_t)a & 15) == 0 && ((uintptr_t)w & 15) == 0, "linear (bfloat16): operands must be 16-byte aligned");
  LEV_REQUIRE(lda >= K && ldo >= N, "linear: row strides lda=%ld ldo=%ld are smaller than K=%d / N=%d", lda, ldo, K, N);
  LEV_REQUIRE(!residual || (ldr >= N && out_dtype == LEV_F32), "linear: a residual needs a float32 output and a row stride >= N");
  LEV_REQUIRE(act >= LEV_ACT_NONE && act <= LEV_ACT_LAST, "linear: unknown activation %d", act);
  if (M == 0) return 0;
  if (out_dtype == LEV_F32)
    return linear_mfma_typed<float>((const bf16_t*)a, lda, (const bf16_t*)w, bias, residual, ldr, (float*)out, ldo,
                                    (float*)workspace, M, N, K, act, leave_ranges, stream);
  if (out_dtype == LEV_BF16)
    return linear_mfma_typed<bf16_t>((const bf16_t*)a, lda, (const bf16_t*)w, bias, residual, ldr, (bf16_t*)out, ldo,
                                     (float*)workspace, M, N, K, act, leave_ranges, stream);
  return lev_fail("linear: unknown output dtype %d", out_dtype);
}

// Which products of a few rows take the norm ahead of them along (gemm_norm.hip, with the figures): those of the skinny kernel whose workgroups make one
// round of the CUs (more would normalise in vain), but none that spreads a short sum over many outputs (11520 x 256 at 4 / 8 rows 6.4 / 6.2, 6.5 / 6.8). Sums
// below 256 have not been measured, half units (up to 2,048 outputs) are shapes of products that follow no norm.
extern "C" int lev_linear_normed_takes(int M, int N, int K) {
  if (M < 1 || M > NORMED_MAX_M || K < 256 || K > NORMED_MAX_K || K % 8 || N <= 2048 || N > 16 * 720 || (K < 512 && N > 8192) || g_force_kernel == 2 || !use_skinny(M, N, K)) return 0;
  return !skinny_shape(M, N, K).half;
}

// out = act(norm(x) . w^T + bias): the norm of lev_norm into bfloat16 and the product of lev_linear_mfma, bit for bit, in one kernel. x [M][K] float32.
extern "C" int lev_linear_normed(const float* x, const float* norm_w, const float* norm_b, float eps, int rms, const void* w, const float* bias, void* out,
                                 long ldo, int M, int N, int K, int act, hipStream_t stream) {
  LEV_REQUIRE(x && norm_w && w && out && lev_linear_normed_takes(M, N, K), "norm and linear: no kernel for M=%d N=%d K=%d", M, N, K);
  LEV_REQUIRE((((uintptr_t)x | (uintptr_t)norm_w | (uintptr_t)norm_b | (uintptr_t)w) & 15) == 0, "norm and linear: operands must be 16-byte aligned");
  LEV_REQUIRE(ldo >= N && eps > 0.f && act >= LEV_ACT_NONE && act <= LEV_ACT_LAST, "norm and linear: bad ldo=%ld, eps=%g or activation %d", ldo, eps, act);
  const SkinnyShape sh = skinny_shape(M, N, K);
  const int rc = lev_normed_launch(sh.waves, sh.units, x, norm_w, norm_b, eps, rms, (const bf16_t*)w, bias, (bf16_t*)out, ldo, M, N, K, act, stream);
  return rc < 0 ? lev_fail("norm and linear: no kernel of %d waves and %d units", sh.waves, sh.units) : rc;
}
