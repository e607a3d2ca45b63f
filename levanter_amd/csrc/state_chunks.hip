// The recurrences of state_recurrence.hip on runs of many tokens, in chunks on the matrix cores. The step's tokens are cut into blocks of 64;
// a chunk is what of one run lies in one block. With cs_i the running sum of the chunk's log decays and S0 the state that enters it:
//   SSD:    P_ij = exp(cs_i - cs_j) w_j (q_i . k_j), j <= i;     o_i = exp(cs_i) S0^T q_i + sum_j P_ij v_j
//           S    = exp(cs_end) S0 + sum_j exp(cs_end - cs_j) w_j k_j v_j^T
//   DELTA:  P_ij = exp(cs_i - cs_j) (q_i . k_j), j <= i;         A_ij = w_i exp(cs_i - cs_j) (k_i . k_j), j < i;     T = (1 + A)^-1
//           R_i  = w_i (v_i - exp(cs_i) S0^T k_i);               U = T R;     o_i = exp(cs_i) S0^T q_i + sum_j P_ij u_j
//           S    = exp(cs_end) S0 + sum_j exp(cs_end - cs_j) k_j u_j^T
// P, T and the running sums do not depend on the state: a first kernel makes them (of the sums exp(cs_i) and exp(cs_end - cs_i)) for all blocks and heads in parallel
// (entries between tokens of different runs are zero, so T is block-diagonal by itself), a second one goes along each run and carries the state from chunk to chunk.
// Its chain of one block after the other is the time of a long prompt: what can be done ahead is, and products that only add up go in sums of their own. Entries of
// T are bounded: with unit keys and write rates below one, 1 - w k k^T does not lengthen a vector.
//
// Exactness. q, k and v are bfloat16 numbers (their unit norms are a float32 factor a row, applied behind the product), so q . k is a
// bfloat16 product with exact terms and a 32-bit sum. Every other product with a bfloat16 side has its 32-bit side (state, weights) split
// into three bfloat16 numbers that hold all its 24 bits, three products for one. Products with two 32-bit sides (T R, DELTA's P U, and those
// that make T) run on the 32-bit matrix instruction. Differences of running sums are taken in 64-bit: one fast decay must not cost the
// digits of the slow ones behind it.
//
// The matrix instruction leaves rows 4 (lane / 16) + r and column lane % 16 in register r of a lane; as the K order of a product is free as
// long as both sides agree, such registers feed the next product directly (k slot of lane group g, register r: row 4 g + r), also two tiles
// side by side for an instruction with K = 32. A 16 x 16 tile M as a left side is then M[lane % 16][4 (lane / 16) + r]; P and T are stored that
// way, [block][head][w (w + 1) / 2 + j][lane][4] for the tile of rows 16 w and columns 16 j, j <= w.
#include "state_recurrence.h"

typedef __attribute__((ext_vector_type(8))) __bf16 sc_bf16x8;
typedef __attribute__((ext_vector_type(4))) float sc_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t sc_u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t sc_u32x2;

#define SC_Q 64   // tokens of a block
#define SC_VB 16  // value columns of a workgroup
#define SC_LDT (SC_Q + 8)

__device__ __forceinline__ sc_f32x4 sc_mfma(sc_u32x4 a, sc_u32x4 b, sc_f32x4 c) {
  union { sc_u32x4 u; sc_bf16x8 v; } x, y;
  x.u = a, y.u = b;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, y.v, c, 0, 0, 0);
}
// the same in four sums that do not wait for each other
__device__ __forceinline__ void sc_mfma32(sc_f32x4 a, sc_f32x4 b, sc_f32x4 (&c)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c[r], 0, 0, 0);
}
__device__ __forceinline__ sc_f32x4 sc_mfma32(sc_f32x4 a, sc_f32x4 b, sc_f32x4 c) {  // 16 of the K dimension: register r is k slot (lane / 16, r)
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}
// eight 32-bit numbers as three times eight bfloat16 numbers whose sum they are
__device__ __forceinline__ void sc_split(const float (&v)[8], sc_u32x4 (&out)[3]) {
  float rest[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) rest[i] = v[i];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = float2_to_bf16x2(rest[2 * i], rest[2 * i + 1]);
      out[p][i] = w;
      rest[2 * i] -= __uint_as_float(w << 16);
      rest[2 * i + 1] -= __uint_as_float(w & 0xffff0000u);
    }
}
// the decays from tokens 4 grp + r of a tile to the token whose running sum is cs_i: zero for tokens of other runs and, in the token's own tile
// (`diagonal`), for those behind it (the condition goes into the exponent: around the exponential it would become a branch per element)
__device__ __forceinline__ sc_f32x4 sc_decays(double cs_i, const double* cs, const bool (&same)[4], bool valid, bool diagonal, int grp, int col) {
  typedef __attribute__((ext_vector_type(2))) double sc_f64x2;
  const sc_f64x2 a = *reinterpret_cast<const sc_f64x2*>(cs), b = *reinterpret_cast<const sc_f64x2*>(cs + 2);
  sc_f32x4 x = {(float)(cs_i - a[0]), (float)(cs_i - a[1]), (float)(cs_i - b[0]), (float)(cs_i - b[1])};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    x[r] = !valid || !same[r] || (diagonal && 4 * grp + r > col) ? -INFINITY : fminf(x[r], 0.f);
    x[r] = expf(x[r]);
  }
  return x;
}
__device__ __forceinline__ sc_u32x4 sc_read16(const bf16_t* p) { return *reinterpret_cast<const sc_u32x4*>(p); }
__device__ __forceinline__ sc_u32x4 sc_read8x2(const bf16_t* p, const bf16_t* q) {
  const sc_u32x2 a = *reinterpret_cast<const sc_u32x2*>(p), b = *reinterpret_cast<const sc_u32x2*>(q);
  return sc_u32x4{a[0], a[1], b[0], b[1]};
}
// eight channels from i0 on of a row of dk. VEC (rows are multiples of 8 channels at 16-byte boundaries): what lies beyond the row is some
// other of its channels and the load stands under no condition (nothing waits for it before it is used); sc_mask8 puts zeros there.
template <bool VEC>
__device__ __forceinline__ sc_u32x4 sc_load8(const bf16_t* row, int i0, int dk) {
  sc_u32x4 v = {0, 0, 0, 0};
  if (VEC) {
    v = *reinterpret_cast<const sc_u32x4*>(row + min(i0, dk - 8));
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (i0 + e < dk) v[e >> 1] |= (uint32_t)row[i0 + e] << (16 * (e & 1));
  }
  return v;
}
__device__ __forceinline__ sc_u32x4 sc_mask8(sc_u32x4 v, int i0, int dk) {
  const uint32_t keep = i0 < dk ? 0xffffffffu : 0u;
  return sc_u32x4{v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
}

// ---- what does not depend on the state ---------------------------------------------------------------------------------------
// One workgroup of four waves per (block, head); wave w has the rows 16 w of the block's matrices.
template <int DKM, int RULE, bool VEC>
__global__ void __launch_bounds__(256)
sc_inner_kernel(const bf16_t* __restrict__ u, const float* __restrict__ scal, const int* __restrict__ token_slots, float* __restrict__ P_out,
                float* __restrict__ T_out, float2* __restrict__ E_out, SrShape s) {
  constexpr int LDK = DKM + 8, KS = DKM / 32, QI = DKM / 32;
  constexpr bool DELTA = RULE == SR_DELTA;
  __shared__ __attribute__((aligned(16))) bf16_t s_q[SC_Q][LDK], s_k[SC_Q][LDK];
  __shared__ __attribute__((aligned(16))) double s_cs[SC_Q];
  __shared__ __attribute__((aligned(16))) float s_w[SC_Q], s_rk[SC_Q], s_rq[SC_Q];
  __shared__ __attribute__((aligned(16))) int s_slot[SC_Q];
  __shared__ __attribute__((aligned(16))) sc_f32x4 s_A[DELTA ? 6 : 1][64], s_T[DELTA ? 4 : 1][64];
  __shared__ __attribute__((aligned(16))) float s_At[DELTA ? 4 : 1][16][16], s_Tr[DELTA ? 4 : 1][16][20];
  const int h = blockIdx.x, tb = blockIdx.y * SC_Q;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, grp = lane >> 4;
  const int g = h / (s.H / s.G), n_scal = 2 * s.H + 2 * s.G, dk = s.dk;
#pragma unroll
  for (int n = 0; n < QI; ++n) {
    const int idx = tid + 256 * n, row = idx / (DKM / 8), i0 = (idx % (DKM / 8)) * 8;
    const bf16_t* ur = u + (size_t)min(tb + row, s.Tn - 1) * s.C + (size_t)g * dk;
    const sc_u32x4 q = sc_load8<VEC>(ur + s.q_off, i0, dk), k = sc_load8<VEC>(ur + s.k_off, i0, dk);
    *reinterpret_cast<sc_u32x4*>(&s_q[row][i0]) = VEC ? sc_mask8(q, i0, dk) : q;
    *reinterpret_cast<sc_u32x4*>(&s_k[row][i0]) = VEC ? sc_mask8(k, i0, dk) : k;
  }
  if (wave == 0) {
    const int t = min(tb + lane, s.Tn - 1), slot = tb + lane < s.Tn ? token_slots[t] : -1;
    const float* sc = scal + (size_t)t * n_scal;
    const float w = sc[s.H + h], rk = sc[2 * s.H + g], rq = sc[2 * s.H + s.G + g];
    double cs = slot >= 0 ? (double)sc[h] : 0.0;
    // running sums within the runs: `begin` is the first of the lane's own, `end` its last
    const int before = __shfl_up(slot, 1, 64);  // by all lanes
    const unsigned long long begins = __ballot(lane == 0 || slot != before), behind = begins >> lane >> 1;
    const int begin = 63 - __clzll(begins & (~0ull >> (63 - lane))), end = behind ? lane + __ffsll(behind) - 1 : 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const double up = __shfl_up(cs, d, 64);
      if (lane - d >= begin) cs += up;
    }
    s_cs[lane] = cs;
    s_slot[lane] = slot;
    s_w[lane] = w;
    s_rk[lane] = rk, s_rq[lane] = rq;
    // what the walk along the runs needs of them: exp(cs_i), and exp(cs_end - cs_i) times the key's weight
    E_out[((size_t)blockIdx.y * s.H + h) * SC_Q + lane] = make_float2(expf((float)cs), expf((float)(__shfl(cs, end, 64) - cs)) * (DELTA ? rk : w));
  }
  __syncthreads();
  const double cs_i = s_cs[16 * wave + col];  // of the token that is this lane's row in the tiles below
  const int slot_i = s_slot[16 * wave + col];
  const float rq_i = s_rq[16 * wave + col], wk_i = DELTA ? s_w[16 * wave + col] * s_rk[16 * wave + col] : 0.f;
  const size_t tile0 = ((size_t)blockIdx.y * s.H + h) * 10;
  sc_u32x4 bq[KS], bk[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    bq[ks] = sc_read16(&s_q[16 * wave + col][32 * ks + 8 * grp]);
    if (DELTA) bk[ks] = sc_read16(&s_k[16 * wave + col][32 * ks + 8 * grp]);
  }
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    if (jt > wave) break;
    sc_f32x4 pq = {0.f, 0.f, 0.f, 0.f}, kk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const sc_u32x4 a = sc_read16(&s_k[16 * jt + col][32 * ks + 8 * grp]);
      pq = sc_mfma(a, bq[ks], pq);
      if (DELTA) kk = sc_mfma(a, bk[ks], kk);
    }
    const int4 slot_j = *reinterpret_cast<const int4*>(&s_slot[16 * jt + 4 * grp]);
    const bool same[4] = {slot_j.x == slot_i, slot_j.y == slot_i, slot_j.z == slot_i, slot_j.w == slot_i};
    sc_f32x4 dec = sc_decays(cs_i, &s_cs[16 * jt + 4 * grp], same, slot_i >= 0, jt == wave, grp, col);
    dec *= *reinterpret_cast<const sc_f32x4*>(DELTA ? &s_rk[16 * jt + 4 * grp] : &s_w[16 * jt + 4 * grp]);
    pq *= dec * rq_i;
    *reinterpret_cast<sc_f32x4*>(P_out + ((tile0 + wave * (wave + 1) / 2 + jt) * 64 + lane) * 4) = pq;
    if (DELTA) {
      kk *= dec * wk_i;
      if (jt < wave) {
        s_A[wave * (wave - 1) / 2 + jt][lane] = sc_f32x4{-kk[0], -kk[1], -kk[2], -kk[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) s_At[wave][4 * grp + r][col] = 4 * grp + r == col ? 0.f : kk[r];  // column 4 grp + r of the diagonal tile
        __builtin_amdgcn_wave_barrier();
        // row `col` of its inverse: y (1 + A) = e_col, from the last column back
        float y[16];
#pragma unroll
        for (int c = 15; c >= 0; --c) {
          float acc[4] = {c == col ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            if (4 * q4 + 3 <= c) continue;
            const sc_f32x4 a4 = *reinterpret_cast<const sc_f32x4*>(&s_At[wave][c][4 * q4]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (4 * q4 + e > c) acc[e] = fmaf(-a4[e], y[4 * q4 + e], acc[e]);
          }
          y[c] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        }
        sc_f32x4 T;
#pragma unroll
        for (int r = 0; r < 4; ++r) T[r] = grp == 0 ? y[r] : grp == 1 ? y[4 + r] : grp == 2 ? y[8 + r] : y[12 + r];
        s_T[wave][lane] = T;
        *reinterpret_cast<sc_f32x4*>(&s_Tr[wave][col][4 * grp]) = T;  // the same by rows, for the product below
        *reinterpret_cast<sc_f32x4*>(T_out + ((tile0 + wave * (wave + 1) / 2 + wave) * 64 + lane) * 4) = T;
      }
    }
  }
  if (!DELTA) return;
  __syncthreads();
  // wave j: the tiles below the diagonal of column tile j of the inverse, T_ij = -T_ii sum_k A_ik T_kj
  sc_f32x4 Tc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i < wave) continue;
    if (i == wave) {
#pragma unroll
      for (int r = 0; r < 4; ++r) Tc[i][r] = s_Tr[wave][4 * grp + r][col];
      continue;
    }
    sc_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k < wave || k >= i) continue;
      acc = sc_mfma32(s_A[i * (i - 1) / 2 + k][lane], Tc[k], acc);
    }
    Tc[i] = sc_mfma32(s_T[i][lane], acc, sc_f32x4{0.f, 0.f, 0.f, 0.f});
    float* dst = T_out + (tile0 + i * (i + 1) / 2 + wave) * 256;
#pragma unroll
    for (int r = 0; r < 4; ++r) dst[((col >> 2) * 16 + 4 * grp + r) * 4 + (col & 3)] = Tc[i][r];
  }
}

// ---- along the runs -------------------------------------------------------------------------------------------------------------
// One workgroup of four waves per (run, head, 16 CT value columns); wave w has the tokens 16 w .. of the block as rows of the result and a quarter
// of the state's key channels, in accumulator registers. SSD takes up to 64 columns at once where there are many runs: what a block stages in LDS (keys, queries, weights)
// is the same for all of them (64 heads of 128 / 64, microseconds with 16 / 64 columns: 32 runs of 40 to 150 tokens 205 / 158, but three of 300 to 999, whose chain is the bound, 62 / 100; with the next block's loads kept
// from waits - copies of registers for a branch's sake, the block's own stores - and operands read ahead of their products 57; DELTA, 16 heads, 64 / 55).
// Runs of several tokens begin first: behind 31 single tokens, as a step has them, one of 1,000 would begin last and its chain be the end of the step (with all that stands around the kernel, 16 columns / 64 / 64 and
// long runs first: 246 / 254 / 188; of 3,000 406 / 484 / 365; 32 of 40 to 150, in a scan that reads every slot once, 386 / 306 / 282). DELTA stays at 16: its products with two 32-bit sides are four times as long.
template <int DKM, int RULE, bool VEC, int CT>
__global__ void __launch_bounds__(256, (DKM == 64 && CT == 4) || (DKM == 128 && RULE == SR_DELTA && !VEC) ? 2 : 1)  // else 260 and 257 registers would leave one workgroup a CU; others lose 2 - 7 % by the bound
sc_chunk_kernel(const bf16_t* __restrict__ u, const float* __restrict__ scal, const float* __restrict__ P_in, const float* __restrict__ T_in,
                const float2* __restrict__ E_in, float* __restrict__ state, const int* __restrict__ token_slots, float* __restrict__ o, SrShape s) {
  constexpr int LDK = DKM + 8, KS = DKM / 32, NTW = DKM / 64, KI = DKM / 64, QI = DKM / 32;
  constexpr bool DELTA = RULE == SR_DELTA;
  static_assert(!DELTA || CT == 1, "one tile of columns");
  __shared__ __attribute__((aligned(16))) bf16_t s_q[SC_Q][LDK], s_k[DELTA ? SC_Q : 1][LDK], s_kt[DKM][SC_LDT], s_S[3][SC_VB * CT][LDK];
  __shared__ __attribute__((aligned(16))) bf16_t s_x[DELTA ? 1 : SC_VB * CT][SC_LDT];
  __shared__ __attribute__((aligned(16))) float s_ecs[SC_Q], s_wend[SC_Q], s_w[SC_Q], s_rk[SC_Q], s_rq[SC_Q];
  __shared__ float s_end;
  __shared__ __attribute__((aligned(16))) sc_f32x4 s_R[DELTA ? 4 : 1][64], s_U[DELTA ? 4 : 1][64];
  __shared__ int tmp[256 + 2];
  // Workgroups go to the 8 chiplets in turn: the runs a step may have and does not must not be every second or fourth of them, so the run is
  // the slowest index; and the heads of a chiplet are neighbours, which read the same keys and queries through its cache.
  const int n_items = gridDim.x, per_xcd = n_items / 8;
  const int item = n_items % 8 == 0 ? (blockIdx.x % 8) * per_xcd + blockIdx.x / 8 : blockIdx.x;
  const int n_blocks = (s.dv + SC_VB * CT - 1) / (SC_VB * CT), h = item / n_blocks;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, grp = lane >> 4;
  const int g = h / (s.H / s.G), n_scal = 2 * s.H + 2 * s.G, dk = s.dk, dv = s.dv;
  const int j = (item - h * n_blocks) * SC_VB * CT + col;  // this lane's value column, and every 16th behind it
  bool live[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) live[c] = j + 16 * c < dv;
  int t0, t_end, slot;
  if (!sr_find_run<256, true>(blockIdx.y, token_slots, s.Tn, tmp, t0, t_end, slot)) return;
  const bf16_t* uk = u + s.k_off + (size_t)g * dk;
  const bf16_t* uq = u + s.q_off + (size_t)g * dk;
  const bf16_t* uv = u + s.v_off + (size_t)h * dv;
  int jc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) jc[c] = live[c] ? j + 16 * c : 0;
  float* sp = state + (size_t)slot * s.slot_stride + (size_t)s.K * s.C + (size_t)h * dk * dv;

  // the state: key channels 16 (wave * NTW + n) + 4 grp + r of column j
  sc_f32x4 S[CT][NTW];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int n = 0; n < NTW; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * (wave * NTW + n) + 4 * grp + r;
        S[c][n][r] = live[c] && i < dk ? sp[(size_t)i * dv + jc[c]] : 0.f;
      }

  // what of the next block is on its way: keys (two neighbouring tokens, eight channels), queries, values, scalars; and, once this block's have been used, this wave's rows
  // of P and T. Raw loads only, under no condition (the last block is written out apart): whatever is computed from them here, or copied for the sake of a branch, would wait for their way
  // through the memory.
  sc_u32x4 nk[KI][2], nq[QI];
  bf16_t nv[CT][4];
  sc_f32x4 P[4], T[4];
  float2 n_e = make_float2(0.f, 0.f);
  float n_w = 0.f, n_rk = 0.f, n_rq = 0.f;
  auto fetch = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < KI; ++n) {
      const int idx = tid + 256 * n, pair = idx & 31, i0 = (idx >> 5) * 8;
#pragma unroll
      for (int e = 0; e < 2; ++e) nk[n][e] = sc_load8<VEC>(uk + (size_t)min(tb + 2 * pair + e, s.Tn - 1) * s.C, i0, dk);
    }
#pragma unroll
    for (int n = 0; n < QI; ++n) {
      const int idx = tid + 256 * n, row = idx / (DKM / 8), i0 = (idx % (DKM / 8)) * 8;
      nq[n] = sc_load8<VEC>(uq + (size_t)min(tb + row, s.Tn - 1) * s.C, i0, dk);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // DELTA: the rows and the column of this lane's part of R; SSD: 16 columns of four tokens per thread, for the transposed copy
      const int t = DELTA ? tb + 16 * wave + 4 * grp + r : tb + (tid >> 4) + 16 * r;
#pragma unroll
      for (int c = 0; c < CT; ++c) nv[c][r] = uv[(size_t)min(t, s.Tn - 1) * s.C + jc[c]];
    }
    const float* sc = scal + (size_t)min(tb + lane, s.Tn - 1) * n_scal;
    n_e = E_in[((size_t)(tb / SC_Q) * s.H + h) * SC_Q + lane];
    if (DELTA) n_w = sc[s.H + h], n_rk = sc[2 * s.H + g], n_rq = sc[2 * s.H + s.G + g];
  };
  auto fetch_tiles = [&](int tb) __attribute__((always_inline)) {
    const size_t tile = ((size_t)(tb / SC_Q) * s.H + h) * 10 + wave * (wave + 1) / 2;
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      const size_t at = ((tile + min(jt, wave)) * 64 + lane) * 4;
      P[jt] = *reinterpret_cast<const sc_f32x4*>(P_in + at);
      if (DELTA) T[jt] = *reinterpret_cast<const sc_f32x4*>(T_in + at);
    }
  };
  auto stage = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < KI; ++n) {
      const int idx = tid + 256 * n, pair = idx & 31, i0 = (idx >> 5) * 8;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (VEC) nk[n][e] = sc_mask8(nk[n][e], i0, dk);
        if (DELTA) *reinterpret_cast<sc_u32x4*>(&s_k[2 * pair + e][i0]) = nk[n][e];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {  // channels i0 + 2 c and i0 + 2 c + 1 of both tokens, transposed
        const uint32_t a = nk[n][0][c], b = nk[n][1][c];
        *reinterpret_cast<uint32_t*>(&s_kt[i0 + 2 * c][2 * pair]) = (a & 0xffffu) | (b << 16);
        *reinterpret_cast<uint32_t*>(&s_kt[i0 + 2 * c + 1][2 * pair]) = (a >> 16) | (b & 0xffff0000u);
      }
    }
#pragma unroll
    for (int n = 0; n < QI; ++n) {
      const int idx = tid + 256 * n, row = idx / (DKM / 8), i0 = (idx % (DKM / 8)) * 8;
      *reinterpret_cast<sc_u32x4*>(&s_q[row][i0]) = VEC ? sc_mask8(nq[n], i0, dk) : nq[n];
    }
    if (!DELTA)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) s_x[16 * c + col][(tid >> 4) + 16 * r] = live[c] ? nv[c][r] : (bf16_t)0;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int n = 0; n < NTW; ++n) {
        float rest[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) rest[r] = S[c][n][r];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const uint32_t lo = float2_to_bf16x2(rest[0], rest[1]), hi = float2_to_bf16x2(rest[2], rest[3]);
          *reinterpret_cast<sc_u32x2*>(&s_S[p][16 * c + col][16 * (wave * NTW + n) + 4 * grp]) = sc_u32x2{lo, hi};
          rest[0] -= __uint_as_float(lo << 16), rest[1] -= __uint_as_float(lo & 0xffff0000u);
          rest[2] -= __uint_as_float(hi << 16), rest[3] -= __uint_as_float(hi & 0xffff0000u);
        }
      }
    if (wave == 0) {
      const bool in = tb + lane >= t0 && tb + lane < t_end;  // the block's tokens of other runs: no weight
      s_ecs[lane] = in ? n_e.x : 0.f;
      s_wend[lane] = in ? n_e.y : 0.f;
      if (DELTA) s_w[lane] = in ? n_w : 0.f, s_rk[lane] = in ? n_rk : 0.f, s_rq[lane] = in ? n_rq : 0.f;
      if (tb + lane == min(t_end, tb + SC_Q) - 1) s_end = n_e.x;  // the decay of the chunk
    }
  };

  const int first = t0 / SC_Q * SC_Q, last = (t_end - 1) / SC_Q * SC_Q;
  fetch(first);
  __builtin_amdgcn_sched_barrier(0);  // in this order, here as in the loop: rows are waited for first
  fetch_tiles(first);
  __builtin_amdgcn_sched_barrier(0);
  auto block = [&](int tb, bool more) __attribute__((always_inline)) {
    float v_now[4];
    stage(tb);
#pragma unroll
    for (int r = 0; r < 4; ++r) v_now[r] = live[0] ? to_float<bf16_t>(nv[0][r]) : 0.f;  // DELTA
    lds_barrier();  // the loads and stores in flight are the thread's own and are not waited for
    if (more) fetch(tb + SC_Q);
    __builtin_amdgcn_sched_barrier(0);

    // rows of the result: tokens 16 wave + .. ; S0^T q and (DELTA) S0^T k, two sums each
    const sc_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    sc_f32x4 oq3[CT][3], ok3[3] = {zero, zero, zero};  // a sum for each part of the state: the longest wait in a block is for products in turn
#pragma unroll
    for (int c = 0; c < CT; ++c) oq3[c][0] = oq3[c][1] = oq3[c][2] = zero;
    // operands of a step of 32 channels and 16 columns, read a step ahead of their products
    sc_u32x4 aq[2], ak[2], sb[2][3];
    auto read = [&](int at) __attribute__((always_inline)) {
      const int ks = at / CT, c = at % CT;
      if (c == 0) {
        aq[ks & 1] = sc_read16(&s_q[16 * wave + col][32 * ks + 8 * grp]);
        if (DELTA) ak[ks & 1] = sc_read16(&s_k[DELTA ? 16 * wave + col : 0][32 * ks + 8 * grp]);
      }
#pragma unroll
      for (int p = 2; p >= 0; --p) sb[at & 1][p] = sc_read16(&s_S[p][16 * c + col][32 * ks + 8 * grp]);
    };
    read(0);
#pragma unroll
    for (int at = 0; at < KS * CT; ++at) {
      const int ks = at / CT, c = at % CT;
      if (at + 1 < KS * CT) read(at + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 2; p >= 0; --p) {
        oq3[c][p] = sc_mfma(aq[ks & 1], sb[at & 1][p], oq3[c][p]);
        if (DELTA) ok3[p] = sc_mfma(ak[ks & 1], sb[at & 1][p], ok3[p]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    sc_f32x4 oq[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) oq[c] = (oq3[c][2] + oq3[c][1]) + oq3[c][0];
    const sc_f32x4 ok = (ok3[2] + ok3[1]) + ok3[0];
    const sc_f32x4 ecs_rows = *reinterpret_cast<const sc_f32x4*>(&s_ecs[16 * wave + 4 * grp]);
    if (DELTA) {
      const sc_f32x4 w_rows = *reinterpret_cast<const sc_f32x4*>(&s_w[16 * wave + 4 * grp]), rk_rows = *reinterpret_cast<const sc_f32x4*>(&s_rk[16 * wave + 4 * grp]);
      const sc_f32x4 rq_rows = *reinterpret_cast<const sc_f32x4*>(&s_rq[16 * wave + 4 * grp]);
      sc_f32x4 R;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        R[r] = w_rows[r] * (v_now[r] - ecs_rows[r] * rk_rows[r] * ok[r]);
        oq[0][r] *= ecs_rows[r] * rq_rows[r];
      }
      s_R[wave][lane] = R;
      lds_barrier();
      sc_f32x4 U4[4] = {zero, zero, zero, zero};
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {
        if (jt > wave) break;
        sc_mfma32(T[jt], s_R[jt][lane], U4);
      }
      s_U[wave][lane] = (U4[0] + U4[1]) + (U4[2] + U4[3]);
      lds_barrier();
      sc_f32x4 U[4];
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) U[jt] = s_U[jt][lane];
      sc_f32x4 PU[4] = {zero, zero, zero, zero};
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {
        if (jt > wave) break;
        sc_mfma32(P[jt], U[jt], PU);
      }
      oq[0] += (PU[0] + PU[1]) + (PU[2] + PU[3]);
      const float dend = s_end;
#pragma unroll
      for (int n = 0; n < NTW; ++n) S[0][n] = S[0][n] * dend;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const sc_f32x4 w0 = *reinterpret_cast<const sc_f32x4*>(&s_wend[32 * half + 4 * grp]), w1 = *reinterpret_cast<const sc_f32x4*>(&s_wend[32 * half + 16 + 4 * grp]);
        float w8[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) w8[e] = U[2 * half][e] * w0[e], w8[4 + e] = U[2 * half + 1][e] * w1[e];
        sc_u32x4 b[3];
        sc_split(w8, b);
#pragma unroll
        for (int n = 0; n < NTW; ++n) {
          const bf16_t* row = s_kt[16 * (wave * NTW + n) + col];
          const sc_u32x4 a = sc_read8x2(row + 32 * half + 4 * grp, row + 32 * half + 16 + 4 * grp);
#pragma unroll
          for (int p = 2; p >= 0; --p) S[0][n] = sc_mfma(a, b[p], S[0][n]);
        }
      }
    } else {
      const float dend = s_end;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        oq[c] = oq[c] * ecs_rows;
#pragma unroll
        for (int n = 0; n < NTW; ++n) S[c][n] = S[c][n] * dend;
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        sc_u32x4 pb[3];
        if (2 * half <= wave) {  // the block's weights, the same for all columns
          const float second = 2 * half + 1 <= wave ? 1.f : 0.f;
          float p8[8];
#pragma unroll
          for (int e = 0; e < 4; ++e) p8[e] = P[2 * half][e], p8[4 + e] = P[2 * half + 1][e] * second;
          sc_split(p8, pb);
        }
        const sc_f32x4 w0 = *reinterpret_cast<const sc_f32x4*>(&s_wend[32 * half + 4 * grp]), w1 = *reinterpret_cast<const sc_f32x4*>(&s_wend[32 * half + 16 + 4 * grp]);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          const int xr = DELTA ? 0 : 16 * c + col;
          const sc_u32x4 x8 = sc_read8x2(&s_x[xr][32 * half + 4 * grp], &s_x[xr][32 * half + 16 + 4 * grp]);
          if (2 * half <= wave)
#pragma unroll
            for (int p = 2; p >= 0; --p) oq[c] = sc_mfma(pb[p], x8, oq[c]);
          float v8[8];
          sc_u32x4 b[3];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float xv = __uint_as_float((e & 1) ? x8[e >> 1] & 0xffff0000u : x8[e >> 1] << 16);
            v8[e] = xv * (e < 4 ? w0[e] : w1[e - 4]);
          }
          sc_split(v8, b);
#pragma unroll
          for (int n = 0; n < NTW; ++n) {
            const bf16_t* row = s_kt[16 * (wave * NTW + n) + col];
            const sc_u32x4 a = sc_read8x2(row + 32 * half + 4 * grp, row + 32 * half + 16 + 4 * grp);
#pragma unroll
            for (int p = 2; p >= 0; --p) S[c][n] = sc_mfma(a, b[p], S[c][n]);
          }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) fetch_tiles(tb + SC_Q);
    // through a buffer of the wave's 16 rows (of at most 65,535 heads of 256 channels, which is all that is let in: 2^30 bytes), beyond whose end nothing is written: a branch round a store makes
    // the next block's loads wait for it
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(o + (size_t)(tb + 16 * wave) * s.H * dv, 0, 16 * s.H * dv * (int)sizeof(float), 0x00027000);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 4 * grp + r, at = tb + 16 * wave + t;
      const bool in = at >= t0 && at < t_end;
#pragma unroll
      for (int c = 0; c < CT; ++c)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(oq[c][r]), rows, in && live[c] ? ((t * s.H + h) * dv + j + 16 * c) * (int)sizeof(float) : 0x7ffffff0, 0, 0);
    }
    lds_barrier();  // the block's tiles have been read by every wave
  };
  int tb = first;
  for (; tb < last; tb += SC_Q) block(tb, true);
  block(last, false);
#pragma unroll
  for (int c = 0; c < CT; ++c)
    if (live[c]) {
#pragma unroll
      for (int n = 0; n < NTW; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * (wave * NTW + n) + 4 * grp + r;
          if (i < dk) sp[(size_t)i * dv + jc[c]] = S[c][n][r];
        }
    }
}

long sr_chunks_workspace(int rule, int Tn, int H) { return (long)((Tn + SC_Q - 1) / SC_Q) * H * (10 * 256 * (rule == SR_DELTA ? 2 : 1) + 2 * SC_Q); }

int sr_chunks_launch(int rule, const bf16_t* u, const float* scal, float* state, const int* token_slots, float* o, float* workspace, int max_runs,
                     const SrShape& s, hipStream_t stream) {
  const int vec = s.C % 8 == 0 && s.dk % 8 == 0 && s.k_off % 8 == 0 && s.q_off % 8 == 0 && ((uintptr_t)u & 15) == 0;
  const int n_blocks = (s.Tn + SC_Q - 1) / SC_Q;
  LEV_REQUIRE(max_runs <= 65535 && n_blocks <= 65535 && ((uintptr_t)workspace & 15) == 0, "state recurrence: too many runs (%d) or tokens (%d)", max_runs, s.Tn);
  float* P = workspace;
  float* T = workspace + (size_t)n_blocks * s.H * 10 * 256;
  float2* E = reinterpret_cast<float2*>(rule == SR_DELTA ? T + (size_t)n_blocks * s.H * 10 * 256 : T);
  const dim3 inner(s.H, n_blocks);
  // columns at once: 64 (or as many as there are) where even so the runs give every CU four workgroups, else 16; of heads of 256 keys, which fill the LDS, 16. A token's
  // sums are the same.
  const long items = (long)max_runs * s.H * ((s.dv + SC_VB - 1) / SC_VB);
  const int tiles = rule == SR_DELTA || s.dk > 128 || items < 4096 ? 1 : s.dv > 32 ? 4 : s.dv > 16 ? 2 : 1;
  const dim3 grid(s.H * ((s.dv + SC_VB * tiles - 1) / (SC_VB * tiles)), max_runs);
#define SC_CHUNK(DKM, RULE, VEC, CT) sc_chunk_kernel<DKM, RULE, VEC, CT><<<grid, 256, 0, stream>>>(u, scal, P, T, E, state, token_slots, o, s)
#define SC_RUN(DKM, RULE, VEC)                                                                                   \
  do {                                                                                                           \
    sc_inner_kernel<DKM, RULE, VEC><<<inner, 256, 0, stream>>>(u, scal, token_slots, P, T, E, s);                 \
    if (lev_check_launch("state recurrence (blocks)")) return -1;                                                \
    if constexpr (RULE == SR_DELTA || DKM > 128) SC_CHUNK(DKM, RULE, VEC, 1);                                    \
    else if (tiles == 4) SC_CHUNK(DKM, RULE, VEC, 4);                                                            \
    else if (tiles == 2) SC_CHUNK(DKM, RULE, VEC, 2);                                                            \
    else SC_CHUNK(DKM, RULE, VEC, 1);                                                                            \
  } while (0)
#define SC_GO(DKM)                                          \
  do {                                                      \
    if (rule == SR_DELTA && vec) SC_RUN(DKM, SR_DELTA, true);   \
    else if (rule == SR_DELTA) SC_RUN(DKM, SR_DELTA, false);    \
    else if (vec) SC_RUN(DKM, SR_SSD, true);                    \
    else SC_RUN(DKM, SR_SSD, false);                            \
  } while (0)
  if (s.dk <= 64) SC_GO(64);
  else if (s.dk <= 128) SC_GO(128);
  else SC_GO(256);
#undef SC_GO
#undef SC_RUN
#undef SC_CHUNK
  return lev_check_launch("state recurrence (chunks)");
}
