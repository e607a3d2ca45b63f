// A feed-forward made of many small experts of which every token uses a few (a mixture of experts), steered from the device:
// no count ever goes to the host, so the launches depend on the number of tokens alone.
//
//   route     per token: scores s of the router's logits z (float32 [T][E]): sigmoid(z) (scoring 0), the softmax of z over all E outputs
//             (1) or z itself (2: the weights are then the softmax over the winners' s alone); the choice goes by c = s + correction;
//             the experts form G equal groups of neighbours, a group's score is the sum of its `group_top` largest c, only the
//             experts of the `keep` best groups can be chosen (the others count as -inf); the `top` largest c win (ties: the
//             lower index); the weights are the winners' s (times 1 / their sum if `renormalize`), in the order of falling c.
//   sort      the T * top (token, choice) pairs by expert: sorted[pos] = pair, pos_of[pair] = pos, and a list of row tiles
//             (expert, first position, rows <= tile_rows) that covers every expert's stretch; n_tiles on the device.
//             tile_rows is 16, or 128 for steps with many rows an expert.
//   linear    for every tile: out[pos][o] = sum_k w[expert][o][k] a[row(pos)][k], row(pos) = the pair's token (gather) or pos
//             itself, through the activation (none for the second product); with glu the expert's matrix is [gate ; up] (2F rows) and
//             out[pos][f] = act(gate_f) * up_f.
//             bfloat16 on the matrix cores (16x16x32): few tiles of 16 rows with K split over a workgroup's waves, many with a
//             wave per tile, tiles of 128 rows with both operands staged through LDS; float32 in plain arithmetic. Workgroups
//             beyond n_tiles return at once.
//             with limit > 0 the gate sum is capped at limit and the up sum clamped to +-limit first, and up_shift is added to
//             the up sum: act(min(gate, limit)) * (clamp(up) + up_shift).
//   combine   y[t] = sum_c weight[t][c] * out[pos_of[t * top + c]], c in order, float32; with `accumulate` added to what y holds.
//   identity  router outputs n_real .. E-1 may stand for experts without weights whose result is their input: sort gives their pairs
//             places but no tiles (the products never see them), and combine takes the token's own row of `identity_in` for them.
#include "moe.h"

#define MOE_TM 16          // rows of a matrix-core row tile, and of a tile of the list in steps of few tokens
#define MOE_MAX_E 1024     // experts (at most 32 a lane)
#define MOE_MAX_TOP 32

// ---- route ------------------------------------------------------------------------------------
// One wave routes one token; s_s, c_s (and g_s with groups) are E (G) numbers of its own in LDS. Every wave of
// the workgroup passes the same barriers. `extra`: a further choice behind the `top` ones, expert E with weight 1 (an expert that runs for
// every token). store: the wave's token is one of the step's.
struct MoeRouteArgs {
  const float* z;
  long z_stride;
  const float* correction;
  int E, G, keep, group_top, top, renormalize, scoring, extra;
  int* chosen;
  float* weights;
};
// chosen_s: a copy of the choices in LDS, for a sort in the same workgroup
__device__ __forceinline__ void moe_route_token(const MoeRouteArgs& a, int t, bool store, float* s_s, float* c_s, float* g_s, int* chosen_s) {
  const int lane = threadIdx.x & 63, E = a.E, G = a.G, top = a.top;
  const int per = E / G;
  const float* zt = a.z + (size_t)t * a.z_stride;
  float z_max = 0.f, inv_sum = 1.0f;
  if (a.scoring == 1) {
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, zt[e]);
    z_max = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < E; e += 64) sum += expf(zt[e] - z_max);
    inv_sum = 1.0f / wave_sum(sum);
  }
  for (int e = lane; e < E; e += 64) {
    const float ze = zt[e];
    const float s = a.scoring == 2 ? ze : a.scoring == 1 ? expf(ze - z_max) * inv_sum : 1.0f / (1.0f + expf(-ze));
    s_s[e] = s;
    c_s[e] = s + (a.correction ? a.correction[e] : 0.f);
  }
  __syncthreads();
  if (G > 1) {
    for (int g = lane; g < G; g += 64) {  // the sum of the group's largest choice scores
      float sum = 0.f;
      float last = INFINITY;
      int last_i = -1;
      for (int n = 0; n < min(a.group_top, per); ++n) {  // the next largest: below (last, last_i) in the order (value falling, index rising)
        float best = -INFINITY;
        int best_i = -1;
        for (int i = 0; i < per; ++i) {
          const float c = c_s[g * per + i];
          const bool after = c < last || (c == last && i > last_i);
          if (after && (best_i < 0 || c > best)) best = c, best_i = i;
        }
        sum += best;
        last = best, last_i = best_i;
      }
      g_s[g] = sum;
    }
    __syncthreads();
    for (int e = lane; e < E; e += 64) {
      const int g = e / per;
      const float mine = g_s[g];
      int ahead = 0;  // groups that come before this one
      for (int o = 0; o < G; ++o) ahead += (g_s[o] > mine || (g_s[o] == mine && o < g)) ? 1 : 0;
      if (ahead >= a.keep) c_s[e] = -INFINITY;
    }
    __syncthreads();
  }
  // the next largest, `top` times: every lane looks through its own experts (e % 64 == lane), the lanes compare; lane n keeps the n-th
  float wsum = 0.f;
  int mine = 0;
  uint32_t taken = 0;  // of this lane's experts: bit e / 64
  for (int n = 0; n < top; ++n) {
    float best = -INFINITY;
    int best_e = 0x7fffffff;
    for (int e = lane, i = 0; e < E; e += 64, ++i) {
      const float c = c_s[e];
      if (!(taken >> i & 1u) && (c > best || (c == best && e < best_e))) best = c, best_e = e;
    }
    // the largest, and of its owners' experts the first: those of the lowest 64 before others, then the lowest lane's
    const float largest = wave_max(best);
    const bool owner = best == largest && best_e < E;
    unsigned long long owners = 0;
    int block = 0;
    for (; block * 64 < E && owners == 0; ++block) owners = __ballot(owner && best_e >> 6 == block);
    best_e = owners != 0 ? (block - 1) * 64 + __ffsll(owners) - 1 : E;
    if (best_e >= E) best_e = 0;  // nothing left to choose from (a configuration that keeps fewer experts than it uses)
    if ((best_e & 63) == lane) taken |= 1u << (best_e >> 6);
    if (lane == n) mine = best_e;
    wsum += s_s[best_e];
  }
  const size_t at = (size_t)t * (top + a.extra);
  float weight = s_s[mine];
  if (a.scoring == 2) {
    const float mx = wave_max(lane < top ? weight : -INFINITY);
    weight = lane < top ? expf(weight - mx) : 0.f;
    weight /= wave_sum(weight);
  } else if (a.renormalize) {
    weight /= wsum;
  }
  if (!store) return;
  if (lane < top) {
    a.chosen[at + lane] = mine;
    if (chosen_s != nullptr) chosen_s[at + lane] = mine;
    a.weights[at + lane] = weight;
  } else if (lane == top && a.extra) {
    a.chosen[at + top] = E;
    if (chosen_s != nullptr) chosen_s[at + top] = E;
    a.weights[at + top] = 1.0f;
  }
}

__global__ void __launch_bounds__(64)
moe_route_kernel(const MoeRouteArgs a) {
  __shared__ float s_s[MOE_MAX_E], c_s[MOE_MAX_E], g_s[MOE_MAX_E];
  moe_route_token(a, blockIdx.x, true, s_s, c_s, g_s, nullptr);
}

// ---- sort --------------------------------------------------------------------------------------
// One workgroup. meta: [0] = n_tiles; tiles: (expert, first position, rows) per tile. The order of an expert's pairs among
// themselves is whatever the atomic counters give: a pair's results do not depend on its place in a tile.
#define MOE_SORT_NT 1024
struct MoeSortLds {
  int count[MOE_MAX_E + 1], start[MOE_MAX_E + 1], tile_start[MOE_MAX_E + 2], cursor[MOE_MAX_E + 1];
};
__device__ __forceinline__ void moe_sort_pairs(MoeSortLds& l, const int* chosen, int P, int E, int n_real, int tile_rows, int* __restrict__ sorted,
                                               int* __restrict__ pos_of, int* __restrict__ tiles, int* __restrict__ meta) {
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += MOE_SORT_NT) l.count[e] = 0, l.cursor[e] = 0;
  lds_barrier();
  for (int p = tid; p < P; p += MOE_SORT_NT) atomicAdd(&l.count[chosen[p]], 1);
  lds_barrier();
  if (tid < 64) {  // running sums over the experts: each lane a stretch of neighbours, then across the lanes
    const int c = (E + 63) / 64, lo = min(E, tid * c), hi = min(E, lo + c);
    int n = 0, nt = 0;
    for (int e = lo; e < hi; ++e) {
      n += l.count[e];
      if (e < n_real) nt += (l.count[e] + tile_rows - 1) / tile_rows;  // experts without weights get places and no tiles
    }
    int at = n, tile = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int a = __shfl_up(at, o, 64), b = __shfl_up(tile, o, 64);
      if (tid >= o) at += a, tile += b;
    }
    if (tid == 63) l.tile_start[E] = tile, meta[0] = tile;
    at -= n, tile -= nt;
    for (int e = lo; e < hi; ++e) {
      l.start[e] = at;
      l.tile_start[e] = tile;
      at += l.count[e];
      if (e < n_real) tile += (l.count[e] + tile_rows - 1) / tile_rows;
    }
  }
  lds_barrier();
  for (int p = tid; p < P; p += MOE_SORT_NT) {
    const int e = chosen[p];
    const int pos = l.start[e] + atomicAdd(&l.cursor[e], 1);
    sorted[pos] = p;
    pos_of[p] = pos;
  }
  for (int e = tid; e < E; e += MOE_SORT_NT) {
    const int n = l.tile_start[e + 1] - l.tile_start[e];
    for (int i = 0; i < n; ++i) {
      int* tl = tiles + 3 * (size_t)(l.tile_start[e] + i);
      tl[0] = e;
      tl[1] = l.start[e] + i * tile_rows;
      tl[2] = min(tile_rows, l.count[e] - i * tile_rows);
    }
  }
}

__global__ void __launch_bounds__(MOE_SORT_NT)
moe_sort_kernel(const int* __restrict__ chosen, int P, int E, int n_real, int tile_rows, int* __restrict__ sorted, int* __restrict__ pos_of,
                int* __restrict__ tiles, int* __restrict__ meta) {
  __shared__ MoeSortLds l;
  moe_sort_pairs(l, chosen, P, E, n_real, tile_rows, sorted, pos_of, tiles, meta);
}

// Both for a step of few tokens, in one workgroup: a wave routes a token, then all of them sort.
#define MOE_SMALL_T (MOE_SORT_NT / 64)
#define MOE_SMALL_E 256
__global__ void __launch_bounds__(MOE_SORT_NT)
moe_route_sort_kernel(const MoeRouteArgs a, int T, int n_real, int tile_rows, int* __restrict__ sorted, int* __restrict__ pos_of, int* __restrict__ tiles,
                      int* __restrict__ meta) {
  __shared__ MoeSortLds l;
  __shared__ float s_s[MOE_SMALL_T][MOE_SMALL_E], c_s[MOE_SMALL_T][MOE_SMALL_E];
  __shared__ int chosen_s[MOE_SMALL_T * (MOE_MAX_TOP + 1)];
  const int wave = threadIdx.x >> 6;
  // the groups' scores take the place of the sort's counters, which nobody needs before the routing is done
  float* g_s = reinterpret_cast<float*>(l.count) + (size_t)wave * MOE_SMALL_E / 4;
  moe_route_token(a, min(wave, T - 1), wave < T, s_s[wave], c_s[wave], g_s, chosen_s);
  lds_barrier();  // (the choices in global memory are on their way: the sort reads the copy)
  moe_sort_pairs(l, chosen_s, T * (a.top + a.extra), a.E + a.extra, n_real, tile_rows, sorted, pos_of, tiles, meta);
}

static int moe_route_check(const MoeRouteArgs& a, int T) {
  LEV_REQUIRE(a.scoring >= 0 && a.scoring <= 2, "experts: unknown scoring %d", a.scoring);
  LEV_REQUIRE(T >= 0 && a.E > 0 && a.E <= MOE_MAX_E, "experts: %d experts (at most %d)", a.E, MOE_MAX_E);
  LEV_REQUIRE(a.G > 0 && a.E % a.G == 0 && a.keep > 0 && a.keep <= a.G && a.group_top > 0, "experts: %d groups of %d experts, %d kept", a.G, a.E, a.keep);
  LEV_REQUIRE(a.top > 0 && a.top <= MOE_MAX_TOP && a.top <= a.keep * (a.E / a.G), "experts: %d experts a token out of %d that can be chosen (at most %d)", a.top,
              a.keep * (a.E / a.G), MOE_MAX_TOP);
  LEV_REQUIRE(a.extra == 0 || a.extra == 1, "experts: one further choice at most");
  LEV_REQUIRE(a.z && a.chosen && a.weights && a.z_stride >= a.E, "experts: a tensor is missing");
  return 0;
}

extern "C" int lev_moe_route(const float* z, long z_stride, const float* correction, int T, int E, int G, int keep, int group_top, int top,
                             int renormalize, int scoring, int extra, int* chosen, float* weights, hipStream_t stream) {
  const MoeRouteArgs a{z, z_stride, correction, E, G, keep, group_top, top, renormalize, scoring, extra, chosen, weights};
  if (moe_route_check(a, T)) return -1;
  if (T == 0) return 0;
  moe_route_kernel<<<T, 64, 0, stream>>>(a);
  return lev_check_launch("moe_route");
}

extern "C" int lev_moe_max_tiles(int P, int E, int tile_rows) { return P / tile_rows + E + 1; }

static int moe_sort_check(const void* chosen, int P, int E, int n_real, int tile_rows, const void* sorted, const void* pos_of, const void* tiles, const void* meta) {
  LEV_REQUIRE(P >= 0 && E > 0 && E <= MOE_MAX_E + 1, "experts: %d experts (at most %d)", E, MOE_MAX_E + 1);
  LEV_REQUIRE(tile_rows == MOE_TM || tile_rows == MOE_BIG, "experts: tiles of %d rows (%d or %d)", tile_rows, MOE_TM, MOE_BIG);
  LEV_REQUIRE(chosen && sorted && pos_of && tiles && meta, "experts: a tensor is missing");
  LEV_REQUIRE(n_real >= 0 && n_real <= E, "experts: %d of %d experts have weights", n_real, E);
  return 0;
}

extern "C" int lev_moe_sort(const int* chosen, int P, int E, int n_real, int tile_rows, int* sorted, int* pos_of, int* tiles, int* meta, hipStream_t stream) {
  if (moe_sort_check(chosen, P, E, n_real, tile_rows, sorted, pos_of, tiles, meta)) return -1;
  moe_sort_kernel<<<1, MOE_SORT_NT, 0, stream>>>(chosen, P, E, n_real, tile_rows, sorted, pos_of, tiles, meta);
  return lev_check_launch("moe_sort");
}

// 1: not for these sizes (nothing has been launched); else as the two above, one after the other
extern "C" int lev_moe_route_sort(const float* z, long z_stride, const float* correction, int T, int E, int G, int keep, int group_top, int top,
                                  int renormalize, int scoring, int extra, int* chosen, float* weights, int n_real, int tile_rows, int* sorted, int* pos_of,
                                  int* tiles, int* meta, hipStream_t stream) {
  const MoeRouteArgs a{z, z_stride, correction, E, G, keep, group_top, top, renormalize, scoring, extra, chosen, weights};
  if (moe_route_check(a, T) || moe_sort_check(chosen, T * (top + extra), E + extra, n_real, tile_rows, sorted, pos_of, tiles, meta)) return -1;
  if (T == 0 || T > MOE_SMALL_T || E > MOE_SMALL_E || G > MOE_SMALL_E / 4) return 1;
  moe_route_sort_kernel<<<1, MOE_SORT_NT, 0, stream>>>(a, T, n_real, tile_rows, sorted, pos_of, tiles, meta);
  return lev_check_launch("moe_route_sort");
}

// ---- the experts' products ------------------------------------------------------------------------
// float32: a thread per (row of the tile, output); 16 x 16 a workgroup
template <typename T, typename TO>
__global__ void __launch_bounds__(256)
moe_linear_plain_kernel(const T* __restrict__ a, long a_stride, const T* __restrict__ w, TO* __restrict__ out, long o_stride,
                        const int* __restrict__ tiles, const int* __restrict__ meta, const int* __restrict__ sorted, int top, int gather,
                        int K, int N, int F, int glu, int act, float limit, float up_shift) {
  const int tile = blockIdx.x;
  if (tile >= meta[0]) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
  const int o = blockIdx.y * 16 + (threadIdx.x & 15);
  if (o >= F) return;
  for (int rr = threadIdx.x >> 4; rr < rows; rr += 16) {  // a tile may have more rows than the workgroup has row threads
    const int pos = first + rr;
    const T* ar = a + (size_t)(gather ? sorted[pos] / top : pos) * a_stride;
    const T* wg = w + ((size_t)e * N + o) * K;
    float acc = 0.f, acc_up = 0.f;
    for (int kk = 0; kk < K; ++kk) acc = fmaf(to_float<T>(wg[kk]), to_float<T>(ar[kk]), acc);
    if (glu) {
      const T* wu = wg + (size_t)F * K;
      for (int kk = 0; kk < K; ++kk) acc_up = fmaf(to_float<T>(wu[kk]), to_float<T>(ar[kk]), acc_up);
      acc = moe_act(acc, acc_up, act, limit, up_shift);
    } else {
      acc = lev_activate(acc, act);
    }
    out[(size_t)pos * o_stride + o] = from_float<TO>(acc);
  }
}

typedef __attribute__((ext_vector_type(8))) __bf16 moe_bf16x8;
typedef __attribute__((ext_vector_type(4))) float moe_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t moe_u32x4;
__device__ __forceinline__ moe_bf16x8 moe_as_bf16x8(moe_u32x4 v) {
  union { moe_u32x4 u; moe_bf16x8 b; } c;
  c.u = v;
  return c.b;
}

template <typename TO>
__device__ __forceinline__ void moe_store4(TO* p, const float (&v)[4], int n, bool vec);
template <>
__device__ __forceinline__ void moe_store4<float>(float* p, const float (&v)[4], int n, bool vec) {
  if (vec && n >= 4) *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  else
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < n) p[r] = v[r];
}
template <>
__device__ __forceinline__ void moe_store4<bf16_t>(bf16_t* p, const float (&v)[4], int n, bool vec) {
  if (vec && n >= 4) *reinterpret_cast<uint2*>(p) = make_uint2(float2_to_bf16x2(v[0], v[1]), float2_to_bf16x2(v[2], v[3]));
  else
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < n) p[r] = float_to_bf16(v[r]);
}

// Tiles of 16 rows (steps of few tokens): the products are bound by reading the chosen experts' weights. A workgroup of KS waves owns one
// tile and 16 outputs (with glu their gate and up rows; the transposed product out^T = w a^T leaves each lane with four neighbouring
// outputs of a row); its waves split K in pairs of k-steps (64 k), U pairs on their way at once, and the partial sums are added through LDS
// in wave order. Weights and rows are read as whole 128-byte lines (8 rows an instruction) and turned into operands in an LDS area of the
// wave's own: read in operand layout, 64 bytes of each of 16 rows, a load costs the vector cache a look-up for every lane, which bounds
// such a kernel at 16 bytes a cycle and CU. 33 experts of 2048 x 2048, 5 a token, microseconds of the up and of the gated product, before
// (operand layout) and now: 1 token 16.6 and 25.5 / 12.6 and 19.8, 8 tokens (20 tiles, 168 MB) 40.7 and 70.5 / 32.6 and 60.3, 64 tokens
// 81.7 and 136.8 / 54.8 and 99.2; 128 experts of 2048 to 768, 8 a token, 8 tokens: 65 and 127 / 30 and 56. Below K = 2,048 four waves are
// enough: 1024 x 1024, 8 tokens 11.4 against 12.2 of eight, 768 to 2,048, 32 tokens 62 / 80; at 2,048 eight are: 1 token 12.6 / 13.8.
#define MOE_SLOTS 72  // 16-byte slots of one staged instruction: 8 rows x (8 chunks + 1 of padding)
template <typename TO, bool GLU, int KS, int U>
__global__ void __launch_bounds__(64 * KS, KS == 4 ? 2 : 1)
moe_linear_few_kernel(const MoeLinearArgs p) {
  constexpr int G = GLU ? 2 : 1;
  __shared__ moe_f32x4 part[KS][G][64];
  __shared__ moe_u32x4 stage[KS][2 * MOE_SLOTS];
  const int tile = blockIdx.x;
  if (tile >= p.meta[0]) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4, lr = lane >> 3, lc = lane & 7;
  const int o0 = blockIdx.y * 16, K = p.K, F = p.F;
  const int e = p.tiles[3 * tile], first = p.tiles[3 * tile + 1], rows = p.tiles[3 * tile + 2];
  const bf16_t *ar[2], *wr[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int pos = first + min(8 * i + lr, rows - 1);  // rows beyond the tile: read again, never stored
    ar[i] = p.a + (size_t)(p.gather ? p.sorted[pos] / p.top : pos) * p.a_stride;
    wr[i] = p.w + (size_t)e * p.N * K + (size_t)min(o0 + 8 * i + lr, F - 1) * K;
  }
  moe_u32x4* mine = stage[wave];
  const int st = lr * 9 + lc, ld = (col >> 3) * MOE_SLOTS + (col & 7) * 9 + g;
  moe_f32x4 acc[G], acc_hi[G];  // a pair's first and second k-steps: 8 or 16 partial sums a workgroup, so that none is a long chain of roundings
#pragma unroll
  for (int x = 0; x < G; ++x) acc[x] = acc_hi[x] = moe_f32x4{0.f, 0.f, 0.f, 0.f};
  const int pairs = (K + 63) / 64;
  for (int p0 = wave; p0 < pairs; p0 += KS * U) {
    moe_u32x4 av[U][2], wv[U][G][2];
    uint32_t keep[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (p0 + u * KS) * 64 + lc * 8, kc = min(k, K - 8);  // loads stand under no condition; a chunk beyond K counts as zeros
      keep[u] = k < K ? 0xffffffffu : 0u;
#pragma unroll
      for (int x = 0; x < G; ++x)
#pragma unroll
        for (int i = 0; i < 2; ++i) wv[u][x][i] = *reinterpret_cast<const moe_u32x4*>(wr[i] + (size_t)x * F * K + kc);
#pragma unroll
      for (int i = 0; i < 2; ++i) av[u][i] = *reinterpret_cast<const moe_u32x4*>(ar[i] + kc);
    }
    __builtin_amdgcn_sched_barrier(0);  // all of them are on their way before the first is waited for
#pragma unroll
    for (int u = 0; u < U; ++u) {  // LDS executes a wave's instructions in order: the area is used again and again without a barrier
      const moe_u32x4 mk = moe_u32x4{keep[u], keep[u], keep[u], keep[u]};
      mine[st] = av[u][0] & mk, mine[MOE_SLOTS + st] = av[u][1] & mk;
      const moe_u32x4 a_lo = mine[ld], a_hi = mine[ld + 4];
#pragma unroll
      for (int x = 0; x < G; ++x) {
        mine[st] = wv[u][x][0] & mk, mine[MOE_SLOTS + st] = wv[u][x][1] & mk;
        const moe_u32x4 w_lo = mine[ld], w_hi = mine[ld + 4];
        acc[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(moe_as_bf16x8(w_lo), moe_as_bf16x8(a_lo), acc[x], 0, 0, 0);
        acc_hi[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(moe_as_bf16x8(w_hi), moe_as_bf16x8(a_hi), acc_hi[x], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int x = 0; x < G; ++x) part[wave][x][lane] = acc[x] += acc_hi[x];
  __syncthreads();
  const int o = o0 + 4 * g;
  if (wave != 0 || col >= rows || o >= F) return;
#pragma unroll
  for (int x = 0; x < G; ++x)
#pragma unroll
    for (int q = 1; q < KS; ++q) acc[x] += part[q][x][lane];
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = GLU ? moe_act(acc[0][r], acc[G - 1][r], p.act, p.limit, p.up_shift) : lev_activate(acc[0][r], p.act);
  moe_store4<TO>(static_cast<TO*>(p.out) + (size_t)(first + col) * p.o_stride + o, v, F - o, p.vec);
}

// Tiles of 128 rows (prompts, large batches) of sums that are no multiple of 128 or below 384, and of fewer units than fill the CUs (moe_ring.hip has the others): a workgroup of four waves owns 128 rows and BN weight rows (with glu: BN / 2 outputs' gate
// rows and the same outputs' up rows), a wave 64 x BN / 2 of them in 32x32x16 products (the transposed product out^T = w a^T: a lane ends
// with four neighbouring outputs of a row). K goes by in steps of 64, the step after next on its way in registers, two buffers in LDS,
// one barrier a step that waits for LDS only; loads, LDS writes and fragment reads are issued one by one between the products. Rows
// beyond the tile are read again and never stored. The workgroups of a tile and of its neighbours in the list (an expert's rows, its
// weights) follow each other on one of the eight chiplets (workgroups are dealt to them in turn).
// What bounds it: the read of the weights with up to about 128 rows an expert (4.7 - 5.0 TB/s), else what the CUs pull through L2 (32 KB a
// step and workgroup at 15 TB/s) and the last round of tiles. The outputs leave through LDS as whole lines, after one decision on the activation
// for all of them: stored from the products' registers, 8 or 16 bytes of each of 32 rows, with the decision at every value, the last 64 KB of a
// workgroup cost 15 us a round: 2048 outputs of 2048 (bfloat16 / 32-bit, microseconds), 32 experts of 256 rows 126 / 137 -> 110 / 116,
// 4 of 2,048 93 / 105 -> 78 / 80. Where the weights' read is the bound the workgroups begin at places of
// their own along K: rows a power of two apart lie in the same channels of the memory, and workgroups that walk together ask those alone: 32
// experts of 128 rows 97 -> 65 us, of 40 72 -> 56, of 160 160 -> 114, 64 of 30 140 -> 103. With many rounds or rows they drift apart by themselves (8 of 4,096
// rows 190 in order, 197 spread; 64 of 160 with gates, 512 workgroups a chiplet, 416 / 463), so: up to one and a half rounds of a chiplet's 64 workgroups,
// counted with as many tiles as the step's sizes allow, and up to three where that is twice what most routings make, at 128 rows an expert on average
// or fewer. How the routing dealt the tokens out has no say: a token's sums would be in another order when others of the step chose otherwise. Over 780
// shapes 2 are slower by 4 - 5 % than with the actual number of tiles (128 experts of 1024 x 1024 with 60 rows), 50 faster by 4 % and up to 40 %.
// Measured and not kept: tiles of 256 rows by 8 waves (32 of 256 rows 107, of 254 drawn ones 153 against 136),
// workgroups that stay and fetch the next tile's first steps ahead of the last outputs (spills; 4 of 2,048 rows 82 - 107), weights three
// steps ahead (no gain), chiplets' shares by cost (of 40 rows 77 against 55).
#define MOE_BN 128
#define MOE_BIG_K 64
#define MOE_BIG_LD (MOE_BIG_K + 8)
#define MOE_BIG_SPREAD 96  // a chiplet's workgroups of one and a half rounds
#define MOE_BIG_LDS(BN) (2 * (MOE_BIG + (BN)) * MOE_BIG_LD * (int)sizeof(bf16_t))
typedef __attribute__((ext_vector_type(16))) float moe_f32x16;
// the sums become outputs in place; with glu the first half of a row's registers takes them
template <int ACT, bool GLU, int TI, int TJ>
__device__ __forceinline__ void moe_big_activate(moe_f32x16 (&acc)[TI][TJ], const MoeLinearArgs& p) {
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < (GLU ? TJ / 2 : TJ); ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = GLU ? moe_act(acc[i][j][r], acc[i][(j + TJ / 2) % TJ][r], ACT, p.limit, p.up_shift) : lev_activate(acc[i][j][r], ACT);
}

// eight (bfloat16) or four (float32) neighbouring outputs of a row; `vec`: 1: rows allow half of such a store, 2: a whole one
__device__ __forceinline__ void moe_big_store(float* to, const moe_u32x4& v, int left, int vec) {
  if (vec && left >= 4) *reinterpret_cast<moe_u32x4*>(to) = v;
  else
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < left) to[r] = __uint_as_float(v[r]);
}
__device__ __forceinline__ void moe_big_store(bf16_t* to, const moe_u32x4& v, int left, int vec) {
  if (vec == 2 && left >= 8) *reinterpret_cast<moe_u32x4*>(to) = v;
  else if (vec && left >= 8) reinterpret_cast<uint2*>(to)[0] = make_uint2(v[0], v[1]), reinterpret_cast<uint2*>(to)[1] = make_uint2(v[2], v[3]);
  else
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (r < left) to[r] = (bf16_t)(v[r / 2] >> (r % 2 * 16));
}

// BM: 128, or 64 for a tile whose rows fit that
template <typename TO, bool GLU, int BN, int BM>
__device__ __forceinline__ void moe_big_tile(const MoeLinearArgs& p, unsigned char* moe_smem, int e, int first, int rows, int ycol) {
  constexpr int LD = MOE_BIG_LD, WM = BM / 2, WN = BN / 2, TI = WM / 32, TJ = WN / 32;
  constexpr int CA = BM * (MOE_BIG_K / 8) / 256, CW = BN * (MOE_BIG_K / 8) / 256;  // 16-byte chunks a thread fetches a step
  constexpr int OUT = GLU ? BN / 2 : BN;  // outputs of a workgroup
  const int K = p.K, N = p.N, F = p.F;
  bf16_t* sa = reinterpret_cast<bf16_t*>(moe_smem);  // [2][BM][LD]
  bf16_t* sw = sa + 2 * BM * LD;                     // [2][BN][LD]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
  const int o0 = ycol * OUT;
  const int kc = (tid & 7) * 8;
  const bf16_t* we = p.w + (size_t)e * N * K;
  const bf16_t *pa[CA], *pw[CW];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int pos = first + min((tid + 256 * i) >> 3, rows - 1);
    pa[i] = p.a + (size_t)(p.gather ? p.sorted[pos] / p.top : pos) * p.a_stride;
  }
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int r = (tid + 256 * i) >> 3, q = r % WN;  // with glu a wave's weight rows are its outputs' gate rows, then their up rows
    const int o = GLU ? min(o0 + r / WN * (WN / 2) + q % (WN / 2), F - 1) + (q >= WN / 2 ? F : 0) : min(o0 + r, F - 1);
    pw[i] = we + (size_t)o * K;
  }
  // the steps in the order they are taken: a partial one (K % 64 != 0) first, so that the loop needs no masks
  const int tail = K % MOE_BIG_K, steps = (K + MOE_BIG_K - 1) / MOE_BIG_K, shift = tail ? 1 : 0;
  const int turn = p.spread && !tail ? ycol * 5 % steps : 0;  // whole steps then begin at a place of the workgroup's own
  auto k_of = [&](int t) {  // t >= 1; beyond the last: loaded again, not used
    const unsigned i = max(min(t, steps - 1) - shift, 0) + turn;
    return (int)min(i, i - (unsigned)steps) * MOE_BIG_K;  // i, or i - steps if that is not below 0
  };
  moe_u32x4 ra[2][CA], rw[2][CW];
  auto fetch_one = [&](int set, int k, int i) {
    if (i < CA) ra[set][i] = *reinterpret_cast<const moe_u32x4*>(pa[i] + k);
    else rw[set][i - CA] = *reinterpret_cast<const moe_u32x4*>(pw[i - CA] + k);
  };
  bf16_t* a_st = sa + (tid >> 3) * LD + kc;
  bf16_t* w_st = sw + (tid >> 3) * LD + kc;
  auto stage_one = [&](int set, int buf, int i) {
    if (i < CA) *reinterpret_cast<moe_u32x4*>(a_st + (buf * BM + i * 32) * LD) = ra[set][i];
    else *reinterpret_cast<moe_u32x4*>(w_st + (buf * BN + (i - CA) * 32) * LD) = rw[set][i - CA];
  };
  moe_f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  {
    const int k0 = tail ? K - tail : turn * MOE_BIG_K, k = min(k0 + kc, K - 8);
    const bool in = k0 + kc < K;
#pragma unroll
    for (int i = 0; i < CA + CW; ++i) fetch_one(0, k, i);
#pragma unroll
    for (int i = 0; i < CA; ++i) if (!in) ra[0][i] = moe_u32x4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < CW; ++i) if (!in) rw[0][i] = moe_u32x4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < CA + CW; ++i) stage_one(0, 0, i);
    const int k1 = min(k_of(1) + kc, K - 8);
#pragma unroll
    for (int i = 0; i < CA + CW; ++i) fetch_one(1, k1, i);
  }
  lds_barrier();
  constexpr int KS = MOE_BIG_K / 16, NM = TI * TJ, NR = TI + TJ, PW = (CA + CW + KS - 2) / (KS - 1);
  const bf16_t* a_rd = sa + (wm * WM + (lane & 31)) * LD + (lane >> 5) * 8;
  const bf16_t* w_rd = sw + (wn * WN + (lane & 31)) * LD + (lane >> 5) * 8;
  moe_u32x4 af[2][TI], wf[2][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i) af[0][i] = *reinterpret_cast<const moe_u32x4*>(a_rd + i * 32 * LD);
#pragma unroll
  for (int j = 0; j < TJ; ++j) wf[0][j] = *reinterpret_cast<const moe_u32x4*>(w_rd + j * 32 * LD);
  // step t: register set `cur` (step t + 1) goes to the other buffer, the other set receives step t + 2; the last products cover the first
  // fragment reads of step t + 1 behind the barrier
  auto step = [&](int t, int cur) {
    const int buf = t & 1, k = min(k_of(t + 2) + kc, K - 8);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int c = ks & 1, nx = c ^ 1, from = ks + 1 < KS ? buf : buf ^ 1, at = ks + 1 < KS ? (ks + 1) * 16 : 0;
      if (ks + 1 == KS) lds_barrier();
#pragma unroll
      for (int i = 0; i < TI; ++i) af[nx][i] = *reinterpret_cast<const moe_u32x4*>(a_rd + (from * BM + i * 32) * LD + at);
#pragma unroll
      for (int j = 0; j < TJ; ++j) wf[nx][j] = *reinterpret_cast<const moe_u32x4*>(w_rd + (from * BN + j * 32) * LD + at);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(moe_as_bf16x8(wf[c][j]), moe_as_bf16x8(af[c][i]), acc[i][j], 0, 0, 0);
      if (ks + 1 < KS) {
#pragma unroll
        for (int q = 0; q < PW; ++q)
          if (ks * PW + q < CA + CW) stage_one(cur, buf ^ 1, ks * PW + q);
#pragma unroll
        for (int q = 0; q < PW; ++q)
          if (ks * PW + q < CA + CW) fetch_one(cur ^ 1, k, ks * PW + q);
      }
      constexpr int others = NR + 2 * PW;
#pragma unroll
      for (int m = 0; m < NM; ++m) {  // the order of issue: a product, then at most a few of the others
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        const int n = ks + 1 < KS ? others : NR, lo = m * n / NM, hi = (m + 1) * n / NM;
#pragma unroll
        for (int o = lo; o < hi; ++o) {
          if (o < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          else if (o < NR + PW) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
          else __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
      }
    }
  };
  int t = 0;
  for (; t + 1 < steps; t += 2) {
    step(t, 1);
    step(t + 1, 0);
  }
  if (t < steps) step(t, 1);
  lds_barrier();  // nobody reads the buffers any more
  switch (p.act) {  // one decision for all outputs
    case LEV_ACT_GELU_TANH: moe_big_activate<LEV_ACT_GELU_TANH, GLU, TI, TJ>(acc, p); break;
    case LEV_ACT_GELU_ERF: moe_big_activate<LEV_ACT_GELU_ERF, GLU, TI, TJ>(acc, p); break;
    case LEV_ACT_RELU: moe_big_activate<LEV_ACT_RELU, GLU, TI, TJ>(acc, p); break;
    case LEV_ACT_SILU: moe_big_activate<LEV_ACT_SILU, GLU, TI, TJ>(acc, p); break;
    case LEV_ACT_QUICK_GELU: moe_big_activate<LEV_ACT_QUICK_GELU, GLU, TI, TJ>(acc, p); break;
    case LEV_ACT_TANH: moe_big_activate<LEV_ACT_TANH, GLU, TI, TJ>(acc, p); break;
    case LEV_ACT_RELU_SQUARED: moe_big_activate<LEV_ACT_RELU_SQUARED, GLU, TI, TJ>(acc, p); break;
    default: moe_big_activate<LEV_ACT_NONE, GLU, TI, TJ>(acc, p);
  }
  // Whole lines go out: 32 rows and 128 bytes of each (64 where a wave has no more) turn round in a part of the LDS that is the wave's own.
  // Register r of a 32 x 32 tile: output 8 (r / 4) + 4 (lane / 32) + r % 4, row lane % 32
  constexpr bool F32 = sizeof(TO) == 4;
  constexpr int TO_J = GLU ? TJ / 2 : TJ, JB = F32 ? 1 : TO_J, PER = 16 / (int)sizeof(TO), WIDTH = 32 * JB, LR = WIDTH / PER;  // lanes a row
  constexpr int STRIDE = 36 * 4 / (int)sizeof(TO);
  TO* lines = reinterpret_cast<TO*>(moe_smem + wave * 32 * 36 * 4);
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int jb = 0; jb < TO_J / JB; ++jb) {
#pragma unroll
      for (int j = 0; j < JB; ++j)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const moe_f32x16& v = acc[i][jb * JB + j];
          TO* at = lines + (lane & 31) * STRIDE + 32 * j + 8 * r4 + 4 * (lane >> 5);
          if constexpr (F32) *reinterpret_cast<float4*>(at) = make_float4(v[4 * r4], v[4 * r4 + 1], v[4 * r4 + 2], v[4 * r4 + 3]);
          else *reinterpret_cast<uint2*>(at) = make_uint2(float2_to_bf16x2(v[4 * r4], v[4 * r4 + 1]), float2_to_bf16x2(v[4 * r4 + 2], v[4 * r4 + 3]));
        }
      lds_wave_order();
#pragma unroll
      for (int x = 0; x < 32 * LR / 64; ++x) {
        const int r = (64 * x + lane) / LR, c = lane % LR * PER, at = wm * WM + 32 * i + r;
        const int o = o0 + wn * (GLU ? WN / 2 : WN) + 32 * jb * JB + c;
        const moe_u32x4 v = *reinterpret_cast<const moe_u32x4*>(lines + r * STRIDE + c);
        if (at < rows && o < F) moe_big_store(static_cast<TO*>(p.out) + (size_t)(first + at) * p.o_stride + o, v, F - o, p.vec);
      }
      lds_wave_order();
    }
}

template <typename TO, bool GLU>
__global__ void __launch_bounds__(256, 2)
moe_linear_big_kernel(const MoeLinearArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char moe_smem[];
  const int n_tiles = p.meta[0], per = (n_tiles + 7) / 8;
  if (per == 0) return;
  const int lo = (blockIdx.x & 7) * per, n = min(per, n_tiles - lo), slot = blockIdx.x >> 3;
  if (slot >= n * p.n_cols) return;  // the whole workgroup (n may be below 1)
  int tile = lo + slot % n, ycol = slot / n;
  if (n <= 64) {  // the chiplet's larger tiles first, in all columns: what runs last is short
    const int lane = threadIdx.x & 63;
    const bool large = lane < n && p.tiles[3 * (lo + lane) + 2] > MOE_BIG / 2;
    const unsigned long long all = __ballot(lane < n), larger = __ballot(large);
    const int n_larger = __popcll(larger);
    const bool mine = slot < n_larger * p.n_cols;
    const unsigned long long of = mine ? larger : all & ~larger;
    const int at = mine ? slot : slot - n_larger * p.n_cols, kind = __popcll(of);
    ycol = at / kind;
    tile = lo + __ffsll(__ballot((of >> lane & 1) && __popcll(of & ((1ull << lane) - 1)) == at % kind)) - 1;
  }
  const int e = p.tiles[3 * tile], first = p.tiles[3 * tile + 1], rows = p.tiles[3 * tile + 2];
  if (rows <= MOE_BIG / 2) moe_big_tile<TO, GLU, MOE_BN, MOE_BIG / 2>(p, moe_smem, e, first, rows, ycol);
  else moe_big_tile<TO, GLU, MOE_BN, MOE_BIG>(p, moe_smem, e, first, rows, ycol);
}

// a [rows][K]; w [E][N][K] with N = F outputs, or with glu N = 2F: gate rows then up rows; out [P][F]
extern "C" int lev_moe_linear(const void* a, long a_rows, long a_stride, const void* w, void* out, long o_stride, const int* tiles, const int* meta,
                              const int* sorted, int max_tiles, int tile_rows, int E, int top, int gather, int K, int N, int glu, int act, float limit,
                              float up_shift, int dtype, int out_dtype, int use_mfma, hipStream_t stream) {
  LEV_REQUIRE(a && w && out && tiles && meta && sorted, "experts: a tensor is missing");
  LEV_REQUIRE(K > 0 && N > 0 && (!glu || N % 2 == 0) && top > 0 && max_tiles >= 0, "experts: bad sizes K=%d N=%d", K, N);
  LEV_REQUIRE(act >= 0 && act <= LEV_ACT_LAST, "experts: unknown activation %d", act);
  LEV_REQUIRE(tile_rows == MOE_TM || tile_rows == MOE_BIG, "experts: tiles of %d rows (%d or %d)", tile_rows, MOE_TM, MOE_BIG);
  LEV_REQUIRE(dtype == LEV_F32 || dtype == LEV_BF16, "experts: unknown dtype %d", dtype);
  LEV_REQUIRE(dtype == LEV_BF16 || out_dtype == LEV_F32, "experts: float32 inputs give float32 outputs");
  const int F = glu ? N / 2 : N;
  LEV_REQUIRE(a_stride >= K && o_stride >= F, "experts: row strides are smaller than the rows");
  if (max_tiles == 0) return 0;
  if (dtype == LEV_BF16 && use_mfma && K % 8 == 0 && a_stride % 8 == 0 && ((uintptr_t)a & 15) == 0 && ((uintptr_t)w & 15) == 0) {
    const int vec = o_stride % 8 == 0 && ((uintptr_t)out & 15) == 0 ? 2 : o_stride % 4 == 0 && ((uintptr_t)out & (out_dtype == LEV_F32 ? 15 : 7)) == 0;
    if (tile_rows == MOE_BIG) {
      const int bn = glu ? MOE_BN / 2 : MOE_BN, n_cols = (F + bn - 1) / bn;
      const long blocks = (long)((max_tiles + 7) / 8) * 8 * n_cols;
      LEV_REQUIRE(blocks <= 0x7fffffffL, "experts: too many tiles (%ld)", blocks);
      const bool spread = blocks / 8 <= (max_tiles <= 2L * E + 1 ? 2 * MOE_BIG_SPREAD : MOE_BIG_SPREAD);  // by sizes alone, not by what the routing made of them
      const MoeLinearArgs args{(const bf16_t*)a, a_stride, (const bf16_t*)w, out, o_stride, tiles, meta, sorted, top, gather, K, N, F, act, limit, up_shift, n_cols, vec, spread};
      const int ring = lev_moe_ring(args, a_rows, out_dtype, glu, max_tiles, stream);
      if (ring <= 0) return ring;
#define MOE_BIG_CASE(TO, G)                                                                                                                       \
  do {                                                                                                                                            \
    hipError_t e = hipFuncSetAttribute((const void*)moe_linear_big_kernel<TO, G>, hipFuncAttributeMaxDynamicSharedMemorySize, MOE_BIG_LDS(MOE_BN)); \
    LEV_REQUIRE(e == hipSuccess, "experts: %d bytes of LDS a workgroup: %s", MOE_BIG_LDS(MOE_BN), hipGetErrorString(e));                           \
    moe_linear_big_kernel<TO, G><<<(unsigned)blocks, 256, MOE_BIG_LDS(MOE_BN), stream>>>(args);                                                   \
  } while (0)
      if (out_dtype == LEV_F32) {
        if (glu) MOE_BIG_CASE(float, true); else MOE_BIG_CASE(float, false);
      } else {
        if (glu) MOE_BIG_CASE(bf16_t, true); else MOE_BIG_CASE(bf16_t, false);
      }
#undef MOE_BIG_CASE
      return lev_check_launch("moe_linear (matrix cores, tiles of 128 rows)");
    }
    const MoeLinearArgs args{(const bf16_t*)a, a_stride, (const bf16_t*)w, out, o_stride, tiles, meta, sorted, top, gather, K, N, F, act, limit, up_shift, 0, vec, false};
    const dim3 grid(max_tiles, (F + 15) / 16);
#define MOE_FEW(TO, G)                                                                              \
  do {                                                                                              \
    if (K < 2048) moe_linear_few_kernel<TO, G, 4, 2><<<grid, 64 * 4, 0, stream>>>(args);            \
    else moe_linear_few_kernel<TO, G, 8, 2><<<grid, 64 * 8, 0, stream>>>(args);                     \
  } while (0)
    if (out_dtype == LEV_F32) {
      if (glu) MOE_FEW(float, true); else MOE_FEW(float, false);
    } else {
      if (glu) MOE_FEW(bf16_t, true); else MOE_FEW(bf16_t, false);
    }
#undef MOE_FEW
    return lev_check_launch("moe_linear (matrix cores)");
  }
  dim3 grid(max_tiles, (F + 15) / 16);
  if (dtype == LEV_F32)
    moe_linear_plain_kernel<float, float><<<grid, 256, 0, stream>>>((const float*)a, a_stride, (const float*)w, (float*)out, o_stride, tiles, meta,
                                                                    sorted, top, gather, K, N, F, glu, act, limit, up_shift);
  else if (out_dtype == LEV_F32)
    moe_linear_plain_kernel<bf16_t, float><<<grid, 256, 0, stream>>>((const bf16_t*)a, a_stride, (const bf16_t*)w, (float*)out, o_stride, tiles, meta,
                                                                     sorted, top, gather, K, N, F, glu, act, limit, up_shift);
  else
    moe_linear_plain_kernel<bf16_t, bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)a, a_stride, (const bf16_t*)w, (bf16_t*)out, o_stride, tiles,
                                                                      meta, sorted, top, gather, K, N, F, glu, act, limit, up_shift);
  return lev_check_launch("moe_linear");
}

// ---- combine -------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
moe_combine_kernel(const float* __restrict__ expert_out, const int* __restrict__ pos_of, const float* __restrict__ weights, float* __restrict__ y,
                   int D, int top, int accumulate, const int* __restrict__ chosen, int n_real, const void* __restrict__ identity_in, long id_stride,
                   int id_dtype) {
  __shared__ int pos_s[MOE_MAX_TOP];
  __shared__ float w_s[MOE_MAX_TOP];
  const int t = blockIdx.x;
  if (threadIdx.x < top) {
    const bool own = identity_in != nullptr && chosen[(size_t)t * top + threadIdx.x] >= n_real;  // an expert that returns its input
    pos_s[threadIdx.x] = own ? -1 : pos_of[(size_t)t * top + threadIdx.x];
    w_s[threadIdx.x] = weights[(size_t)t * top + threadIdx.x];
  }
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += 256) {
    float acc = accumulate ? y[(size_t)t * D + d] : 0.f;
    float own = 0.f;
    if (identity_in != nullptr)
      own = id_dtype == LEV_F32 ? ((const float*)identity_in)[(size_t)t * id_stride + d] : bf16_to_float(((const bf16_t*)identity_in)[(size_t)t * id_stride + d]);
    for (int c = 0; c < top; ++c) acc = fmaf(w_s[c], pos_s[c] < 0 ? own : expert_out[(size_t)pos_s[c] * D + d], acc);
    y[(size_t)t * D + d] = acc;
  }
}

extern "C" int lev_moe_combine(const float* expert_out, const int* pos_of, const float* weights, float* y, int T, int D, int top, int accumulate,
                               const int* chosen, int n_real, const void* identity_in, long id_stride, int id_dtype, hipStream_t stream) {
  LEV_REQUIRE(expert_out && pos_of && weights && y && T >= 0 && D > 0 && top > 0 && top <= MOE_MAX_TOP, "experts: bad arguments of the weighted sum");
  LEV_REQUIRE(identity_in == nullptr || (chosen && id_stride >= D && (id_dtype == LEV_F32 || id_dtype == LEV_BF16)), "experts: experts that return their input need the choices and the input's rows");
  if (T == 0) return 0;
  moe_combine_kernel<<<T, 256, 0, stream>>>(expert_out, pos_of, weights, y, D, top, accumulate, chosen, n_real, identity_in, id_stride, id_dtype);
  return lev_check_launch("moe_combine");
}
