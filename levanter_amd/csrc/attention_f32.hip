// Attention of a ragged batch over the paged cache in 32 bits, on the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32), for head sizes
// of 16 .. 128 in steps of 16. The problem is transposed, S^T = K Q^T and O^T = V^T P^T: both page layouts are then read 16 bytes a lane as
// the instruction's first operand, and the probabilities leave the first product in the registers that the second one reads.
//   q [T][H*HD] (row stride q_stride), out likewise; keys [page][kv_head][HD/8][PS][8], values [page][kv_head][HD][PS]
//   scores, mask, pages that are not there and queries without a key as in attention_simple.hip
//
// A workgroup of W waves owns 16 columns: 16 consecutive query rows of one head (runs of several tokens), or up to 16 query heads of one
// key/value head (single tokens). Its waves take the blocks of 16 KB keys in turn and merge through LDS in wave order.
// What bounds it: prompts, the vector instructions and round trips between a block's two products, and the waves there are to fill the matrix pipe meanwhile:
// blocks of 16 keys (KB = 1) leave registers for three waves on a SIMD at head size 64 and two at 128, where blocks of 64 and 32 keys left two and one, and a
// prompt's last keys fill them better (777 rows of 16 heads of 64, 1.2 GFLOP of visible products: 35.0 -> 25.4 us; 4 x 777 rows: 106 -> 81; 8 key/value
// heads of 128, 4 x 777 rows: 225 -> 152; the next block's keys and values loaded ahead take the registers instead: 54 us at 777 rows); single tokens, the chain of one block's loads, products and merge (4 tokens of 12 heads over
// 200 keys: 9.6 us). The plain kernel gives a wave one query row, reads keys 4 bytes at a time and walks the values key by key:
// 1,187 us and 70 us. A step of single tokens alone brings its new keys and values along: the wave whose keys they are takes them from the projection's output, and
// the wave behind it, which has none in a short context, writes them to their page; the kernel that wrote them first took 4 us a layer (GPT-2 small, 4 requests of
// 100 to 200 tokens, with the arguments of the first loads in registers besides: 10.78 -> 9.99 ms a session, same bits).
#include "common.h"
#include <math.h>

typedef __attribute__((ext_vector_type(4))) float af_f32x4;

struct AttentionF32Args {
  const float* q;
  long q_stride;
  float* out;
  long o_stride;
  float *k_pages, *v_pages;
  int window, bias_len;
  float scale, softcap;
  const float* score_bias;
  const float *k_new, *v_new;  // single tokens: the step's new keys and values (rows kv_stride apart), not in their pages yet; or null
  long kv_stride;
  const int* dest;  // where they go, by token: page * PS + offset
};

// over the four lanes of a column, neighbouring groups of 16 first; register swaps, where the shuffles of two numbers would wait for LDS four times a block
template <class Op>
static __device__ __forceinline__ float af_over_groups(float v, Op op) {
  typedef __attribute__((ext_vector_type(2))) unsigned pair_t;
  const pair_t a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);  // {groups 0 0 2 2, groups 1 1 3 3}
  v = op(__uint_as_float(a.x), __uint_as_float(a.y));
  const pair_t b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);  // {lower half twice, upper half twice}
  return op(__uint_as_float(b.x), __uint_as_float(b.y));
}

template <int HD, int KB, int W, bool RUNS>
__global__ void __launch_bounds__(64 * W, 8 / W)  /* two waves on a SIMD, runs need 137 registers at head size 64 and 256 at 128 */
attention_f32_kernel(const int* __restrict__ work,  // runs: (first token, rows) per tile of the list; single tokens: their indexes
                     const int* __restrict__ positions, const int* __restrict__ token_seq, const int* __restrict__ block_tables, int bt_stride, int H, int KVH, int PS,
                     int tile_rows, int columns, int n_positions,  // rows of a tile of the list (runs); columns in use (single tokens: query heads of a key/value head, at most 16); entries of positions (single tokens)
                     const AttentionF32Args p) {  // all before p is in registers when the waves start
  extern __shared__ __attribute__((aligned(16))) float af_lds[];  // [W][HD/16][4][columns] of four outputs, then maxima and sums [2][W][16] and a tile's weights [W][16][16]
  constexpr int DT = HD / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
  const int group = H / KVH, nc = RUNS ? 16 : columns;
  int token, head, pos, seq;
  bool mine;  // this lane's column is one
  if (RUNS) {
    const int subs = (tile_rows + 15) / 16;
    head = blockIdx.x % H;
    const int sub = blockIdx.x / H % subs, tile = blockIdx.x / H / subs;
    const int first = work[2 * tile], rows = work[2 * tile + 1] - 16 * sub;
    if (rows <= 0) return;  // the whole workgroup
    mine = col < rows;
    token = first + 16 * sub + min(col, rows - 1);
    pos = positions[token], seq = token_seq[token];
  } else {
    const int sets = (group + 15) / 16, kvh = blockIdx.x / sets % KVH, set = blockIdx.x % sets;
    // which token, its position and its row in one trip: the i-th single token of a step is mostly its i-th token, and if not they are asked for again. With no
    // exchange over the columns below (they are one token's) a session of 4 requests on 12 layers of 12 heads, which waits for one load after another, 9.29 -> 9.19 ms.
    const int i = blockIdx.x / sets / KVH, guess = min(i, n_positions - 1);
    token = work[i], pos = positions[guess], seq = token_seq[guess];
    if (token != guess) pos = positions[token], seq = token_seq[token];
    const int n = min(16, group - 16 * set);
    mine = col < n;
    head = kvh * group + 16 * set + min(col, n - 1);
  }
  const int kvh = head / group;
  const int first = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  int last = pos, lo = first;  // over the columns
  if (RUNS)
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      last = max(last, __shfl_xor(last, o, 64));
      lo = min(lo, __shfl_xor(lo, o, 64));
    }
  const int* bt = block_tables + (size_t)seq * bt_stride;
  const size_t head_elems = (size_t)HD * PS;
  const float* qr = p.q + (size_t)token * p.q_stride + (size_t)head * HD;
  constexpr int SUMS = !RUNS && W == 4 ? KB : 1;  // four waves have longer chains of sums than eight: a tile of a block to each keeps their roundings
  af_f32x4 q[DT], o_acc[SUMS][DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    q[d] = *reinterpret_cast<const af_f32x4*>(qr + 16 * d + 4 * g) * p.scale;
#pragma unroll
    for (int a = 0; a < SUMS; ++a) o_acc[a][d] = af_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float* ml = af_lds + (size_t)W * DT * 4 * nc * 4;
  float* weights = ml + 2 * W * 16 + wave * 256;
  // l: of the weights of this lane's keys, every fourth four. Four sums of a quarter each have half the roundings of one over the column that each block joins (1 / the sum of 16,384 weights,
  // rms in 2^-24, over the block's lanes first / so: runs of four waves 2.1 / 1.3, of eight 1.5 / 1.1, single tokens of four 1.6 / 1.1, of eight 1.4 / 1.1; times level)
  float m = -INFINITY, l = 0.f;
  const int t_last = last / 16;
  const bool fused = !RUNS && p.k_new != nullptr;
  const float* kn = fused ? p.k_new + (size_t)token * p.kv_stride + (size_t)kvh * HD : qr;  // not fused: read, not used
  const float* vn = fused ? p.v_new + (size_t)token * p.kv_stride + (size_t)kvh * HD : qr;
  float nv[DT];  // the token's new value in this lane's dimensions
  int to = -1;
  if (!RUNS) {
#pragma unroll
    for (int d = 0; d < DT; ++d) nv[d] = vn[16 * d + col];
    to = *(fused ? p.dest + token : work);
    to = fused ? to : -1;
  }
  for (int t0 = lo / 16 + wave * KB; t0 <= t_last; t0 += W * KB) {
    int page[KB], off[KB];
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      const int key = min(t0 + t, t_last) * 16;  // tiles behind the last are read again and masked
      page[t] = bt[key / PS];
      off[t] = key % PS;
    }
    af_f32x4 s[KB], k[KB][DT], v[KB][DT];  // all of the block's loads are on their way before the first product
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      const bool is_new = fused && (t0 + t) * 16 + col == pos;
      const float* kb = is_new ? kn + 4 * g : p.k_pages + ((size_t)max(page[t], 0) * KVH + kvh) * head_elems + (size_t)(off[t] + col) * 8 + (g & 1) * 4 + (size_t)(g >> 1) * PS * 8;
      const size_t next = is_new ? 16 : (size_t)PS * 16;
#pragma unroll
      for (int d = 0; d < DT; ++d) k[t][d] = *reinterpret_cast<const af_f32x4*>(kb + d * next);
    }
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      const float* vb = p.v_pages + ((size_t)max(page[t], 0) * KVH + kvh) * head_elems + off[t] + 4 * g;
#pragma unroll
      for (int d = 0; d < DT; ++d) v[t][d] = *reinterpret_cast<const af_f32x4*>(vb + (size_t)(16 * d + col) * PS);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!RUNS) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[t][d][e] = fused && (t0 + t) * 16 + 4 * g + e == pos ? nv[d] : v[t][d][e];
    }
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      s[t] = af_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][d][e], q[d][e], s[t], 0, 0, 0);
    }
    if (p.score_bias || p.softcap > 0.f) {
#pragma unroll
      for (int t = 0; t < KB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (p.score_bias) s[t][r] += p.score_bias[(size_t)head * p.bias_len + min(max(pos - (t0 + t) * 16 - 4 * g - r, 0), p.bias_len - 1)];
          if (p.softcap > 0.f) s[t][r] = p.softcap * tanhf(s[t][r] / p.softcap);
        }
    }
    float mx = -INFINITY;
    bool masked = false;  // some column does not see some key of the block
#pragma unroll
    for (int t = 0; t < KB; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = (t0 + t) * 16 + 4 * g + r;
        const bool live = key <= pos && key >= first && page[t] >= 0;
        masked |= !live;
        s[t][r] = live ? s[t][r] : -INFINITY;
        mx = fmaxf(mx, s[t][r]);
      }
    mx = af_over_groups(mx, [](float a, float b) { return fmaxf(a, b); });
    const float m_new = fmaxf(m, mx);
    const float corr = m == -INFINITY ? 0.f : expf(m - m_new);
    float sum = 0.f;  // this lane's keys
#pragma unroll
    for (int t = 0; t < KB; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = s[t][r] == -INFINITY ? 0.f : expf(s[t][r] - m_new);  // no live key so far: m_new = -inf, all are 0
        s[t][r] = e;
        sum += e;
      }
    l = l * corr + sum;
    m = m_new;
#pragma unroll
    for (int a = 0; a < SUMS; ++a)
#pragma unroll
      for (int d = 0; d < DT; ++d) o_acc[a][d] *= corr;
    const bool any_masked = __any(masked);
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      if (any_masked) {  // the whole wave
        // keys that nobody sees (a page may hold anything behind the last token): zeros. Keys that some columns see and others do not:
        // their weight is 0 in the others, and 0 times infinity or NaN must not reach those: such a tile takes the sum column by column.
        bool odd = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = (t0 + t) * 16 + 4 * g + r;
          const bool there = key <= last && page[t] >= 0;
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            if (!there) v[t][d][r] = 0.f;
            odd |= !(fabsf(v[t][d][r]) < INFINITY);
          }
        }
        if (__any(odd)) {  // rare, and kept small: the weights through LDS, a key at a time
#pragma unroll
          for (int r = 0; r < 4; ++r) weights[(4 * g + r) * 16 + col] = s[t][r];
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // within the wave
          const float* at = p.v_pages + ((size_t)max(page[t], 0) * KVH + kvh) * head_elems + off[t] + (size_t)4 * g * PS;
#pragma unroll 1
          for (int j = 0; j < 16; ++j) {
            const int key = (t0 + t) * 16 + j;
            const bool live = key <= pos && key >= first && page[t] >= 0;
            const float weight = weights[j * 16 + col];
            const bool is_new = fused && key == pos;  // not in its page yet
            const float* row = is_new ? vn + 4 * g : at + j;
            const int next = is_new ? 1 : PS;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                asm volatile("" : "+v"(row));  // one address, moved on: the compiler would keep one for each of the sums
                if (live) o_acc[t % SUMS][d][e] = fmaf(weight, *row, o_acc[t % SUMS][d][e]);
                row += e < 3 ? next : 13 * next;
              }
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          continue;
        }
      }
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) o_acc[t % SUMS][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][d][e], s[t][e], o_acc[t % SUMS][d], 0, 0, 0);
    }
  }
  if (SUMS == 2) {
#pragma unroll
    for (int d = 0; d < DT; ++d) o_acc[0][d] += o_acc[SUMS - 1][d];
  }
  // the new key and value go to their page: read by later steps only. By the wave behind the one with the last keys, which has none where there are few
  if (!RUNS && to >= 0 && blockIdx.x % ((group + 15) / 16) == 0 && wave == ((t_last - lo / 16) / KB + 1) % W) {
    const size_t page = ((size_t)(to / PS) * KVH + kvh) * head_elems;
    const int at = to % PS;
#pragma unroll
    for (int i = lane; i < HD; i += 64) {
      p.k_pages[page + ((size_t)(i >> 3) * PS + at) * 8 + (i & 7)] = kn[i];
      p.v_pages[page + (size_t)i * PS + at] = vn[i];
    }
  }
  if (col < nc) {
#pragma unroll
    for (int d = 0; d < DT; ++d) *reinterpret_cast<af_f32x4*>(af_lds + ((size_t)((wave * DT + d) * 4 + g) * nc + col) * 4) = o_acc[0][d];
  }
  l = af_over_groups(l, [](float a, float b) { return a + b; });
  if (g == 0) ml[wave * 16 + col] = m, ml[(W + wave) * 16 + col] = l;
  __syncthreads();
  if (!mine) return;
  float top = -INFINITY, total = 0.f, factor[W];
#pragma unroll
  for (int w = 0; w < W; ++w) top = fmaxf(top, ml[w * 16 + col]);
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const float mw = ml[w * 16 + col];
    factor[w] = mw == -INFINITY ? 0.f : expf(mw - top);
    total += ml[(W + w) * 16 + col] * factor[w];
  }
  const float inv = total > 0.f || total != total ? 1.0f / total : 0.f;  // a query without a key gives zeros, a score that is NaN gives NaN
  float* orow = p.out + (size_t)token * p.o_stride + (size_t)head * HD;
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    if (d % W != wave) continue;  // the waves finish 16 dimensions each in turn
    af_f32x4 sum = af_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const af_f32x4 part = *reinterpret_cast<const af_f32x4*>(af_lds + ((size_t)((w * DT + d) * 4 + g) * nc + col) * 4);
      if (factor[w] != 0.f) sum += part * factor[w];
    }
    *reinterpret_cast<af_f32x4*>(orow + 16 * d + 4 * g) = sum * inv;
  }
}

template <int HD, int W>
static int attention_f32_runs(const AttentionF32Args& p, const int* positions, const int* token_seq, const int* block_tables, int bt_stride, int H, int KVH, int PS,
                              const int* tiles, long blocks, int tile_rows, hipStream_t stream) {
  constexpr int lds = W * (HD / 16) * 4 * 16 * 16 + 2 * W * 16 * 4 + W * 1024;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)attention_f32_kernel<HD, 1, W, true>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    LEV_REQUIRE(e == hipSuccess, "attention: %d bytes of LDS a workgroup: %s", lds, hipGetErrorString(e));
  }
  attention_f32_kernel<HD, 1, W, true><<<(unsigned)blocks, 64 * W, lds, stream>>>(tiles, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tile_rows, 16, 0, p);
  return 0;
}

template <int HD, int KB, int W>
static int attention_f32_singles(const AttentionF32Args& p, const int* positions, const int* token_seq, const int* block_tables, int bt_stride, int H, int KVH, int PS,
                                 const int* tokens, long blocks, int n_positions, hipStream_t stream) {
  const int group = H / KVH, columns = group < 16 ? group : 16;
  const int lds = W * (HD / 16) * 4 * columns * 16 + 2 * W * 16 * 4 + W * 1024;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)attention_f32_kernel<HD, KB, W, false>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    LEV_REQUIRE(e == hipSuccess, "attention: %d bytes of LDS a workgroup: %s", lds, hipGetErrorString(e));
  }
  attention_f32_kernel<HD, KB, W, false><<<(unsigned)blocks, 64 * W, lds, stream>>>(tokens, positions, token_seq, block_tables, bt_stride, H, KVH, PS, 0, columns, n_positions, p);
  return 0;
}

template <int HD>
static int attention_f32_launch(const AttentionF32Args& p, const int* positions, const int* token_seq, const int* block_tables, int bt_stride, int H, int KVH, int PS,
                                const int* tiles, int n_tiles, int tile_rows, const int* tokens, int n_tokens, int n_positions, hipStream_t stream) {
  constexpr int KB1 = HD <= 96 ? 2 : 1;  // single tokens: as many tiles of keys as fit the registers
  if (n_tiles > 0) {
    const long blocks = (long)n_tiles * ((tile_rows + 15) / 16) * H;
    LEV_REQUIRE(blocks <= 0x7fffffffL, "attention: too many tiles (%ld)", blocks);
    // Eight waves a workgroup up to one and a half for a CU (not all rows of a tile are there): the keys are then walked in half the steps (65 rows behind 935 keys, 16 heads of 64: 21.2 us
    // with four, 18.8 with eight; 256 rows, 12 heads: 8.3 and 8.1; 3 x 64 rows, 16 heads of 128: 8.8 and 7.2; 500 rows, 8 heads of 32: 10.1 and 8.8). With more of them the merges cost more than that
    // (777 rows, 16 heads of 64: 25.4 and 31.3; 300 + 500 rows, 16 heads of 112: 28.7 and 36.4).
    const int rc = blocks <= 384 ? attention_f32_runs<HD, 8>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, blocks, tile_rows, stream)
                                 : attention_f32_runs<HD, 4>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, blocks, tile_rows, stream);
    if (rc) return rc;
  }
  if (n_tokens > 0) {
    const int sets = (H / KVH + 15) / 16;
    const long blocks = (long)n_tokens * KVH * sets;
    LEV_REQUIRE(blocks <= 0x7fffffffL, "attention: too many single tokens (%ld)", blocks);
    // Eight waves use up a CU's registers, so that a grid of more workgroups than CUs came in rounds; four leave room for two workgroups (24 tokens of 12 heads of 64
    // over 150 keys: 16.9 -> 13.0 us; 16 of 25 over 200: 19.0 -> 15.7; 32 of 25 over 1,000: 96.9 -> 88.0; 64 of 16 heads of 96 over 200: 51.8 -> 42.2; 64 of 12 over
    // 600: level). With no more workgroups than CUs the shorter walk over the keys is the better one (20 of 12 over 150: 10.3 and 11.3; 2 of 12 over 1,000: 20.2 and
    // 26.7). Head sizes of 112 and 128 have no registers for a second set of sums, without which four waves' error is 2 - 15 % larger.
    const bool four = KB1 == 2 && blocks > 256;
    const int rc = four ? attention_f32_singles<HD, KB1, KB1 == 2 ? 4 : 8>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tokens, blocks, n_positions, stream)
                        : attention_f32_singles<HD, KB1, 8>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tokens, blocks, n_positions, stream);
    if (rc) return rc;
  }
  return lev_check_launch("attention (32-bit)");
}

// 1: not for these operands (nothing has been launched): head sizes in steps of 16 up to 128, rows at 16-byte addresses. tiles: (first token,
// rows <= tile_rows) of runs of several consecutive tokens; tokens: the single ones; n_positions: entries of positions and token_seq. k_new (a step of single tokens alone): the step's keys and values (rows kv_stride
// apart) are not in the cache yet and are written to dest[t] = page * PS + offset on the way.
extern "C" int lev_attention_f32(const float* q, long q_stride, float* out, long o_stride, float* k_pages, float* v_pages, const int* positions,
                                 const int* token_seq, const int* block_tables, int bt_stride, const int* tiles, int n_tiles, int tile_rows, const int* tokens,
                                 int n_tokens, int n_positions, const float* k_new, const float* v_new, long kv_stride, const int* dest, int H, int KVH, int HD, int PS, float scale, int window, float softcap, const float* score_bias, int bias_len,
                                 hipStream_t stream) {
  LEV_REQUIRE(H > 0 && KVH > 0 && H % KVH == 0, "attention: bad head counts heads=%d kv_heads=%d", H, KVH);
  LEV_REQUIRE(PS > 0 && PS % 16 == 0, "attention: page_size=%d must be a multiple of 16", PS);
  LEV_REQUIRE(window >= 0, "attention: window=%d must not be negative", window);
  LEV_REQUIRE(softcap >= 0.f && (!score_bias || bias_len >= 1), "attention: soft cap %g must not be negative and a bias table needs entries (%d)", (double)softcap, bias_len);
  LEV_REQUIRE(n_tiles >= 0 && n_tokens >= 0 && (n_tiles == 0 || (tiles && tile_rows > 0)) && (n_tokens == 0 || (tokens && n_positions > 0)), "attention: a work list is missing");
  LEV_REQUIRE(!k_new || (v_new && dest && n_tiles == 0), "attention: new keys come with values and destinations, in steps of single tokens");
  if (HD % 16 != 0 || HD < 16 || HD > 128 || q_stride % 4 != 0 || o_stride % 4 != 0 || (k_new && kv_stride % 4 != 0)) return 1;
  if ((((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_pages | (uintptr_t)v_pages | (uintptr_t)k_new) & 15) != 0) return 1;
  const AttentionF32Args p{q, q_stride, out, o_stride, k_pages, v_pages, window, bias_len, scale, softcap, score_bias, k_new, v_new, kv_stride, dest};
  switch (HD / 16) {
    case 1: return attention_f32_launch<16>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    case 2: return attention_f32_launch<32>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    case 3: return attention_f32_launch<48>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    case 4: return attention_f32_launch<64>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    case 5: return attention_f32_launch<80>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    case 6: return attention_f32_launch<96>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    case 7: return attention_f32_launch<112>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
    default: return attention_f32_launch<128>(p, positions, token_seq, block_tables, bt_stride, H, KVH, PS, tiles, n_tiles, tile_rows, tokens, n_tokens, n_positions, stream);
  }
}
