// The attention of attention_values.hip on the matrix cores, bfloat16 in, 32-bit softmax and accumulation. Compiled once
// per pair of head sizes: -DLEV_HD=<key head size> -DLEV_VD=<value head size>, both multiples of 16.
//
// As in attention_mfma.hip the problem is transposed so that no operand needs a transposition:
//   S^T = K . Q^T      A operand: 16 keys x 32 head dims from the key pages, B operand: Q^T, in registers
//   O^T = V^T . P^T    A operand: 16 value dims x 32 keys from the transposed value pages, B operand: P^T, which is what
//                      the lanes hold after the softmax
// with the 16x16x32 MFMA (A lane l: row l%16, k = 8*(l/16) .. +7; B lane l: column l%16, the same k; accumulator register
// r of lane l: row 4*(l/16) + r, column l%16). The rows of score tile (u, h) are the keys 32u + 8*(row/4) + 4h + row%4 of
// a block of 64, so that lane group g = l/16 holds the weights of the keys 32u + 8g .. +7 in its two tiles.
//
// One wave owns 16 columns that share a request and a key/value head:
//   * a run of several tokens: 16 consecutive query tokens of one query head; the 8 waves of a workgroup are a tile of up
//     to 128 tokens and share every block of keys and values through LDS (attention_values_mfma_runs_kernel);
//   * a single token: the query heads of one key/value head (up to 16 at a time); operands go from the pages straight
//     into registers, and a token's keys may be split over several waves, whose results their workgroup merges through LDS or, where there
//     are too many or their reads would crowd one CU, a second kernel.
// A wave walks the keys in blocks of 64, keeps a running maximum and sum per column, and applies the weights to the
// values of up to NVC value heads (blockIdx.z picks which): its own one, or, for layers that mix the weights over the
// heads afterwards, every key/value head in turn.
//
//   score(t, key) = cap(scale * q . k) - slope[h] * (position(t) - position(key)),  cap(s) = softcap * tanh(s / softcap)
//   out [T][H][NV][VD] float32, as attention_values.hip writes it.
//   sinks (float32 [H] or null): exp(sinks[h]) is added to the denominator of head h's softmax, once per query (a token whose
//   keys are split over waves gets it in the merge).
#include "common.h"
#include "attention_config.h"

#if !defined(LEV_HD) || !defined(LEV_VD)
#error "compile with -DLEV_HD=<key head size> -DLEV_VD=<value head size>"
#endif

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

#define HD LEV_HD
#define VD LEV_VD
#define NKS ((HD + 31) / 32)  // k-steps of the score product
#define NDT (VD / 16)         // 16-row tiles of O^T per value head
// value heads per wave: at most 16 accumulator tiles (64 registers)
#define NVC (NDT <= 2 ? 8 : (NDT <= 4 ? 4 : (NDT <= 8 ? 2 : 1)))
#define SUB_TILES (PF_ROWS / 16)

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}

// all but the first n of eight consecutive keys' values (two to a word) made zero: what lies behind the last key that was
// written may be anything, NaN too, and zero times that would reach the sum
__device__ __forceinline__ u32x4 first_keys(u32x4 v, int n) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] &= n >= 2 * e + 2 ? 0xffffffffu : (n == 2 * e + 1 ? 0x0000ffffu : 0u);
  return v;
}

__device__ __forceinline__ float fast_tanh(float x) {  // 1 - 2 / (1 + e^(2x)) with the hardware's exp2 and reciprocal
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * 2.8853900817779268f));
}

// NC: value heads that a wave has room for (1, or a power of two up to NVC). The operands of all of them are on their way together, so room
// for more than there are costs registers and a launch that is 0.3 - 0.5 us longer (16 x 16 heads of 64 / 64, 8 tokens of 60 keys 5.1 us, 5.6 with
// room for four; 16 x 4 of 64 / 32 with all 4 value heads 6.2 us, 6.6 with room for eight).
// WAVES > 1: up to so many ranges of a single token's keys are the waves of one workgroup, which merge through LDS; more of them go through scratch
// memory and a second kernel.
template <bool SINGLE, int NC, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
attention_values_mfma_kernel(const bf16_t* __restrict__ q, long q_stride, float* __restrict__ out, const bf16_t* __restrict__ k_pages,
                             const bf16_t* __restrict__ v_pages, const int* __restrict__ positions, const int* __restrict__ token_seq,
                             const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ work, int n_positions, int H, int KVH, int NV,
                             int PS, float scale, int window, int chunk, int keep, float softcap, const float* __restrict__ slopes, int splits,
                             float* __restrict__ part_o, float* __restrict__ part_ml, const float* __restrict__ sinks) {
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int group = H / KVH;
  int tok = 0, head = 0, kvh = 0, pos, seq;
  bool valid;
  if (SINGLE) {
    const int col_sets = (group + 15) / 16;
    kvh = blockIdx.y / col_sets;
    const int c = (blockIdx.y % col_sets) * 16 + col;
    valid = c < group;
    head = kvh * group + (valid ? c : 0);
    // which token, its position and its row in one trip: the i-th single token of a step is mostly its i-th token, and if not they are asked for again
    const int i = WAVES > 1 ? blockIdx.x : blockIdx.x / splits, guess = min(i, n_positions - 1);
    tok = work[i], pos = positions[guess], seq = token_seq[guess];
    if (tok != guess) pos = positions[tok], seq = token_seq[tok];
  } else {
    const int tile = blockIdx.x / SUB_TILES, sub = blockIdx.x % SUB_TILES;
    const int first = work[2 * tile], n = work[2 * tile + 1];
    if (sub * 16 >= n) return;  // the whole wave
    head = blockIdx.y;
    kvh = head / group;
    valid = sub * 16 + col < n;
    tok = first + (valid ? sub * 16 + col : sub * 16);
    pos = positions[tok], seq = token_seq[tok];
  }
  const int lo = lev_first_visible(pos, window, chunk);
  // the wave's range of keys; every column belongs to the same request, those of a single token to one position
  int p_max = SINGLE || valid ? pos : -1, lo_min = SINGLE || valid ? lo : 0x7fffffff;
  if (!SINGLE)
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      p_max = max(p_max, __shfl_xor(p_max, o, 64));
      lo_min = min(lo_min, __shfl_xor(lo_min, o, 64));
    }
  const int* bt = block_tables + (size_t)seq * bt_stride;
  const float slope = slopes ? slopes[head] : 0.f;
  const int c0 = NV == 1 ? kvh : blockIdx.z * NC;              // first value head of this wave
  const int n_c = NV == 1 ? 1 : min(NC, NV - blockIdx.z * NC);  // and how many

  u32x4 qf[NKS];
#pragma unroll
  for (int s = 0; s < NKS; ++s) {
    qf[s] = u32x4{0u, 0u, 0u, 0u};
    if (valid && 32 * s + 8 * g < HD)
      qf[s] = *reinterpret_cast<const u32x4*>(q + (size_t)tok * q_stride + (size_t)head * HD + 32 * s + 8 * g);
  }
  f32x4 o[NC][NDT];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[c][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  constexpr float LOG2E = 1.4426950408889634f;
  const size_t k_head = (size_t)HD * PS, v_head = (size_t)VD * PS;

  // a single token's keys may be split over `splits` waves (blockIdx.x % splits): each takes a run of whole blocks
  // the blocks of 64 keys: those of the kept first positions that lie before the window's first block, then the window's
  const int first_block = lo_min / 64, n_kept = lev_kept_blocks(lo_min, keep);
  int block_first = 0, block_last = n_kept + p_max / 64 - first_block;
  if (SINGLE && splits > 1) {
    const int per = (block_last + splits) / splits, z = WAVES > 1 ? (int)threadIdx.x >> 6 : blockIdx.x % splits;
    block_first = z * per;
    block_last = min(block_last, block_first + per - 1);
  }
  // Page ids of a block: of this lane's two groups of 8 keys (32u + 8g .. +7) and of its four operand rows. They are read one block
  // ahead, behind the block's own loads, and a block's keys and values are asked for together: with the values behind the softmax and a
  // key's page id ahead of each key, a short context (a block or two a wave) was a chain of round trips (8 tokens of 240 keys, heads of 256 and
  // 224: 15.0 -> 7.7 us; 32 tokens, heads of 64: 10.4 -> 7.9).
  // Loads stand under no condition: a branch would wait for everything in flight.
  int pgv[2], pgk[2][2];
  auto page_ids = [&](int bi) {
    const int key0 = lev_block_key(bi, n_kept, first_block);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      pgv[u] = bt[min(key0 + 32 * u + 8 * g, p_max) / PS];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) pgk[u][hh] = bt[min(key0 + 32 * u + 8 * (col >> 2) + 4 * hh + (col & 3), p_max) / PS];
    }
  };
  page_ids(block_first);
  for (int bi = block_first; bi <= block_last; ++bi) {
    const int key0 = lev_block_key(bi, n_kept, first_block);
    u32x4 kf[2][2][NKS], vf[NC][NDT][2];
    int page_of[2];  // of the two groups, -1: none
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int kpc = min(key0 + 32 * u + 8 * (col >> 2) + 4 * hh + (col & 3), p_max);  // the key of this lane's operand row
        const int page = max(pgk[u][hh], 0);  // a key without a page or beyond the range is masked below; its operand may be anything that can be read
        const bf16_t* kb = k_pages + ((size_t)page * KVH + kvh) * k_head + (size_t)(kpc % PS) * 8;
#pragma unroll
        for (int s = 0; s < NKS; ++s) kf[u][hh][s] = *reinterpret_cast<const u32x4*>(kb + (size_t)min(4 * s + g, HD / 8 - 1) * PS * 8);
      }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int kp = key0 + 32 * u + 8 * g;
      page_of[u] = kp <= p_max ? pgv[u] : -1;
      const bf16_t* vb = v_pages + (size_t)max(page_of[u], 0) * KVH * v_head + (size_t)col * PS + kp % PS;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (c == 0 || c < n_c) {  // the same for the whole wave
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) vf[c][dt][u] = *reinterpret_cast<const u32x4*>(vb + (size_t)(c0 + c) * v_head + (size_t)(16 * dt) * PS);
        }
    }
    page_ids(bi + 1);
    __builtin_amdgcn_sched_barrier(0);  // all of them are on their way before the first is waited for
    // scores: S^T tiles (u, h)
    f32x4 st[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NKS; ++s) {
          u32x4 k = kf[u][hh][s];
          if (HD % 32 != 0 && 4 * s + g >= HD / 8) k = u32x4{0u, 0u, 0u, 0u};
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(qf[s]), acc, 0, 0, 0);
        }
        st[u][hh] = acc;
      }
    // scale, cap, distance term, mask; in base 2 from here on
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int kp = key0 + 32 * u + 8 * g + 4 * hh + r;
          const bool ok = valid && lev_key_visible(kp, pos, lo, keep) && page_of[u] >= 0;
          float s = st[u][hh][r] * scale;
          if (softcap > 0.f) s = softcap * fast_tanh(s * __builtin_amdgcn_rcpf(softcap));
          s = (s - slope * (float)(pos - kp)) * LOG2E;
          s = ok ? s : -INFINITY;
          st[u][hh][r] = s;
          mx = fmaxf(mx, s);
        }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __builtin_amdgcn_exp2f(m - m_use);  // m = -inf: 0
    m = m_new;
    float psum = 0.f;
    u32x4 pf[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float p[8];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[4 * hh + r] = __builtin_amdgcn_exp2f(st[u][hh][r] - m_use);
          psum += p[4 * hh + r];
        }
#pragma unroll
      for (int e = 0; e < 4; ++e) pf[u][e] = float2_to_bf16x2(p[2 * e], p[2 * e + 1]);
    }
    l = l * corr + psum;
    // values of every value head of this wave
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c < n_c) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          f32x4 acc = o[c][dt] * corr;
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int kp = key0 + 32 * u + 8 * g;
            const u32x4 v = first_keys(vf[c][dt][u], page_of[u] >= 0 ? min(8, max(0, p_max - kp + 1)) : 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v), as_bf16x8(pf[u]), acc, 0, 0, 0);
          }
          o[c][dt] = acc;
        }
      }
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (WAVES > 1) {  // the merge of the kernel below (the same sums in the same order), a wave some tiles of the result
    extern __shared__ __attribute__((aligned(16))) unsigned char av_merge[];
    f32x4* po = reinterpret_cast<f32x4*>(av_merge);                       // [splits][NC * NDT][64]
    float2* ml = reinterpret_cast<float2*>(po + splits * NC * NDT * 64);  // [splits][16]
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (c == 0 || c < n_c) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) po[(wave * NC * NDT + c * NDT + dt) * 64 + lane] = o[c][dt];
      }
    if (g == 0) ml[wave * 16 + col] = make_float2(m, l);
    lds_barrier();
    float w[8], M = -INFINITY;
#pragma unroll
    for (int s = 0; s < WAVES; ++s) M = fmaxf(M, ml[min(s, splits - 1) * 16 + col].x);
    float v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const float2 q2 = ml[min(s, splits - 1) * 16 + col];
      w[s] = s < splits ? __builtin_amdgcn_exp2f(q2.x - (M == -INFINITY ? 0.f : M)) : 0.f;
      v[s] = s < splits ? w[s] * q2.y : 0.f;
    }
    float L = ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
    if (sinks != nullptr) L = M == -INFINITY ? 1.0f : L + __builtin_amdgcn_exp2f(sinks[head] * LOG2E - M);
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    float* ob = out + (((size_t)tok * H + head) * NV + (NV == 1 ? 0 : c0)) * VD + 4 * g;
    for (int t = wave; t < n_c * NDT; t += splits) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < WAVES; ++s) {  // beyond the ranges: weight 0
        const f32x4 part = po[(min(s, splits - 1) * NC * NDT + t) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(w[s], part[r], acc[r]);
      }
      if (valid) *reinterpret_cast<f32x4*>(ob + 16 * t) = acc * inv;
    }
    return;
  }
  if (!valid) return;
  if (SINGLE && splits > 1) {  // unnormalised sums, the maximum and the sum of weights: merged by the kernel below
    const size_t slot = ((size_t)blockIdx.x * H + head);  // (token index, split) major, then head
    if (g == 0 && blockIdx.z == 0) {
      part_ml[2 * slot] = m;
      part_ml[2 * slot + 1] = l;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c < n_c) {
        float* ob = part_o + (slot * NV + (NV == 1 ? 0 : c0 + c)) * VD;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<f32x4*>(ob + 16 * dt + 4 * g) = o[c][dt];
      }
    }
    return;
  }
  if (sinks != nullptr) l = m == -INFINITY ? 1.0f : l + __builtin_amdgcn_exp2f(sinks[head] * LOG2E - m);  // m is in base 2
  const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c < n_c) {
      float* ob = out + (((size_t)tok * H + head) * NV + (NV == 1 ? 0 : c0 + c)) * VD;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<f32x4*>(ob + 16 * dt + 4 * g) = o[c][dt] * inv;
    }
  }
}

// Runs of several tokens: one workgroup per (tile of up to PF_ROWS consecutive query tokens or half of one, query head,
// set of value heads). The keys and values of a block of 64 positions are staged once for all waves: global -> registers
// (requested a block ahead) -> LDS, with everything beyond the last written key made zero on the way (from the registers, not when they are asked
// for: that would wait for them).
// What bounds it: the chain of a block (two barriers, scores, softmax, values) in the workgroups of the longest tiles, few of which share a CU; in short runs the trips to memory ahead of the first
// block. So the operands of the products come from LDS four at a time, a group ahead, instead of each ahead of its product; a block has no branch for its scores; the maximum goes over the lanes by swaps, and the outputs
// are scaled only when one was raised. The next block is asked for in one set of registers (of two sets, one of which a branch picked, the loads went to a third, were waited for
// and copied there, in every block), behind the last none; the queries are asked for under no condition: in a branch each, they were waited for one by one (wide heads, twelve runs of 150: 29 -> 24 us).
// Microseconds a layer, 16 heads, two sets of registers and each operand ahead of its product / all that now:
//                    128 / 64      64 / 64      144 / 112    256 / 224
//   1,000 tokens     36.9 / 23.8   31.6 / 22.4  44.3 / 33.2  58.8 / 45.4
//   two of 1,015     40.1 / 30.8   33.8 / 26.5  47.3 / 34.7  62.7 / 48.6
//   six of 1,000     79.5 / 67     68.3 / 59    130 / 99     176 / 137
//   twelve of 150    12.6 / 11.1   10.7 / 10.4  18.6 / 17.5  26.6 / 23.8
//   32 of 60          9.5 /  9.1    9.3 /  9.2  13.0 / 12.2  18.8 / 17.4
//   64 of 30         13.7 / 12.6   12.2 / 12.0  18.8 / 17.2  29.1 / 26.6
//   32 of 70, 200 keys  16.8 / 14.9  15.9 / 14.3  27.3 / 23.4  37.7 / 31.7
#define RUN_MAX_LDS (80 * 1024)  // bytes a workgroup may take: two workgroups a CU
#define RUN_PAGES 2048  // page ids of a tile's key range that are kept in LDS

// Waves of a workgroup, 16 query tokens each: half a tile's, where three such workgroups fit a CU's registers (heads of 128 / 64, microseconds, whole tiles / halves: 1,000 tokens 28.3 / 24.5,
// two of 1,015 30.7 / 30.4; of 256 / 224 two of 1,015 55 / 100: the loads of a block are twice as many registers a thread).
#define RUN_WAVES (HD + VD <= 192 ? PF_WAVES / 2 : PF_WAVES)

// Whole tiles whose operands are read without a group ahead, in registers for two workgroups a CU (of 16 heads of 128 / 64, us, so / as above): where tiles are half empty, so that so
// are the halves (64 runs of 30: 12.6 / 15.9; of 30 behind 60 keys 17.0 / 22.6), and where there are more of them than the 768 halves that three a CU are (32 of 70, 200 keys 14.9 / 21.1; 32 of 128 12.8 / 16.2; 24 of 128
// still 11.6 / 11.2; eight of 1,000 79 / 88), but for the smallest heads, of whose halves a CU holds four (12 heads of 64 / 32, 64 runs of 96: 14.1 / 12.5). Heads beyond 192 numbers, which have no halves: where tiles are half
// empty and contexts short (144 / 112, 64 runs of 30: 17.2 / 21.5; 16 of 64 over 1,000 keys 32.3 / 29.7); beyond 256 never: their registers leave one workgroup a CU either way (256 / 224, 64 of 30: 27.3 / 26.6).
static bool av_whole_tiles(int n_tiles, int tokens, int H, int max_keys) {
  const bool half_empty = tokens <= PF_ROWS / 2 * n_tiles;
  if (HD + VD > 192) return HD + VD <= 256 && half_empty && max_keys <= 256;
  return half_empty || (HD + VD >= 128 && (long)n_tiles * H > 384);
}

// NC: value heads that a wave has room for, as above: 1, or NVC for layers with more
// D - 1: groups of operands that are read ahead
template <int NC, int WAVES, int D>
__global__ void __launch_bounds__(64 * WAVES, WAVES == PF_WAVES ? 2 : 3)
attention_values_mfma_runs_kernel(const bf16_t* __restrict__ q, long q_stride, float* __restrict__ out, const bf16_t* __restrict__ k_pages,
                                  const bf16_t* __restrict__ v_pages, const int* __restrict__ positions, const int* __restrict__ token_seq,
                                  const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tiles, int H, int KVH, int NV,
                                  int PS, float scale, int window, int chunk, int keep, float softcap, const float* __restrict__ slopes,
                                  const float* __restrict__ sinks) {
  constexpr int THREADS = 64 * WAVES, PARTS = PF_ROWS / (16 * WAVES);
  constexpr int K_STAGE = (HD * 8 + THREADS - 1) / THREADS, V_STAGE = (NC * VD * 8 + THREADS - 1) / THREADS;  // 16-byte chunks of a block of keys, of values per thread
  extern __shared__ __attribute__((aligned(16))) unsigned char av_smem[];
  bf16_t* ks = reinterpret_cast<bf16_t*>(av_smem);  // [HD/8][64][8]
  bf16_t* vs = ks + HD * 64;                        // [8 chunks][n_c VD][8]
  __shared__ int pages_s[RUN_PAGES];                // page ids of the blocks that the tile's keys lie in
  __shared__ __attribute__((aligned(16))) bf16_t zeros[HD % 32 != 0 ? 3 * 128 + 8 : 8];  // keys' dimensions beyond HD, read from as far apart as those of keys are
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, g = lane >> 4;
  const int tile = blockIdx.x / PARTS, skip = (blockIdx.x - tile * PARTS) * 16 * WAVES;
  const int first = tiles[2 * tile] + skip, n = min(tiles[2 * tile + 1] - skip, 16 * WAVES);
  if (n <= 0) return;  // the whole workgroup
  const int head = blockIdx.y, group = H / KVH, kvh = head / group;
  const bool active = wave * 16 < n;            // this wave has query rows
  const bool valid = wave * 16 + col < n;       // this lane's column is one of them
  const int tok = first + (valid ? wave * 16 + col : 0);
  const int pos0 = positions[first];
  const int pos = pos0 + (tok - first);         // a run's tokens stand at consecutive positions
  const int lo = lev_first_visible(pos, window, chunk);
  const int p_max_wg = pos0 + n - 1, lo_wg = lev_first_visible(pos0, window, chunk);
  const int p_min = pos0 + wave * 16, p_max = min(p_max_wg, p_min + 15);                    // this wave's rows
  const int lo_min = lev_first_visible(p_min, window, chunk), lo_max = lev_first_visible(p_max, window, chunk);
  const int* bt = block_tables + (size_t)token_seq[first] * bt_stride;
  const float slope = slopes ? slopes[head] : 0.f;
  const int c0 = NV == 1 ? kvh : blockIdx.z * NC;
  const int n_c = NV == 1 ? 1 : min(NC, NV - blockIdx.z * NC);
  const int key_begin = (lo_wg / 64) * 64;
  // A key's page: from LDS, where the page ids of the tile's whole key range were put once (a look-up in global memory ahead
  // of every operand load would put two memory latencies in a row into every block). Pages are powers of two in practice:
  // a shift then, a division otherwise.
  const int sh = (PS & (PS - 1)) == 0 ? __builtin_ctz(PS) : -1;
  auto block_of = [&](int kp) { return sh >= 0 ? kp >> sh : kp / PS; };
  const int pg0 = block_of(key_begin), n_pg = block_of(p_max_wg) - pg0 + 1;
  // with kept first positions the tile also reads the n_kept blocks of 64 keys that hold them and lie before key_begin: their
  // page ids stand at the table's start, those of the range from key_begin on behind them
  const int first_block = lo_wg / 64, n_kept = lev_kept_blocks(lo_wg, keep), n_blocks = n_kept + p_max_wg / 64 - first_block + 1;
  const int n_kpg = n_kept > 0 ? block_of(n_kept * 64 - 1) + 1 : 0;
  int none = 0;  // negative: a page that holds a key in sight is missing
  for (int i = tid; i < min(n_kpg, RUN_PAGES); i += THREADS) {
    const int page = bt[i];
    pages_s[i] = page, none |= i * PS < keep ? page : 0;
  }
  for (int i = tid; i < min(n_pg, RUN_PAGES - n_kpg); i += THREADS) {  // the host sends longer ranges elsewhere
    const int page = bt[pg0 + i];
    pages_s[n_kpg + i] = page, none |= (pg0 + i + 1) * PS > lo_wg ? page : 0;
  }
  // The page of a key of the block at key0 (within the tile's range or among the kept blocks) and the key's place in it, from the number and the
  // first key of the page that key0 lies in (one division a block). The distance from there is below PS + 64: its quotient in 16 bits is exact.
  const int sixteenths = PS < 64 ? (65536 + PS - 1) / PS : 0;
  auto place_of = [&](int kp, int page_no, int page_key, int& at) {
    const int r = kp - page_key, over = PS < 64 ? r * sixteenths >> 16 : r >= PS, b = page_no + over;
    at = r - over * PS;
    return pages_s[b >= pg0 ? n_kpg + b - pg0 : b];
  };

  u32x4 qf[NKS];
#pragma unroll
  for (int s = 0; s < NKS; ++s) {
    qf[s] = *reinterpret_cast<const u32x4*>(q + (size_t)tok * q_stride + (size_t)head * HD + (HD % 32 == 0 ? 32 * s + 8 * g : min(32 * s + 8 * g, HD - 8)));
  }
  f32x4 o[NC][NDT];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[c][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  constexpr float LOG2E = 1.4426950408889634f;
  const size_t k_head = (size_t)HD * PS, v_head = (size_t)VD * PS;
  const bool all_pages = __syncthreads_or(none < 0) == 0;  // the page ids are there, and every key in sight has a page

  // In LDS a chunk of 8 dimensions has its 64 keys in the order in which the score tiles have them as rows, and a chunk of 8 keys' values its rows in their
  // order but for a turn by twice the chunk's number: 16 lanes' reads, and what neighbouring lanes write, fall on all banks.
  const int v_rows = NC == 1 ? VD : n_c * VD;
  const bf16_t* ks_get = ks + (g * 64 + col) * 8;
  const bf16_t* ks_get_last = 32 * (NKS - 1) + 8 * g < HD ? ks_get + 4 * (NKS - 1) * 64 * 8 : zeros;
  const bf16_t* vs_get[2] = {vs + (g * v_rows + (col ^ 2 * g)) * 8, vs + ((4 + g) * v_rows + (col ^ (8 + 2 * g))) * 8};
  bf16_t* ks_put = ks + ((tid & ~63) + (tid & 32) + 16 * (tid >> 2 & 1) + 4 * (tid >> 3 & 3) + (tid & 3)) * 8;
  u32x4 kst[K_STAGE], vst[V_STAGE];  // the next block, on its way
  // This thread's chunks of the block at key0, from the pages into registers: chunks of one key, and of one group of 8 keys' values.
  // Every load stands under no condition (a load in a branch makes the compiler wait for all loads in flight where the
  // branch ends): addresses are clamped into what can be read, what must not count is made zero when it goes to LDS.
  auto fetch = [&](int key0) __attribute__((always_inline)) {
    const int page_no = block_of(key0), page_key = page_no * PS;
    int ka, va;
    const int kpage = place_of(min(key0 + (tid & 63), p_max_wg), page_no, page_key, ka);
    const int vpage = place_of(min(key0 + 8 * (tid & 7), p_max_wg & ~7), page_no, page_key, va);
    const bf16_t* kb = k_pages + ((size_t)max(kpage, 0) * KVH + kvh) * k_head + (size_t)ka * 8;
    const bf16_t* vb = v_pages + ((size_t)max(vpage, 0) * KVH + c0) * v_head + va;
#pragma unroll
    for (int i = 0; i < K_STAGE; ++i) kst[i] = *reinterpret_cast<const u32x4*>(kb + min((tid >> 6) + THREADS / 64 * i, HD / 8 - 1) * PS * 8);
#pragma unroll
    for (int i = 0; i < V_STAGE; ++i) vst[i] = *reinterpret_cast<const u32x4*>(vb + (size_t)min((tid >> 3) + THREADS / 8 * i, n_c * VD - 1) * PS);
  };
  auto stage = [&](int key0) __attribute__((always_inline)) {
    if (!all_pages || key0 + 63 > p_max_wg || !(key0 >= lo_wg || key0 + 63 < keep)) {  // keys without values: the same for the whole workgroup
      const int page_no = block_of(key0), page_key = page_no * PS, kp = key0 + (tid & 63), vp = key0 + 8 * (tid & 7);
      int at;
      const bool in = kp <= p_max_wg && place_of(min(kp, p_max_wg), page_no, page_key, at) >= 0;
      const int count = place_of(min(vp, p_max_wg & ~7), page_no, page_key, at) >= 0 ? min(8, max(0, p_max_wg - vp + 1)) : 0;
#pragma unroll
      for (int i = 0; i < K_STAGE; ++i)
        if (!in) kst[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < V_STAGE; ++i) vst[i] = first_keys(vst[i], count);
    }
#pragma unroll
    for (int i = 0; i < K_STAGE; ++i)
      if (HD * 8 % THREADS == 0 || tid + THREADS * i < HD * 8) *reinterpret_cast<u32x4*>(ks_put + THREADS * 8 * i) = kst[i];
#pragma unroll
    for (int i = 0; i < V_STAGE; ++i) {
      const int row = (tid >> 3) + THREADS / 8 * i;
      if ((NC == 1 && VD * 8 % THREADS == 0) || row < v_rows) *reinterpret_cast<u32x4*>(vs + ((tid & 7) * v_rows + (row ^ 2 * (tid & 7))) * 8) = vst[i];
    }
  };

  if (HD % 32 != 0 && tid < 4 * 8) zeros[(tid >> 3) * 128 + (tid & 7)] = 0;
  fetch(lev_block_key(0, n_kept, first_block));
  if (HD % 32 != 0 && 32 * (NKS - 1) + 8 * g >= HD) qf[NKS - 1] = u32x4{0u, 0u, 0u, 0u};
  for (int it = 0; it < n_blocks; ++it) {
    const int key0 = lev_block_key(it, n_kept, first_block);
    lds_barrier();  // the block before has been read by every wave (a barrier for LDS only: the loads on their way stay there)
    stage(key0);
    if (it + 1 < n_blocks) fetch(lev_block_key(it + 1, n_kept, first_block));  // the same for the workgroup
    lds_barrier();
    if (!active || key0 > p_max || (key0 + 63 < lo_min && key0 >= keep)) continue;  // none of this wave's rows sees a key of this block
    // Four operands at a time come from LDS, two such groups ahead of the products: keys (a score tile and up to four k-steps; the tiles in turn), then values (two tiles of 16
    // dimensions), the first of them before the softmax.
    constexpr int KC = (NKS + 3) / 4, NGK = 4 * KC, NGV1 = (NDT + 1) / 2, NGV = NC * NGV1;
    u32x4 fr[D][4];
    f32x4 st[2][2];
    auto read = [&](int group) __attribute__((always_inline)) {
      u32x4 (&to)[4] = fr[group % D];
      if (group < NGK) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int s = group / 4 * 4 + e;
          if (s >= NKS) break;
          to[e] = *reinterpret_cast<const u32x4*>((HD % 32 != 0 && s == NKS - 1 ? ks_get_last : ks_get + 4 * s * 64 * 8) + 16 * (group % 4) * 8);
        }
      } else if (group < NGK + NGV) {
        const int c = (group - NGK) / NGV1, dt0 = (group - NGK) % NGV1 * 2;
        const int row0 = (NC == 1 ? 0 : min(c, n_c - 1)) * VD + 16 * dt0;  // of heads beyond the last: read, not used
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (dt0 + e / 2 < NDT) to[e] = *reinterpret_cast<const u32x4*>(vs_get[e & 1] + (row0 + e / 2 * 16) * 8);
      }
    };
#pragma unroll
    for (int group = 0; group < D - 1; ++group) read(group);
#pragma unroll
    for (int group = 0; group < NGK; ++group) {
      read(group + D - 1);
      __builtin_amdgcn_sched_barrier(0);
      f32x4& acc = st[group % 4 >> 1][group & 1];
      if (group < 4) acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (group / 4 * 4 + e < NKS) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fr[group % D][e]), as_bf16x8(qf[group / 4 * 4 + e]), acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // scale, cap, distance term; in base 2 from here on
    float mx = -INFINITY;
    const float dist0 = (float)(pos - key0 - 8 * g);  // whole numbers: exact
    if (softcap > 0.f) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int r = 0; r < 4; ++r) st[u][hh][r] = fmaf(-slope, dist0 - (float)(32 * u + 4 * hh + r), softcap * fast_tanh(st[u][hh][r] * scale * __builtin_amdgcn_rcpf(softcap))) * LOG2E;
    } else {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int r = 0; r < 4; ++r) st[u][hh][r] = fmaf(-slope, dist0 - (float)(32 * u + 4 * hh + r), st[u][hh][r] * scale) * LOG2E;
    }
    if (!all_pages || key0 + 63 > p_min || !(key0 >= lo_max || key0 + 63 < keep)) {  // a row that does not see every key: the same for the whole wave
      const int page_no = block_of(key0), page_key = page_no * PS;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int kg = key0 + 32 * u + 8 * g;
        int at;
        const bool there = valid && kg <= p_max && place_of(min(kg, p_max_wg), page_no, page_key, at) >= 0;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int r = 0; r < 4; ++r) st[u][hh][r] = there && lev_key_visible(kg + 4 * hh + r, pos, lo, keep) ? st[u][hh][r] : -INFINITY;
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[u][hh][r]);
    {  // over the lanes 16, 32 and 48 further on, by the lane-swap instructions
      typedef __attribute__((ext_vector_type(2))) uint32_t pair_t;
      const pair_t a = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
      const pair_t b = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
    }
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __builtin_amdgcn_exp2f(m - m_use);
    m = m_new;
    float psum = 0.f;
    u32x4 pf[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float p[8];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma clang fp contract(off)  // the rounded score, as the maximum holds it
          const float below = st[u][hh][r] - m_use;
          p[4 * hh + r] = __builtin_amdgcn_exp2f(below);
          psum += p[4 * hh + r];
        }
#pragma unroll
      for (int e = 0; e < 4; ++e) pf[u][e] = float2_to_bf16x2(p[2 * e], p[2 * e + 1]);
    }
    l = l * corr + psum;
    if (__any(corr != 1.f)) {  // some row's maximum was raised
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[c][dt] *= corr;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NGV; ++v) {
      const int c = v / NGV1, dt0 = v % NGV1 * 2;
      if (NC > 1 && c > 0 && c >= n_c) break;
      if (v + D - 1 < NGV) read(NGK + v + D - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (dt0 + t < NDT) o[c][dt0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fr[(NGK + v) % D][2 * t + u]), as_bf16x8(pf[u]), o[c][dt0 + t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (!valid) return;
  if (sinks != nullptr) l = m == -INFINITY ? 1.0f : l + __builtin_amdgcn_exp2f(sinks[head] * LOG2E - m);  // m is in base 2
  const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c < n_c) {
      float* ob = out + (((size_t)tok * H + head) * NV + (NV == 1 ? 0 : c0 + c)) * VD;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<f32x4*>(ob + 16 * dt + 4 * g) = o[c][dt] * inv;
    }
  }
}

// Merges the splits of a single token's keys: out[tok][head] = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s, in the order of s.
#define MERGE_MAX_SPLITS 32
__global__ void __launch_bounds__(64)
attention_values_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ singles,
                              float* __restrict__ out, int H, int n_out, int splits, const float* __restrict__ sinks) {
  __shared__ float w_s[MERGE_MAX_SPLITS + 8];
  const int idx = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  // lane s holds split s's maximum and sum; loads stand under no condition (clamped index, the value replaced afterwards)
  const float* ml = part_ml + 2 * (((size_t)idx * splits + min(lane, splits - 1)) * H + head);
  const float mv = ml[0], lv = ml[1];
  const float ms = lane < splits ? mv : -INFINITY;
  const float M = wave_max(ms);
  const float w = __builtin_amdgcn_exp2f(ms - (M == -INFINITY ? 0.f : M));  // a split without keys, a lane without a split: 0
  float L = wave_sum(w * (lane < splits ? lv : 0.f));
  if (sinks != nullptr) L = M == -INFINITY ? 1.0f : L + __builtin_amdgcn_exp2f(sinks[head] * 1.4426950408889634f - M);
  if (lane < MERGE_MAX_SPLITS + 8) w_s[lane] = w;
  __syncthreads();
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  float* o = out + ((size_t)singles[idx] * H + head) * n_out;
  const float* po = part_o + ((size_t)idx * splits * H + head) * n_out;
  for (int e = lane; e < n_out; e += 64) {
    float acc = 0.f;
    for (int s0 = 0; s0 < splits; s0 += 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j)  // lanes beyond the splits hold weight 0: what they read twice does not count
        acc = fmaf(w_s[s0 + j], po[(size_t)min(s0 + j, splits - 1) * H * n_out + e], acc);
    }
    o[e] = acc * inv;
  }
}

// Key ranges that one workgroup's waves take: eight where a wave's operands and sums leave it half of a lane's 512 registers, else four
template <int NC>
constexpr int av_waves() { return 20 * NKS + 12 * NDT * NC > 160 ? 4 : 8; }
static int av_room(int NV) {  // value heads of a wave of the kernels without shared operands
  int room = 1;
  while (room < NV && room < NVC) room *= 2;
  return room;
}
// Whether a token's ranges are the waves of one workgroup. That saves a launch and a way through memory and puts their reads on one CU, which takes about 50
// KB a microsecond: not where that CU then reads over 192 KB more than if the waves lay apart. Over 11 pairs of head sizes, 1 .. 128 tokens of 70 .. 2,000 keys (pages that
// no cache holds) 541 launches merge, at 0.94 - 1.61 times the speed of two, 1.29 on average; 5 of them, with ranges of 1,000 keys or right at the limit, are 3 - 6 % slower. 8 tokens
// of 240 keys, four ranges, before / now: heads of 256 / 224 (180 KB more) 11.3 / 8.7 us, 4 heads of 128 / 64 (72 KB) 8.6 / 6.9.
static bool av_merged(int n_singles, int splits, int H, int KVH, int NV, int window, int chunk, int keep, int max_keys) {
  const int room = av_room(NV);
  if (splits <= 1 || splits > (room == 1 ? av_waves<1>() : room == 2 ? av_waves<2>() : room == 4 ? av_waves<4>() : av_waves<8>())) return false;
  const long groups = (long)n_singles * KVH * ((H / KVH + 15) / 16) * (NV == 1 ? 1 : (NV + NVC - 1) / NVC);
  long reach = window > 0 && window < max_keys ? window : max_keys;
  if (chunk > 0 && chunk < reach) reach = chunk;
  reach += keep > 0 ? keep : 0;
  const long wave_bytes = ((reach + 63) / 64 + splits - 1) / splits * 64 * (HD + (NV < room ? NV : room) * VD) * 2;
  const long apart = (groups * splits + 255) / 256, together = (groups + 255) / 256 * splits;
  return (together - apart) * wave_bytes <= 192 * 1024;
}

// bytes of scratch memory for n single tokens whose keys are split `splits` ways; none where a workgroup merges them
extern "C" long lev_attention_values_mfma_workspace(int n_singles, int splits, int H, int KVH, int NV, int window, int chunk, int keep, int max_keys) {
  if (splits <= 1 || n_singles <= 0 || KVH <= 0 || av_merged(n_singles, splits, H, KVH, NV, window, chunk, keep, max_keys)) return 0;
  return (long)n_singles * splits * H * ((long)NV * VD + 2) * (long)sizeof(float);
}

extern "C" int lev_attention_values_mfma(const void* q, long q_stride, float* out, const void* k_pages, const void* v_pages,
                                         const int* positions, const int* token_seq, const int* block_tables, int bt_stride,
                                         const int* tiles, int n_tiles, const int* singles, int n_singles, int n_positions, int H, int KVH, int HD_,
                                         int VD_, int NV, int PS, float scale, int window, int chunk, int keep, float softcap, const float* slopes,
                                         const float* sinks, int splits, float* workspace, int max_keys, hipStream_t stream) {
  LEV_REQUIRE(HD_ == HD && VD_ == VD, "attention: this library was built for head sizes %d / %d, not %d / %d", HD, VD, HD_, VD_);
  LEV_REQUIRE(H > 0 && KVH > 0 && H % KVH == 0, "attention: bad head counts heads=%d kv_heads=%d", H, KVH);
  LEV_REQUIRE(NV == 1 || NV == KVH, "attention: %d value heads per query head (1 or kv_heads=%d)", NV, KVH);
  LEV_REQUIRE(PS > 0 && PS % 16 == 0, "attention: page_size=%d must be a multiple of 16", PS);
  LEV_REQUIRE(window >= 0 && chunk >= 0 && keep >= 0 && softcap >= 0.f, "attention: window=%d, chunk=%d, kept positions %d and soft cap %g must not be negative", window, chunk, keep, (double)softcap);
  LEV_REQUIRE(splits >= 1 && splits <= MERGE_MAX_SPLITS, "attention: %d splits (at most %d)", splits, MERGE_MAX_SPLITS);
  const bool merged = n_singles > 0 && av_merged(n_singles, splits, H, KVH, NV, window, chunk, keep, max_keys);
  LEV_REQUIRE(splits == 1 || merged || workspace, "attention: %d splits (at most %d) need scratch memory", splits, MERGE_MAX_SPLITS);
  LEV_REQUIRE(n_tiles >= 0 && n_singles >= 0 && (n_tiles == 0 || tiles) && (n_singles == 0 || (singles && n_positions > 0)), "attention: bad work lists");
  LEV_REQUIRE(((uintptr_t)q & 15) == 0 && q_stride % 8 == 0 && ((uintptr_t)k_pages & 15) == 0 && ((uintptr_t)v_pages & 15) == 0 &&
                  ((uintptr_t)out & 15) == 0,
              "attention: operands must be 16-byte aligned");
  const int chunks = NV == 1 ? 1 : (NV + NVC - 1) / NVC;
  const int room = av_room(NV);
  LEV_REQUIRE(H <= 65535 && chunks <= 65535, "attention: too many heads (%d)", H);
#define AV_ROOM(SINGLE, NC, WAVES, LDS, GRID, WORK, SPLITS, PART_O, PART_ML)                                                                              \
  if constexpr (NC <= NVC)                                                                                                                              \
    if (room == NC) {                                                                                                                                   \
      const size_t lds = LDS(NC);                                                                                                                       \
      if (lds > 64 * 1024) { /* more than a kernel gets unasked */                                                                                      \
        hipError_t e = hipFuncSetAttribute((const void*)attention_values_mfma_kernel<SINGLE, NC, WAVES>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
        LEV_REQUIRE(e == hipSuccess, "attention: %zu bytes of LDS a workgroup: %s", lds, hipGetErrorString(e));                                         \
      }                                                                                                                                                 \
      attention_values_mfma_kernel<SINGLE, NC, WAVES><<<GRID, WAVES > 1 ? 64 * SPLITS : 64, lds, stream>>>(                                             \
          (const bf16_t*)q, q_stride, out, (const bf16_t*)k_pages, (const bf16_t*)v_pages, positions, token_seq, block_tables, bt_stride, WORK, n_positions, H, KVH, \
          NV, PS, scale, window, chunk, keep, softcap, slopes, SPLITS, PART_O, PART_ML, sinks);                                                         \
    }
#define AV_NO_LDS(NC) 0
#define AV_MERGE_LDS(NC) ((size_t)splits * (NC * NDT * 64 * sizeof(f32x4) + 16 * sizeof(float2)))
#define AV_ROOMS(SINGLE, WAVES, LDS, GRID, WORK, SPLITS, PART_O, PART_ML)       \
  do {                                                                          \
    AV_ROOM(SINGLE, 1, WAVES(1), LDS, GRID, WORK, SPLITS, PART_O, PART_ML);     \
    AV_ROOM(SINGLE, 2, WAVES(2), LDS, GRID, WORK, SPLITS, PART_O, PART_ML);     \
    AV_ROOM(SINGLE, 4, WAVES(4), LDS, GRID, WORK, SPLITS, PART_O, PART_ML);     \
    AV_ROOM(SINGLE, 8, WAVES(8), LDS, GRID, WORK, SPLITS, PART_O, PART_ML);     \
  } while (0)
#define AV_ONE_WAVE(NC) 1
#define AV_MANY_WAVES(NC) av_waves<NC>()
  if (n_tiles > 0) {
    const size_t lds = ((size_t)HD * 64 + (size_t)(NV == 1 ? 1 : (NV < NVC ? NV : NVC)) * VD * 64) * sizeof(bf16_t);
    // the page ids of a tile's key range (the window, or all keys so far, and the tile itself) must fit their LDS table
    long reach = window > 0 && window < max_keys ? window : max_keys;
    if (chunk > 0 && chunk < reach) reach = chunk;
    reach += PF_ROWS + 64 + (keep > 0 ? keep + 64 + PS : 0);
    const size_t all_lds = lds + RUN_PAGES * sizeof(int) + (HD % 32 != 0 ? 1024 : 0);
#define AV_RUNS(NC, WAVES, D)                                                                                                                          \
  do {                                                                                                                                                 \
    if (all_lds > 64 * 1024) { /* more than a kernel gets unasked */                                                                                   \
      hipError_t e = hipFuncSetAttribute((const void*)attention_values_mfma_runs_kernel<NC, WAVES, (D)>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
      LEV_REQUIRE(e == hipSuccess, "attention: %zu bytes of LDS a workgroup: %s", all_lds, hipGetErrorString(e));                                      \
    }                                                                                                                                                  \
    attention_values_mfma_runs_kernel<NC, WAVES, (D)><<<dim3(n_tiles * (PF_WAVES / (WAVES)), H, chunks), 64 * (WAVES), lds, stream>>>(                   \
        (const bf16_t*)q, q_stride, out, (const bf16_t*)k_pages, (const bf16_t*)v_pages, positions, token_seq, block_tables, bt_stride, tiles, H, KVH, NV, PS, scale, window, \
        chunk, keep, softcap, slopes, sinks);                                                                                                          \
  } while (0)
    if (all_lds <= RUN_MAX_LDS && reach / PS + 2 <= RUN_PAGES) {
      if (NV > 1) AV_RUNS(NVC, PF_WAVES, 2);
      else if (av_whole_tiles(n_tiles, n_positions - n_singles, H, max_keys)) AV_RUNS(1, PF_WAVES, HD + VD <= 256 ? 1 : 2);
      else AV_RUNS(1, RUN_WAVES, 2);
    }
#undef AV_RUNS
    else  // the longest ranges: every wave by itself, operands straight from the pages
      AV_ROOMS(false, AV_ONE_WAVE, AV_NO_LDS, dim3(n_tiles * SUB_TILES, H, chunks), tiles, 1, nullptr, nullptr);
    if (lev_check_launch("attention_values_mfma (runs)")) return -1;
  }
  if (n_singles > 0) {
    const int group = H / KVH;
    dim3 grid(merged ? n_singles : n_singles * splits, KVH * ((group + 15) / 16), chunks);
    float* part_o = workspace;
    float* part_ml = splits > 1 && !merged ? workspace + (size_t)n_singles * splits * H * NV * VD : nullptr;
    if (merged) AV_ROOMS(true, AV_MANY_WAVES, AV_MERGE_LDS, grid, singles, splits, nullptr, nullptr);
    else AV_ROOMS(true, AV_ONE_WAVE, AV_NO_LDS, grid, singles, splits, part_o, part_ml);
#undef AV_MANY_WAVES
#undef AV_ONE_WAVE
#undef AV_ROOMS
#undef AV_MERGE_LDS
#undef AV_NO_LDS
#undef AV_ROOM
    if (lev_check_launch("attention_values_mfma (single tokens)")) return -1;
    if (splits > 1 && !merged) {
      attention_values_merge_kernel<<<dim3(n_singles, H), 64, 0, stream>>>(part_o, part_ml, singles, out, H, NV * VD, splits, sinks);
      if (lev_check_launch("attention_values_mfma (merge)")) return -1;
    }
  }
  return 0;
}
