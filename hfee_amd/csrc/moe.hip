// A feed-forward of many small gated experts, of which every token uses `top`.
//
// Which experts a token uses is given from outside as int32 [n, top] (`chosen`), or looked up here in
// a table [vocabulary, top] under the token's id; expert e of a token counts with pair_weights[t][j]
// or, without them, with the one number `weight`.
//
//   up:    act[t][j][f] = silu(W_gate[e][f] . h_t) * (W_up[e][f] . h_t),   e = the j-th expert of t
//   down:  x[t][c] (+)= sum_j weight_tj (W_down[e_j][c] . act[t][j])
//
// With gate_act GATE_CLIPPED the experts' gate is the clipped one of common.h (two numbers, `limit` and `sharpness`).
//
// Experts without a gate (`form` 1, no W_gate): act[t][j][f] = relu(w_tj (W_up[e][f] . h_t))^2, where w_tj
// (in_weights, or one) multiplies the expert's input: a product is linear, so the number meets the sum in
// float32 before the activation instead of every element of h before it is rounded.
//
// router_topk: scores of router logits z (float32 [n, experts], plus a bias an expert where one is given); the
// `top` largest choose a token's experts (the lower number of two equal ones), its pair weights are the chosen
// scores: sigmoids, or the softmax over all experts, as they are, or the softmax over the chosen ones only; or the
// chosen scores divided by their sum and multiplied by a number.  With groups the experts are cut into equal groups of
// neighbours, and only those of the groups with the largest best scores can be chosen.
//
// An expert number at or beyond the number of stacked matrices stands for no matrix: the kernels here leave such a
// pair alone (grouped_rows.hip adds what it stands for).
//
// The experts' matrices are stacked [experts][rows][columns].  Two forms:
//
// Token by token (moe_up, moe_down): a wave a dot product, lanes over the summed dimension, added up in a
// fixed order; every token reads the rows of its own experts.  For steps of few tokens, whose time is
// the experts' bytes, and for float32.  In bfloat16 up to 64 (token, expert) pairs also go expert by expert
// (moe_up_by_expert, moe_down_by_expert), an expert's rows once for up to four of its pairs, with the same sums.
//
// Grouped (moe_group, moe_group_tiled, moe_combine; bfloat16): the (token, expert) pairs of a step are put
// in the order of their experts on the device, cut into tiles of up to 192 pairs of one expert, and a workgroup
// multiplies a tile by 256 rows of that expert's matrix on the matrix cores, both operands straight into LDS
// (moe_direct; sizes that are no multiples of 64 and many pairs of a width of 64: tiles of 64 pairs by way of registers):
// an expert's matrices are read once for its pairs and not once a pair.  A pair's numbers do not depend on which pairs share its tile.
#include "common.h"

#include <cmath>
#include <type_traits>

using namespace hfee;

namespace {

__device__ __forceinline__ int expert_of(const int* chosen, const int* table, const int* token_ids, int t, int j, int top) {
  return chosen != nullptr ? chosen[(int64_t)t * top + j] : table[(int64_t)token_ids[t] * top + j];
}

constexpr int kRowsPerWave = 4;

// sum_c a[c] b[c] and sum_c a2[c] b[c] over `count` elements, a lane's share: lanes take turns of one
// element, or of eight bfloat16 (sixteen bytes) where count is a multiple of eight and the rows are aligned.
template <typename T>
__device__ __forceinline__ void two_dots(const T* a, const T* a2, const T* b, int count, int lane, bool wide, float& s, float& s2) {
  s = s2 = 0.f;
  if constexpr (sizeof(T) == 2) {
    if (wide) {
      typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
      for (int c = lane * 8; c < count; c += 64 * 8) {
        const u32x4_t va = load_streamed(reinterpret_cast<const u32x4_t*>(a + c));
        const u32x4_t vb = *reinterpret_cast<const u32x4_t*>(b + c);
        u32x4_t va2 = va;
        if (a2 != nullptr) va2 = load_streamed(reinterpret_cast<const u32x4_t*>(a2 + c));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float b0 = __uint_as_float(vb[i] << 16), b1 = __uint_as_float(vb[i] & 0xffff0000u);
          s = fmaf(__uint_as_float(va[i] << 16), b0, s);
          s = fmaf(__uint_as_float(va[i] & 0xffff0000u), b1, s);
          if (a2 != nullptr) {
            s2 = fmaf(__uint_as_float(va2[i] << 16), b0, s2);
            s2 = fmaf(__uint_as_float(va2[i] & 0xffff0000u), b1, s2);
          }
        }
      }
      return;
    }
  }
  for (int c = lane; c < count; c += 64) {
    const float x = to_float<T>(b[c]);
    s = fmaf(to_float<T>(a[c]), x, s);
    if (a2 != nullptr) s2 = fmaf(to_float<T>(a2[c]), x, s2);
  }
}

// The same for R rows and P vectors at once (bfloat16, wide): a wave has two turns of R loads in flight, and a row's bytes
// serve every vector.
template <int R, int P>
__device__ __forceinline__ void many_dots(const bf16_t* const (&rows)[R], const bf16_t* const (&b)[P], int count, int lane, float (&s)[P][R]) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int q = 0; q < P; ++q)
#pragma unroll
    for (int k = 0; k < R; ++k) s[q][k] = 0.f;
#pragma unroll 2
  for (int c = lane * 8; c < count; c += 64 * 8) {
    u32x4_t v[R], vb[P];
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = load_streamed(reinterpret_cast<const u32x4_t*>(rows[k] + c));
#pragma unroll
    for (int q = 0; q < P; ++q) vb[q] = *reinterpret_cast<const u32x4_t*>(b[q] + c);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < P; ++q) {
        const float b0 = __uint_as_float(vb[q][i] << 16), b1 = __uint_as_float(vb[q][i] & 0xffff0000u);
#pragma unroll
        for (int k = 0; k < R; ++k) {
          s[q][k] = fmaf(__uint_as_float(v[k][i] << 16), b0, s[q][k]);
          s[q][k] = fmaf(__uint_as_float(v[k][i] & 0xffff0000u), b1, s[q][k]);
        }
      }
  }
}

// wave_sum of N values (a power of two), with its additions: in a step a lane hands the half of the values that it does not
// keep to the lane that does, so that 2 N moves do what 6 N did.  Lane l ends with the sum of value l / (64 / N).
template <int N, int OFF = 32>
__device__ __forceinline__ float wave_sums(const float (&v)[N], int lane) {
  if constexpr (OFF == 0) {
    return v[0];
  } else if constexpr (N == 1) {
    const float one[1] = {v[0] + __shfl_xor(v[0], OFF, kWave)};
    return wave_sums<1, OFF / 2>(one, lane);
  } else {
    const bool upper = (lane & OFF) != 0;
    float half[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const float keep = upper ? v[i + N / 2] : v[i], give = upper ? v[i] : v[i + N / 2];
      half[i] = keep + __shfl_xor(give, OFF, kWave);
    }
    return wave_sums<N / 2, OFF / 2>(half, lane);
  }
}

template <typename T>
__device__ __forceinline__ bool rows_aligned(const T* a, const T* b, int count, int64_t row_stride_b) {
  return sizeof(T) == 2 && count % 8 == 0 && row_stride_b % 8 == 0 && ((uintptr_t)a | (uintptr_t)b) % 16 == 0;
}

template <typename T>
__global__ __launch_bounds__(256) void moe_up_kernel(T* __restrict__ act, const T* __restrict__ h, int64_t ldh,
                                                     const T* __restrict__ w_gate, const T* __restrict__ w_up,
                                                     const int* __restrict__ chosen, const int* __restrict__ table,
                                                     const int* __restrict__ token_ids, int top, int experts, int F,
                                                     int width, const float* __restrict__ in_weights, int gate_act,
                                                     GateNumbers numbers) {
  const int pair = blockIdx.x, t = pair / top, j = pair - t * top;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = expert_of(chosen, table, token_ids, t, j, top);
  if (e < 0 || e >= experts) return;                       // (a table that names no such expert: nothing is read)
  const T* hr = h + (int64_t)t * ldh;
  const bool wide = rows_aligned<T>(w_up, h, width, ldh) && (uintptr_t)w_gate % 16 == 0;
  const int f0 = (blockIdx.y * 4 + wave) * kRowsPerWave;
  const float wt = in_weights != nullptr ? in_weights[pair] : 1.0f;
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const int f = f0 + r;
    if (f >= F) break;
    const T* u = w_up + ((int64_t)e * F + f) * width;
    float sg, su;
    if (w_gate == nullptr) {        // no gate: the square of relu
      two_dots<T>(u, nullptr, hr, width, lane, wide, su, sg);
      su = fmaxf(wave_sum(su) * wt, 0.f);
      if (lane == 0) act[(int64_t)pair * F + f] = from_float<T>(su * su);
      continue;
    }
    const T* g = w_gate + ((int64_t)e * F + f) * width;
    two_dots<T>(g, u, hr, width, lane, wide, sg, su);
    sg = wave_sum(sg);
    su = wave_sum(su);
    if (lane == 0)
      act[(int64_t)pair * F + f] = from_float<T>(gate_act == GATE_CLIPPED ? clipped_gate_exact(sg, su, numbers)
                                                                          : sg / (1.0f + expf(-sg)) * su);
  }
}

// The next (up to) four of a set of pairs; the set loses them.
__device__ __forceinline__ uint64_t take_four(uint64_t& users) {
  const uint64_t all = users;
#pragma unroll
  for (int i = 0; i < 4; ++i) users &= users - 1;
  return all & ~users;
}

// Of at most 64 pairs, lane p the expert of pair p (negative: none): the `which`-th group of up to four pairs of one expert;
// none where there are not so many.
__device__ __forceinline__ uint64_t users_of(int e, int which) {
  for (uint64_t left = __ballot(e >= 0); left != 0;) {
    const int mine = __builtin_amdgcn_readlane(e, __builtin_ctzll(left));
    uint64_t users = __ballot(e == mine);
    left &= ~users;
    const int groups = (__popcll(users) + 3) / 4;
    if (which < groups) {
      for (; which > 0; --which) take_four(users);
      return take_four(users);
    }
    which -= groups;
  }
  return 0;
}

// A group of one to four pairs as the bytes of a word, in go<P> of one, two or four (of three the third is there twice).  (As an
// array, of which a lane picks, they would lie in LDS, whose place comes from the launch's packet in host memory: 14 us.)
template <typename GO>
__device__ __forceinline__ void with_pairs(uint64_t users, const GO& go) {
  const int many = __popcll(users);
  const auto next = [&]() {
    const uint32_t p = __builtin_ctzll(users);
    users &= users - 1;
    return p;
  };
  if (many >= 3) {
    const uint32_t a = next(), b = next(), c = next(), d = many == 4 ? next() : c;
    go(std::integral_constant<int, 4>{}, a | b << 8 | c << 16 | d << 24);
  } else if (many == 2) {
    const uint32_t a = next(), b = next();
    go(std::integral_constant<int, 2>{}, a | b << 8);
  } else if (many == 1) {
    go(std::integral_constant<int, 1>{}, next());
  }
}

__device__ __forceinline__ int pair_of(uint32_t pairs, int q) { return (pairs >> (8 * q)) & 0xff; }

// The most groups of up to four pairs of one expert that so many pairs make.
int most_groups(int pairs, int experts) {
  const int different = pairs < experts ? pairs : experts;
  return different + (pairs - different) / 4;
}

// moe_up for gated experts in bfloat16 and at most 64 pairs, expert by expert: grid (blocks of 16 rows, groups), a column of
// workgroups up to four pairs of one expert, so that an expert's rows come through every XCD (with the experts as the faster
// index all of an expert's blocks went to one: 94 us for 64) and once for four pairs; many pairs of one expert are many
// columns, side by side.  What bounds small experts is the chain of loads, sums over the wave and the code's own way from L2.
// us pair by pair / an expert's pairs four after four in one column, six moves a sum / as now: 16 experts of 2,048, width
// 4,096, one token on two 35 / 17.6 / 14.1, 8 tokens on two each 78 / 64 / 60, 64 on two in all 233 / 132 / 62; 128 experts of
// 768, width 2,048, 64 tokens on two in all 49 / 94 / 12.9; 16 of 256, width 512, 16 on two 8.8 / 15.8 / 4.5.
template <int P>
__device__ __forceinline__ void up_for_pairs(bf16_t* act, const bf16_t* h, int64_t ldh, const bf16_t* const (&rows)[2 * kRowsPerWave],
                                             uint32_t pairs, int top, int f0, int F, int width, int lane, int gate_act,
                                             GateNumbers numbers) {
  const bf16_t* b[P];
  float s[P][2 * kRowsPerWave], gate[kRowsPerWave * P], up[kRowsPerWave * P];
#pragma unroll
  for (int q = 0; q < P; ++q) b[q] = h + (int64_t)(pair_of(pairs, q) / top) * ldh;
  many_dots<2 * kRowsPerWave, P>(rows, b, width, lane, s);
#pragma unroll
  for (int i = 0; i < kRowsPerWave * P; ++i) {
    gate[i] = s[i / kRowsPerWave][i % kRowsPerWave];
    up[i] = s[i / kRowsPerWave][kRowsPerWave + i % kRowsPerWave];
  }
  constexpr int LANES = 64 / (kRowsPerWave * P);       // that end with the same sum
  const float sg = wave_sums(gate, lane), su = wave_sums(up, lane);
  const int at = lane / LANES, r = at % kRowsPerWave;
  if (lane % LANES == 0 && f0 + r < F)
    act[(int64_t)pair_of(pairs, at / kRowsPerWave) * F + f0 + r] =
        float_to_bf16(gate_act == GATE_CLIPPED ? clipped_gate_exact(sg, su, numbers) : sg / (1.0f + expf(-sg)) * su);
}

__global__ __launch_bounds__(256) void moe_up_by_expert_kernel(bf16_t* __restrict__ act, const bf16_t* __restrict__ h, int64_t ldh,
                                                               const bf16_t* __restrict__ w_gate, const bf16_t* __restrict__ w_up,
                                                               const int* __restrict__ chosen, const int* __restrict__ table,
                                                               const int* __restrict__ token_ids, int n_pairs, int top, int experts, int F,
                                                               int width, int gate_act, GateNumbers numbers) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), f0 = (blockIdx.x * 4 + wave) * kRowsPerWave;
  int own = -1;
  if (lane < n_pairs) own = expert_of(chosen, table, token_ids, lane / top, lane % top, top);
  if (own >= experts) own = -1;
  const uint64_t users = users_of(own, blockIdx.y);
  if (users == 0 || f0 >= F) return;
  const int e = __builtin_amdgcn_readlane(own, __builtin_ctzll(users));
  const bf16_t* rows[2 * kRowsPerWave];
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const int64_t row = (int64_t)e * F + min(f0 + r, F - 1);
    rows[r] = w_gate + row * width;
    rows[kRowsPerWave + r] = w_up + row * width;
  }
  with_pairs(users, [&](auto many, uint32_t pairs) {
    up_for_pairs<decltype(many)::value>(act, h, ldh, rows, pairs, top, f0, F, width, lane, gate_act, numbers);
  });
}

template <typename T>
__global__ __launch_bounds__(256) void moe_down_kernel(float* __restrict__ x, int64_t ldx, const T* __restrict__ act,
                                                       const T* __restrict__ w_down, const int* __restrict__ chosen,
                                                       const int* __restrict__ table, const int* __restrict__ token_ids,
                                                       const float* __restrict__ pair_weights, float weight, int top,
                                                       int experts, int F, int width, int accumulate) {
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = (blockIdx.y * 4 + wave) * kRowsPerWave;
  const bool wide = rows_aligned<T>(w_down, act, F, F);
  if constexpr (sizeof(T) == 2) {
    if (wide) {                             // a wave's four rows side by side
      if (c0 >= width) return;
      float total = 0.f;
      for (int j = 0; j < top; ++j) {
        const int e = expert_of(chosen, table, token_ids, t, j, top);
        if (e < 0 || e >= experts) continue;
        const bf16_t* rows[kRowsPerWave];
        float s[1][kRowsPerWave];
#pragma unroll
        for (int r = 0; r < kRowsPerWave; ++r) rows[r] = w_down + ((int64_t)e * width + min(c0 + r, width - 1)) * F;
        const bf16_t* const one[1] = {act + ((int64_t)t * top + j) * F};
        many_dots<kRowsPerWave, 1>(rows, one, F, lane, s);
        const float w = pair_weights != nullptr ? pair_weights[(int64_t)t * top + j] : weight;
        total = fmaf(wave_sums(s[0], lane), w, total);
      }
      const int r = lane / (64 / kRowsPerWave);
      if (lane % (64 / kRowsPerWave) == 0 && c0 + r < width) {
        float* o = x + (int64_t)t * ldx + c0 + r;
        *o = accumulate ? *o + total : total;
      }
      return;
    }
  }
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const int c = c0 + r;
    if (c >= width) break;
    float total = 0.f;
    for (int j = 0; j < top; ++j) {
      const int e = expert_of(chosen, table, token_ids, t, j, top);
      if (e < 0 || e >= experts) continue;
      const T* w = w_down + ((int64_t)e * width + c) * F;
      const T* a = act + ((int64_t)t * top + j) * F;
      float s, unused;
      two_dots<T>(w, nullptr, a, F, lane, wide, s, unused);
      total = fmaf(wave_sum(s), pair_weights != nullptr ? pair_weights[(int64_t)t * top + j] : weight, total);
    }
    if (lane == 0) {
      float* o = x + (int64_t)t * ldx + c;
      *o = accumulate ? *o + total : total;
    }
  }
}

// moe_down in bfloat16 for at most 64 pairs, expert by expert: a workgroup has four rows of the result, its waves take groups
// of up to four pairs of one expert in turn, on the same bytes; the pairs' sums meet in LDS, where a token's are added up in the
// order of its experts, as above.  What bounds it is loads in flight: rows of a narrow result are few workgroups, which then
// have more waves (16 waves at width 4,096 took half as long again).
template <int P>
__device__ __forceinline__ void down_for_pairs(float (*sums)[kRowsPerWave], const bf16_t* act, const bf16_t* const (&rows)[kRowsPerWave],
                                               uint32_t pairs, int F, int lane) {
  const bf16_t* b[P];
  float s[P][kRowsPerWave], all[kRowsPerWave * P];
#pragma unroll
  for (int q = 0; q < P; ++q) b[q] = act + (int64_t)pair_of(pairs, q) * F;
  many_dots<kRowsPerWave, P>(rows, b, F, lane, s);
#pragma unroll
  for (int i = 0; i < kRowsPerWave * P; ++i) all[i] = s[i / kRowsPerWave][i % kRowsPerWave];
  constexpr int LANES = 64 / (kRowsPerWave * P);       // that end with the same sum
  const float sum = wave_sums(all, lane);
  const int at = lane / LANES;
  if (lane % LANES == 0) sums[pair_of(pairs, at / kRowsPerWave)][at % kRowsPerWave] = sum;
}

template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void moe_down_by_expert_kernel(float* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ act,
                                                                 const bf16_t* __restrict__ w_down, const int* __restrict__ chosen,
                                                                 const int* __restrict__ table, const int* __restrict__ token_ids,
                                                                 const float* __restrict__ pair_weights, float weight, int n_pairs, int top,
                                                                 int experts, int F, int width, int accumulate) {
  __shared__ float sums[64][kRowsPerWave];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c0 = blockIdx.x * kRowsPerWave;
  int e = -1;
  if (lane < n_pairs) e = expert_of(chosen, table, token_ids, lane / top, lane % top, top);
  if (e >= experts) e = -1;
  int turn = 0;
  for (uint64_t left = __ballot(e >= 0); left != 0;) {
    uint64_t users = __ballot(e == __builtin_amdgcn_readlane(e, __builtin_ctzll(left)));
    left &= ~users;
    while (users != 0) {
      const uint64_t some = take_four(users);
      if ((turn++ & (WAVES - 1)) != wave) continue;
      // (read from the group, or the rows' addresses are made in front of the turns of other waves as well)
      const int mine = __builtin_amdgcn_readlane(e, __builtin_ctzll(some));
      const bf16_t* rows[kRowsPerWave];
#pragma unroll
      for (int r = 0; r < kRowsPerWave; ++r) rows[r] = w_down + ((int64_t)mine * width + min(c0 + r, width - 1)) * F;
      with_pairs(some, [&](auto many, uint32_t pairs) { down_for_pairs<decltype(many)::value>(sums, act, rows, pairs, F, lane); });
    }
  }
  __syncthreads();
  const int t = threadIdx.x / kRowsPerWave, r = threadIdx.x % kRowsPerWave;
  if (t >= n_pairs / top || c0 + r >= width) return;
  float total = 0.f;
  for (int j = 0; j < top; ++j) {
    const int p = t * top + j, ep = expert_of(chosen, table, token_ids, t, j, top);
    if (ep < 0 || ep >= experts) continue;
    total = fmaf(sums[p][r], pair_weights != nullptr ? pair_weights[p] : weight, total);
  }
  float* o = x + (int64_t)t * ldx + c0 + r;
  *o = accumulate ? *o + total : total;
}

// ---------------------------------------------------------------------------- grouped
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kTilePairs = 64, kTileRows = 256;

// How many pairs of one expert a tile holds at most: `pairs`, or `more` (0: never) where the step's pairs lie so that larger tiles are
// faster, by the blocks of rows and the columns of the two products.
struct TileSizes {
  int pairs, more, up_blocks, up_columns, down_blocks, down_columns;
};

// What the two products take in tiles of which the largest has `groups` groups of 32 pairs, in a unit of its own: rounds of a workgroup a
// CU, each as long as that tile.
__device__ __forceinline__ float tiles_cost(const TileSizes& s, int tiles, int groups) {
  constexpr int CUS = 256;
  const float rounds = (float)((tiles * s.up_blocks + CUS - 1) / CUS) * s.up_columns + (float)((tiles * s.down_blocks + CUS - 1) / CUS) * s.down_columns;
  return rounds * ((float)max(groups, 2) + 0.5f);
}

// One workgroup.  order: the pairs (t * top + j) by expert; tiles: (expert, first place in order, pairs)
// for every tile, tiles[3 * most_tiles] holds their number.  An expert's pairs make as few tiles of up to the step's tile size as they
// can, of whole 32s but the last one and alike to within one 32.  Which of an expert's pairs comes first is
// left to chance; nothing that is computed depends on it.  The first wave goes over the experts, 64 at a time.  (One thread took 128 of
// them one by one, 6 us of the feed-forward: 512 tokens on eight 281 us -> 275 with the choice of a size.)
__global__ __launch_bounds__(1024) void moe_group_kernel(int* __restrict__ order, int* __restrict__ tiles, int most_tiles,
                                                         const int* __restrict__ chosen, const int* __restrict__ table,
                                                         const int* __restrict__ token_ids, int n, int top, int experts,
                                                         TileSizes sizes) {
  extern __shared__ int lds[];
  int* counts = lds;                  // [experts]
  int* starts = lds + experts;        // [experts]
  int* cursor = lds + 2 * experts;    // [experts]
  const int pairs = n * top;
  for (int e = threadIdx.x; e < experts; e += blockDim.x) counts[e] = cursor[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
    const int e = expert_of(chosen, table, token_ids, p / top, p % top, top);
    if (e >= 0 && e < experts) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int tile_pairs = sizes.pairs;
    if (sizes.more > 0) {
      int number[2] = {0, 0}, largest[2] = {0, 0};      // of tiles, and groups of 32 pairs in one, by either size
      for (int e = lane; e < experts; e += 64)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int count = counts[e], size = i == 0 ? sizes.pairs : sizes.more, mine = (count + size - 1) / size;
          number[i] += mine;
          if (mine > 0) largest[i] = max(largest[i], ((count + 31) / 32 + mine - 1) / mine);
        }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          number[i] += __shfl_xor(number[i], off, kWave);
          largest[i] = max(largest[i], __shfl_xor(largest[i], off, kWave));
        }
      if (tiles_cost(sizes, number[1], largest[1]) < 0.93f * tiles_cost(sizes, number[0], largest[0])) tile_pairs = sizes.more;
    }
    int at = 0, tile = 0;             // of the experts behind
    for (int e0 = 0; e0 < experts; e0 += 64) {
      const int e = e0 + lane, count = e < experts ? counts[e] : 0, n_tiles = (count + tile_pairs - 1) / tile_pairs;
      int pairs_to = count, tiles_to = n_tiles;      // of the lanes up to this one
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int p = __shfl_up(pairs_to, off, kWave), t = __shfl_up(tiles_to, off, kWave);
        if (lane >= off) {
          pairs_to += p;
          tiles_to += t;
        }
      }
      const int start = at + pairs_to - count, first_tile = tile + tiles_to - n_tiles, groups = (count + 31) / 32;
      if (e < experts) starts[e] = start;
      for (int i = 0, to = 0; i < n_tiles; ++i) {
        const int mine = 32 * (groups / n_tiles + (i < groups % n_tiles ? 1 : 0));
        int* tl = tiles + 3 * (first_tile + i);
        tl[0] = e;
        tl[1] = start + to;
        tl[2] = min(mine, count - to);
        to += mine;
      }
      at += __shfl(pairs_to, 63, kWave);
      tile += __shfl(tiles_to, 63, kWave);
    }
    if (lane == 0) tiles[3 * most_tiles] = tile;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
    const int e = expert_of(chosen, table, token_ids, p / top, p % top, top);
    if (e >= 0 && e < experts) order[starts[e] + atomicAdd(&cursor[e], 1)] = p;
  }
}

// The grouped products through LDS.  A workgroup takes a tile of up to 64 pairs of one expert and 256 rows of
// weights (KIND 0: 128 rows of the gate's matrix and the same 128 of the up matrix); K in steps of 32: every
// thread asks for its 16-byte pieces of the next step (one of the pairs' rows, four of the weights') while the
// matrix cores work on the current one out of LDS, then lays them into the other buffer; rows of 40 elements
// so that the operand reads of 32 rows spread over the banks.  A wave owns 64 weight rows (KIND 0: 32 of each
// matrix) x 64 pairs as 2 x 2 tiles of `32x32x16`, the weights as the row operand, so that a lane ends with
// four neighbouring rows of the matrix for one pair and stores them at once.  A sum runs over K in the same
// order whichever pairs share the tile.
//   KIND 0: act = silu(gate) * up, or the clipped gate's product      KIND 1: act = relu(weight * up)^2      KIND 2: out (+)= scale * down
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kStageK = 32, kStagePitch = 40;

template <int KIND>
__global__ __launch_bounds__(256) void moe_group_tiled_kernel(
    void* __restrict__ dst, int64_t ldo, const bf16_t* __restrict__ src, int64_t lds_rows, const bf16_t* __restrict__ w0,
    const bf16_t* __restrict__ w1, const int* __restrict__ order, const int* __restrict__ tiles, int most_tiles, int top,
    int n_rows, int K, int add, const float* __restrict__ pair_weights, float weight, int gate_act, GateNumbers numbers) {
  __shared__ __attribute__((aligned(16))) bf16_t As[2][kTilePairs * kStagePitch];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[2][kTileRows * kStagePitch];
  if ((int)blockIdx.x >= tiles[3 * most_tiles]) return;
  const int* tl = tiles + 3 * blockIdx.x;
  const int e = tl[0], first = tl[1], count = tl[2];
  constexpr int kRowsOut = KIND == 0 ? kTileRows / 2 : kTileRows;      // rows of the result a workgroup makes
  const int row0 = blockIdx.y * kRowsOut;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // what this thread brings of every step: piece (tid & 3) of pair row tid / 4, and of weight rows tid / 4 + 64 p
  const int piece = (tid & 3) * 8, srow = tid >> 2;
  const int my_pair = order[first + (srow < count ? srow : 0)];
  const bf16_t* a_src = src + (int64_t)(KIND == 2 ? my_pair : my_pair / top) * lds_rows + piece;
  const bf16_t* w_src[4];
  bool w_ok[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int s = srow + 64 * p;                                        // the row's place in the staged tile
    const bf16_t* base = KIND == 0 && s >= kRowsOut ? w1 : w0;
    const int row = row0 + (KIND == 0 && s >= kRowsOut ? s - kRowsOut : s);
    w_ok[p] = row < n_rows;
    w_src[p] = base + ((int64_t)e * n_rows + (w_ok[p] ? row : 0)) * K + piece;
  }
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 ra = *reinterpret_cast<const u32x4*>(a_src), rw[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) rw[p] = w_ok[p] ? *reinterpret_cast<const u32x4*>(w_src[p]) : zero;
  *reinterpret_cast<u32x4*>(&As[0][srow * kStagePitch + piece]) = ra;
#pragma unroll
  for (int p = 0; p < 4; ++p) *reinterpret_cast<u32x4*>(&Ws[0][(srow + 64 * p) * kStagePitch + piece]) = rw[p];
  __syncthreads();

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int lrow = lane & 31, lk = (lane >> 5) * 8;
  // the wave's two groups of 32 staged weight rows
  const int base_i[2] = {KIND == 0 ? wave * 32 : wave * 64, KIND == 0 ? kRowsOut + wave * 32 : wave * 64 + 32};
  const int steps = K / kStageK;
  int buf = 0;
  for (int kt = 0; kt < steps; ++kt) {
    if (kt + 1 < steps) {
      const int k = (kt + 1) * kStageK;
      ra = *reinterpret_cast<const u32x4*>(a_src + k);
#pragma unroll
      for (int p = 0; p < 4; ++p) rw[p] = w_ok[p] ? *reinterpret_cast<const u32x4*>(w_src[p] + k) : zero;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(&Ws[buf][(base_i[i] + lrow) * kStagePitch + ks * 16 + lk]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = *reinterpret_cast<const bf16x8*>(&As[buf][(j * 32 + lrow) * kStagePitch + ks * 16 + lk]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < steps) {
      *reinterpret_cast<u32x4*>(&As[buf ^ 1][srow * kStagePitch + piece]) = ra;
#pragma unroll
      for (int p = 0; p < 4; ++p) *reinterpret_cast<u32x4*>(&Ws[buf ^ 1][(srow + 64 * p) * kStagePitch + piece]) = rw[p];
    }
    __syncthreads();
    buf ^= 1;
  }

  // register r of lane l in tile (i, j): row 8 (r / 4) + 4 (l / 32) + r % 4 of the wave's group i, pair 32 j + l % 32
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int at = j * 32 + lrow;
    if (at >= count) continue;
    const int pair = order[first + at];
    if constexpr (KIND == 0) {
      bf16_t* o = (bf16_t*)dst + (int64_t)pair * ldo;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int f = row0 + wave * 32 + 8 * q + 4 * (lane >> 5);
        if (f >= n_rows) continue;
        bf16_t four[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = acc[0][j][4 * q + r], u = acc[1][j][4 * q + r];
          four[r] = float_to_bf16(gate_act == GATE_CLIPPED ? clipped_gate(g, u, numbers) : g / (1.0f + expf(-g)) * u);
        }
        *reinterpret_cast<u32x2*>(o + f) = *reinterpret_cast<const u32x2*>(four);
      }
    } else {
      const float scale = KIND == 1 ? (pair_weights != nullptr ? pair_weights[pair] : 1.0f)
                                    : add ? (pair_weights != nullptr ? pair_weights[pair] : weight) : 1.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = row0 + wave * 64 + 32 * i + 8 * q + 4 * (lane >> 5);
          if (f >= n_rows) continue;
          if constexpr (KIND == 1) {
            bf16_t four[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float u = fmaxf(acc[i][j][4 * q + r] * scale, 0.f);
              four[r] = float_to_bf16(u * u);
            }
            *reinterpret_cast<u32x2*>((bf16_t*)dst + (int64_t)pair * ldo + f) = *reinterpret_cast<const u32x2*>(four);
          } else {
            float* o = (float*)dst + (int64_t)pair * ldo + f;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = add ? fmaf(acc[i][j][4 * q + r], scale, o[r]) : acc[i][j][4 * q + r];
          }
        }
    }
  }
}

// What becomes of four neighbouring rows' sums of one pair.
template <int KIND>
__device__ __forceinline__ void store_pair_rows(void* dst, int64_t ldo, int pair, int f, const f32x4& v, const f32x4& up, int add,
                                                float scale, int gate_act, GateNumbers numbers) {
  if constexpr (KIND == 2) {
    float* o = (float*)dst + (int64_t)pair * ldo + f;
    if (add || ldo % 4 != 0 || (uintptr_t)dst % 16 != 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = add ? fmaf(v[r], scale, o[r]) : v[r];
    } else {
      *reinterpret_cast<f32x4*>(o) = v;
    }
  } else {
    bf16_t four[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (KIND == 0) {
        four[r] = float_to_bf16(gate_act == GATE_CLIPPED ? clipped_gate(v[r], up[r], numbers) : v[r] / (1.0f + expf(-v[r])) * up[r]);
      } else {
        const float u = fmaxf(v[r] * scale, 0.f);
        four[r] = float_to_bf16(u * u);
      }
    }
    *reinterpret_cast<u32x2*>((bf16_t*)dst + (int64_t)pair * ldo + f) = *reinterpret_cast<const u32x2*>(four);
  }
}

// The same products for K in multiples of 64: tiles of up to 192 pairs and 256 rows of weights, four waves with all the
// pairs and 64 rows each (KIND 0: 32 of each matrix).  The instruction and the order of a sum over K are those of
// moe_group_tiled, so a pair has the same bits in both.  Rows go from memory straight into one of three or four buffers in LDS,
// asked for as many steps before they are read less one.  A tile brings and multiplies its pairs in groups of 32.  Up to 128
// pairs a step is 64 columns, 128 bytes a row, whose eight 16-byte chunks lie at chunk ^ (row % 8), so that the rows that a
// read asks the same chunk of spread over the banks (up to 64 pairs leave room for a fourth buffer); with more pairs a step is
// 32 columns, 64 bytes a row, its four chunks at chunk ^ (bit 3 of the row | bit 2 << 1), and there are four buffers.
//
// Why so many pairs: with 64 pairs a step's 20 KB fed 256 cycles of the matrix cores, more than the 64 bytes a cycle that a CU
// gets from L2, and an expert's rows came once for every tile of its pairs.  The whole feed-forward, 9 / 128 / 800 / 2,048 tokens
// on two of 16 experts of 2,048, width 4,096 (206 GFLOP at 2,048; 805 MB of weights): moe_group_tiled 225 / 252 / 428 / 804
// us, tiles of 128 pairs 128 / 178 / 213 / 374 (380 with weights that are in no cache), this 356 for 2,048; 1,200 276 -> 266;
// 16 of 1,024, width 2,048, 2,048 tokens 155 -> 115 (an expert's 256 pairs, and a few more, are two tiles instead of three).
// What bounds it now is memory: all workgroups walk the same columns of rows that lie 8 KB apart, and such a walk alone, 128
// bytes of 65,536 rows a step without any product, gets 4.4 TB/s whatever is in flight (121 us of the up product's 537 MB).
// (Blocks of rows that begin their walk over K at places of their own get 6.0 TB/s, but then a pair's sums have another order
// of additions, and bits, than in moe_group_tiled; so would 512 bytes a row, 5.1, for which LDS has no room.)
constexpr int kMostGroups = 6;                                        // of 32 pairs a tile
constexpr int direct_row(int groups) { return groups <= 4 ? 128 : 64; }                       // bytes of a row in a buffer
constexpr int direct_buffers(int groups) { return groups == 3 || groups == 4 ? 3 : 4; }
constexpr int direct_pair_rows(int groups) { return groups <= 4 ? 32 * groups : (groups + 1) / 2 * 64; }      // (a request of 64-byte rows is 16 of them a wave)
constexpr int direct_lds(int groups) { return direct_buffers(groups) * (direct_pair_rows(groups) + kTileRows) * direct_row(groups); }
constexpr int kDirectLds = direct_lds(2);                             // the most of all
static_assert(kDirectLds >= direct_lds(4) && kDirectLds >= direct_lds(kMostGroups) && kDirectLds <= 160 * 1024);

template <int KIND>
__global__ __launch_bounds__(256) void moe_direct_kernel(
    void* __restrict__ dst, int64_t ldo, const bf16_t* __restrict__ src, int64_t ld_src, const bf16_t* __restrict__ w0,
    const bf16_t* __restrict__ w1, const int* __restrict__ order, const int* __restrict__ tiles, int most_tiles, int top,
    int n_rows, int K, int add, const float* __restrict__ pair_weights, float weight, int gate_act, GateNumbers numbers,
    uint32_t src_bytes) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass has no buffer resources; it only needs the stub
  constexpr int kRowsOut = KIND == 0 ? kTileRows / 2 : kTileRows;      // rows of the result a workgroup makes
  extern __shared__ __attribute__((aligned(1024))) char lds_bytes[];
  const int n_tiles = tiles[3 * most_tiles], row_blocks = (n_rows + kRowsOut - 1) / kRowsOut, items = n_tiles * row_blocks;
  if ((int)blockIdx.x >= items) return;
  // An XCD gets a run of items; an expert's items follow one another, its tiles of pairs within its blocks of rows, so that
  // weight rows are read from memory once and the pairs' rows by the one or two XCDs that have the expert.
  const int xcd = blockIdx.x % 8, item = xcd * (items / 8) + min(xcd, items % 8) + (int)blockIdx.x / 8;
  const int lane = threadIdx.x & 63, some_tile = item / row_blocks, e = tiles[3 * some_tile];       // (a tile of the item's expert)
  int tile0 = some_tile, tile1 = some_tile + 1;                                                     // the expert's tiles
  for (bool more = true; more;) {
    const int at = tile0 - 1 - lane;
    const uint64_t other = __ballot(at < 0 || tiles[3 * max(at, 0)] != e);
    tile0 -= other ? __builtin_ctzll(other) : 64;
    more = other == 0;
  }
  for (bool more = true; more;) {
    const int at = tile1 + lane;
    const uint64_t other = __ballot(at >= n_tiles || tiles[3 * min(at, n_tiles - 1)] != e);
    tile1 += other ? __builtin_ctzll(other) : 64;
    more = other == 0;
  }
  const int within = item - tile0 * row_blocks, row0 = within / (tile1 - tile0) * kRowsOut;
  const int* tl = tiles + 3 * (tile0 + within % (tile1 - tile0));
  const int first = tl[1], count = tl[2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, g = lane >> 5;

  typedef __attribute__((address_space(3))) void* lds_ptr;
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, (int)src_bytes, 0x00020000);
  const int64_t expert = (int64_t)e * n_rows * K;
  const int matrix_bytes = (int)((uint32_t)n_rows * (uint32_t)K * 2u);
  const __amdgpu_buffer_rsrc_t w0_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(w0 + expert), 0, matrix_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t w1_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)((KIND == 0 ? w1 : w0) + expert), 0, matrix_bytes, 0x00020000);
  const auto work = [&](auto subtiles) {
    constexpr int PT = decltype(subtiles)::value;                    // groups of 32 pairs
    constexpr int ROW = direct_row(PT), BUFFERS = direct_buffers(PT), A_ROWS = direct_pair_rows(PT), BUFFER = (A_ROWS + kTileRows) * ROW;
    constexpr int CHUNKS = ROW / 16;                                  // of a row
    // (a request a wave is a kilobyte, REQUEST rows of the four waves; what a wave reads and multiplies of half a step's
    // columns, which are SIXTEENS instructions' 16 each)
    constexpr int REQUEST = 4096 / ROW, SIXTEENS = ROW / 64;
    constexpr int A_LOADS = A_ROWS / REQUEST, LOADS = A_LOADS + kTileRows / REQUEST, READS = SIXTEENS * (2 + PT), PRODUCTS = SIXTEENS * 2 * PT;
    constexpr int EARLY = LOADS / 2;                                  // of a step's requests that go out in a step's second half
    const int steps = K * 2 / ROW;
    // where a row's chunk lies in it
    const auto turned = [](int row, int chunk) { return CHUNKS == 8 ? chunk ^ (row & 7) : chunk ^ (((row >> 3) & 1) | ((row >> 1) & 2)); };
    const int lrow = (64 / CHUNKS) * wave + lane / CHUNKS, chunk = turned(lrow, lane % CHUNKS);      // of the rows that a wave's request t brings: + REQUEST t
    uint32_t a_off[A_LOADS], w_off[kTileRows / REQUEST];
#pragma unroll
    for (int t = 0; t < A_LOADS; ++t) {
      const int pair = order[first + min(lrow + REQUEST * t, count - 1)];
      a_off[t] = (uint32_t)((KIND == 2 ? pair : pair / top) * ld_src + 8 * chunk) * 2;
    }
#pragma unroll
    for (int t = 0; t < kTileRows / REQUEST; ++t) {
      const int s = lrow + REQUEST * t;                                // the row's place in the staged tile
      w_off[t] = ((uint32_t)min(row0 + (KIND == 0 && s >= kRowsOut ? s - kRowsOut : s), n_rows - 1) * (uint32_t)K + 8 * chunk) * 2;
    }
    const auto load_one = [&](int step, int buffer, int t) {
      const int at = min(step, steps - 1) * ROW;                     // (past the end: a repeat that nobody uses)
      char* to = lds_bytes + buffer * BUFFER + wave * 1024;
      if (t < A_LOADS) __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr)(to + t * 4096), 16, a_off[t], at, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(t - A_LOADS < kTileRows / REQUEST / 2 ? w0_rsrc : w1_rsrc,
                                                    (lds_ptr)(to + t * 4096), 16, w_off[t - A_LOADS], at, 0, 0);
    };
    struct Operands {
      bf16x8 w[SIXTEENS][2], a[SIXTEENS][PT];
    };
    const auto read_one = [&](int buffer, int half, Operands& o, int i) {      // in the order in which the products need them
      const int sixteen = i / (2 + PT), t = i % (2 + PT);
      const char* tile = lds_bytes + buffer * BUFFER + r * ROW + (turned(r, 2 * SIXTEENS * half + 2 * sixteen + g) << 4);
      if (t < 2) o.w[sixteen][t] = *reinterpret_cast<const bf16x8*>(tile + (A_ROWS + (KIND == 0 ? t * kRowsOut + wave * 32 : wave * 64 + t * 32)) * ROW);
      else o.a[sixteen][t - 2] = *reinterpret_cast<const bf16x8*>(tile + (t - 2) * 32 * ROW);
    };
    f32x16 acc[2][PT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int m = 0; m < PT; ++m)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[i][m][q] = 0.f;
    const auto multiply_one = [&](const Operands& o, int p) {
      const int sixteen = p / (2 * PT), i = p & 1, m = p / 2 % PT;
      acc[i][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(o.w[sixteen][i], o.a[sixteen][m], acc[i][m], 0, 0, 0);
    };

    if (steps < BUFFERS) {                                           // a buffer for every step, and no repeats
      for (int s = 0; s < steps; ++s)
#pragma unroll
        for (int t = 0; t < LOADS; ++t) load_one(s, s, t);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      barrier_no_fence();
      for (int half = 0; half < 2 * steps; ++half) {
        Operands o;
#pragma unroll
        for (int i = 0; i < READS; ++i) read_one(half / 2, half % 2, o, i);
#pragma unroll
        for (int p = 0; p < PRODUCTS; ++p) multiply_one(o, p);
      }
    } else {
      // A step's buffer is free from the middle of its step on (its reads end before the barrier there): the first EARLY
      // requests of step s + BUFFERS go out in the second half of step s, the others in the first half of step s + 1, so
      // that they stand between matrix instructions one by one.
#pragma unroll
      for (int s = 0; s < BUFFERS; ++s)
#pragma unroll
        for (int t = 0; t < (s < BUFFERS - 1 ? LOADS : EARLY); ++t) load_one(s, s, t);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUFFERS - 2) * LOADS + EARLY) : "memory");
      barrier_no_fence();
      Operands o[2];
#pragma unroll
      for (int i = 0; i < READS; ++i) read_one(0, 0, o[0], i);
      int now = 0, before = BUFFERS - 1;                               // the step's buffer, and that of the step before
      for (int s = 0; s < steps; ++s) {
        const int next = now == BUFFERS - 1 ? 0 : now + 1;
        // the first half of the columns, with the reads of the others
#pragma unroll
        for (int p = 0; p < PRODUCTS; ++p) {
          multiply_one(o[0], p);
#pragma unroll
          for (int i = 0; i < READS; ++i)
            if (i >= 2 * READS * p / PRODUCTS && i < 2 * READS * (p + 1) / PRODUCTS) read_one(now, 1, o[1], i);
#pragma unroll
          for (int l = 0; l < LOADS - EARLY; ++l)
            if (l >= (LOADS - EARLY) * p / PRODUCTS && l < (LOADS - EARLY) * (p + 1) / PRODUCTS) load_one(s + BUFFERS - 1, before, EARLY + l);
          __builtin_amdgcn_sched_barrier(0);
        }
        // this wave's part of step s + 1 has landed and its reads of step s are done; behind the barrier everybody's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((BUFFERS - 2) * LOADS) : "memory");
        barrier_no_fence();
#pragma unroll
        for (int p = 0; p < PRODUCTS; ++p) {
          multiply_one(o[1], p);
#pragma unroll
          for (int i = 0; i < READS; ++i)
            if (i >= 2 * READS * p / PRODUCTS && i < 2 * READS * (p + 1) / PRODUCTS) read_one(next, 0, o[0], i);
#pragma unroll
          for (int l = 0; l < EARLY; ++l)
            if (l >= EARLY * p / PRODUCTS && l < EARLY * (p + 1) / PRODUCTS) load_one(s + BUFFERS, now, l);
          __builtin_amdgcn_sched_barrier(0);
        }
        before = now;
        now = next;
      }
      // the repeats asked for past the end still write into this workgroup's LDS: they land before the wave ends
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    // register q of lane l in (i, m): row 8 (q / 4) + 4 (l / 32) + q % 4 of the wave's group i, pair 32 m + l % 32
#pragma unroll
    for (int m = 0; m < PT; ++m) {
      if (32 * m + r >= count) continue;
      const int pair = order[first + 32 * m + r];
      const float scale = KIND == 0 ? 1.0f : KIND == 1 ? (pair_weights != nullptr ? pair_weights[pair] : 1.0f)
                                          : add ? (pair_weights != nullptr ? pair_weights[pair] : weight) : 1.0f;
#pragma unroll
      for (int i = 0; i < (KIND == 0 ? 1 : 2); ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = row0 + (KIND == 0 ? wave * 32 : wave * 64 + 32 * i) + 8 * q + 4 * g;
          const f32x4 v = {acc[i][m][4 * q], acc[i][m][4 * q + 1], acc[i][m][4 * q + 2], acc[i][m][4 * q + 3]};
          const f32x4 up = {acc[1][m][4 * q], acc[1][m][4 * q + 1], acc[1][m][4 * q + 2], acc[1][m][4 * q + 3]};      // (KIND 0)
          if (f < n_rows) store_pair_rows<KIND>(dst, ldo, pair, f, v, up, add, scale, gate_act, numbers);
        }
    }
  };
  switch ((count + 31) / 32) {
    case 0: case 1: case 2: return work(std::integral_constant<int, 2>{});
    case 3: return work(std::integral_constant<int, 3>{});
    case 4: return work(std::integral_constant<int, 4>{});
    case 5: return work(std::integral_constant<int, 5>{});
    default: return work(std::integral_constant<int, kMostGroups>{});
  }
#endif
}

template <int KIND>
int launch_direct(int most, void* dst, int64_t ldo, const bf16_t* src, int64_t ld_src, int64_t src_rows, const bf16_t* w0,
                  const bf16_t* w1, const int* order, const int* tiles, int top, int n_rows, int K, int add,
                  const float* pair_weights, float weight, int gate_act, GateNumbers numbers, hipStream_t stream) {
  constexpr int rows_out = KIND == 0 ? kTileRows / 2 : kTileRows;
  static const hipError_t raised =
      hipFuncSetAttribute((const void*)moe_direct_kernel<KIND>, hipFuncAttributeMaxDynamicSharedMemorySize, kDirectLds);
  HFEE_REQUIRE(raised == hipSuccess, "moe_grouped: %s", hipGetErrorString(raised));
  const int64_t grid = (int64_t)most * ((n_rows + rows_out - 1) / rows_out);
  HFEE_REQUIRE(grid < (int64_t)1 << 31, "moe_grouped: too many tiles");
  moe_direct_kernel<KIND><<<(unsigned)grid, 256, kDirectLds, stream>>>(dst, ldo, src, ld_src, w0, w1, order, tiles, most, top, n_rows, K, add,
                                                              pair_weights, weight, gate_act, numbers,
                                                              (uint32_t)(((src_rows - 1) * ld_src + K) * 2));
  HFEE_CHECK_LAUNCH("moe_grouped");
  return 0;
}

// The tiles of moe_direct.  Tiles of up to 192 pairs read an expert's rows fewer times, and are fewer: a gain where the workgroups (one
// a CU) then are fewer rounds and the last one's CUs are not idle for as long as the tiles are larger.  How many tiles there are
// depends on how the pairs lie, which only the device knows, and so does the largest tile, for which an XCD with few pairs of many
// experts waits for another one: rounds times the largest tile is what a step is expected to take, and the larger tiles are taken where that
// is 7 % less.  Fitted to 160 steps (8 to 128 experts, 512 to 2,048 tokens; pairs spread evenly, over half or a quarter of the
// experts, by a power law, all on as few as a token uses): of the better of 128 and 192 it misses 0.05 %, and none is more than 1.5 % slower than
// with 128.  (By the mean number of pairs instead, which is known on the host, steps whose pairs are not spread evenly lost up to a third.)
// The feed-forward with weights that are in no cache, us with 128 / 192: 16 experts of 2,048, width 4,096, 2,048 tokens on two, evenly
// 359 / 342, on two experts 248 / 320, by a power law 350 / 366; on one expert each, evenly 289 / 246, by a power law 271 / 355; 1,200 on two 255 / 249 and 262 /
// 328; 16 of 1,024, width 2,048, 2,048 on two 152 / 109; 64 of 1,408, 2,048 on six 437 / 451; 128 of 768, 2,048 on eight 422 / 398 and 432 / 490; 8 of 4,096,
// width 4,096, 2,048 on two 541 / 525 and 543 / 622.  (Tiles of more than 192: 256 pairs leave CUs idle, 440 us in the first case; more do not fit the
// accumulation registers.)
TileSizes direct_tiles(int ff, int width, bool gated) {
  const int rows_up = gated ? kTileRows / 2 : kTileRows;
  return TileSizes{128, 32 * kMostGroups, (ff + rows_up - 1) / rows_up, width, (width + kTileRows - 1) / kTileRows, ff};
}

// x[t] += sum_j weight_tj y[t * top + j], j ascending.
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ x, int64_t ldx, const float* __restrict__ y,
                                                          const float* __restrict__ pair_weights, float weight, int top,
                                                          int width) {
  const int64_t t = blockIdx.x;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < width; c += gridDim.y * blockDim.x) {
    float total = 0.f;
    for (int j = 0; j < top; ++j)
      total = fmaf(y[(t * top + j) * width + c], pair_weights != nullptr ? pair_weights[t * top + j] : weight, total);
    x[t * ldx + c] += total;
  }
}

// The same for rows on 16 bytes, four values a thread, the pairs' rows asked for two at a time: bound by its bytes.  2,048 tokens of
// 4,096 on two experts each (134 MB) 37 us by single values, 22 so (6.1 TB/s).
__global__ __launch_bounds__(256) void moe_combine_fours_kernel(float* __restrict__ x, int64_t ldx, const float* __restrict__ y,
                                                                const float* __restrict__ pair_weights, float weight, int top,
                                                                int width) {
  const int64_t t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= width) return;
  f32x4* to = reinterpret_cast<f32x4*>(x + t * ldx + c);
  const f32x4 before = *to;
  const float* from = y + t * top * width + c;
  f32x4 total = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < top; j += 2) {
    const bool two = j + 1 < top;
    const f32x4 one = *reinterpret_cast<const f32x4*>(from + (int64_t)j * width);
    const f32x4 other = *reinterpret_cast<const f32x4*>(from + (int64_t)(two ? j + 1 : j) * width);
    const float w1 = pair_weights != nullptr ? pair_weights[t * top + j] : weight;
    const float w2 = pair_weights != nullptr ? pair_weights[t * top + (two ? j + 1 : j)] : weight;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      total[i] = fmaf(one[i], w1, total[i]);
      if (two) total[i] = fmaf(other[i], w2, total[i]);
    }
  }
  *to = before + total;
}

// One wave a token.  A lane looks through its share of the experts (lane, lane + 64, ...) for the largest
// logit that is not chosen yet (a bit a share in the lane's own registers says which are); the wave's lanes
// meet over (logit, number), the larger logit and of two equal ones the lower number, and every lane ends
// with the same answer.  The sigmoid grows with its argument, so the largest scores are the largest logits.
constexpr int kRouterMostExperts = 64 * 128, kRouterMostGroups = 512;

struct RouterGroups {
  int count, keep;       // count 0: no groups
};

// score_kind 0: a score is sigmoid(z); 1: the softmax of z over all experts; 2: the softmax of z over the chosen
// experts.  bias (float32 [experts] or null) is part of z.  correction (the same; not with kind 2) is added to a
// score where the experts are chosen and nowhere else: the weights are the scores.  groups: an expert can be chosen
// where fewer than `keep` groups come before its own (a larger best choice score, or an equal one and a lower number).
// renormalize (not with kind 2): the weights are the chosen scores / (their sum + 1e-20) * scale.
__global__ __launch_bounds__(256) void router_topk_kernel(const float* __restrict__ logits, int64_t ld, int n, int experts,
                                                          int top, int* __restrict__ chosen, float* __restrict__ weights,
                                                          int score_kind, const float* __restrict__ correction,
                                                          const float* __restrict__ bias, RouterGroups groups,
                                                          int renormalize, float scale) {
  extern __shared__ float group_best[];      // [waves][2][groups.count]: a group's best, and whether it is kept
  const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= n) return;
  const float* row = logits + (int64_t)t * ld;
  auto z = [&](int e) { return bias != nullptr ? row[e] + bias[e] : row[e]; };
  float zmax = 0.f, inv_sum = 1.f;
  if (score_kind == 1) {
    zmax = -INFINITY;
    for (int e = lane; e < experts; e += 64) zmax = fmaxf(zmax, z(e));
    zmax = wave_max(zmax);
    float sum = 0.f;
    for (int e = lane; e < experts; e += 64) sum += expf(z(e) - zmax);
    inv_sum = 1.0f / wave_sum(sum);
  }
  auto score = [&](int e) { return score_kind == 1 ? expf(z(e) - zmax) * inv_sum : 1.0f / (1.0f + expf(-z(e))); };
  // without a correction the order of the scores is the order of the logits (both scores grow with them)
  auto choice = [&](int e) { return correction != nullptr ? score(e) + correction[e] : z(e); };
  float* best_of = group_best + (threadIdx.x >> 6) * 2 * groups.count;
  float* kept = best_of + groups.count;
  const int each = groups.count > 0 ? experts / groups.count : experts;
  if (groups.count > 0) {      // (a wave's own part of LDS: what its lanes wrote is there behind the wave's own wait)
    for (int g = lane; g < groups.count; g += 64) {
      float best = choice(g * each);
      for (int e = g * each + 1; e < (g + 1) * each; ++e) best = fmaxf(best, choice(e));
      best_of[g] = best;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int g = lane; g < groups.count; g += 64) {
      int before = 0;
      for (int o = 0; o < groups.count; ++o) before += best_of[o] > best_of[g] || (best_of[o] == best_of[g] && o < g);
      kept[g] = before < groups.keep ? 1.f : 0.f;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  auto open = [&](int e) { return groups.count == 0 || kept[e / each] != 0.f; };
  float first = 0.f, chosen_sum = 0.f;       // (kind 2: the largest logit, and the sum of the chosen ones' exponentials)
  unsigned long long taken[2] = {0ull, 0ull};
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane, i = 0; e < experts; e += 64, ++i) {
      const float v = choice(e);
      if (!((taken[i >> 6] >> (i & 63)) & 1ull) && open(e) && (at == 0x7fffffff || v > best)) { best = v; at = e; }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const int oa = __shfl_xor(at, off, 64);
      if (oa != 0x7fffffff && (at == 0x7fffffff || ob > best || (ob == best && oa < at))) { best = ob; at = oa; }
    }
    if ((at & 63) == lane) taken[(at >> 6) >> 6] |= 1ull << ((at >> 6) & 63);
    if (lane == 0) {
      chosen[(int64_t)t * top + j] = at;
      if (score_kind == 2) {
        if (j == 0) first = best;
        const float w = expf(best - first);
        chosen_sum += w;
        weights[(int64_t)t * top + j] = w;
      } else {
        const float w = score(at);
        chosen_sum += w;
        weights[(int64_t)t * top + j] = w;
      }
    }
  }
  if (score_kind == 2 && lane == 0) {
    const float inv = 1.0f / chosen_sum;
    for (int j = 0; j < top; ++j) weights[(int64_t)t * top + j] *= inv;
  }
  if (renormalize && lane == 0) {
    const float by = scale / (chosen_sum + 1e-20f);
    for (int j = 0; j < top; ++j) weights[(int64_t)t * top + j] *= by;
  }
}

// The same for up to 64 experts, one a lane: a lane keeps its expert's score and choice score in registers.
__global__ __launch_bounds__(256) void router_topk_few_kernel(const float* __restrict__ logits, int64_t ld, int n, int experts,
                                                              int top, int* __restrict__ chosen, float* __restrict__ weights,
                                                              int score_kind, const float* __restrict__ correction,
                                                              const float* __restrict__ bias, RouterGroups groups,
                                                              int renormalize, float scale) {
  const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= n) return;
  const bool mine = lane < experts;
  const int e = mine ? lane : 0;
  float z = logits[(int64_t)t * ld + e];
  if (bias != nullptr) z += bias[e];
  const float shift = correction != nullptr ? correction[e] : 0.f;
  float score = z;                                       // (kind 2: the exponential comes when the largest is known)
  if (score_kind == 0) score = 1.0f / (1.0f + expf(-z));
  if (score_kind == 1) {
    const float zmax = wave_max(mine ? z : -INFINITY);
    const float w = expf(z - zmax);
    score = w * (1.0f / wave_sum(mine ? w : 0.f));
  }
  // without a correction the order of the scores is the order of the logits (both scores grow with them)
  const float choice = correction != nullptr ? score + shift : z;
  bool open = mine;
  if (groups.count > 0) {
    const int each = experts / groups.count, first = e / each * each;
    float best = -INFINITY;
    for (int i = 0; i < each; ++i) best = fmaxf(best, __shfl(choice, first + i, 64));
    int before = 0;
    for (int o = 0; o < experts; o += each) {
      const float other = __shfl(best, o, 64);
      before += other > best || (other == best && o < first);
    }
    open = mine && before < groups.keep;
  }
  float first_choice = 0.f, sum = 0.f, kept = 0.f;       // kept: lane j's weight of the j-th chosen
  int kept_at = 0;
  for (int j = 0; j < top; ++j) {
    float best = choice;
    int at = open ? lane : 0x7fffffff;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const int oa = __shfl_xor(at, off, 64);
      if (oa != 0x7fffffff && (at == 0x7fffffff || ob > best || (ob == best && oa < at))) { best = ob; at = oa; }
    }
    if (j == 0) first_choice = best;
    const float w = score_kind == 2 ? expf(best - first_choice) : __shfl(score, at & 63, 64);
    sum += w;
    if (at == lane) open = false;
    if (j == lane) {
      kept = w;
      kept_at = at;
    }
  }
  if (lane >= top) return;                               // (top is at most the number of experts)
  if (score_kind == 2) kept *= 1.0f / sum;
  if (renormalize) kept *= scale / (sum + 1e-20f);
  chosen[(int64_t)t * top + lane] = kept_at;
  weights[(int64_t)t * top + lane] = kept;
}

}  // namespace

HFEE_API int hfee_router_topk(const float* logits, int64_t ld, int n, int experts, int top, int* chosen, float* weights,
                              int score_kind, const float* correction, const float* bias, int group_count, int group_keep,
                              int renormalize, float scale, hipStream_t stream) {
  HFEE_REQUIRE(score_kind >= 0 && score_kind <= 2, "router_topk: the scores are sigmoids (0), a softmax (1) or a softmax over the chosen (2)");
  HFEE_REQUIRE(score_kind != 2 || correction == nullptr, "router_topk: a softmax over the chosen experts takes no correction");
  HFEE_REQUIRE(n >= 0 && experts >= 1 && experts <= kRouterMostExperts && top >= 1 && top <= experts && ld >= experts,
               "router_topk: a token uses 1 to %d experts (of at most %d), not %d", experts, kRouterMostExperts, top);
  HFEE_REQUIRE(group_count >= 0 && group_count <= kRouterMostGroups && (group_count == 0 || (experts % group_count == 0 &&
               group_keep >= 1 && group_keep <= group_count && top <= group_keep * (experts / group_count))),
               "router_topk: %d experts in %d groups of which %d are kept cannot give a token %d", experts, group_count, group_keep, top);
  HFEE_REQUIRE(!renormalize || score_kind != 2, "router_topk: a softmax over the chosen experts adds up to one already");
  if (n == 0) return 0;
  if (experts <= 64) {
    router_topk_few_kernel<<<(n + 3) / 4, 256, 0, stream>>>(logits, ld, n, experts, top, chosen, weights, score_kind, correction,
                                                            bias, RouterGroups{group_count, group_keep}, renormalize, scale);
    HFEE_CHECK_LAUNCH("router_topk");
    return 0;
  }
  router_topk_kernel<<<(n + 3) / 4, 256, 4 * 2 * group_count * sizeof(float), stream>>>(
      logits, ld, n, experts, top, chosen, weights, score_kind, correction, bias, RouterGroups{group_count, group_keep}, renormalize, scale);
  HFEE_CHECK_LAUNCH("router_topk");
  return 0;
}

// The whole feed-forward in its grouped form, bfloat16: x (float32 [n, width]) += the experts' weighted
// outputs; x null: a pair's output, not weighted, is left in its row of y (whatever top is).  order: int32 [n * top]; tiles: int32 [3 * hfee_moe_group_tiles(n, top, experts) + 1]; act:
// bfloat16 [n * top, ff]; y: float32 [n * top, width], needed where top > 1.
HFEE_API int hfee_moe_group_tiles(int n, int top, int experts) {
  return (int)(((int64_t)n * top + kTilePairs - 1) / kTilePairs) + experts;
}

HFEE_API int hfee_moe_grouped(float* x, int64_t ldx, const void* h, int64_t ldh, const void* w_gate, const void* w_up,
                              const void* w_down, const int* chosen, const int* table, const int* token_ids,
                              const float* pair_weights, float weight, int top, int experts, int ff, int width, int n,
                              int* order, int* tiles, void* act, float* y, const float* in_weights, int gate_act, float limit,
                              float sharpness, hipStream_t stream) {
  HFEE_REQUIRE(gate_act == GATE_SILU || (gate_act == GATE_CLIPPED && w_gate != nullptr), "moe_grouped: unknown gate %d", gate_act);
  const GateNumbers numbers{limit, sharpness};
  HFEE_REQUIRE(n >= 0 && top >= 1 && experts >= 1 && experts <= 8192 && ff >= 1 && width >= 1, "moe_grouped: bad sizes");
  HFEE_REQUIRE(chosen != nullptr || (table != nullptr && token_ids != nullptr), "moe_grouped: the experts of a token, or a table and the ids");
  HFEE_REQUIRE(width % 32 == 0 && ff % 32 == 0 && ldh % 8 == 0 && (x == nullptr || ldx >= width) && ldh >= width,
               "moe_grouped: the width and the experts' size must be multiples of 32");
  HFEE_REQUIRE(w_gate != nullptr || pair_weights == nullptr, "moe_grouped: experts without a gate take their weights on the input");
  HFEE_REQUIRE(((uintptr_t)h | (uintptr_t)w_gate | (uintptr_t)w_up | (uintptr_t)w_down | (uintptr_t)act) % 16 == 0,
               "moe_grouped: operands must be 16-byte aligned");
  HFEE_REQUIRE(order != nullptr && tiles != nullptr && act != nullptr && ((top == 1 && x != nullptr) || y != nullptr), "moe_grouped: scratch missing");
  HFEE_REQUIRE((int64_t)n * top < (1 << 30), "moe_grouped: too many pairs");
  if (n == 0) return 0;
  // Tiles through LDS loads: steps of 64 columns, and offsets of 32 bits from the first row of an operand.  (Not for many pairs
  // of a width of one such step, which is no work to have a whole CU's LDS for.  us by way of registers / straight into LDS, width
  // 64: 8 experts of 64, 500 pairs 27 / 25, 1,000 18.2 / 25, 16,384 35 / 41; 8 of 4,096, 130 pairs 78 / 40, 2,048 105 / 94,
  // 16,384 172 / 252.)
  const int64_t limit32 = (int64_t)1 << 31;
  const bool direct = width % 64 == 0 && ff % 64 == 0 && (width > 64 || (int64_t)n * top < 960) && ((int64_t)n * ldh) * 2 < limit32 && (int64_t)n * top * ff * 2 < limit32 &&
                      (int64_t)ff * width * 2 < limit32;
  const TileSizes sizes = direct ? direct_tiles(ff, width, w_gate != nullptr) : TileSizes{kTilePairs, 0, 0, 0, 0, 0};
  const int most = (int)(((int64_t)n * top + sizes.pairs - 1) / sizes.pairs) + experts;      // (larger tiles are not more)
  moe_group_kernel<<<1, 1024, 3 * experts * sizeof(int), stream>>>(order, tiles, most, chosen, table, token_ids, n, top, experts, sizes);
  HFEE_CHECK_LAUNCH("moe_group");
  const bool straight = top == 1 && x != nullptr;
  void* down = straight ? (void*)x : (void*)y;
  const int64_t ld_down = straight ? ldx : (int64_t)width;
  if (direct) {
    if (w_gate != nullptr ? launch_direct<0>(most, act, ff, (const bf16_t*)h, ldh, n, (const bf16_t*)w_gate, (const bf16_t*)w_up, order,
                                             tiles, top, ff, width, 0, nullptr, 1.0f, gate_act, numbers, stream)
                          : launch_direct<1>(most, act, ff, (const bf16_t*)h, ldh, n, (const bf16_t*)w_up, nullptr, order, tiles, top, ff,
                                             width, 0, in_weights, 1.0f, GATE_SILU, numbers, stream))
      return 1;
    if (launch_direct<2>(most, down, ld_down, (const bf16_t*)act, ff, (int64_t)n * top, (const bf16_t*)w_down, nullptr, order, tiles, top,
                         width, ff, straight ? 1 : 0, pair_weights, weight, GATE_SILU, numbers, stream))
      return 1;
  } else {
    // (rows in whole groups of four: ff and width are multiples of 32)
    if (w_gate != nullptr)
      moe_group_tiled_kernel<0><<<dim3(most, (ff + kTileRows / 2 - 1) / (kTileRows / 2)), 256, 0, stream>>>(
          act, ff, (const bf16_t*)h, ldh, (const bf16_t*)w_gate, (const bf16_t*)w_up, order, tiles, most, top, ff, width, 0,
          nullptr, 1.0f, gate_act, numbers);
    else
      moe_group_tiled_kernel<1><<<dim3(most, (ff + kTileRows - 1) / kTileRows), 256, 0, stream>>>(
          act, ff, (const bf16_t*)h, ldh, (const bf16_t*)w_up, nullptr, order, tiles, most, top, ff, width, 0, in_weights, 1.0f,
          GATE_SILU, numbers);
    HFEE_CHECK_LAUNCH("moe_group_up");
    moe_group_tiled_kernel<2><<<dim3(most, (width + kTileRows - 1) / kTileRows), 256, 0, stream>>>(
        down, ld_down, (const bf16_t*)act, ff, (const bf16_t*)w_down, nullptr, order, tiles, most, top, width, ff, straight ? 1 : 0,
        pair_weights, weight, GATE_SILU, numbers);
    HFEE_CHECK_LAUNCH("moe_group_down");
  }
  if (top > 1 && x != nullptr) {
    // (the width is a multiple of 32)
    if (ldx % 4 == 0 && (((uintptr_t)x | (uintptr_t)y) & 15) == 0 && width <= 65535 * 1024) {
      moe_combine_fours_kernel<<<dim3(n, (width / 4 + 255) / 256), 256, 0, stream>>>(x, ldx, y, pair_weights, weight, top, width);
    } else {
      int parts = (width + 255) / 256;
      if (parts > 64) parts = 64;
      moe_combine_kernel<<<dim3(n, parts), 256, 0, stream>>>(x, ldx, y, pair_weights, weight, top, width);
    }
    HFEE_CHECK_LAUNCH("moe_combine");
  }
  return 0;
}

HFEE_API int hfee_moe_up(void* act, const void* h, int64_t ldh, const void* w_gate, const void* w_up, int dtype,
                         const int* chosen, const int* table, const int* token_ids, int top, int experts, int ff,
                         int width, int n, const float* in_weights, int gate_act, float limit, float sharpness,
                         hipStream_t stream) {
  HFEE_REQUIRE(gate_act == GATE_SILU || (gate_act == GATE_CLIPPED && w_gate != nullptr), "moe_up: unknown gate %d", gate_act);
  const GateNumbers numbers{limit, sharpness};
  HFEE_REQUIRE(n >= 0 && top >= 1 && experts >= 1 && ff >= 1 && width >= 1 && ldh >= width, "moe_up: bad sizes");
  HFEE_REQUIRE(chosen != nullptr || (table != nullptr && token_ids != nullptr), "moe_up: the experts of a token, or a table and the ids");
  if (n == 0) return 0;
  const int per_block = 4 * kRowsPerWave;
  HFEE_REQUIRE((ff + per_block - 1) / per_block <= 65535, "moe_up: experts too wide");
  dim3 grid((unsigned)((int64_t)n * top), (ff + per_block - 1) / per_block);
  if (dtype == 0)
    moe_up_kernel<float><<<grid, 256, 0, stream>>>((float*)act, (const float*)h, ldh, (const float*)w_gate, (const float*)w_up,
                                                   chosen, table, token_ids, top, experts, ff, width, in_weights,
                                                    gate_act, numbers);
  // (expert by expert where the pairs fit a wave's lanes, but for many pairs of next to no work: 8 experts of 64, width 64, 32
  // pairs 5.8 us pair by pair, 6.8 by expert; 8 pairs 6.4 / 4.9)
  else if (dtype == 1 && w_gate != nullptr && (int64_t)n * top <= 64 && width % 8 == 0 && ldh % 8 == 0 &&
           (n * top <= 16 || (int64_t)n * top * ff * width > 1 << 18) && (((uintptr_t)h | (uintptr_t)w_gate | (uintptr_t)w_up) & 15) == 0)
    moe_up_by_expert_kernel<<<dim3(grid.y, most_groups(n * top, experts)), 256, 0, stream>>>(
        (bf16_t*)act, (const bf16_t*)h, ldh, (const bf16_t*)w_gate, (const bf16_t*)w_up, chosen, table, token_ids, n * top, top, experts,
        ff, width, gate_act, numbers);
  else if (dtype == 1)
    moe_up_kernel<bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)act, (const bf16_t*)h, ldh, (const bf16_t*)w_gate,
                                                    (const bf16_t*)w_up, chosen, table, token_ids, top, experts, ff, width, in_weights,
                                                    gate_act, numbers);
  else
    return fail("moe_up: unknown dtype %d", dtype);
  HFEE_CHECK_LAUNCH("moe_up");
  return 0;
}

HFEE_API int hfee_moe_down(float* x, int64_t ldx, const void* act, const void* w_down, int dtype, const int* chosen,
                           const int* table, const int* token_ids, const float* pair_weights, float weight, int top,
                           int experts, int ff, int width, int accumulate, int n, hipStream_t stream) {
  HFEE_REQUIRE(n >= 0 && top >= 1 && experts >= 1 && ff >= 1 && width >= 1 && ldx >= width, "moe_down: bad sizes");
  HFEE_REQUIRE(chosen != nullptr || (table != nullptr && token_ids != nullptr), "moe_down: the experts of a token, or a table and the ids");
  if (n == 0) return 0;
  const int per_block = 4 * kRowsPerWave;
  HFEE_REQUIRE((width + per_block - 1) / per_block <= 65535, "moe_down: rows too wide");
  dim3 grid(n, (width + per_block - 1) / per_block);
  // Token by token reads an expert's rows for every pair and walks a token's experts one after the other; expert by expert
  // has every wave look through all groups.  The latter for many bytes of pairs, unless they may lie on many experts, for
  // several experts a token with few groups, and where the former makes thousands of workgroups.  us token by token / expert
  // by expert: 16 experts of 2,048, width 4,096, 4 tokens on one each 12.6 / 10.8, 8 on two each 41 / 31; 128 of 768, width 2,048,
  // one on eight 18.2 / 9.6; 32 of 320, width 1,536, 16 on two each 9.1 / 16.8; 256 of 64, width 1,024, 64 on one each 10.6 / 19.0;
  // 8 of 64, width 4,096, 32 on one each 19.6 / 10.5.
  const int64_t pairs = (int64_t)n * top;
  const int groups = pairs <= 64 ? most_groups((int)pairs, experts) : 0, blocks = (width + kRowsPerWave - 1) / kRowsPerWave;
  const int64_t work = pairs * ff * width;
  const bool by_expert = dtype == 1 && pairs <= 64 && ff % 8 == 0 && (((uintptr_t)act | (uintptr_t)w_down) & 15) == 0 &&
                         ((work >= (int64_t)1 << 24 && groups <= 32) || work >= (int64_t)1 << 26 ||
                          (groups <= 16 && (top >= 3 || (int64_t)top * ff >= 8192)) || (groups <= 24 && (int64_t)n * blocks >= 8192));
  if (by_expert) {
    const auto go = [&](auto kernel, int waves) {
      kernel<<<blocks, 64 * waves, 0, stream>>>(x, ldx, (const bf16_t*)act, (const bf16_t*)w_down, chosen, table, token_ids, pair_weights,
                                                weight, n * top, top, experts, ff, width, accumulate);
    };
    // (as many waves as there can be groups, and as make sixteen a CU)
    const int waves = groups < 4096 / blocks ? groups : 4096 / blocks;
    if (waves <= 4) go(moe_down_by_expert_kernel<4>, 4);
    else if (waves <= 8) go(moe_down_by_expert_kernel<8>, 8);
    else go(moe_down_by_expert_kernel<16>, 16);
  } else if (dtype == 0)
    moe_down_kernel<float><<<grid, 256, 0, stream>>>(x, ldx, (const float*)act, (const float*)w_down, chosen, table,
                                                     token_ids, pair_weights, weight, top, experts, ff, width, accumulate);
  else if (dtype == 1)
    moe_down_kernel<bf16_t><<<grid, 256, 0, stream>>>(x, ldx, (const bf16_t*)act, (const bf16_t*)w_down, chosen, table,
                                                      token_ids, pair_weights, weight, top, experts, ff, width, accumulate);
  else
    return fail("moe_down: unknown dtype %d", dtype);
  HFEE_CHECK_LAUNCH("moe_down");
  return 0;
}
