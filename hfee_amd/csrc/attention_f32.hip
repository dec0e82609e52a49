// Paged attention of the 32-bit path for head sizes that are multiples of 16, on the float32 matrix instruction.
//
// The reference's sums (/root/reference/internal/llm/forward.go:144-178): score_j = dot(q, k_j) * scale over the keys of
// the token's own sequence up to its position, softmax, weighted values.  Everything is float32; exponentials are the
// library's.
//
// A workgroup has up to 16 query rows that read the same KV head: neighbouring tokens times the heads of the group.  Keys
// come in tiles of 32 at multiples of 32; wave w of four takes the tiles t with t % 4 == w, keeps its own running
// maximum, sum and values (softmax as it goes), and the four are joined in their order at the end.  Which wave and which
// place in it adds a key depends only on the key's position, and a tile of which a row sees nothing leaves the row's
// numbers as they are: a token's result has the same bits however the work was cut into steps, whatever stands around it
// in the batch, and wherever its pages lie.  (An infinity or NaN in a tile would not leave them: rows that share a workgroup
// and come out with a NaN are done once more, one by one.)
//
// The operands need no rearrangement.  Keys lie in chunks of 16 dims by slot, so a lane's 16 bytes as the rows operand
// stand in a kilobyte that the wave reads front to back; the scores come out with four keys of one query a lane, which is
// the columns operand of the product with the values, whose columns lie in the cache by dimension.
//
// What bounds it: the wait for keys and values of the few tiles a wave has; the products of 500 tokens of 32 heads of 64 on 8
// key heads are 7 us of a layer's 29.  So nothing is waited for one by one: a lane holds each token's sequence and position and
// each page's number, a tile is asked for without a condition, q comes and results go by 16 bytes, and the token groups with
// the most keys start first.  That layer 45 -> 28.6 us, 2,048 tokens 353 -> 240, 180 tokens of 32 heads of 128 30 -> 17, 3
// requests that decode at 60 tokens 9.7 -> 8.3, 8 at 1,000 50 -> 44.  (One wave a token and head, every key read twice and a
// lane a key: 1,453 us.)
#include "common.h"

using namespace hfee;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVES = 4, TILE = 32, ROWS = 16;

__device__ __forceinline__ f32x4 mfma(float rows, float columns, const f32x4& acc) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(rows, columns, acc, 0, 0, 0);
}

// Over the four lanes that hold a query's keys.
__device__ __forceinline__ float query_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, kWave));
  return fmaxf(v, __shfl_xor(v, 32, kWave));
}

__device__ __forceinline__ float query_sum(float v) {
  v += __shfl_xor(v, 16, kWave);
  return v + __shfl_xor(v, 32, kWave);
}

struct Args {
  float* out;
  int64_t ld_out;
  const float* q;
  int64_t ldq;
  const float* cache;
  const int* positions;
  const int* token_segment;
  const int* block_tables;
  const int* items;                                 // (first token, how many) of each workgroup; null: `tokens` each
  int bt_stride, num_heads, n, tokens, window, count;
  float scale;
  bool in_fours, out_fours;                         // rows of q (of out) begin on 16 bytes
};

template <int CHUNKS>      // of 16 dims
__global__ __launch_bounds__(64 * WAVES) void attention_f32_kernel(Args p, CacheLayout lay) {
  constexpr bool BOTH = CHUNKS <= 8;        // keys and values of both halves of a tile in registers at once
  __shared__ f32x4 values[WAVES][CHUNKS][kWave];
  __shared__ float most[WAVES][ROWS], sums[WAVES][ROWS];
  __shared__ bool no_number[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int per = p.num_heads / lay.kv_heads, heads = min(per, ROWS), parts = (per + heads - 1) / heads;
  // (all heads of a token group side by side, and the groups back to front: in a prompt the last have the most keys)
  const int group = p.count - 1 - blockIdx.x / (lay.kv_heads * parts), part = blockIdx.x % (lay.kv_heads * parts);
  const int kvh = part / parts, head0 = (part % parts) * heads;
  const int t0 = p.items != nullptr ? p.items[2 * group] : group * p.tokens;
  const int t1 = min(t0 + min(p.items != nullptr ? p.items[2 * group + 1] : p.tokens, ROWS), p.n);
  if (t0 >= t1) return;
  // lane i keeps the sequence and the position of token t0 + i
  const int token_of_lane = min(t0 + lane, t1 - 1);
  const int segment_of_lane = p.token_segment[token_of_lane], position_of_lane = p.positions[token_of_lane];
  const int token = t0 + r / heads, head = kvh * per + head0 + r % heads;
  const bool valid = token < t1 && head0 + r % heads < per;

  // (rows that do not exist repeat one that does: their weights are all zero)
  const float* q_row = p.q + (int64_t)(valid ? token : t0) * p.ldq + (valid ? head : kvh * per + head0) * (16 * CHUNKS) + 4 * g;
  f32x4 q[CHUNKS];
  if (p.in_fours) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) q[c] = *reinterpret_cast<const f32x4*>(q_row + 16 * c);
  } else {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) q[c][i] = q_row[16 * c + i];
  }
  const int position = __shfl(position_of_lane, r / heads, kWave), pos = valid ? position : -1;
  const int lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;

  // one run of tokens of the same sequence after the other (with items there is one)
  int longest_run = ROWS;
  for (int from = t0; from < t1;) {
    const int segment = __builtin_amdgcn_readlane(segment_of_lane, from - t0);
    int to = from, last = -1, first = 0x7fffffff;
    for (; to < t1 && to - from < longest_run && __builtin_amdgcn_readlane(segment_of_lane, to - t0) == segment; ++to) {
      const int at = __builtin_amdgcn_readlane(position_of_lane, to - t0);
      last = max(last, at);
      first = min(first, p.window > 0 ? max(0, at - p.window + 1) : 0);
    }
    const bool mine = valid && token >= from && token < to;
    const int* bt = p.block_tables + (int64_t)segment * p.bt_stride;
    // lane i keeps the page of block first_block + i, of those that hold a key of the run (without one, where every position is
    // below zero, the table's first entry is read and no tile)
    const int last_block = max(last, 0) >> lay.page_shift;
    int first_block = first >> lay.page_shift;
    int page_of_lane = bt[min(first_block + lane, last_block)];

    f32x4 o[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, sum = 0.f;
    const int tile0 = first / TILE, tile1 = last < 0 ? -1 : last / TILE;
    for (int t = tile0 + ((wave - tile0) & (WAVES - 1)); t <= tile1; t += WAVES) {
      bool there[2];
      int slot[2];
      const float* at[2];       // the half's page
      f32x4 k[2][CHUNKS], v[2][CHUNKS];
      const auto load_keys = [&](int u) {
        const float* keys = at[u] + lay.key_offset(0, kvh, slot[u] + r, 4 * g);
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) k[u][c] = *reinterpret_cast<const f32x4*>(keys + (int64_t)c * lay.key_chunk_stride());
      };
      const auto load_values = [&](int u) {
        // (a lane group's four keys; slots 8 .. 11 and 4 .. 7 of sixteen have changed places)
        const float* columns = at[u] + lay.value_column(0, kvh, r) + lay.value_slot(slot[u] + 4 * g);
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) v[u][c] = *reinterpret_cast<const f32x4*>(columns + (int64_t)16 * c * lay.page_size);
      };
      // (a half without a key of the run reads the run's first or last block instead: everything is asked for at once, with
      // no condition between, and what such a half gives is masked)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int key0 = TILE * t + 16 * u, block = min(max(key0 >> lay.page_shift, first >> lay.page_shift), last_block);
        there[u] = key0 <= last && key0 + 15 >= first;
        if (block >= first_block + kWave) {
          first_block = block;
          page_of_lane = bt[min(first_block + lane, last_block)];
        }
        slot[u] = key0 & (lay.page_size - 1);
        at[u] = p.cache + (int64_t)__builtin_amdgcn_readlane(page_of_lane, __builtin_amdgcn_readfirstlane(block - first_block)) * lay.page_stride;
      }
      if (BOTH) {
        load_keys(0);
        load_keys(1);
        load_values(0);
        load_values(1);
      }
      f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      if (BOTH) {
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int u = 0; u < 2; ++u) s[u] = mfma(k[u][c][j], q[c][j], s[u]);
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          load_keys(u);
#pragma unroll
          for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) s[u] = mfma(k[u][c][j], q[c][j], s[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = TILE * t + 16 * u + 4 * g + i;
          s[u][i] = mine && there[u] && key <= pos && key >= lo ? s[u][i] * p.scale : -INFINITY;
        }
      float top = m;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) top = fmaxf(top, s[u][i]);
      top = query_max(top);
      const float keep = top == -INFINITY ? 1.f : expf(m - top);       // (a row that has seen no key yet stays at zero)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[u][i] = s[u][i] == -INFINITY ? 0.f : expf(s[u][i] - top);
      m = top;
      sum = sum * keep + (((s[0][0] + s[0][1]) + (s[0][2] + s[0][3])) + ((s[1][0] + s[1][1]) + (s[1][2] + s[1][3])));
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) o[c] *= keep;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (!there[u]) continue;
        if (!BOTH) load_values(u);
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            // (slots that no row of the run sees may hold anything: times a weight of zero they must stay out)
            const int key = TILE * t + 16 * u + 4 * g + j;
            o[c] = mfma(key <= last && key >= first ? v[u][c][j] : 0.f, s[u][j], o[c]);
          }
      }
    }

    // the four waves' shares, joined in their order; each wave does every fourth chunk of dims
    sum = query_sum(sum);
    if (lane < ROWS) {
      most[wave][r] = m;
      sums[wave][r] = sum;
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) values[wave][c][lane] = o[c];
    __syncthreads();
    float top = most[0][r], weight[WAVES], total = 0.f;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, most[w][r]);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      weight[w] = most[w][r] == -INFINITY ? 0.f : expf(most[w][r] - top);
      total += sums[w][r] * weight[w];
    }
    bool nan = false;
    for (int c = wave; c < CHUNKS; c += WAVES) {
      f32x4 all = values[0][c][lane] * weight[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) all += values[w][c][lane] * weight[w];
      if (mine) {
        float* to_row = p.out + (int64_t)token * p.ld_out + head * (16 * CHUNKS) + 16 * c + 4 * g;
        f32x4 result;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          result[i] = all[i] / total;
          nan = nan || isnan(all[i]);
        }
        if (p.out_fours) *reinterpret_cast<f32x4*>(to_row) = result;
        else
#pragma unroll
          for (int i = 0; i < 4; ++i) to_row[i] = result[i];
      }
    }
    // A key's values meet the weights of all rows, those that are zero because a row does not see the key as well, and zero
    // times an infinity or NaN is NaN: a run with a NaN is done once more, token by token, where rows see the same keys.
    if (to - from > 1) {
      const bool some = __ballot(nan) != 0;
      if (lane == 0) no_number[wave] = some;
      __syncthreads();
      if (no_number[0] || no_number[1] || no_number[2] || no_number[3]) {
        longest_run = 1;
        continue;
      }
    }
    from = to;
    if (from < t1) __syncthreads();       // (the next run's shares go to the same places)
  }
}

template <int CHUNKS>
void launch(const Args& p, const CacheLayout& lay, dim3 grid, hipStream_t stream) {
  attention_f32_kernel<CHUNKS><<<grid, 64 * WAVES, 0, stream>>>(p, lay);
}

}  // namespace

// A workgroup takes up to 16 rows, which are 16 / heads of a KV head (up to 16) tokens; tokens of different sequences in one
// would be one after the other, each through its own keys.  items: int32 [item_count][2], the tokens of each workgroup
// (first, how many); null: neighbours, whatever their sequences, or with singles != 0 one each.  16 requests that decode at
// 4,000 tokens beside a portion of 64, 4 heads of 64 on as many key heads: 2,250 us neighbour by neighbour, 149 with items
// (1,610 with a wave a token and head); at 1,000 tokens, 32 heads of 128 on 8 key heads, 213 and 61 (760): times of the kernel
// that waited for every load.
HFEE_API int hfee_attention_f32(float* out, int64_t ld_out, const float* q, int64_t ldq, const float* cache,
                                const int* positions, const int* token_segment, const int* block_tables, int bt_stride,
                                int num_heads, int kv_heads, int head_dim, int page_size, float scale, int window, const int* items,
                                int item_count, int singles, int n, hipStream_t stream) {
  HFEE_REQUIRE(n >= 0, "attention_f32: bad token count");
  if (n == 0) return 0;
  HFEE_REQUIRE(num_heads > 0 && kv_heads > 0 && num_heads % kv_heads == 0,
               "attention_f32: %d heads are not a multiple of %d kv heads", num_heads, kv_heads);
  HFEE_REQUIRE(head_dim >= 16 && head_dim <= 256 && head_dim % 16 == 0, "attention_f32: head_dim %d is no multiple of 16 up to 256", head_dim);
  HFEE_REQUIRE(num_heads <= 65535, "attention_f32: too many heads");
  HFEE_REQUIRE(window >= 0, "attention_f32: negative window");
  HFEE_REQUIRE(items == nullptr || item_count > 0, "attention_f32: no items");
  HFEE_REQUIRE(ldq >= (int64_t)num_heads * head_dim && ld_out >= (int64_t)num_heads * head_dim, "attention_f32: q/out row too short");
  HFEE_REQUIRE((uintptr_t)cache % 16 == 0, "attention_f32: the cache layer must start on 16 bytes");
  CacheLayout lay;
  if (make_cache_layout(&lay, kv_heads, head_dim, page_size)) return 1;
  const int per = num_heads / kv_heads, heads = per < ROWS ? per : ROWS, tokens = singles ? 1 : ROWS / heads;
  const int count = items != nullptr ? item_count : (n + tokens - 1) / tokens;
  const int64_t groups = (int64_t)count * kv_heads * ((per + heads - 1) / heads);
  HFEE_REQUIRE(groups <= 0x7fffffff, "attention_f32: too many tokens");
  const dim3 grid((unsigned)groups);
  const Args p{out, ld_out, q, ldq, cache, positions, token_segment, block_tables, items, bt_stride, num_heads, n, tokens, window, count, scale,
               (uintptr_t)q % 16 == 0 && ldq % 4 == 0, (uintptr_t)out % 16 == 0 && ld_out % 4 == 0};
  switch (head_dim / 16) {
#define HFEE_CHUNKS(C) case C: launch<C>(p, lay, grid, stream); break;
    HFEE_CHUNKS(1) HFEE_CHUNKS(2) HFEE_CHUNKS(3) HFEE_CHUNKS(4) HFEE_CHUNKS(5) HFEE_CHUNKS(6) HFEE_CHUNKS(7) HFEE_CHUNKS(8)
    HFEE_CHUNKS(9) HFEE_CHUNKS(10) HFEE_CHUNKS(11) HFEE_CHUNKS(12) HFEE_CHUNKS(13) HFEE_CHUNKS(14) HFEE_CHUNKS(15) HFEE_CHUNKS(16)
#undef HFEE_CHUNKS
  }
  HFEE_CHECK_LAUNCH("attention_f32");
  return 0;
}
