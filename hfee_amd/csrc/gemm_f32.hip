// True 32-bit matrix product for the check path: C[M,N] (+)= A[M,K] * W[N,K]^T.
//
// The role of /root/reference/internal/ggml/ops.go:54-71 (out[t,r] = W[r,:] . x[t,:]).
// Every product and sum is float32, on the float32 matrix instruction (v_mfma_f32_16x16x4_f32, 154 TFLOP/s here
// against half of that on the vector units without packed instructions).
//
// One order of additions for every kernel in this file.  K is cut into at most eight segments of equal length (a
// multiple of 32).  In a segment the columns go through the matrix instruction 32 at a time, as eight instructions of
// which number 4 b + j takes columns 4 b + j, 8 + 4 b + j, 16 + 4 b + j, 24 + 4 b + j (a lane group holds eight
// neighbours); an instruction is a chain of four fused multiply-adds.  The segments' sums are added up in their order.  An
// element's value therefore does not depend on M, on where its row sits in the batch, or on which kernel or tile it
// falls in: a row has the same bits alone and among others.
//
// Three kernels.  Few rows: the weights' way from memory bounds the product, and `stream_kernel` gives a workgroup 16
// weight rows, each of its eight waves a segment of K.  More rows: `direct_kernel`, tiles of A and W that go straight
// into LDS, bound by the matrix instruction, which at float32 runs on the vector units' multipliers: every other vector
// instruction in the loop takes its time from it, so the loop has none.  Sizes and alignments that those loads do not
// take go through `general_kernel`, tiles by way of registers.
//
// Measured, with one thread a 4 x 4 block of a 64 x 64 tile on the vector units (before) and now: 8 B shape, 3 rows, down
// product (4,096 x 14,336) 1,400 -> 42 us (5.6 TB/s of weights), gate and up (28,672 x 4,096) 850 -> 93 us; 500 rows of
// the 1 B shape, gate and up (16,384 x 2,048) 1,900 -> 273 us (123 TFLOP/s; the instruction alone reaches 154), head 3,500
// -> 2,030 us.
#include "common.h"

using namespace hfee;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int SEGMENTS = 8;

// Columns of a segment: K in eight, up to a multiple of 32.
__host__ __device__ __forceinline__ int segment_columns(int K) { return (K + 32 * SEGMENTS - 1) / (32 * SEGMENTS) * 32; }

// Columns k .. k + 3 of a row, whatever lies within it from K on.  VEC: the row starts on 16 bytes and K is a multiple of 4.
// (Zeros come in where the values are used: a select behind the load would make the wave wait for it there.)
template <bool VEC>
__device__ __forceinline__ f32x4 load_columns(const float* __restrict__ row, int k, int K) {
  if constexpr (VEC) return *reinterpret_cast<const f32x4*>(row + min(k, K - 4));
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = row[min(k + i, K - 1)];
  return v;
}

__device__ __forceinline__ f32x4 zero_from(const f32x4& v, int k, int K) {
  f32x4 z;
#pragma unroll
  for (int i = 0; i < 4; ++i) z[i] = k + i < K ? v[i] : 0.f;
  return z;
}

// Four sums that lie side by side in a row of C.
template <bool ACCUMULATE>
__device__ __forceinline__ void store_four(float* c, const f32x4& v, int left, bool wide) {
  if (wide) {        // (on 16 bytes, and all four are columns of C)
    f32x4* p = reinterpret_cast<f32x4*>(c);
    *p = ACCUMULATE ? *p + v : v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < left) c[i] = ACCUMULATE ? c[i] + v[i] : v[i];
  }
}

// The weights as the rows operand, so that a lane's four results are neighbours in a row of C: lane l holds batch row
// l % 16, weight rows 4 (l / 16) .. + 3.
__device__ __forceinline__ f32x4 mfma(float w, float a, const f32x4& acc) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, acc, 0, 0, 0);
}

// Sixteen weight rows of one step of 32 columns, whole 128-byte lines an instruction: eight rows' lines each.  Lane l asks
// for chunk l / 8 (four columns) of rows l % 8 and 8 + l % 8; the products want row l % 16 in lane l, chunks 2 (l / 16) and
// that + 1, which is one exchange of neighbouring groups of eight lanes.
struct SixteenRows {
  f32x4 low, high;

  __device__ __forceinline__ void load(const float* row_low, const float* row_high, int k0) {
    low = load_streamed(reinterpret_cast<const f32x4*>(row_low + k0));
    high = load_streamed(reinterpret_cast<const f32x4*>(row_high + k0));
  }
  __device__ __forceinline__ void exchange(f32x4& first, f32x4& second) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int l = __float_as_int(low[i]), h = __float_as_int(high[i]);
      // (row_ror:8: the lane eight further on in its row of 16; the bank mask picks who takes it)
      first[i] = __int_as_float(__builtin_amdgcn_update_dpp(l, h, 0x128, 0xf, 0xc, false));
      second[i] = __int_as_float(__builtin_amdgcn_update_dpp(h, l, 0x128, 0xf, 0x3, false));
    }
  }
};

template <int MT, bool VEC, bool ACCUMULATE>
__global__ __launch_bounds__(64 * SEGMENTS) void stream_kernel(float* __restrict__ C, int64_t ldc, const float* __restrict__ A,
                                                               int64_t lda, const float* __restrict__ W, int64_t ldw, int M,
                                                               int N, int K, bool wide_stores) {
  constexpr int AHEAD = 4;                         // steps of 32 columns in flight
  __shared__ f32x4 sums[SEGMENTS][MT][kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int seg = segment_columns(K), first = wave * seg, end = min(first + seg, K);
  const int steps = VEC ? max(end - first, 0) / 32 : 0;      // whole ones (a segment that lies behind K has none)

  const float* arow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) arow[t] = A + (int64_t)min(16 * t + r, M - 1) * lda;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const auto multiply = [&](int b, const f32x4& w, const f32x4 (&a)[2][MT]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = mfma(w[j], a[b][m][j], acc[m]);
  };

  if (VEC && steps > 0) {
    const float* row_low = W + (int64_t)min(n0 + (lane & 7), N - 1) * ldw + 4 * (lane >> 3);
    const float* row_high = W + (int64_t)min(n0 + 8 + (lane & 7), N - 1) * ldw + 4 * (lane >> 3);
    SixteenRows w[AHEAD];
    f32x4 a[AHEAD][2][MT];
    const auto load = [&](int i, int k0) {
      w[i].load(row_low, row_high, k0);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int t = 0; t < MT; ++t) a[i][b][t] = *reinterpret_cast<const f32x4*>(arow[t] + k0 + 8 * g + 4 * b);
    };
    const auto multiply_step = [&](int i) {
      f32x4 one, two;
      w[i].exchange(one, two);
      multiply(0, one, a[i]);
      multiply(1, two, a[i]);
    };
    const int last = first + 32 * (steps - 1);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) load(i, min(first + 32 * i, last));
    int s = 0;
    for (; s + AHEAD <= steps; s += AHEAD) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        multiply_step(i);
        __builtin_amdgcn_sched_barrier(0);                    // (else every load of the loop ends up behind its last product)
        load(i, min(first + 32 * (s + i + AHEAD), last));     // (past the end: the last step once more, not used)
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (s + i < steps) multiply_step(i);
  }
  // columns behind the last whole step, zeros from K on (and all columns of rows that 16-byte loads do not take)
  for (int k0 = first + 32 * steps; k0 < end; k0 += 32) {
    const float* wrow = W + (int64_t)min(n0 + r, N - 1) * ldw;
    f32x4 w[2], a[2][MT];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int k = k0 + 8 * g + 4 * b;
      w[b] = zero_from(load_columns<VEC>(wrow, k, K), k, K);
#pragma unroll
      for (int t = 0; t < MT; ++t) a[b][t] = zero_from(load_columns<VEC>(arow[t], k, K), k, K);
    }
    multiply(0, w[0], a);
    multiply(1, w[1], a);
  }

  // the segments' sums, added in their order; wave t does the t-th sixteen rows of the batch
#pragma unroll
  for (int m = 0; m < MT; ++m) sums[wave][m][lane] = acc[m];
  __syncthreads();
  if (wave >= MT) return;
  f32x4 total = sums[0][wave][lane];
  for (int i = 1; i < SEGMENTS && i * seg < K; ++i) total += sums[i][wave][lane];
  const int row = 16 * wave + r, n = n0 + 4 * g;
  if (row < M && n < N) store_four<ACCUMULATE>(C + (int64_t)row * ldc + n, total, N - n, wide_stores && n + 4 <= N);
}

// Which tile a workgroup does.  Neighbouring workgroups go to different XCDs: each XCD gets a run of tiles, of which those
// that follow one another share their weight rows in its L2.
struct TilePlace {
  int m0, n0;
  __device__ __forceinline__ TilePlace(int M, int rows, int columns) {
    const int tiles_m = (M + rows - 1) / rows, share = gridDim.x / 8, rest = gridDim.x % 8, xcd = blockIdx.x % 8;
    const int tile = xcd * share + min(xcd, rest) + (int)blockIdx.x / 8;
    m0 = tile % tiles_m * rows;
    n0 = tile / tiles_m * columns;
  }
};

// The sums of a tile, as two by two waves hold them.
template <int TM, int TN, bool ACCUMULATE>
__device__ __forceinline__ void store_tile(float* C, int64_t ldc, int M, int N, int m0, int n0, int lane, const f32x4 (&total)[TM][TN],
                                           bool wide_stores) {
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = m0 + 16 * m + (lane & 15);
    if (row >= M) continue;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const int n = n0 + 16 * t + 4 * (lane >> 4);
      if (n < N) store_four<ACCUMULATE>(C + (int64_t)row * ldc + n, total[m][t], N - n, wide_stores && n + 4 <= N);
    }
  }
}

// Tiles of 32 TM rows of A and 32 TN rows of W, two by two waves with 16 TM x 16 TN each.  K in steps of 32 columns; a
// step's rows, 128 bytes each, go from memory straight into one of four buffers in LDS, asked for three steps before they
// are read and read one step before they are multiplied.  A row's eight 16-byte chunks lie at chunk ^ (row % 8), so that
// the rows that a read asks the same chunk of spread over the banks.  K is a multiple of 32, rows start on 16 bytes.
template <int TM, int TN, bool ACCUMULATE>
__global__ __launch_bounds__(256) void direct_kernel(float* __restrict__ C, int64_t ldc, const float* __restrict__ A, int64_t lda,
                                                     const float* __restrict__ W, int64_t ldw, int M, int N, int K,
                                                     bool wide_stores) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass has no buffer resources; it only needs the stub
  constexpr int BUFFERS = 4, ROW = 128, BUFFER = 32 * (TM + TN) * ROW;
  extern __shared__ __attribute__((aligned(1024))) char lds_bytes[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const TilePlace place(M, 32 * TM, 32 * TN);
  const int wave_m = (wave & 1) * 16 * TM, wave_n = (wave >> 1) * 16 * TN;
  const int steps = K / 32, per_segment = segment_columns(K) / 32;

  // Buffer loads from the tile's first row on: a lane's offset is a register that never changes, the step a scalar.
  // Request t of a wave fills rows 32 t + 8 wave .. + 7 of the tile: lane -> row lane / 8, chunk lane % 8 of the LDS.
  typedef __attribute__((address_space(3))) void* lds_ptr;
  const int lrow = 8 * wave + (lane >> 3), chunk = (lane & 7) ^ (lrow & 7);
  const auto bytes = [&](int rows, int64_t ld) { return (int)min(((int64_t)(rows - 1) * ld + K) * 4, (int64_t)0x7fffffff); };
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(A + place.m0 * lda), 0, bytes(min(32 * TM, M - place.m0), lda), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(W + place.n0 * ldw), 0, bytes(min(32 * TN, N - place.n0), ldw), 0x00020000);
  uint32_t a_off[TM], w_off[TN];
#pragma unroll
  for (int t = 0; t < TM; ++t) a_off[t] = (uint32_t)(min(lrow + 32 * t, M - 1 - place.m0) * lda + 4 * chunk) * 4;
#pragma unroll
  for (int t = 0; t < TN; ++t) w_off[t] = (uint32_t)(min(lrow + 32 * t, N - 1 - place.n0) * ldw + 4 * chunk) * 4;
  const auto load_one = [&](int step, int t) {
    const int at = min(step, steps - 1) * ROW;                // (past the end: a repeat that nobody uses)
    char* dst = lds_bytes + (step & (BUFFERS - 1)) * BUFFER + wave * 1024;
    if (t < TM) __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr)(dst + t * 4096), 16, a_off[t], at, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_ptr)(dst + t * 4096), 16, w_off[t - TM], at, 0, 0);
  };

  constexpr int LOADS = TM + TN, READS = 2 * (TM + TN), PRODUCTS = 8 * TM * TN;
  struct Operands {
    f32x4 a[2][TM], w[2][TN];
  };
  // what a lane reads of a buffer: columns 8 g + 4 b of its row
  const char* from[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) from[b] = lds_bytes + r * ROW + (((2 * g + b) ^ (r & 7)) << 4);
  const auto read_one = [&](int buffer, Operands& o, int i) {      // in the order in which the products need them
    const int b = i / LOADS, t = i % LOADS;
    const char* tile = from[b] + buffer * BUFFER;
    if (t < TN) o.w[b][t] = *reinterpret_cast<const f32x4*>(tile + (32 * TM + wave_n + 16 * t) * ROW);
    else o.a[b][t - TN] = *reinterpret_cast<const f32x4*>(tile + (wave_m + 16 * (t - TN)) * ROW);
  };

  f32x4 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[m][t] = total[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < BUFFERS; ++s)
#pragma unroll
    for (int t = 0; t < LOADS; ++t) load_one(s, t);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LOADS) : "memory");
  barrier_no_fence();
  Operands o[2];
#pragma unroll
  for (int i = 0; i < READS; ++i) read_one(0, o[0], i);

  // One step.  In front of the barrier this wave's part of step s + 1 has landed (at most the loads of two later steps are
  // outstanding) and its reads of step s are done; behind it everybody's, so that step s + 1 can be read and the buffer of
  // step s asked into.  Every product with what follows it stands between two scheduling barriers.
  int until_sum = per_segment;
  const auto step = [&](int s, const Operands& now, Operands& next) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * LOADS) : "memory");
    barrier_no_fence();
    const int buffer = (s + 1) & (BUFFERS - 1);
#pragma unroll
    for (int p = 0; p < PRODUCTS; ++p) {
      const int t = p % TN, m = p / TN % TM, j = p / (TN * TM) % 4, b = p / (4 * TN * TM);
      acc[m][t] = mfma(now.w[b][t][j], now.a[b][m][j], acc[m][t]);
#pragma unroll
      for (int i = 0; i < READS; ++i)        // (the reads under the first half of the products, the requests under all)
        if (i >= 2 * READS * p / PRODUCTS && i < 2 * READS * (p + 1) / PRODUCTS) read_one(buffer, next, i);
#pragma unroll
      for (int l = 0; l < LOADS; ++l)
        if (l >= LOADS * p / PRODUCTS && l < LOADS * (p + 1) / PRODUCTS) load_one(s + BUFFERS, l);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (--until_sum == 0 || s + 1 == steps) {       // the end of a segment
      until_sum = per_segment;
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          total[m][t] = s < per_segment ? acc[m][t] : total[m][t] + acc[m][t];
          acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  int s = 0;
  for (; s + 1 < steps; s += 2) {
    step(s, o[0], o[1]);
    step(s + 1, o[1], o[0]);
  }
  if (s < steps) step(s, o[0], o[1]);
  // the repeats asked for past the end still write into this workgroup's LDS: they land before the wave ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  store_tile<TM, TN, ACCUMULATE>(C, ldc, M, N, place.m0 + wave_m, place.n0 + wave_n, lane, total, wide_stores);
#endif
}

// The same tiles for any K and any alignment: 32 columns of both lie in LDS twice, the next ones on their way through
// registers meanwhile, where what lies behind K becomes zero.
template <int TM, int TN, bool VEC, bool ACCUMULATE>
__global__ __launch_bounds__(256) void general_kernel(float* __restrict__ C, int64_t ldc, const float* __restrict__ A, int64_t lda,
                                                      const float* __restrict__ W, int64_t ldw, int M, int N, int K,
                                                      bool wide_stores) {
  __shared__ f32x4 tile_a[2][32 * TM * 8];
  __shared__ f32x4 tile_w[2][32 * TN * 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const TilePlace at(M, 32 * TM, 32 * TN);
  const int wave_m = (wave & 1) * 16 * TM, wave_n = (wave >> 1) * 16 * TN;

  const int lrow = tid >> 3, chunk = tid & 7;       // what a thread brings: this chunk of every 32nd row
  const float* arow[TM];
  const float* wrow[TN];
#pragma unroll
  for (int t = 0; t < TM; ++t) arow[t] = A + (int64_t)min(at.m0 + lrow + 32 * t, M - 1) * lda;
#pragma unroll
  for (int t = 0; t < TN; ++t) wrow[t] = W + (int64_t)min(at.n0 + lrow + 32 * t, N - 1) * ldw;
  const int place = lrow * 8 + (chunk ^ (lrow & 7));

  f32x4 acc[TM][TN], total[TM][TN], in_a[TM], in_w[TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[m][t] = total[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const auto load = [&](int k0) {
#pragma unroll
    for (int t = 0; t < TM; ++t) in_a[t] = load_columns<VEC>(arow[t], k0 + 4 * chunk, K);
#pragma unroll
    for (int t = 0; t < TN; ++t) in_w[t] = load_columns<VEC>(wrow[t], k0 + 4 * chunk, K);
  };
  const auto put = [&](int buffer, int k0) {
#pragma unroll
    for (int t = 0; t < TM; ++t) tile_a[buffer][place + 256 * t] = zero_from(in_a[t], k0 + 4 * chunk, K);
#pragma unroll
    for (int t = 0; t < TN; ++t) tile_w[buffer][place + 256 * t] = zero_from(in_w[t], k0 + 4 * chunk, K);
  };

  const int steps = (K + 31) / 32, per_segment = segment_columns(K) / 32;
  load(0);
  put(0, 0);
  __syncthreads();
  int until_sum = per_segment;
  for (int s = 0; s < steps; ++s) {
    if (s + 1 < steps) load(32 * (s + 1));
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x4 a[TM], w[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m) a[m] = tile_a[s & 1][(wave_m + 16 * m + r) * 8 + ((2 * g + b) ^ (r & 7))];
#pragma unroll
      for (int t = 0; t < TN; ++t) w[t] = tile_w[s & 1][(wave_n + 16 * t + r) * 8 + ((2 * g + b) ^ (r & 7))];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int t = 0; t < TN; ++t) acc[m][t] = mfma(w[t][j], a[m][j], acc[m][t]);
    }
    if (--until_sum == 0 || s + 1 == steps) {       // the end of a segment
      until_sum = per_segment;
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          total[m][t] = s < per_segment ? acc[m][t] : total[m][t] + acc[m][t];
          acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (s + 1 < steps) put((s + 1) & 1, 32 * (s + 1));      // (whoever read that buffer has passed the barrier behind it)
    __syncthreads();
  }
  store_tile<TM, TN, ACCUMULATE>(C, ldc, M, N, at.m0 + wave_m, at.n0 + wave_n, lane, total, wide_stores);
}

struct Product {
  float* C;
  int64_t ldc;
  const float* A;
  int64_t lda;
  const float* W;
  int64_t ldw;
  int M, N, K;
  bool vec, wide_stores, accumulate;
};

template <int MT>
void launch_stream(const Product& p, hipStream_t stream) {
  const dim3 grid((p.N + 15) / 16), block(64 * SEGMENTS);
  const auto go = [&](auto kernel) {
    kernel<<<grid, block, 0, stream>>>(p.C, p.ldc, p.A, p.lda, p.W, p.ldw, p.M, p.N, p.K, p.wide_stores);
  };
  if (p.vec) p.accumulate ? go(stream_kernel<MT, true, true>) : go(stream_kernel<MT, true, false>);
  else p.accumulate ? go(stream_kernel<MT, false, true>) : go(stream_kernel<MT, false, false>);
}

template <int TM, int TN>
int64_t tile_count(const Product& p) {
  return (int64_t)((p.M + 32 * TM - 1) / (32 * TM)) * ((p.N + 32 * TN - 1) / (32 * TN));
}

// What a product in these tiles takes, in rounds of 64 x 64 tiles over the 256 CUs: a tile of half the size takes a little
// more than half the time (it reads more of its operands a product).  us measured with 64 x 64 / 32 x 64 /
// 32 x 32 tiles: N = 4,096, K = 14,336, 96 rows 242 / 152 / 156; 500 rows 480 / 502 / 541; N = 3,072, K = 2,048, 500 rows
// 79 / 67 / 73; N = 28,672, K = 4,096, 24 rows 138 / 99 / 101, 256 rows 451 / 487 / 534 (133 TFLOP/s).
template <int TM, int TN>
double tile_cost(const Product& p) {
  const double size = TM * TN / 4.0, rounds = (double)((tile_count<TM, TN>(p) + 255) / 256);
  return rounds * size * (TM * TN == 4 ? 1.0 : TM * TN == 2 ? 1.07 : 1.2);
}

template <int TM, int TN>
void launch_direct(const Product& p, hipStream_t stream) {
  const dim3 grid((unsigned)tile_count<TM, TN>(p)), block(256);
  constexpr size_t lds = (size_t)4 * 32 * (TM + TN) * 128;
  static_assert(lds <= 64 * 1024, "a kernel gets more LDS only after hipFuncSetAttribute");
  const auto go = [&](auto kernel) {
    kernel<<<grid, block, lds, stream>>>(p.C, p.ldc, p.A, p.lda, p.W, p.ldw, p.M, p.N, p.K, p.wide_stores);
  };
  p.accumulate ? go(direct_kernel<TM, TN, true>) : go(direct_kernel<TM, TN, false>);
}

void launch_general(const Product& p, hipStream_t stream) {
  const dim3 grid((unsigned)tile_count<2, 2>(p)), block(256);
  const auto go = [&](auto kernel) {
    kernel<<<grid, block, 0, stream>>>(p.C, p.ldc, p.A, p.lda, p.W, p.ldw, p.M, p.N, p.K, p.wide_stores);
  };
  if (p.vec) p.accumulate ? go(general_kernel<2, 2, true, true>) : go(general_kernel<2, 2, true, false>);
  else p.accumulate ? go(general_kernel<2, 2, false, true>) : go(general_kernel<2, 2, false, false>);
}

}  // namespace

// accumulate != 0: C += A W^T (the residual add of forward.go:106-107, 113-114).
HFEE_API int hfee_gemm_f32(float* C, int64_t ldc, const float* A, int64_t lda, const float* W, int64_t ldw,
                           int M, int N, int K, int accumulate, hipStream_t stream) {
  HFEE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  HFEE_REQUIRE(ldc >= N && lda >= K && ldw >= K, "gemm_f32: a leading dimension is shorter than its row");
  if (M == 0) return 0;
  HFEE_REQUIRE(M <= 65535 * 64, "gemm_f32: too many rows (%d)", M);
  HFEE_REQUIRE((int64_t)((M + 31) / 32) * ((N + 31) / 32) < (int64_t)1 << 31, "gemm_f32: too many tiles (M=%d N=%d)", M, N);
  const auto on16 = [](const void* p, int64_t ld) { return (uintptr_t)p % 16 == 0 && ld % 4 == 0; };
  Product p{C, ldc, A, lda, W, ldw, M, N, K, K % 4 == 0 && on16(A, lda) && on16(W, ldw), on16(C, ldc), accumulate != 0};
  // (the offsets of a tile's rows are 32-bit)
  const bool direct = p.vec && K % 32 == 0 && lda < (1 << 21) && ldw < (1 << 21);
  // Streaming reads the batch from L2 once for every 16 weight rows and leaves most of an instruction's columns empty, so
  // tiles win from few rows on where there are enough of them for the chip.  us streaming / tiles: N = 28,672, K = 4,096,
  // 3 rows 93 / 99, 16 rows 134 / 99; N = 4,096, K = 14,336, 16 rows 63 / 117, 32 rows 89 / 117, 48 rows 124 / 117;
  // N = K = 2,048, 16 rows 20 / 21, 32 rows 26 / 21.
  const bool few_tiles = N < 6144;
  if (M <= 8 || (M <= 16 && (few_tiles || !direct))) launch_stream<1>(p, stream);
  else if (M <= 32 && (!direct || (few_tiles && K >= 4096))) launch_stream<2>(p, stream);
  else if (!direct) launch_general(p, stream);
  else {
    const double whole = tile_cost<2, 2>(p), half = tile_cost<1, 2>(p), quarter = tile_cost<1, 1>(p);
    if (whole <= half && whole <= quarter) launch_direct<2, 2>(p, stream);
    else if (half <= quarter) launch_direct<1, 2>(p, stream);
    else launch_direct<1, 1>(p, stream);
  }
  HFEE_CHECK_LAUNCH("gemm_f32");
  return 0;
}
