// bfloat16 products on the matrix cores (MFMA), float32 accumulation.
//
// Up to 16 rows of x, the shape of decoding, are gemm_flow's below, 17 to 128 gemm_stream's, gemm_medium's and gemm_ring's.
//
// gemm_skinny: out[M, N] = x[M, K] . w[N, K]^T (+ bias) for M <= 64 at the sizes and operands that those do not take: a K that is no multiple of 64 (up to 16
// rows) or 128, and operands that begin inside a piece of 16 bytes.  Such a product is a stream of the weight matrix from HBM:
// a workgroup owns 16 weight rows and its waves split K between them; every
// lane keeps two groups of four 16-byte loads of its weight row in flight; the weights go
// straight from global memory into the A operand of v_mfma_f32_16x16x32_bf16 (lane l holds
// row l % 16, k = (l / 16) * 8 .. + 8 of a 32-wide step), the few activation rows into the B
// operand, so the result tile D[n][m] leaves four consecutive n of one token in each lane.
// The waves' partial tiles are added through LDS in wave order, so a row's bits depend on
// the shape of the weight only, not on what else is in the batch.
//
// With `gated`, weight rows alternate gate_j, up_j and the epilogue writes
// silu(gate) * up (reference model.py:188) to out[M, N / 2].
#include "common.h"
#include <type_traits>
#include <utility>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Loads into LDS, and of vectors, bring 16 bytes from a multiple of 16.
static bool in_pieces(const void* a, const void* b) { return (((size_t)a | (size_t)b) & 15) == 0; }

#define STEP 32   // k per MFMA
#define GROUP 4   // MFMA steps a wave loads at once: 128 k, 256 bytes of each weight row

__device__ __forceinline__ bf16x8 load8(const bf16_t* p) { return *(const bf16x8*)p; }
// (Plain loads: a load here takes half a cache line of sixteen rows, the next the other half; past the caches they were 8-12 % slower.  gemm_flow takes whole lines, and past them.)
__device__ __forceinline__ bf16x8 load8_stream(const bf16_t* p) { return *(const bf16x8*)p; }
#ifndef TARGET_WAVES
#define TARGET_WAVES 2048
#endif

// GATED in the kernels for up to 64 rows below: 0 a plain product, 1 silu(gate) * up, 2 relu(gate) * up, 3 a plain product
// whose columns from `Tail::first` on are activated (relu(z)^2) and go to rows of their own
struct Tail {
  bf16_t* rows;  // column n of row m, n >= first, goes to rows[m * stride + n - first]; a column below `first` to out[m * first + n]
  int first, stride;
};

template <typename TO>
__device__ __forceinline__ void store_with_tail(TO* out, const Tail& tail, int m, int n_first, int N, f32x4 total) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n_first + i;
    if (n >= N) break;
    if (n < tail.first) {
      out[(size_t)m * tail.first + n] = from_float<TO>(total[i]);
    } else {
      const float z = fmaxf(total[i], 0.f);
      tail.rows[(size_t)m * tail.stride + n - tail.first] = (bf16_t)(z * z);
    }
  }
}

template <int GATED>
__device__ __forceinline__ float gate_value(float gate) {
  return GATED == 2 ? fmaxf(gate, 0.f) : gate / (1.f + expf(-gate));
}

// Two products with a norm between them, without a kernel for the norm (up to 64 rows).  The first one
// (INTO_NORM) holds whole sums over K, adds them to the residual stream in its epilogue, and writes what the second reads:
// x * weight in bfloat16, not yet divided by the row's root mean square, and each tile's sum of squares of x a row.  The second
// one (SCALED) multiplies its float32 results by rsqrt(mean of squares + eps), which is the same for all of a row's
// products: rounding x * weight loses what rounding the normed row loses.  A norm's kernel is a launch, two trips to
// memory and a sum over a workgroup, 4 to 5 us whatever the rows.  Against that the first product needs whole sums over K, and the second one brings the sums of
// squares.  A pass of four steps, us, the three apart -> linked: 1.5B sizes 1 row 4,130 -> 3,899, 8 rows 4,406 -> 4,160 (contexts of 4,000: 5,460 -> 5,166), 16 rows 4,666 -> 4,440, 64
// rows 6,182 -> 6,059; 7B sizes 1 row 10,478 -> 10,187, 8 rows 10,773 -> 10,496, 16 rows 11,783 -> 11,597, 64 rows (no link there) 14,187.
enum { NO_LINK = 0, INTO_NORM = 1, SCALED = 2 };
struct Link {
  float* hidden;             // INTO_NORM: [M, N], added to in place
  const void* weight;        // INTO_NORM: the norm's [N]
  int weight_is_float;
  bf16_t* rows;              // INTO_NORM: [M, N]
  float* sums;               // [tiles, stride]: of 16 columns of x each, row by row
  int stride, tiles;
  float inverse_width, eps;  // SCALED
};

// The end of a product into a norm: `total` four neighbouring columns from n_first of row m, of 16 (tile) that the lanes
// r, r + 16, r + 32, r + 48 share; they are in the branch together.  N is a multiple of 16.
struct LinkedColumns {
  f32x4 hidden;
  uint2 low, high;  // of the weight: four bfloat16 (twice) or the halves of four float32
};
// (asked for at the start and used at the end; without a branch, at whose end the loads inside would be waited for: that cost
// the 1.5B sizes' output projection 1.5 us)
__device__ __forceinline__ LinkedColumns linked_columns(const Link& link, int m, int n_first, int M, int N) {
  LinkedColumns columns;
  columns.hidden = *(const f32x4*)(link.hidden + (size_t)min(m, M - 1) * N + n_first);
  const char* weight = (const char*)link.weight + (size_t)n_first * (link.weight_is_float ? 4 : 2);
  columns.low = *(const uint2*)weight;
  columns.high = *(const uint2*)(weight + (link.weight_is_float ? 8 : 0));
  asm volatile("" ::: "memory");  // (asked for here)
  return columns;
}
__device__ __forceinline__ void store_into_norm(const Link& link, const LinkedColumns& columns, f32x4 total, int m, int n_first, int N) {
  const f32x4 x = columns.hidden + total;
  *(f32x4*)(link.hidden + (size_t)m * N + n_first) = x;
  const unsigned halves[4] = {columns.low.x << 16, columns.low.x & 0xffff0000u, columns.low.y << 16, columns.low.y & 0xffff0000u};
  const unsigned words[4] = {columns.low.x, columns.low.y, columns.high.x, columns.high.y};
  bf16_t row[4];
  float squares = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    row[i] = (bf16_t)(x[i] * __uint_as_float(link.weight_is_float ? words[i] : halves[i]));
    squares = fmaf(x[i], x[i], squares);
  }
  *(uint2*)(link.rows + (size_t)m * N + n_first) = *(const uint2*)row;
  squares += __shfl_xor(squares, 16, WAVE);
  squares += __shfl_xor(squares, 32, WAVE);
  if (n_first % 16 == 0) link.sums[(size_t)(n_first / 16) * link.stride + m] = squares;
}

// This thread's share of the sums of squares of row threadIdx.x % ROWS: the tiles threadIdx.x / ROWS, + THREADS / ROWS, ...
template <int THREADS, int ROWS>
__device__ __forceinline__ float squares_share(const Link& link, int M) {
  const float* of_row = link.sums + min((int)threadIdx.x % ROWS, M - 1);
  float share = 0.f;
#pragma unroll 8
  for (int tile = threadIdx.x / ROWS; tile < link.tiles; tile += THREADS / ROWS) share += of_row[(size_t)tile * link.stride];
  return share;
}
// The factor of row m, once every thread's share is in LDS (`shares`, a thread after the other) and a barrier has passed.
template <int THREADS, int ROWS>
__device__ __forceinline__ float row_factor(const Link& link, const float* shares, int m) {
  float squares = 0.f;
#pragma unroll
  for (int part = 0; part < THREADS / ROWS; ++part) squares += shares[part * ROWS + m];
  return rsqrtf(squares * link.inverse_width + link.eps);
}

template <int WAVES, int MT, typename TO, int GATED>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(const bf16_t* __restrict__ x,
                                                                 const bf16_t* __restrict__ w,
                                                                 const void* __restrict__ bias, int bias_is_float,
                                                                 TO* __restrict__ out, int M, int N, int K,
                                                                 int k_split, Tail tail) {
  extern __shared__ float partial[];  // [WAVES][MT][64 lanes][4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int n = min((int)blockIdx.x * 16 + r, N - 1);
  // blockIdx.y picks a slice of K, `k_split` long; its sums go to its own copy of `out`
  const int k_first = blockIdx.y * k_split;
  const bf16_t* w_row = w + (size_t)n * K + k_first + g * 8;
  const bf16_t* x_row[MT];
  bool x_live[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + r;
    x_live[t] = m < M;
    x_row[t] = x + (size_t)min(m, M - 1) * K + k_first + g * 8;
  }
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  // the bias of this lane's four outputs is asked for now and used at the end
  const bool with_bias = bias && blockIdx.y == 0;
  // (as 16-bit halves, so that both types of bias take the same loads: a float32 is two of them, a
  // bfloat16 the upper one alone)
  // (without a branch: where there is no bias the same loads read the start of the weights and
  // their result is dropped; loads inside a branch would be waited for at its end)
  unsigned short bias_low[4], bias_high[4];
  {
    const unsigned short* source = with_bias ? (const unsigned short*)bias : (const unsigned short*)w;
    const int halves = with_bias && bias_is_float ? 2 : 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = min((int)blockIdx.x * 16 + g * 4 + i, N - 1) * halves;
      bias_low[i] = source[at];
      bias_high[i] = source[at + halves - 1];
    }
  }

  const int groups = k_split / (STEP * GROUP);
  bf16x8 a[GROUP], a_next[GROUP];
  int group = wave;
  if (group < groups) {
#pragma unroll
    for (int u = 0; u < GROUP; ++u) a[u] = load8_stream(w_row + (group * GROUP + u) * STEP);
  }
  while (group < groups) {
    const int next = group + WAVES;
    // this group's x is asked for before the next group's weights: loads come back in the order they
    // were asked for, and the products below wait for x
    bf16x8 b[MT][GROUP];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < GROUP; ++u) b[t][u] = x_live[t] ? load8(x_row[t] + (group * GROUP + u) * STEP) : zero;
    asm volatile("" ::: "memory");  // (the compiler would put the weights first again)
    if (next < groups) {
#pragma unroll
      for (int u = 0; u < GROUP; ++u) a_next[u] = load8_stream(w_row + (next * GROUP + u) * STEP);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < GROUP; ++u) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[t][u], acc[t], 0, 0, 0);
#pragma unroll
    for (int u = 0; u < GROUP; ++u) a[u] = a_next[u];
    group = next;
  }
  // the steps left over when K is not a multiple of 128
  for (int step = groups * GROUP + wave; step < k_split / STEP; step += WAVES) {
    const bf16x8 a_tail = load8_stream(w_row + step * STEP);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const bf16x8 b_tail = x_live[t] ? load8(x_row[t] + step * STEP) : zero;
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_tail, b_tail, acc[t], 0, 0, 0);
    }
  }

#pragma unroll
  for (int t = 0; t < MT; ++t) *(f32x4*)(partial + ((wave * MT + t) * 64 + lane) * 4) = acc[t];
  __syncthreads();
  if (wave >= MT) return;
  // wave t finishes token tile t: lane holds token m = t * 16 + r, rows n0 + g * 4 .. + 4
  const int t = wave;
  f32x4 total = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int v = 0; v < WAVES; ++v) total += *(const f32x4*)(partial + ((v * MT + t) * 64 + lane) * 4);
  const int m = t * 16 + r;
  const int n_first = blockIdx.x * 16 + g * 4;
  if (m >= M) return;
  if (with_bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      total[i] += __uint_as_float((unsigned)bias_high[i] << 16 | (bias_is_float ? (unsigned)bias_low[i] : 0u));
  }
  if (GATED == 3) {
    store_with_tail(out, tail, m, n_first, N, total);
  } else if (GATED) {
    TO* dst = out + (size_t)m * (N / 2) + n_first / 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (n_first + 2 * i + 1 < N) {
        const float gate = total[2 * i], up = total[2 * i + 1];
        dst[i] = from_float<TO>(gate_value<GATED>(gate) * up);
      }
    }
  } else {
    TO* dst = out + ((size_t)blockIdx.y * M + m) * N + n_first;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n_first + i < N) dst[i] = from_float<TO>(total[i]);
  }
}

template <int WAVES, int MT, typename TO, int GATED>
static int launch_skinny(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N,
                         int K, int splits, hipStream_t stream, Tail tail = {}) {
  const size_t lds = (size_t)WAVES * MT * 64 * 4 * sizeof(float);
  hipLaunchKernelGGL((gemm_skinny_kernel<WAVES, MT, TO, GATED>), dim3((N + 15) / 16, splits), dim3(WAVES * 64), lds,
                     stream, (const bf16_t*)x, (const bf16_t*)w, bias, bias_is_float, (TO*)out, M, N, K, K / splits, tail);
  return LAUNCH_STATUS();
}

template <int WAVES, typename TO, int GATED>
static int pick_tiles(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                      int splits, hipStream_t stream, Tail tail = {}) {
  if (M <= 16) return launch_skinny<WAVES, 1, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, tail);
  if (M <= 32) return launch_skinny<WAVES, 2, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, tail);
  return launch_skinny<WAVES, 4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, tail);
}

template <typename TO, int GATED>
static int pick_waves(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                      int splits, hipStream_t stream, Tail tail = {}) {
  // enough waves to cover the chip (about 2,048), but no more than there are 128-wide groups of K
  const int tiles = (N + 15) / 16 * splits, groups = max(1, K / splits / (STEP * GROUP));
  int waves = 4;
  while (waves < 16 && waves * tiles < TARGET_WAVES && waves * 2 <= groups) waves *= 2;
  if (waves == 4) return pick_tiles<4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, tail);
  if (waves == 8) return pick_tiles<8, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, tail);
  return pick_tiles<16, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, tail);
}

// ---------------------------------------------------------------------------- the streams through LDS
// gemm_stream: 17 to 64 rows of x and a small weight, both operands brought through LDS.
// The matrix cores take a weight row as a row of the A operand, lane (r, g) holding k = 8g .. 8g+7 of
// row r, so the four lanes the address unit serves together (r .. r+3 at one g) would read 16 bytes
// of four different rows, four cache lines, and a load of a wave costs that unit four times what
// 64 bytes in a row cost it; x is read the same way.  Here lane L instead asks for piece L % 4 of row
// L / 4 (a quad reads 64 bytes of one row), straight into LDS (global_load_lds_dwordx4: the wave's 1 KB
// lands in lane order), and lane (r, g) reads its operand back from slot 4 r + g.  The pieces of a
// row are swizzled by bits 1-2 of the row so that the eight lanes LDS serves together hit all banks.
// Every wave has STAGES stages of its own, a stage holding one group of G steps of 32 k of its NT
// weight tiles and of x; nothing is shared between waves before the end, so the only waits are the
// wave's own: for its loads to land (counted, so that the younger stage may still be under way) and
// for its reads to come back before the stage is asked for anew.  The reads of LDS are written as
// instructions: left to the compiler, every read of LDS waits for all loads into LDS under way.
#define STREAM_STAGES 2
#define STREAM_CHUNK 1024  // one 32-k step of 16 rows

template <int OFFSET>
__device__ __forceinline__ void stream_read(bf16x8& operand, unsigned at) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(operand) : "v"(at), "n"(OFFSET) : "memory");
}
template <int I, int COUNT>
struct StreamReads {
  static __device__ __forceinline__ void run(bf16x8* operands, unsigned at) {
    stream_read<I * STREAM_CHUNK>(operands[I], at);
    StreamReads<I + 1, COUNT>::run(operands, at);
  }
};
template <int COUNT>
struct StreamReads<COUNT, COUNT> {
  static __device__ __forceinline__ void run(bf16x8*, unsigned) {}
};
// What a lane reads of a tile of sixteen rows, step by step: the tile's chunks are its upper and lower eight rows of 64 k, then of the next 64.
template <int I, int COUNT>
struct RingReads {
  static __device__ __forceinline__ void run(bf16x8* operands, unsigned even, unsigned odd) {
    stream_read<I / 2 * 2 * STREAM_CHUNK>(operands[I], I % 2 ? odd : even);
    RingReads<I + 1, COUNT>::run(operands, even, odd);
  }
};
template <int COUNT>
struct RingReads<COUNT, COUNT> {
  static __device__ __forceinline__ void run(bf16x8*, unsigned, unsigned) {}
};

template <int N>
__device__ __forceinline__ void stream_wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// MT: 16-row tiles of x (up to 16 MT rows).  A stage then holds MT chunks of x beside the NT of the
// weights for every step, and each weight operand meets MT operands of x.
template <int WAVES, int NT, int MT, int G, typename TO, int GATED, int LINK = NO_LINK>
__global__ __launch_bounds__(WAVES * 64) void gemm_stream_kernel(const bf16_t* __restrict__ x,
                                                                 const bf16_t* __restrict__ w,
                                                                 const void* __restrict__ bias, int bias_is_float,
                                                                 TO* __restrict__ out, int M, int N, int K,
                                                                 int k_split, Link link) {
  extern __shared__ __attribute__((aligned(16))) unsigned char stream_lds[];
  constexpr int OPERANDS = (NT + MT) * G;                // of one group: the weight tiles' steps, then x's
  constexpr int STAGE_BYTES = OPERANDS * STREAM_CHUNK;
  constexpr int WAVE_BYTES = STREAM_STAGES * STAGE_BYTES;
  constexpr int TILES = NT * MT;                         // of the result
  static_assert(OPERANDS <= 31, "a group's loads are counted in vmcnt beside a second group's");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int k_first = blockIdx.y * k_split;
  // what this lane asks for: piece (L % 4) ^ f(row) of row L / 4, and where lane (r, g) finds its own
  const int load_row = lane >> 2, load_piece = (lane & 3) ^ ((load_row >> 1) & 3);
  const bf16_t* w_src[NT];
#pragma unroll
  for (int s = 0; s < NT; ++s)
    w_src[s] = w + (size_t)min(((int)blockIdx.x * NT + s) * 16 + load_row, N - 1) * K + k_first + load_piece * 8;
  // rows of x beyond M are read as row M - 1: their columns of the result are dropped at the end
  const bf16_t* x_src[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) x_src[t] = x + (size_t)min(t * 16 + load_row, M - 1) * K + k_first + load_piece * 8;
  unsigned char* mine = stream_lds + (size_t)wave * WAVE_BYTES;
  const unsigned read_at = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)mine +
                           (unsigned)(4 * r + (g ^ ((r >> 1) & 3))) * 16;

  // the bias of the four outputs this lane will finish first (wave v finishes tile v, of weight tile
  // v / MT) is asked for now
  float bias_here[4] = {0.f, 0.f, 0.f, 0.f};
  if (bias && blockIdx.y == 0 && wave < TILES) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      bias_here[i] =
          load_as_float(bias, bias_is_float, min(((int)blockIdx.x * NT + wave / MT) * 16 + g * 4 + i, N - 1));
  }
  static_assert(LINK != INTO_NORM || (TILES <= WAVES && sizeof(TO) == 4), "a wave finishes one tile of whole sums");
  static_assert(LINK != SCALED, "gemm_flow and gemm_ring read such rows");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // so that the counts below count the stream alone
  LinkedColumns columns;  // (ahead of the stream, whose first wait covers them)
  if (LINK == INTO_NORM) columns = linked_columns(link, (wave % MT) * 16 + r, ((int)blockIdx.x * NT + min(wave, TILES - 1) / MT) * 16 + g * 4, M, N);
  auto request = [&](int group, int stage) {
    unsigned char* to = mine + (size_t)stage * STAGE_BYTES;
    const int k = group * G * STEP;
#pragma unroll
    for (int u = 0; u < G; ++u) {
#pragma unroll
      for (int s = 0; s < NT; ++s)
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(w_src[s] + k + u * STEP),
                                         (void __attribute__((address_space(3)))*)(to + (s * G + u) * STREAM_CHUNK), 16,
                                         0, 0);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(x_src[t] + k + u * STEP),
                                         (void __attribute__((address_space(3)))*)(to + ((NT + t) * G + u) * STREAM_CHUNK),
                                         16, 0, 0);
    }
  };

  f32x4 acc[NT][MT];
#pragma unroll
  for (int s = 0; s < NT; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[s][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int groups = k_split / (STEP * G);
  int group = wave;
  if (group < groups) request(group, 0);
  if (group + WAVES < groups) request(group + WAVES, 1);
  for (int stage = 0; group < groups; group += WAVES, stage ^= 1) {
    // this stage has landed once at most the next group's loads are under way
    if (group + WAVES < groups) stream_wait_loads<OPERANDS>();
    else stream_wait_loads<0>();
    bf16x8 operands[OPERANDS];
    StreamReads<0, OPERANDS>::run(operands, read_at + (unsigned)stage * STAGE_BYTES);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < OPERANDS; ++i) asm volatile("" : "+v"(operands[i]));  // used only after the wait
    if (group + 2 * WAVES < groups) request(group + 2 * WAVES, stage);       // the stage is read: ask anew
#pragma unroll
    for (int u = 0; u < G; ++u)
#pragma unroll
      for (int s = 0; s < NT; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operands[s * G + u], operands[(NT + t) * G + u],
                                                              acc[s][t], 0, 0, 0);
  }

  __syncthreads();  // every wave is done with its stages: LDS is free for the waves' sums
  float* partial = (float*)stream_lds;  // [WAVES][TILES][64 lanes][4]
#pragma unroll
  for (int s = 0; s < NT; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) *(f32x4*)(partial + ((wave * TILES + s * MT + t) * 64 + lane) * 4) = acc[s][t];
  __syncthreads();
  for (int tile = wave; tile < TILES; tile += WAVES) {
    const int s = tile / MT;
    f32x4 total = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int v = 0; v < WAVES; ++v) total += *(const f32x4*)(partial + ((v * TILES + tile) * 64 + lane) * 4);
    const int m = (tile % MT) * 16 + r;
    const int n_first = ((int)blockIdx.x * NT + s) * 16 + g * 4;
    if (m >= M) continue;
    if (tile == wave) {
#pragma unroll
      for (int i = 0; i < 4; ++i) total[i] += bias_here[i];
    } else if (bias && blockIdx.y == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) total[i] += load_as_float(bias, bias_is_float, min(n_first + i, N - 1));
    }
    if (LINK == INTO_NORM) {
      store_into_norm(link, columns, total, m, n_first, N);
    } else if (GATED) {
      TO* dst = out + (size_t)m * (N / 2) + n_first / 2;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (n_first + 2 * i + 1 < N) {
          const float gate = total[2 * i], up = total[2 * i + 1];
          dst[i] = from_float<TO>(gate_value<GATED>(gate) * up);
        }
      }
    } else {
      TO* dst = out + ((size_t)blockIdx.y * M + m) * N + n_first;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n_first + i < N) dst[i] = from_float<TO>(total[i]);
    }
  }
}

template <int WAVES, int NT, int MT, int G, typename TO, int GATED, int LINK = NO_LINK>
static int launch_stream(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N,
                         int K, int splits, hipStream_t stream, Link link = {}) {
  const size_t stages = (size_t)WAVES * STREAM_STAGES * (NT + MT) * G * STREAM_CHUNK;
  const size_t sums = (size_t)WAVES * NT * MT * 64 * 4 * sizeof(float);
  const size_t lds = stages > sums ? stages : sums;
  if (lds > 64 * 1024) {
    static bool asked = false;
    if (!asked) {
      if (hipFuncSetAttribute((const void*)gemm_stream_kernel<WAVES, NT, MT, G, TO, GATED, LINK>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return ERR_BAD_ARGUMENT;
      asked = true;
    }
  }
  hipLaunchKernelGGL((gemm_stream_kernel<WAVES, NT, MT, G, TO, GATED, LINK>), dim3((N + 16 * NT - 1) / (16 * NT), splits),
                     dim3(WAVES * 64), lds, stream, (const bf16_t*)x, (const bf16_t*)w, bias, bias_is_float, (TO*)out, M,
                     N, K, K / splits, link);
  return LAUNCH_STATUS();
}

// 17 to 64 rows: two or four tiles of x.  nt, g: 0 = by the sizes, else as asked (measurements).  K / splits a multiple of 128.
template <typename TO, int GATED>
static int pick_stream(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                       int splits, hipStream_t stream, int nt = 0, int g = 0) {
  const long tiles = (N + 15) / 16;
  if (nt == 0) nt = tiles * splits >= 2048 ? 2 : 1;
  if (g == 0) g = 1;
#define ROWS_CASE(NT_, MT_, G_)                                                                              \
  if (nt == NT_ && g == G_ && M <= 16 * MT_)                                                                 \
    return launch_stream<4, NT_, MT_, G_, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
  ROWS_CASE(1, 2, 1)
  ROWS_CASE(2, 2, 1)
  ROWS_CASE(1, 2, 2)
  ROWS_CASE(2, 2, 2)
  ROWS_CASE(1, 4, 1)
  ROWS_CASE(2, 4, 1)
  ROWS_CASE(1, 4, 2)
  ROWS_CASE(2, 4, 2)
  ROWS_CASE(4, 2, 1)
  ROWS_CASE(4, 4, 1)
#undef ROWS_CASE
  return ERR_BAD_ARGUMENT;
}

// ---------------------------------------------------------------------------- up to 16 rows
// gemm_flow: up to 16 rows of x, the shape of decoding, which is a stream of the weight from memory and nothing else.  What the rate of that stream hangs on,
// measured: whole cache lines (a load of a wave is 8 rows x 128 bytes; 16 rows x 64 bytes ask for every line twice), past the caches (non-temporal: a
// line that is read once pushes nothing out, 8-20 % of a large weight's time), and the same number of rows for every CU.  So a workgroup takes
// `rows_each` weight rows, any even number up to 8 NH, rather than a tile of sixteen (flow_shape), and its four waves take the units of 64 k in
// turn.  Lane L asks for piece (L % 8) ^ (L / 8) of row L / 8 of every eight rows, straight into LDS, where lane (r, g) reads its operand of step s, piece
// 4 s + g of row r, from slot 8 r + ((4 s + g) ^ (r % 8)): the eight lanes that LDS serves together hit all banks.  Every wave has STAGES units of its
// own under way (XH eights of rows of x, then NH of weights), asks for a pair of eights anew as soon as it is read, and waits for its own loads alone, counted;
// the waves' sums meet in LDS at the end, added up in wave order: a row's bits depend on sizes, not on what the other rows hold.
// Rows past the last are asked for as the last one: their results are dropped.
// Us in a captured chain over different weights at 1 / 8 / 16 rows, the kernels before (one and two tiles of sixteen rows through LDS, four through registers, the ring)
// -> this one: 1.5B sizes gate/up 11.6 / 12.9 / 13.8 -> 10.5 / 10.5 / 11.3, down 6.8 / 7.4 / 7.9 -> 6.2 / 6.3 / 6.7, head 75 / 90 / 99 -> 72 / 73 / 79 (6.4 TB/s
// at 8 rows); 7B sizes gate/up 46.6 / 49.1 / 49.0 -> 42.4 / 42.8 / 44.6, down 26.0 / 24.9 / 25.3 -> 21.7 / 21.9 / 23.1, qkv 9.9 / 10.4 / 11.3 -> 8.3 / 8.1 / 8.5.
#define FLOW_UNIT 64    // k a unit
#define FLOW_ROWS 40    // rows a workgroup at most
#define FLOW_SCALED_K 8192  // a row's sums of 16 columns, which a workgroup's threads hold in registers

template <typename F, int... I>
__device__ __forceinline__ void flow_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// Units that a wave has under way for so many eights of weight rows and of x, so that a workgroup has 32 KB of weights or more, and its LDS.
constexpr int flow_stages(int eights, int x_eights) { return eights == 1 ? 6 : eights == 2 ? 4 : eights == 3 && x_eights == 1 ? 3 : 2; }
constexpr size_t flow_lds_bytes(int eights, int x_eights) {
  const size_t stages = (size_t)4 * flow_stages(eights, x_eights) * (eights + x_eights) * 1024 + eights % 2 * 1024;  // (what an odd number reads beyond its own)
  const size_t sums = (size_t)4 * ((eights + 1) / 2) * 1024 + 4 * 16 * sizeof(float);
  return stages > sums ? stages : sums;
}

// TEMPORAL: the weight is small, and may have been brought into the caches.  SUMS (SCALED): pieces of four sums a thread holds.
// (On a page of its own: which kernels of a step share one, and which lie across two, otherwise hangs on all that the library holds before them.  With seven instances of
// another kernel gone, which no step launches, a pass of 8 rows took 6,200 -> 6,250 us over 8,192 keys and 5,156 -> 5,199 over 3,000; on pages 6,213 and 5,155.)
template <int NH, int XH, bool TEMPORAL, typename TO, int GATED, int LINK, int SUMS>
__global__ __attribute__((aligned(4096))) __launch_bounds__(256) void gemm_flow_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, int M, int N, int K, int k_split,
                                                        int rows_each, int bias_is_float, const void* __restrict__ bias, TO* __restrict__ out, Tail tail,
                                                        Link link) {
  extern __shared__ __attribute__((aligned(16))) unsigned char flow_lds[];
  constexpr int STAGES = flow_stages(NH, XH), WAVES = 4, NT = (NH + 1) / 2, LOADS = NH + XH, STAGE_BYTES = LOADS * 1024;
  static_assert(STAGES * LOADS <= 63, "a wave's loads are counted in vmcnt");
  static_assert(NT <= WAVES, "a wave finishes one tile");
  static_assert(LINK != INTO_NORM || (NH == 2 && sizeof(TO) == 4), "whole tiles of sixteen columns");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int n_begin = (int)blockIdx.x * rows_each, n_end = min(N, n_begin + rows_each);
  const int k_first = (int)blockIdx.y * k_split;
  const int row8 = lane >> 3, piece = (lane & 7) ^ row8;
  const bf16_t* w_src[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) w_src[h] = w + (size_t)min(n_begin + h * 8 + row8, n_end - 1) * K + k_first + piece * 8;
  const bf16_t* x_src[XH];
#pragma unroll
  for (int h = 0; h < XH; ++h) x_src[h] = x + (size_t)min(h * 8 + row8, M - 1) * K + k_first + piece * 8;
  unsigned char* mine = flow_lds + (size_t)wave * STAGES * STAGE_BYTES;
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)mine;
  // (an odd number of eights: the upper half of the last tile reads what lies behind, and its results are dropped)
  const unsigned read_w = base + XH * 1024 + (unsigned)r * 128, read_x = base + (unsigned)(XH == 1 ? r & 7 : r) * 128;
  const unsigned at[2] = {(unsigned)(g ^ (r & 7)) * 16, (unsigned)((g + 4) ^ (r & 7)) * 16};

  auto ask = [&](const bf16_t* from, int unit, int stage, int slot) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(from + unit * FLOW_UNIT),
                                     (void __attribute__((address_space(3)))*)(mine + stage * STAGE_BYTES + slot * 1024), 16, 0, 0);
  };
  auto ask_weight = [&](int h, int unit, int stage) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(w_src[h] + unit * FLOW_UNIT),
                                     (void __attribute__((address_space(3)))*)(mine + stage * STAGE_BYTES + (XH + h) * 1024), 16, 0, TEMPORAL ? 0 : 2);
  };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int units = k_split / FLOW_UNIT;
  const int count = (units - wave + WAVES - 1) / WAVES;  // this wave's: wave, wave + 4, ...
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < count) {
#pragma unroll
      for (int h = 0; h < XH; ++h) ask(x_src[h], wave + s * WAVES, s, h);
#pragma unroll
      for (int h = 0; h < NH; ++h) ask_weight(h, wave + s * WAVES, s);
    }
  // What the end needs is asked for behind the first units, which therefore wait for no argument beyond those that come with the wave.  (The counts
  // below do not know of these loads, and so wait for as many of the stream's more, until they have come.)
  const int n_first = n_begin + wave * 16 + g * 4;  // of the four columns that this lane finishes, where wave < NT
  // (the bias without a branch, at whose end its loads would be waited for, and the stream with them: as 16-bit halves, a float32 two and a bfloat16 the
  // upper one alone; where there is none the same loads read the weights' start)
  unsigned short bias_low[4], bias_high[4];
  const bool with_bias = LINK != SCALED && bias && blockIdx.y == 0;
  if (LINK != SCALED) {
    const unsigned short* source = with_bias ? (const unsigned short*)bias : (const unsigned short*)w;
    const int halves = with_bias && bias_is_float ? 2 : 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = min(n_first + i, N - 1) * halves;
      bias_low[i] = source[at];
      bias_high[i] = source[at + halves - 1];
    }
  }
  LinkedColumns columns;
  if (LINK == INTO_NORM) columns = linked_columns(link, r, n_begin + g * 4, M, N);
  f32x4 sums[SUMS > 0 ? SUMS : 1];
  if (LINK == SCALED) {
#pragma unroll
    for (int c = 0; c < SUMS; ++c) sums[c] = *(const f32x4*)(link.sums + min((int)threadIdx.x + c * 256, link.tiles * 4 - 1) * 4);
  }
  asm volatile("" ::: "memory");
  // This wave's unit i, in `stage`; AFTER units behind it are under way, and with AGAIN unit i + STAGES is asked for into the same places.
  auto one_unit = [&](int i, int stage, auto after, auto again) {
    constexpr int AFTER = decltype(after)::value;
    constexpr bool AGAIN = decltype(again)::value;
    const unsigned here = (unsigned)stage * STAGE_BYTES;
    const int next = wave + (i + STAGES) * WAVES;
    bf16x8 b[2];
    flow_each([&](auto tile) {
      constexpr int t = decltype(tile)::value, EIGHTS = 2 * t + 2 <= NH ? 2 : 1;
      // asked for behind this tile's: the unit's other eights, the units behind, what has been asked for anew
      stream_wait_loads<NH - 2 * t - EIGHTS + AFTER * LOADS + (AGAIN && t > 0 ? XH + 2 * t : 0)>();
      bf16x8 a[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (t == 0) stream_read<0>(b[s], read_x + here + at[s]);
        stream_read<2048 * t>(a[s], read_w + here + at[s]);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int s = 0; s < 2; ++s) {  // used only after the wait
        asm volatile("" : "+v"(a[s]));
        if (t == 0) asm volatile("" : "+v"(b[s]));
      }
      if (AGAIN) {
        if (t == 0) {
#pragma unroll
          for (int h = 0; h < XH; ++h) ask(x_src[h], next, stage, h);
        }
#pragma unroll
        for (int h = 0; h < EIGHTS; ++h) ask_weight(2 * t + h, next, stage);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s], b[s], acc[t], 0, 0, 0);
    }, std::make_integer_sequence<int, NT>{});
  };
  int i = 0, stage = 0;
  for (; i + STAGES < count; ++i) {
    one_unit(i, stage, std::integral_constant<int, STAGES - 1>{}, std::true_type{});
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  }
  flow_each([&](auto done) {  // the last STAGES units (or as many as there are)
    constexpr int AFTER = STAGES - 1 - decltype(done)::value;
    if (count - i != AFTER + 1) return;
    one_unit(i, stage, std::integral_constant<int, AFTER>{}, std::false_type{});
    ++i;
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  }, std::make_integer_sequence<int, STAGES>{});

  __syncthreads();  // every wave is done with its stages: LDS is free for the waves' sums
  float* partial = (float*)flow_lds;  // [WAVES][NT][64 lanes][4]
  float* shares = partial + WAVES * NT * 256;  // [WAVES][16 rows]
#pragma unroll
  for (int t = 0; t < NT; ++t) *(f32x4*)(partial + ((wave * NT + t) * 64 + lane) * 4) = acc[t];
  if (LINK == SCALED) {  // piece threadIdx.x + 256 c holds rows 4 (threadIdx.x % 4) .. + 3 of a tile of columns
    f32x4 squares = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < SUMS; ++c)
      if ((int)threadIdx.x + c * 256 < link.tiles * 4) squares += sums[c];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int offset = 4; offset < WAVE; offset *= 2) squares[i] += __shfl_xor(squares[i], offset, WAVE);
    }
    if (lane < 4) *(f32x4*)(shares + wave * 16 + lane * 4) = squares;
  }
  __syncthreads();
  if (wave >= NT) return;
  f32x4 total = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < WAVES; ++v) total += *(const f32x4*)(partial + ((v * NT + wave) * 64 + lane) * 4);
  const int m = r;
  if (m >= M) return;
  if (with_bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i) total[i] += __uint_as_float((unsigned)bias_high[i] << 16 | (bias_is_float ? (unsigned)bias_low[i] : 0u));
  }
  if (LINK == SCALED) {
    const float squares = ((shares[m] + shares[16 + m]) + shares[32 + m]) + shares[48 + m];
    const float factor = rsqrtf(squares * link.inverse_width + link.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) total[i] *= factor;  // (such a product has no bias)
  }
  if (LINK == INTO_NORM) {
    store_into_norm(link, columns, total, m, n_first, N);
  } else if (GATED == 3) {
    store_with_tail(out, tail, m, n_first, n_end, total);
  } else if (GATED) {
    TO* dst = out + (size_t)m * (N / 2) + n_first / 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (n_first + 2 * i + 1 < n_end) {
        const float gate = total[2 * i], up = total[2 * i + 1];
        dst[i] = from_float<TO>(gate_value<GATED>(gate) * up);
      }
    }
  } else {
    TO* dst = out + ((size_t)blockIdx.y * M + m) * N + n_first;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n_first + i < n_end) dst[i] = from_float<TO>(total[i]);
  }
}

template <int NH, int XH, bool TEMPORAL, typename TO, int GATED, int LINK, int SUMS>
static int launch_flow(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K, int splits, int rows_each,
                       hipStream_t stream, Tail tail, Link link) {
  constexpr size_t lds = flow_lds_bytes(NH, XH);
  if (lds > 64 * 1024) {
    static bool asked = false;
    if (!asked) {
      if (hipFuncSetAttribute((const void*)gemm_flow_kernel<NH, XH, TEMPORAL, TO, GATED, LINK, SUMS>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return ERR_BAD_ARGUMENT;
      asked = true;
    }
  }
  hipLaunchKernelGGL((gemm_flow_kernel<NH, XH, TEMPORAL, TO, GATED, LINK, SUMS>), dim3((N + rows_each - 1) / rows_each, splits), dim3(256), lds,
                     stream, (const bf16_t*)x, (const bf16_t*)w, M, N, K, K / splits, rows_each, bias_is_float, bias, (TO*)out, tail, link);
  return LAUNCH_STATUS();
}

// A weight of up to 8 MB is read as any other memory: the kernel before may have brought it into the caches, and a model of such weights may
// live in them.  (Its rows give every CU a workgroup with no more than 16 rows.)
static bool flow_temporal(int N, int K) { return (long)N * K <= (1L << 22); }

// The rows a workgroup takes: what a CU has to bring, weight rows and rows of x, is least.  Workgroups that share a CU's LDS run
// at once, so that CUs get whole numbers of them; of more, CUs take the next as they finish.  Gate/up of the 1.5B sizes (17,920 rows) at 8 rows of x: 18 rows each, four
// a CU at most, 10.7 us; 24, three, 10.5; 32, three, 11.8; 40, two, 10.6.  The head (151,936 rows) at 8 and 16 rows of x: 24 rows
// each 78.5 and 93.8 us, 32 72.6 and 79.0, 40 75.5 and 83.8 (hence the 1.06 and 1.12).
// Of 128 or more workgroups side by side, those whose weights lie 256 or 512 KB apart walk them in step and ask the same few channels of memory at a time (1.3).  Us at one row,
// the kernels before -> 32 rows each, which they are apart -> as it is picked now: gate/up of N 57,344 K 8,192 174 -> 193 -> 147, N 24,576 K 4,096 35.1 -> 38.8 -> 32.6, a head of
// N 128,256 K 4,096 169 -> 186 -> 161; 16 rows each of K 8,192 cost a tenth too (N 57,344 160).  Three times 256 KB costs nothing (N 40,000 K 12,288 154 at 32 rows each, 154-160
// about it), a million bytes little (N 32,768 K 16,384 193, 180 and at 16 rows of x 180, 193).
struct FlowShape {
  int rows_each;
  double load;  // rows of K / splits that a CU brings
};
static FlowShape flow_shape(int M, int N, int K, int splits) {
  FlowShape best = {0, 0.0};
  const int most = flow_temporal(N, K) ? 16 : FLOW_ROWS;
  for (int rows = 8; rows <= most; rows += 2) {
    const int eights = (rows + 7) / 8;
    const long workgroups = (long)((N + rows - 1) / rows) * splits;
    const int held = (int)(160 * 1024 / flow_lds_bytes(eights, M <= 8 ? 1 : 2));
    const double each = rows + 0.3 * (8 * eights - rows) + M + 2.0;
    double load = workgroups <= 256L * held ? (double)((workgroups + 255) / 256) * each : (workgroups / 256.0 + 0.5) * each;
    if (eights == 5) load *= M <= 8 ? 1.06 : 1.12;
    const long apart = 2L * rows * K;
    if ((apart == 256 << 10 || apart == 512 << 10) && (N + rows - 1) / rows >= 128) load *= 1.3;
    if (best.rows_each == 0 || load < best.load) best = {rows, load};
  }
  return best;
}

template <typename TO, int GATED, int LINK, int SUMS>
static int pick_flow(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K, int splits,
                     hipStream_t stream, Tail tail = {}, Link link = {}) {
  const int rows_each = flow_shape(M, N, K, splits).rows_each, eights = (rows_each + 7) / 8;
#define FLOW_CASE(NH_, TEMPORAL_)                                                                                                             \
  if (eights == NH_)                                                                                                                          \
    return M <= 8 ? launch_flow<NH_, 1, TEMPORAL_, TO, GATED, LINK, SUMS>(x, w, bias, bias_is_float, out, M, N, K, splits,  \
                                                                                            rows_each, stream, tail, link)                    \
                  : launch_flow<NH_, 2, TEMPORAL_, TO, GATED, LINK, SUMS>(x, w, bias, bias_is_float, out, M, N, K, splits,  \
                                                                                            rows_each, stream, tail, link);
  if (flow_temporal(N, K)) {
    FLOW_CASE(1, true)
    FLOW_CASE(2, true)
  } else {
    FLOW_CASE(1, false)
    FLOW_CASE(2, false)
    FLOW_CASE(3, false)
    FLOW_CASE(4, false)
    FLOW_CASE(5, false)
  }
#undef FLOW_CASE
  return ERR_BAD_ARGUMENT;
}

// K % 128 == 0, N % 16 == 0: tiles of sixteen columns, whose squares the reader adds up
static int pick_flow_into_norm(const void* x, const void* w, const void* bias, int bias_is_float, int M, int N, int K, hipStream_t stream, Link link) {
#define NORM_CASE(XH_, TEMPORAL_) \
  launch_flow<2, XH_, TEMPORAL_, float, 0, INTO_NORM, 0>(x, w, bias, bias_is_float, nullptr, M, N, K, 1, 16, stream, Tail{}, link)
  if (flow_temporal(N, K)) return M <= 8 ? NORM_CASE(1, true) : NORM_CASE(2, true);
  return M <= 8 ? NORM_CASE(1, false) : NORM_CASE(2, false);
#undef NORM_CASE
}

static int pick_flow_scaled(const void* rows, const void* w, void* out, int M, int N, int K, hipStream_t stream, Link link) {
  if (K <= 2048) return pick_flow<bf16_t, 1, SCALED, 2>(rows, w, nullptr, 0, out, M, N, K, 1, stream, {}, link);
  if (K <= 4096) return pick_flow<bf16_t, 1, SCALED, 4>(rows, w, nullptr, 0, out, M, N, K, 1, stream, {}, link);
  return pick_flow<bf16_t, 1, SCALED, 8>(rows, w, nullptr, 0, out, M, N, K, 1, stream, {}, link);
}

static bool flow_takes(const void* x, const void* w, int out_is_float, int gated, int M, int N, int K, int splits) {
  return M > 0 && M <= 16 && K % splits == 0 && (K / splits) % FLOW_UNIT == 0 && !(gated && out_is_float) && in_pieces(x, w);
}
static int flow_entry(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int out_is_float, int gated, int M, int N, int K,
                      int splits, hipStream_t stream, Tail tail) {
  if (gated == 3) return pick_flow<bf16_t, 3, NO_LINK, 0>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, tail);
  if (gated == 2) return pick_flow<bf16_t, 2, NO_LINK, 0>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  if (gated) return pick_flow<bf16_t, 1, NO_LINK, 0>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  return out_is_float ? pick_flow<float, 0, NO_LINK, 0>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)
                      : pick_flow<bf16_t, 0, NO_LINK, 0>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
}

// The weight rows that a workgroup of the product of M <= 16 rows takes (splits parts of K, a multiple of 64 each), for who brings them ahead.
extern "C" int llmserve_gemm_flow_rows(int M, int N, int K, int splits) { return flow_shape(M, N, K, splits).rows_each; }

// Into how many parts of K such a product is best cut when its float32 result may stay in parts, 1 to 8: by what a CU brings, and 0.12 us a part for
// writing and adding it up (a CU brings 26 bytes a ns).  A part has two units a wave or more.  The same at every M, as parts decide in which order a row's
// sums meet: by what eight rows take, and the fewest that the estimate has within 7 percent of the best.  Us with the norm that adds them up, in the parts that M itself
// would have -> these: 1 row of N 1,152 K 6,912 (three -> four) 7.1 -> 7.2, 8 rows (six -> four) 7.8 -> 7.6; 16 rows of N 1,536 K 8,960 (five -> four) 9.8 -> 9.8; 1 row
// of N 1,024 K 3,072 (two -> four) 5.8 -> 5.9.  By what one row takes 16 rows of N 1,024 K 2,048 go from 5.6 to 5.9, of N 2,560 K 4,096 from 8.7 to 9.0.
extern "C" int llmserve_gemm_flow_parts(int, int N, int K) {
  const int rows = 8, units = K / FLOW_UNIT;
  double us[9], least = 0.0;
  for (int splits = 1; splits <= 8; ++splits) {
    us[splits] = -1.0;
    if (splits > 1 && (K % FLOW_UNIT || units % splits || units / splits < 8)) continue;
    us[splits] = flow_shape(rows, N, K, splits).load * (K / splits) * 2.0 / 26e3 + 0.12 * splits;
    if (splits == 1 || us[splits] < least) least = us[splits];
  }
  int splits = 1;
  while (us[splits] < 0.0 || us[splits] > 1.07 * least) ++splits;
  return splits;
}

// The same product as llmserve_gemm_skinny, always through gemm_flow or, beyond 16 rows, gemm_stream (tests and measurements); up to 64 rows.
static int stream_entry(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int out_is_float,
                        int gated, int M, int N, int K, int splits, hipStream_t stream, int nt, int g) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || splits < 1 || K % splits || (K / splits) % (STEP * GROUP) || (gated && N % 2) || gated > 1)
    return ERR_BAD_ARGUMENT;
  if ((splits > 1 && (gated || !out_is_float)) || !in_pieces(x, w)) return ERR_BAD_ARGUMENT;
  if (M <= 16) return flow_takes(x, w, out_is_float, gated, M, N, K, splits) ? flow_entry(x, w, bias, bias_is_float, out, out_is_float, gated, M, N, K, splits, stream, Tail{}) : ERR_BAD_ARGUMENT;
  if (gated)
    return out_is_float ? pick_stream<float, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, nt, g)
                        : pick_stream<bf16_t, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, nt, g);
  return out_is_float ? pick_stream<float, false>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, nt, g)
                      : pick_stream<bf16_t, false>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, nt, g);
}

extern "C" int llmserve_gemm_stream(const void* x, const void* w, const void* bias, int bias_is_float, void* out,
                                    int out_is_float, int gated, int M, int N, int K, int splits,
                                    hipStream_t stream) {
  return stream_entry(x, w, bias, bias_is_float, out, out_is_float, gated, M, N, K, splits, stream, 0, 0);
}

// The same for 17 to 64 rows with the shape asked for (measurements): nt weight tiles a workgroup (1, 2),
// groups of g steps (1, 2).
extern "C" int llmserve_gemm_stream_shaped(const void* x, const void* w, const void* bias, int bias_is_float,
                                           void* out, int out_is_float, int gated, int M, int N, int K, int splits,
                                           int nt, int g, hipStream_t stream) {
  if (M <= 16) return ERR_BAD_ARGUMENT;
  return stream_entry(x, w, bias, bias_is_float, out, out_is_float, gated, M, N, K, splits, stream, nt, g);
}

// ---------------------------------------------------------------------------- key splits merged on the way in
// gemm_merged: gemm_skinny for up to 16 rows whose x is the output of decode attention that was left in
// key splits (attention_bf16.hip, `unmerged`): for every (row, head) S results, each divided by its own sum
// of weights, with each split's maximum m_s (in units of log2) and sum of weights l_s.  The row's true
// x[head] = sum_s c_s x_s[head] with c_s = l_s 2^(m_s - m) / sum_t l_t 2^(m_t - m), m the largest m_s.
// A kernel of its own that merges costs a decode step as much as the attention itself (a launch and two
// trips to memory); here every split's x is multiplied as it is, into sums of its own, and those of a head are added up times c_s: lane (r, g) of
// the result holds row r, whose coefficients it has.  What bounds the kernel is what a CU can ask for: all of x, S times, comes to each of
// the 96 workgroups (1.5B sizes), and the address unit takes four lanes a cycle, so lanes without a row ask for nothing and the weights come by whole
// lines, as in gemm_flow (by operands, 16 bytes of four rows to four lanes, and with every lane asking, the first wave had its loads after 3.3 us
// and the last after 5.5; merging x before the product cost 450 instructions a lane and head besides).  A pass of four steps with 20 MB of the next weight brought
// beside it: 1 row 4,272 -> 4,141 us, 8 rows 4,525 -> 4,422.  Heads are
// 128 wide, a group of K (128 k), so a wave's group is one head and its S coefficients are made once.
template <int WAVES, int S, int LINK>
__global__ __launch_bounds__(WAVES * 64) void gemm_merged_kernel(const bf16_t* __restrict__ split_x, const float* __restrict__ split_ml,
                                                                 const bf16_t* __restrict__ w, int M, int N, int K, int k_split, int tiles,
                                                                 int bias_is_float, const void* __restrict__ bias, float* __restrict__ out,
                                                                 Link link, Ahead ahead) {
  extern __shared__ __attribute__((aligned(16))) unsigned char merged_lds[];  // [WAVES][4 KB]: the weights of a wave's head; then [WAVES][64 lanes][4] sums
  if (LINK == INTO_NORM && (int)blockIdx.x >= tiles) {
    bring_ahead(ahead, blockIdx.x, tiles, gridDim.x);
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int head_first = blockIdx.y * (k_split / (STEP * GROUP));
  // (the weights as in gemm_flow: eight rows of 64 k a load, straight into LDS)
  unsigned char* mine = merged_lds + (size_t)wave * 4096;
  const bf16_t* w_src[2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
    w_src[e] = w + (size_t)min((int)blockIdx.x * 16 + e * 8 + (lane >> 3), N - 1) * K + (size_t)head_first * (STEP * GROUP) + ((lane & 7) ^ (lane >> 3)) * 8;
  const unsigned even = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)mine + (unsigned)(8 * r + (g ^ (r & 7))) * 16;
  const unsigned odd = even + (unsigned)(((4 + g) ^ (r & 7)) - (g ^ (r & 7))) * 16;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const bool with_bias = bias && blockIdx.y == 0;
  float bias_here[4] = {0.f, 0.f, 0.f, 0.f};
  if (with_bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      bias_here[i] = load_as_float(bias, bias_is_float, min((int)blockIdx.x * 16 + g * 4 + i, N - 1));
  }
  LinkedColumns columns;  // (asked for behind the first head's loads, which wait for no argument beyond those that come with the wave, and used at the end, by the first wave)
  const int groups = k_split / (STEP * GROUP);
  bf16x8 a[GROUP];
  float2 ml[S];
  bf16x8 piece[S][GROUP];
  auto ask = [&](int group) {
#pragma unroll
    for (int chunk = 0; chunk < 4; ++chunk)
      __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(w_src[chunk % 2] + group * (STEP * GROUP) + chunk / 2 * 64),
                                       (void __attribute__((address_space(3)))*)(mine + chunk * 1024), 16, 0, 0);
    // split_x is [head][split][piece of 8][16 rows][8]: this lane's piece 4 u + g of row r, beside the
    // same piece of the next rows, which the next lanes ask for.  (Lanes of rows that are not there ask for nothing: the CU's address unit takes a cycle
    // for every four lanes, and all of x comes through it.)
    const size_t slot = (size_t)(head_first + group) * S;
    if (r < M) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        ml[s] = *(const float2*)(split_ml + ((slot + s) * 16 + r) * 2);
#pragma unroll
        for (int u = 0; u < GROUP; ++u)
          piece[s][u] = load8(split_x + (((slot + s) * (STEP * GROUP / 8) + u * 4 + g) * 16 + r) * 8);
      }
    }
    asm volatile("" ::: "memory");  // (asked for here)
  };
  ask(min(wave, groups - 1));
  if (LINK == INTO_NORM) columns = linked_columns(link, r, (int)blockIdx.x * 16 + g * 4, M, N);
  for (int group = wave; group < groups; group += WAVES) {
    if (group > wave) ask(group);
    stream_wait_loads<0>();
    RingReads<0, GROUP>::run(a, even, odd);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int u = 0; u < GROUP; ++u) asm volatile("" : "+v"(a[u]));  // used only after the wait
    float best = -INFINITY;
#pragma unroll
    for (int s = 0; s < S; ++s) best = fmaxf(best, ml[s].x);
    float share[S], total = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      share[s] = ml[s].x == -INFINITY ? 0.f : ml[s].y * __builtin_amdgcn_exp2f(ml[s].x - best);  // a split that saw no key
      total += share[s];
    }
    const float inverse = total > 0.f ? 1.f / total : 0.f;
    f32x4 of_split[S];
#pragma unroll
    for (int s = 0; s < S; ++s) of_split[s] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < GROUP; ++u)
#pragma unroll
      for (int s = 0; s < S; ++s) of_split[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], piece[s][u], of_split[s], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < S; ++s) {  // (a split that saw no key holds whatever was there, in this row's column alone; one whose share is NaN, from a key of
                                   // NaN or a score of +inf, is none of those, and reaches the row)
      const float c = share[s] * inverse;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = share[s] != 0.f ? fmaf(c, of_split[s][i], acc[i]) : acc[i];
    }
  }
  __syncthreads();  // (every wave has read its weights)
  float* partial = (float*)merged_lds;
  *(f32x4*)(partial + (wave * 64 + lane) * 4) = acc;
  __syncthreads();
  if (wave > 0) return;
  f32x4 total_tile = {0.f, 0.f, 0.f, 0.f};
  for (int v = 0; v < WAVES; ++v) total_tile += *(const f32x4*)(partial + (v * 64 + lane) * 4);
  const int n_first = blockIdx.x * 16 + g * 4;
  if (r >= M) return;
  if (LINK == INTO_NORM) {
#pragma unroll
    for (int i = 0; i < 4; ++i) total_tile[i] += bias_here[i];
    store_into_norm(link, columns, total_tile, r, n_first, N);
    return;
  }
  float* dst = out + ((size_t)blockIdx.y * M + r) * N + n_first;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n_first + i < N) dst[i] = total_tile[i] + bias_here[i];
}

template <int WAVES, int S, int LINK>
static int launch_merged_as(const void* split_x, const float* split_ml, const void* w, const void* bias, int bias_is_float,
                            float* out, int M, int N, int K, int k_splits, hipStream_t stream, Link link, int helpers, Ahead ahead) {
  const int tiles = (N + 15) / 16;
  hipLaunchKernelGGL((gemm_merged_kernel<WAVES, S, LINK>), dim3(tiles + helpers, k_splits), dim3(WAVES * 64), WAVES * 4096, stream,
                     (const bf16_t*)split_x, split_ml, (const bf16_t*)w, M, N, K, K / k_splits, tiles, bias_is_float, bias, out, link, ahead);
  return LAUNCH_STATUS();
}

// Twelve waves for whole sums over more than eight heads, a head each or two, of which a wave has 168 registers.  Eight splits of a head take 128 for x and 32 for their
// sums (six 96 and 24): in twelve waves that went to memory and came back, and a register put away before its read of LDS has come would come back with what
// it held before.  Those have eight waves of 256.  A pass of four steps over contexts of about 1,500, which attention leaves in eight splits, us, in twelve waves ->
// eight: 1 row 5,640 -> 4,386, 8 rows 5,935 -> 4,710, 16 rows 6,450 -> 5,290 (twelve waves that take eight splits as two runs of four: 4,385, 4,687 and 5,290,
// and of more than twelve heads they would make four trips to memory for two or three).
template <int S, int LINK>
static int launch_merged(const void* split_x, const float* split_ml, const void* w, const void* bias, int bias_is_float,
                         float* out, int M, int N, int K, int k_splits, hipStream_t stream, Link link, int helpers, Ahead ahead) {
#define MERGED(WAVES) launch_merged_as<WAVES, S, LINK>(split_x, split_ml, w, bias, bias_is_float, out, M, N, K, k_splits, stream, link, helpers, ahead)
  const int groups = K / k_splits / (STEP * GROUP);
  if constexpr (LINK == INTO_NORM && S <= 4) {
    if (groups > 8) return MERGED(12);
  }
  return groups <= 4 ? MERGED(4) : MERGED(8);
#undef MERGED
}

// out [k_splits, M, N] float32 partial sums of x . w^T (+ bias in the first), x [M, K] being the merge of
// split_x bfloat16 [K / 128, splits, 16, 16 rows, 8] with split_ml float32 [K / 128, splits, 16 rows, 2] as above.
// M <= 16; K a multiple of 128 * k_splits; splits 2, 3, 4, 6 or 8.
template <int LINK>
static int pick_merged(const void* split_x, const float* split_ml, int splits, const void* w, const void* bias, int bias_is_float,
                       float* out, int M, int N, int K, int k_splits, hipStream_t stream, Link link, int helpers = 0, Ahead ahead = {}) {
  switch (splits) {
    case 2: return launch_merged<2, LINK>(split_x, split_ml, w, bias, bias_is_float, out, M, N, K, k_splits, stream, link, helpers, ahead);
    case 3: return launch_merged<3, LINK>(split_x, split_ml, w, bias, bias_is_float, out, M, N, K, k_splits, stream, link, helpers, ahead);
    case 4: return launch_merged<4, LINK>(split_x, split_ml, w, bias, bias_is_float, out, M, N, K, k_splits, stream, link, helpers, ahead);
    case 6: return launch_merged<6, LINK>(split_x, split_ml, w, bias, bias_is_float, out, M, N, K, k_splits, stream, link, helpers, ahead);
    case 8: return launch_merged<8, LINK>(split_x, split_ml, w, bias, bias_is_float, out, M, N, K, k_splits, stream, link, helpers, ahead);
    default: return ERR_BAD_ARGUMENT;
  }
}

extern "C" int llmserve_gemm_merged(const void* split_x, const float* split_ml, int splits, const void* w,
                                    const void* bias, int bias_is_float, float* out, int M, int N, int K,
                                    int k_splits, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K <= 0 || k_splits < 1 || K % (STEP * GROUP * k_splits) || !in_pieces(split_x, w)) return ERR_BAD_ARGUMENT;
  return pick_merged<NO_LINK>(split_x, split_ml, splits, w, bias, bias_is_float, out, M, N, K, k_splits, stream, Link{});
}

static int sums_stride(int M) { return M <= 16 ? 16 : M <= 32 ? 32 : 64; }

// The product (split_x null: of x; else of the merge of its key splits, as above, M <= 16) into a norm: hidden [M, N] float32 +=
// x . w^T (+ bias); rows [M, N] bfloat16 = hidden * weight; sums float32 [N / 16, 16 rows, or 32 or 64: as many as hold M].
// M <= 64, N a multiple of 16, K of 128; every operand begins at a multiple of 16 bytes.  With split_x `helpers` further workgroups bring the runs of `ahead` into the caches (common.h: Ahead).
extern "C" int llmserve_gemm_into_norm(const void* x, const void* split_x, const float* split_ml, int splits, const void* w, const void* bias,
                                       int bias_is_float, float* hidden, const void* weight, int weight_is_float, void* rows, float* sums,
                                       int M, int N, int K, int helpers, const void* ahead, int stripe, int stripes,
                                       hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || N % 16 || K <= 0 || K % (STEP * GROUP) || (split_x && M > 16) || (!x && !split_x)) return ERR_BAD_ARGUMENT;
  if (!in_pieces(split_x ? split_x : x, w) || !in_pieces(hidden, weight) || !in_pieces(rows, sums)) return ERR_BAD_ARGUMENT;
  if (!ahead_fits(helpers, ahead, stripe, stripes) || (helpers && !split_x)) return ERR_BAD_ARGUMENT;
  const Ahead next = {(const unsigned char*)ahead, (unsigned)stripe, (unsigned)stripes};
  const Link link{hidden, weight, weight_is_float, (bf16_t*)rows, sums, sums_stride(M), N / 16, 0.f, 0.f};
  if (split_x) return pick_merged<INTO_NORM>(split_x, split_ml, splits, w, bias, bias_is_float, nullptr, M, N, K, 1, stream, link, helpers, next);
  if (M <= 16) return pick_flow_into_norm(x, w, bias, bias_is_float, M, N, K, stream, link);
  if (M <= 32) return launch_stream<4, 1, 2, 2, float, 0, INTO_NORM>(x, w, bias, bias_is_float, nullptr, M, N, K, 1, stream, link);
  return launch_stream<4, 1, 4, 1, float, 0, INTO_NORM>(x, w, bias, bias_is_float, nullptr, M, N, K, 1, stream, link);
}

// ---------------------------------------------------------------------------- 16 < M <= 64
// gemm_medium: the same product for up to 64 rows of x.  With more than one 16-row tile of x,
// loading x per wave would cost more than streaming the weights, so a workgroup takes 64
// weight rows (four waves, one 16-row tile each) times four slices of its K range (sixteen
// waves), and the four waves of a K slice share the slice's 128 columns of x through LDS
// (rows padded by 16 bytes, so that the 16-byte reads of an MFMA operand spread over all
// banks).  K may be cut over workgroups too (blockIdx.y), leaving partial sums as above.
#define MEDIUM_ROWS 64
#define X_STRIDE (STEP * GROUP + 8)  // bf16 elements per staged row of x: 128 + padding

template <int MT, typename TO, bool GATED>
__global__ __launch_bounds__(1024) void gemm_medium_kernel(const bf16_t* __restrict__ x,
                                                           const bf16_t* __restrict__ w,
                                                           const void* __restrict__ bias, int bias_is_float,
                                                           TO* __restrict__ out, int M, int N, int K,
                                                           int groups_per_block) {
  extern __shared__ float shared_medium[];
  bf16_t* staged = (bf16_t*)shared_medium;  // [4 slices][MT * 16 rows][X_STRIDE]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row_tile = wave & 3, slice = wave >> 2;
  const int r = lane & 15, g = lane >> 4;
  const int n = min((int)blockIdx.x * MEDIUM_ROWS + row_tile * 16 + r, N - 1);
  const int total_groups = K / (STEP * GROUP);
  const int group_begin = blockIdx.y * groups_per_block;
  const int group_end = min(total_groups, group_begin + groups_per_block);
  const bf16_t* w_row = w + (size_t)n * K + g * 8;
  bf16_t* my_stage = staged + (size_t)slice * (MT * 16) * X_STRIDE;
  const int slice_thread = threadIdx.x & 255;  // index among the four waves of this K slice

  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // The slice's 256 threads bring x[0 .. MT*16)[a group's 128 columns] into LDS, 16 bytes a piece,
  // MT pieces a thread: first into registers (issued a round ahead), then into LDS.
  bf16x8 x_piece[MT];
  auto fetch_x = [&](int group) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int piece = slice_thread + i * 256, row = piece >> 4, part = piece & 15;
      x_piece[i] = (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
      if (row < M) x_piece[i] = load8(x + (size_t)row * K + (size_t)group * (STEP * GROUP) + part * 8);
    }
  };
  auto stage_x = [&]() {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int piece = slice_thread + i * 256, row = piece >> 4, part = piece & 15;
      *(bf16x8*)(my_stage + (size_t)row * X_STRIDE + part * 8) = x_piece[i];
    }
  };
  // Rounds go in runs of three whose weights are all requested before the first is used, so the
  // weight stream never waits for the arithmetic or for x.
  constexpr int RUN = 3;
  const int rounds = (groups_per_block + 3) / 4;
  auto group_of = [&](int round) { return group_begin + round * 4 + slice; };
  if (rounds > 0 && group_of(0) < group_end) fetch_x(group_of(0));
  for (int base = 0; base < rounds; base += RUN) {
    bf16x8 a[RUN][GROUP];
#pragma unroll
    for (int j = 0; j < RUN; ++j) {
      if (base + j < rounds && group_of(base + j) < group_end) {
#pragma unroll
        for (int u = 0; u < GROUP; ++u) a[j][u] = load8_stream(w_row + (group_of(base + j) * GROUP + u) * STEP);
      }
    }
#pragma unroll
    for (int j = 0; j < RUN; ++j) {
      const int round = base + j;
      if (round >= rounds) break;
      const bool live = group_of(round) < group_end;
      __syncthreads();  // the previous round's reads of the staged x are done
      if (live) stage_x();
      if (round + 1 < rounds && group_of(round + 1) < group_end) fetch_x(group_of(round + 1));
      __syncthreads();
      if (live) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
          for (int u = 0; u < GROUP; ++u) {
            const bf16x8 b = *(const bf16x8*)(my_stage + (size_t)(t * 16 + r) * X_STRIDE + u * STEP + g * 8);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][u], b, acc[t], 0, 0, 0);
          }
        }
      }
    }
  }
  __syncthreads();
  // add the four K slices of each row tile through LDS: [slice][row_tile][MT][64 lanes][4]
  float* partial = shared_medium;
#pragma unroll
  for (int t = 0; t < MT; ++t) *(f32x4*)(partial + (((slice * 4 + row_tile) * MT + t) * 64 + lane) * 4) = acc[t];
  __syncthreads();
  if (slice != 0) return;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    f32x4 total = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int v = 0; v < 4; ++v) total += *(const f32x4*)(partial + (((v * 4 + row_tile) * MT + t) * 64 + lane) * 4);
    const int m = t * 16 + r;
    const int n_first = blockIdx.x * MEDIUM_ROWS + row_tile * 16 + g * 4;
    if (m >= M) continue;
    if (bias && blockIdx.y == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n_first + i < N) total[i] += load_as_float(bias, bias_is_float, n_first + i);
    }
    if (GATED) {
      TO* dst = out + (size_t)m * (N / 2) + n_first / 2;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (n_first + 2 * i + 1 < N) {
          const float gate = total[2 * i], up = total[2 * i + 1];
          dst[i] = from_float<TO>(gate / (1.f + expf(-gate)) * up);
        }
      }
    } else {
      TO* dst = out + ((size_t)blockIdx.y * M + m) * N + n_first;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n_first + i < N) dst[i] = from_float<TO>(total[i]);
    }
  }
}

template <int MT, typename TO, bool GATED>
static int launch_medium(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N,
                         int K, int splits, hipStream_t stream) {
  const size_t stage = (size_t)4 * MT * 16 * X_STRIDE * sizeof(bf16_t);
  const size_t merge = (size_t)4 * 4 * MT * 64 * 4 * sizeof(float);
  const size_t lds = stage > merge ? stage : merge;
  if (lds > 64 * 1024) {
    static bool asked = false;
    if (!asked) {
      if (hipFuncSetAttribute((const void*)gemm_medium_kernel<MT, TO, GATED>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return ERR_BAD_ARGUMENT;
      asked = true;
    }
  }
  const int groups = K / (STEP * GROUP);
  const int per_block = (groups + splits - 1) / splits;
  hipLaunchKernelGGL((gemm_medium_kernel<MT, TO, GATED>), dim3((N + MEDIUM_ROWS - 1) / MEDIUM_ROWS, splits),
                     dim3(1024), lds, stream, (const bf16_t*)x, (const bf16_t*)w, bias, bias_is_float, (TO*)out, M, N,
                     K, per_block);
  return LAUNCH_STATUS();
}

template <typename TO, bool GATED>
static int pick_medium(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N,
                       int K, int splits, hipStream_t stream) {
  if (M <= 32) return launch_medium<2, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
  return launch_medium<4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
}

// As llmserve_gemm_skinny, for 16 < M <= 64 and K a multiple of 128.  With splits > 1 the K
// range is cut into `splits` runs of ceil(K / 128 / splits) groups of 128 and `out` is
// [splits, M, N] partial sums.
extern "C" int llmserve_gemm_medium(const void* x, const void* w, const void* bias, int bias_is_float, void* out,
                                    int out_is_float, int gated, int M, int N, int K, int splits,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || K % (STEP * GROUP) || (gated && N % 2) || splits < 1 || gated > 1) return ERR_BAD_ARGUMENT;  // (these epilogues know silu alone)
  if (splits > 1 && (gated || !out_is_float)) return ERR_BAD_ARGUMENT;
  if (gated)
    return out_is_float ? pick_medium<float, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream)
                        : pick_medium<bf16_t, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  return out_is_float ? pick_medium<float, false>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)
                      : pick_medium<bf16_t, false>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
}

// ---------------------------------------------------------------------------- 17 to 128 rows through a ring
// gemm_ring: the product for 17 to 128 rows of x (and few of a large weight), bound by how fast the weights come from memory.  A
// workgroup of four waves owns NT tiles of 16 weight rows over its whole K range and MT tiles of x; both
// go through a ring of DEPTH stages of KSTEPS * 32 k in LDS that the waves share, filled straight from
// memory (global_load_lds_dwordx4, a chunk of eight rows x 64 k in lane order, laid out and swizzled as in
// gemm_flow; the weights, which one workgroup alone reads, past the caches: with chunks of 16 rows x 32 k, half a cache line of
// each, and through them, steps of 64 rows took 2 % longer, prompts of 77 tokens 1.8) DEPTH - 1 stages ahead of the one being multiplied: what a CU has under way is then that
// many stages of weights whatever the compiler does with the registers, and a weight row is read from memory
// once for all rows of x.  The waves divide a stage's chunks between them; one barrier a stage says that
// everyone's loads have landed and that the stage before may be filled again.  A wave multiplies one tile of x
// (two, with six or eight tiles of x: up to 96 and 128 rows) with its share of the weight tiles, so no sums meet at the end.
__device__ __forceinline__ void ring_load(const bf16_t* from, unsigned to, bool once) {
  // (M0 names the place in LDS; it is put back, the compiler keeps other things there)
  unsigned kept;
  if (once)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off nt\n\ts_mov_b32 m0, %0"
                 : "=&s"(kept)
                 : "s"(to), "v"(from)
                 : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(kept)
                 : "s"(to), "v"(from)
                 : "memory");
}
// waits until at most `younger` stages' loads of this wave (PER_WAVE each) are under way; younger <= MOST
template <int PER_WAVE, int MOST>
__device__ __forceinline__ void ring_wait(int younger) {
  if constexpr (MOST == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (younger >= MOST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MOST * PER_WAVE) : "memory");
    else ring_wait<PER_WAVE, MOST - 1>(younger);
  }
}

template <int NT, int MT, int KSTEPS, int DEPTH, typename TO, bool GATED, int LINK = NO_LINK>
__global__ __launch_bounds__(256) void gemm_ring_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                        const void* __restrict__ bias, int bias_is_float,
                                                        TO* __restrict__ out, int M, int N, int K, int k_split, Link link) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  constexpr int XPW = MT > 4 ? 2 : 1;        // tiles of x a wave multiplies
  constexpr int XGROUPS = MT > 4 ? 4 : MT;   // groups of waves by their tiles of x
  constexpr int WAYS = 4 / XGROUPS;          // groups of waves that divide the weight tiles between them
  constexpr int MINE = NT / WAYS;            // weight tiles a wave multiplies
  constexpr int TILES = NT + MT;        // of a stage, each KSTEPS chunks of 1 KB
  constexpr int STAGE_BYTES = TILES * KSTEPS * STREAM_CHUNK;
  constexpr int PER_WAVE = TILES * KSTEPS / 4;  // chunks a wave brings per stage
  constexpr int APART = 4 / KSTEPS;             // tiles between two chunks of a wave
  static_assert(MT == 2 || MT == 4 || MT == 6 || MT == 8, "two, four, six or eight tiles of x");
  static_assert(KSTEPS == 2 || KSTEPS == 4, "stages of 64 or 128 k");
  static_assert(NT % APART == 0, "a wave's chunks are weights up to one number of them, then x");
  static_assert(NT % WAYS == 0, "the waves divide the weight tiles evenly");
  static_assert(TILES * KSTEPS % 4 == 0, "the waves divide a stage's chunks evenly");
  static_assert((DEPTH - 2) * PER_WAVE <= 63, "the loads under way are counted in vmcnt");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int k_first = blockIdx.y * k_split;
  // chunk j of this wave: chunk wave % KSTEPS of tile j * APART + wave / KSTEPS (the weight tiles, then x's): eight rows of 64 k
  const int my_step = wave % KSTEPS, my_first = wave / KSTEPS;
  const int load_row = my_step % 2 * 8 + (lane >> 3), load_piece = (lane & 7) ^ (lane >> 3);
  const bf16_t* src[PER_WAVE];  // this lane's piece of each, in the first stage
#pragma unroll
  for (int j = 0; j < PER_WAVE; ++j) {
    const int tile = j * APART + my_first;
    // rows of x beyond M are read as row M - 1: their columns of the result are dropped at the end
    const bf16_t* row = tile < NT ? w + (size_t)min(((int)blockIdx.x * NT + tile) * 16 + load_row, N - 1) * K
                                  : x + (size_t)min((tile - NT) * 16 + load_row, M - 1) * K;
    src[j] = row + k_first + my_step / 2 * (2 * STEP) + load_piece * 8;
  }
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)ring;
  // the wave's first tile of x, of weights (of six tiles of x the fourth wave multiplies what the third does: the same sums to the same places)
  const int x_tile = min((wave % XGROUPS) * XPW, MT - XPW), first_tile = wave / XGROUPS;
  const unsigned even = base + (unsigned)(8 * r + (g ^ (r & 7))) * 16, to_odd = (unsigned)(((4 + g) ^ (r & 7)) - (g ^ (r & 7))) * 16;
  const unsigned read_w = even + (unsigned)first_tile * KSTEPS * STREAM_CHUNK;
  const unsigned read_x = even + (unsigned)(NT + x_tile) * KSTEPS * STREAM_CHUNK;

  // the bias of the outputs this lane will finish: all asked for at once, of either type
  float bias_here[MINE][4];
  bf16_t bias_short[MINE][4];
  const bool biased = bias && blockIdx.y == 0;
#pragma unroll
  for (int i = 0; i < MINE; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = min(((int)blockIdx.x * NT + first_tile + WAYS * i) * 16 + g * 4 + j, N - 1);
      bias_here[i][j] = 0.f;
      if (biased && bias_is_float) bias_here[i][j] = ((const float*)bias)[n];
      if (biased && !bias_is_float) bias_short[i][j] = ((const bf16_t*)bias)[n];
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // so that the counts below count the ring's loads alone
  if (biased && !bias_is_float) {
#pragma unroll
    for (int i = 0; i < MINE; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) bias_here[i][j] = (float)bias_short[i][j];
  }

  const int stages = k_split / (KSTEPS * STEP);
  auto request = [&](int stage) {
    const unsigned to = base + (unsigned)(stage % DEPTH) * STAGE_BYTES + (unsigned)(my_first * KSTEPS + my_step) * STREAM_CHUNK;
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j)
      ring_load(src[j] + (size_t)stage * (KSTEPS * STEP), to + (unsigned)(j * APART * KSTEPS) * STREAM_CHUNK, j * APART < NT);
  };
  f32x4 acc[MINE][XPW];
#pragma unroll
  for (int i = 0; i < MINE; ++i)
#pragma unroll
    for (int j = 0; j < XPW; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < DEPTH - 1; ++s)
    if (s < stages) request(s);
  auto one_stage = [&](int stage) {
    // this wave's loads of the stage have landed once only the younger stages' are under way
    ring_wait<PER_WAVE, DEPTH - 2>(stages - 1 - stage);
    // everyone's have, and everyone has read the stage before this one: it may be filled again
    asm volatile("s_barrier" ::: "memory");
    if (stage + DEPTH - 1 < stages) request(stage + DEPTH - 1);
    const unsigned slot = (unsigned)(stage % DEPTH) * STAGE_BYTES;
    bf16x8 from_x[XPW][KSTEPS], from_w[MINE][KSTEPS];
#pragma unroll
    for (int j = 0; j < XPW; ++j) {
      const unsigned at = read_x + slot + (unsigned)(j * KSTEPS) * STREAM_CHUNK;
      RingReads<0, KSTEPS>::run(from_x[j], at, at + to_odd);
    }
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const unsigned at = read_w + slot + (unsigned)(WAYS * i * KSTEPS) * STREAM_CHUNK;
      RingReads<0, KSTEPS>::run(from_w[i], at, at + to_odd);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < XPW; ++j)
#pragma unroll
      for (int u = 0; u < KSTEPS; ++u) asm volatile("" : "+v"(from_x[j][u]));  // used only after the wait
#pragma unroll
    for (int i = 0; i < MINE; ++i)
#pragma unroll
      for (int u = 0; u < KSTEPS; ++u) asm volatile("" : "+v"(from_w[i][u]));
#pragma unroll
    for (int u = 0; u < KSTEPS; ++u)
#pragma unroll
      for (int i = 0; i < MINE; ++i)
#pragma unroll
        for (int j = 0; j < XPW; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(from_w[i][u], from_x[j][u], acc[i][j], 0, 0, 0);
  };
  int stage = 0;
  float share = 0.f;
  if constexpr (LINK == SCALED) {
    // The sums of squares are asked for two stages before the end, when the last stage has been asked for too: a thread waits
    // for its own here, and as loads come back in order for those stages with them.
    for (; stage < stages - 2; ++stage) one_stage(stage);
    share = squares_share<256, 16 * MT>(link, M);
  }
  for (; stage < stages; ++stage) one_stage(stage);
  float factor[XPW];
#pragma unroll
  for (int t = 0; t < XPW; ++t) factor[t] = 1.f;
  if constexpr (LINK == SCALED) {
    // The shares meet in the ring itself (six weight tiles beside four of x leave no byte of a CU's LDS, and eight beside two
    // no byte of half of it): everyone has read the last stage, and everyone has its factors before results go there.
    float* shares = (float*)ring;
    __syncthreads();
    shares[threadIdx.x] = share;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < XPW; ++t) factor[t] = row_factor<256, 16 * MT>(link, shares, (x_tile + t) * 16 + r);
    __syncthreads();
  }

  // The results leave through LDS as whole rows of the workgroup's tile, 16 bytes a lane, where the sizes allow it
  // (each lane holds four neighbouring columns of one row: stored from the registers, an instruction writes 8 or 16
  // bytes to each of sixteen rows).
  constexpr int COLUMNS = GATED ? NT * 8 : NT * 16;        // of the workgroup's tile of the result
  constexpr int PER_PIECE = 16 / (int)sizeof(TO);           // columns in 16 bytes
  const int pitch = GATED ? N / 2 : N;                      // of a row of out
  const int column0 = (int)blockIdx.x * COLUMNS;
  const int valid = min(COLUMNS, pitch - column0);
  TO* plane = out + (size_t)blockIdx.y * M * pitch;
  const bool whole_pieces = pitch % PER_PIECE == 0 && valid % PER_PIECE == 0 && COLUMNS % PER_PIECE == 0 &&
                            ((size_t)out & 15) == 0;
  if (whole_pieces) {
    asm volatile("s_barrier" ::: "memory");  // everyone has read the last stage: the ring is free
    TO* tile = (TO*)ring;                    // [16 MT rows][COLUMNS]
#pragma unroll
    for (int t = 0; t < XPW; ++t) {
      const int m = (x_tile + t) * 16 + r;
#pragma unroll
      for (int i = 0; i < MINE; ++i) {
        f32x4 total = acc[i][t];
#pragma unroll
        for (int j = 0; j < 4; ++j) total[j] = LINK == SCALED ? total[j] * factor[t] : total[j] + bias_here[i][j];
        const int c_first = (first_tile + WAYS * i) * 16 + g * 4;  // column of the tile before gating
        if (GATED) {
          TO* dst = tile + m * COLUMNS + c_first / 2;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float gate = total[2 * j], up = total[2 * j + 1];
            dst[j] = from_float<TO>(gate / (1.f + expf(-gate)) * up);
          }
        } else {
          TO* dst = tile + m * COLUMNS + c_first;
#pragma unroll
          for (int j = 0; j < 4; ++j) dst[j] = from_float<TO>(total[j]);
        }
      }
    }
    __syncthreads();
    const int pieces_a_row = valid / PER_PIECE;
    const int rows_here = min(M, 16 * MT);
    for (int piece = threadIdx.x; piece < rows_here * pieces_a_row; piece += 256) {
      const int row = piece / pieces_a_row, at = (piece - row * pieces_a_row) * PER_PIECE;
      *(f32x4*)(plane + (size_t)row * pitch + column0 + at) = *(const f32x4*)(tile + row * COLUMNS + at);
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < XPW; ++t) {
    const int m = (x_tile + t) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const int n_first = ((int)blockIdx.x * NT + first_tile + WAYS * i) * 16 + g * 4;
      f32x4 total = acc[i][t];
#pragma unroll
      for (int j = 0; j < 4; ++j) total[j] = LINK == SCALED ? total[j] * factor[t] : total[j] + bias_here[i][j];
      if (GATED) {
        TO* dst = out + (size_t)m * (N / 2) + n_first / 2;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (n_first + 2 * j + 1 < N) {
            const float gate = total[2 * j], up = total[2 * j + 1];
            dst[j] = from_float<TO>(gate / (1.f + expf(-gate)) * up);
          }
        }
      } else {
        TO* dst = out + ((size_t)blockIdx.y * M + m) * N + n_first;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n_first + j < N) dst[j] = from_float<TO>(total[j]);
      }
    }
  }
}

template <int NT, int MT, int KSTEPS, int DEPTH, typename TO, bool GATED, int LINK = NO_LINK>
static int launch_ring(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                       int splits, hipStream_t stream, Link link = {}) {
  constexpr size_t lds = (size_t)DEPTH * (NT + MT) * KSTEPS * STREAM_CHUNK;
  static_assert(lds <= 160 * 1024, "a CU's LDS");
  if ((K / splits) % (KSTEPS * STEP)) return ERR_BAD_ARGUMENT;
  if (lds > 64 * 1024) {
    static bool asked = false;
    if (!asked) {
      if (hipFuncSetAttribute((const void*)gemm_ring_kernel<NT, MT, KSTEPS, DEPTH, TO, GATED, LINK>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return ERR_BAD_ARGUMENT;
      asked = true;
    }
  }
  hipLaunchKernelGGL((gemm_ring_kernel<NT, MT, KSTEPS, DEPTH, TO, GATED, LINK>), dim3((N + 16 * NT - 1) / (16 * NT), splits),
                     dim3(256), lds, stream, (const bf16_t*)x, (const bf16_t*)w, bias, bias_is_float, (TO*)out, M, N, K,
                     K / splits, link);
  return LAUNCH_STATUS();
}

// nt tiles of 16 weight rows a workgroup, stages of 128 k; four stages, or three with six or eight tiles of x (65 to 128
// rows), which fill the LDS with five weight tiles beside them.
// Up to 96 rows six tiles of x, where eight would bring rows that are not there: a quarter less of x a stage.  (The instructions are as many: the fourth
// wave repeats the third's tiles.)  The same bits.  Us at 65 / 96 rows, eight -> six, in the shape that the products get: gated, two weight tiles N 4,864
// K 896 7.3 / 7.5 -> 7.0 / 7.1, N 7,168 K 1,024 8.3 / 8.4 -> 7.6 / 7.6; four N 9,728 K 896 10.9 / 11.0 -> 9.9 / 10.0, N 12,288 K 2,048 21.0 / 21.2 -> 19.9 /
// 20.2, N 13,824 K 2,304 25.0 / 25.0 -> 23.0 / 22.3; five N 17,920 K 1,536 22.8 / 22.8 -> 20.2 / 20.1, N 18,944 K 3,584 44.5 / 44.5 -> 39.2 / 38.9;
// eight N 24,576 K 3,072 44.2 / 46.5 -> 43.0 / 45.4, N 28,672 K 4,096 58.7 / 59.5 -> 58.1 / 58.3; ten N 37,888 K 3,584 63.0 / 63.2 -> 60.2 / 61.6; in
// parts, two N 2,048 K 1,408 9.4 / 9.6 -> 8.5 / 8.7, N 2,560 K 1,920 6.8 / 7.1 -> 6.5 / 6.6.
template <typename TO, bool GATED>
static int pick_ring(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                     int splits, hipStream_t stream, int nt) {
#define RING_CASE(NT_)                                                                                                  \
  if (nt == NT_ && M <= 64)                                                                                             \
    return M <= 32 ? launch_ring<NT_, 2, 4, 4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)      \
                   : launch_ring<NT_, 4, 4, 4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
  RING_CASE(2)
  RING_CASE(4)
  RING_CASE(6)
#undef RING_CASE
  if (nt == 5 && M > 32 && M <= 64) return launch_ring<5, 4, 4, 4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
#define ROWS_CASE(NT_, KSTEPS_, DEPTH_)                                                                                  \
  if (nt == NT_ && M > 64)                                                                                               \
    return M <= 96 ? launch_ring<NT_, 6, KSTEPS_, DEPTH_, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream) \
                   : launch_ring<NT_, 8, KSTEPS_, DEPTH_, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
  ROWS_CASE(2, 4, 3)
  ROWS_CASE(4, 4, 3)
  ROWS_CASE(5, 4, 3)
  ROWS_CASE(8, 2, 4)
  ROWS_CASE(10, 2, 4)
#undef ROWS_CASE
  // many weight tiles a workgroup, in stages of 64 k: for a weight of so many rows that fewer tiles make several rounds
#define MANY_CASE(NT_)                                                                                                  \
  if (nt == NT_ && M <= 64)                                                                                             \
    return M <= 32 ? launch_ring<NT_, 2, 2, 4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)      \
                   : launch_ring<NT_, 4, 2, 4, TO, GATED>(x, w, bias, bias_is_float, out, M, N, K, splits, stream);
  MANY_CASE(8)
  MANY_CASE(10)
  MANY_CASE(12)
  MANY_CASE(14)
#undef MANY_CASE
  return ERR_BAD_ARGUMENT;
}

// As llmserve_gemm_skinny, for M <= 128 and K / splits a multiple of 128, through gemm_ring with `nt` tiles of
// 16 weight rows a workgroup: 2, 4 or 6 (up to 64 rows), 5 (more than 32 rows), 8 or 10, or 12 or 14 (up to 64 rows).
extern "C" int llmserve_gemm_ring(const void* x, const void* w, const void* bias, int bias_is_float, void* out,
                                  int out_is_float, int gated, int M, int N, int K, int splits, int nt,
                                  hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 128 || K <= 0 || splits < 1 || K % splits || (gated && N % 2) || gated > 1 || !in_pieces(x, w)) return ERR_BAD_ARGUMENT;  // (these epilogues know silu alone)
  if (splits > 1 && (gated || !out_is_float)) return ERR_BAD_ARGUMENT;
  if (gated)
    return out_is_float ? pick_ring<float, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, nt)
                        : pick_ring<bf16_t, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, nt);
  return out_is_float ? pick_ring<float, false>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, nt)
                      : pick_ring<bf16_t, false>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, nt);
}

// silu(gate) * up, bfloat16 [M, N / 2], of rows that a product into a norm has left (`rows` [M, K], `sums` as there, in a
// buffer of whole KB): every result
// times rsqrt(sum of the row's sums / K + eps).  Up to 16 rows and FLOW_SCALED_K through gemm_flow, whatever `tiles` is; else through
// gemm_ring with so many weight tiles a workgroup.
extern "C" int llmserve_gemm_scaled(const void* rows, float* sums, float eps, const void* w, void* out, int tiles, int M, int N, int K,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || K % (STEP * GROUP) || N % 2 || (tiles == 0 && (M > 16 || K > FLOW_SCALED_K))) return ERR_BAD_ARGUMENT;
  if (!in_pieces(rows, w) || !in_pieces(sums, sums)) return ERR_BAD_ARGUMENT;
  const Link link{nullptr, nullptr, 0, nullptr, sums, sums_stride(M), K / 16, 1.f / (float)K, eps};
  if (M <= 16 && K <= FLOW_SCALED_K) return pick_flow_scaled(rows, w, out, M, N, K, stream, link);
#define SCALED_CASE(NT_, KSTEPS_)                                                                                      \
  if (tiles == NT_)                                                                                                    \
    return M <= 32 ? launch_ring<NT_, 2, KSTEPS_, 4, bf16_t, true, SCALED>(rows, w, nullptr, 0, out, M, N, K, 1, stream, link) \
                   : launch_ring<NT_, 4, KSTEPS_, 4, bf16_t, true, SCALED>(rows, w, nullptr, 0, out, M, N, K, 1, stream, link);
  SCALED_CASE(2, 4)
  SCALED_CASE(4, 4)
  SCALED_CASE(6, 4)
  SCALED_CASE(8, 2)
  SCALED_CASE(10, 2)
  SCALED_CASE(12, 2)
  SCALED_CASE(14, 2)
#undef SCALED_CASE
  if (tiles == 5 && M > 32) return launch_ring<5, 4, 4, 4, bf16_t, true, SCALED>(rows, w, nullptr, 0, out, M, N, K, 1, stream, link);
  return ERR_BAD_ARGUMENT;
}

// Whether llmserve_gemm_scaled takes these sizes with tiles 0.
extern "C" int llmserve_gemm_scaled_streams(int M, int N, int K) {
  return M > 0 && M <= 16 && K > 0 && K <= FLOW_SCALED_K && K % (STEP * GROUP) == 0;
}

// x, w bfloat16; out bfloat16 or float32.  Needs 1 <= M <= 64, K a multiple of 32, and with
// `gated` (1: silu(gate) * up, 2: relu(gate) * up) an even N.  Any N.  With splits > 1 (float32 out, not gated, K / splits a multiple of
// 32) `out` is [splits, M, N]: slice s holds the sums over the s-th part of K (the bias in slice 0),
// and whoever reads it adds the slices in order.
static int skinny_entry(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int out_is_float, int gated,
                        int M, int N, int K, int splits, hipStream_t stream, Tail tail) {
  if (splits > 1 && (gated || !out_is_float || K % splits || (K / splits) % STEP)) return ERR_BAD_ARGUMENT;
  if (flow_takes(x, w, out_is_float, gated, M, N, K, splits))
    return flow_entry(x, w, bias, bias_is_float, out, out_is_float, gated, M, N, K, splits, stream, tail);
  if (M > 16 && !gated && K % splits == 0 && (K / splits) % (STEP * GROUP) == 0 && (long)N * K <= (1L << 22) && in_pieces(x, w)) {
    // A small weight at 17 to 64 rows: two or four tiles of x beside one weight tile a workgroup, through
    // LDS.  In a captured chain over different weights, the 1.5B sizes' qkv and o: 4.8 and 4.0 us at 17
    // rows, 5.0 and 4.5 at 32, 6.0 and 5.6 at 48, 6.7 and 6.2 at 64 (the library 7.1-7.7 throughout, the
    // kernel below 5.9 and 4.8 at 17 rows, 6.8 and 5.5 at 32).  Larger weights stay with the library.
    // With K cut in two (float32 partial sums) o takes 3.5 us at 17 rows, 3.7 at 32, 4.6 at 64 (the kernel
    // below, in three parts: 4.9, 5.6, 8.0).
    const int g = M <= 32 && splits == 1 ? 2 : 1;
    return out_is_float ? pick_stream<float, false>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, 1, g)
                        : pick_stream<bf16_t, false>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, 1, g);
  }
  if (gated == 3) return pick_waves<bf16_t, 3>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, tail);
  if (gated == 2)
    return out_is_float ? pick_waves<float, 2>(x, w, bias, bias_is_float, out, M, N, K, 1, stream)
                        : pick_waves<bf16_t, 2>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  if (gated)
    return out_is_float ? pick_waves<float, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream)
                        : pick_waves<bf16_t, true>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  return out_is_float ? pick_waves<float, false>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)
                      : pick_waves<bf16_t, false>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
}

extern "C" int llmserve_gemm_skinny(const void* x, const void* w, const void* bias, int bias_is_float, void* out,
                                    int out_is_float, int gated, int M, int N, int K, int splits,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || K % STEP || (gated && N % 2) || gated > 2 || splits < 1) return ERR_BAD_ARGUMENT;
  return skinny_entry(x, w, bias, bias_is_float, out, out_is_float, gated, M, N, K, splits, stream, Tail{});
}

// The same for a bfloat16 result in two places: columns below `first` to out [M, first] (may be null where first is 0), the
// others, as relu(z)^2, to the first N - first columns of `tail`, whose rows begin every `tail_stride` elements.
extern "C" int llmserve_gemm_skinny_tail(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int first,
                                         void* tail, int tail_stride, int M, int N, int K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || K % STEP || first < 0 || first >= N || tail_stride < N - first || !tail || (first && !out)) return ERR_BAD_ARGUMENT;
  return skinny_entry(x, w, bias, bias_is_float, out, 0, 3, M, N, K, 1, stream, Tail{(bf16_t*)tail, first, tail_stride});
}
