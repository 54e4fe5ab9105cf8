// float32 products on the matrix cores: out[M, N] = x[M, K] . w[N, K]^T (+ bias), every operand,
// product and sum in 32 bits (v_mfma_f32_16x16x4_f32 and v_mfma_f32_32x32x2_f32 multiply and add
// float32 as they stand; no reduced-precision matrix mode, no packed forms).  This is the true 32-bit
// path of every product in the model (the reference runs its float32 products through its BLAS,
// model.py:60-66 via nn.Linear); gemm_generic.hip remains for operands of mixed types and for a K
// that is no multiple of 4.
//
// gemm_f32_stream (M <= 64, decoding): the product is a stream of the weight matrix from HBM.  A
// workgroup owns 16 weight rows (from 33 rows of x on 32) and its waves split K between them; lane (r, g) keeps groups of four
// 16-byte loads of weight row r in flight, k = 16 s + 4 g .. + 3 of every 16-wide step s.  An MFMA
// takes a 16 x 4 piece of the weights as its A operand (lane (r, g) gives A[r][g]) and 4 x 16 of x^T as
// B; which four k an instruction covers is free as long as A and B agree, so instruction j of a step
// takes element j of each lane's load: k = 16 s + 4 g + j.  The waves' partial tiles are added through
// LDS in wave order, so a row's bits depend on the shape of the weight only, never on the batch (the tiled kernel's, for
// larger ones, on the number of rows too).
//
// gemm_f32_whole (65 to 512 rows where its tiles are estimated ahead, see `pick_tile`) is described at its code.
//
// gemm_f32_tiled (more rows, prompt portions): a tile of weight rows by rows of x a workgroup of four waves, each
// one to four tiles of v_mfma_f32_32x32x2_f32; K in steps of 16 (of 32 or 64 where two or four waves share a tile
// and take 16 each) through two LDS buffers.  A staged row is padded by 4 floats, so that the 16-byte reads of an
// operand spread over all banks.  The matrix cores' float32 rate bounds it (a 64 x 64 tile over K 1,536 is 20 us of
// it); what kept the kernel from it was one tile size, 128 x 128: 129 rows cost what 256 do, and a product of few
// tiles left most CUs idle (2,048 x 1,536 weights at 192 rows: 32 workgroups of 122 us each).  So there are five
// tiles, and `pick_tile` takes the one that the sizes are done with first; and the 16-byte pieces are asked for four
// steps ahead, in registers (one step, 512 clocks, is less than a trip to memory: 128 x 128 tiles 120 -> 118 us, 32 x
// 32 ones 18 -> 17).  Us before -> now, a captured chain over different weights: N 17,920 K 1,536 gated: 65 rows
// 130 -> 67, 129 rows 217 -> 99, 192 rows 219 -> 114, 512 rows 319 -> 247; N 1,536 K 8,960 in parts: 65 rows 91 -> 37, 192
// rows 94 -> 58, 2,048 rows 462 -> 453; N 2,048 K 1,536: 65 rows 120 -> 17, 192 rows 122 -> 23, 2,048 rows 127 -> 113.
//
// With `gated`, weight rows alternate gate_j, up_j and the epilogue writes silu(gate) * up (reference
// model.py:188) to out[M, N / 2].  With `splits` > 1, K is cut over workgroups and `out` is
// [splits, M, N] partial sums (bias in the first) that the reader adds in order.
#include "common.h"
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define STREAM_GROUP 4  // 16-byte loads of a weight row a lane has in flight: 64 k

__device__ __forceinline__ f32x4 load4(const float* p) { return *(const f32x4*)p; }

__device__ __forceinline__ float silu(float gate) { return gate / (1.f + expf(-gate)); }

// NT: 16-row tiles of weights a workgroup, MT: 16-row tiles of x (up to 16 MT rows).  Every weight operand meets MT operands of
// x, which each wave reads for itself (M / (16 NT) of what it reads of the weights, from L2).
template <int WAVES, int NT, int MT, bool GATED>
__global__ __launch_bounds__(WAVES * 64) void gemm_f32_stream_kernel(const float* __restrict__ x,
                                                                     const float* __restrict__ w,
                                                                     const float* __restrict__ bias,
                                                                     float* __restrict__ out, int M, int N, int K,
                                                                     int k_split) {
  extern __shared__ float partial[];  // [WAVES][NT MT tiles][64 lanes][4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int k_first = blockIdx.y * k_split;
  const int k_count = min(k_split, K - k_first);  // the last slice may be shorter
  const float* w_row[NT];
#pragma unroll
  for (int s = 0; s < NT; ++s) w_row[s] = w + (size_t)min(((int)blockIdx.x * NT + s) * 16 + r, N - 1) * K + k_first + g * 4;
  bool x_live[MT];
  const float* x_row[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    x_live[t] = t * 16 + r < M;
    x_row[t] = x + (size_t)min(t * 16 + r, M - 1) * K + k_first + g * 4;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[NT][MT];
#pragma unroll
  for (int s = 0; s < NT; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[s][t] = zero;

  const int groups = k_count / (16 * STREAM_GROUP);
  f32x4 a[NT][STREAM_GROUP], a_next[NT][STREAM_GROUP];
  int group = wave;
  if (group < groups) {
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
      for (int u = 0; u < STREAM_GROUP; ++u) a[s][u] = load4(w_row[s] + (group * STREAM_GROUP + u) * 16);
  }
  while (group < groups) {
    const int next = group + WAVES;
    // this group's x is asked for before the next group's weights: loads come back in the order
    // they were asked for, and the products below wait for x
    f32x4 b[MT][STREAM_GROUP];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < STREAM_GROUP; ++u) b[t][u] = x_live[t] ? load4(x_row[t] + (group * STREAM_GROUP + u) * 16) : zero;
    asm volatile("" ::: "memory");
    if (next < groups) {
#pragma unroll
      for (int s = 0; s < NT; ++s)
#pragma unroll
        for (int u = 0; u < STREAM_GROUP; ++u) a_next[s][u] = load4(w_row[s] + (next * STREAM_GROUP + u) * 16);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < STREAM_GROUP; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int s = 0; s < NT; ++s)
            acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][u][j], b[t][u][j], acc[s][t], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
      for (int u = 0; u < STREAM_GROUP; ++u) a[s][u] = a_next[s][u];
    group = next;
  }
  // the steps left over when the slice is no multiple of 64; the last may be cut (K is a multiple of 4)
  for (int step = groups * STREAM_GROUP + wave; step * 16 < k_count; step += WAVES) {
    const bool inside = step * 16 + g * 4 < k_count;
    f32x4 a_tail[NT];
#pragma unroll
    for (int s = 0; s < NT; ++s) a_tail[s] = inside ? load4(w_row[s] + step * 16) : zero;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const f32x4 b_tail = inside && x_live[t] ? load4(x_row[t] + step * 16) : zero;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < NT; ++s)
          acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a_tail[s][j], b_tail[j], acc[s][t], 0, 0, 0);
    }
  }

  constexpr int TILES = NT * MT;
#pragma unroll
  for (int s = 0; s < NT; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) *(f32x4*)(partial + ((wave * TILES + s * MT + t) * 64 + lane) * 4) = acc[s][t];
  __syncthreads();
  // a wave finishes tiles wave, wave + WAVES, ...  D[n][m]: the lane holds token m = 16 t + r and rows n0 + 4 g .. + 3
  for (int tile = wave; tile < TILES; tile += WAVES) {
    f32x4 total = zero;
    for (int v = 0; v < WAVES; ++v) total += *(const f32x4*)(partial + ((v * TILES + tile) * 64 + lane) * 4);
    const int m = tile % MT * 16 + r;
    const int n_first = ((int)blockIdx.x * NT + tile / MT) * 16 + g * 4;
    if (m >= M) continue;
    if (bias && blockIdx.y == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) total[i] += bias[min(n_first + i, N - 1)];
    }
    if (GATED) {
      float* dst = out + (size_t)m * (N / 2) + n_first / 2;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (n_first + 2 * i + 1 < N) dst[i] = silu(total[2 * i]) * total[2 * i + 1];
    } else {
      float* dst = out + ((size_t)blockIdx.y * M + m) * N + n_first;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n_first + i < N) dst[i] = total[i];
    }
  }
}

template <int WAVES, int NT, int MT, bool GATED>
static int launch_stream(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int splits,
                         int k_split, hipStream_t stream) {
  constexpr size_t lds = (size_t)WAVES * NT * MT * 64 * 4 * sizeof(float);
  static_assert(lds <= 64 * 1024, "what a launch has without asking");
  hipLaunchKernelGGL((gemm_f32_stream_kernel<WAVES, NT, MT, GATED>), dim3((N + 16 * NT - 1) / (16 * NT), splits), dim3(WAVES * 64), lds,
                     stream, x, w, bias, out, M, N, K, k_split);
  return LAUNCH_STATUS();
}

template <int WAVES, bool GATED>
static int pick_tiles(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int splits,
                      int k_split, hipStream_t stream) {
  if (M <= 16) return launch_stream<WAVES, 1, 1, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
  if (M <= 32) return launch_stream<WAVES, 1, 2, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
  // From 33 rows on x costs the caches more than the weights cost memory, so two tiles of weights share it (a wave's walk and the order
  // of its sums stay as they are; sixteen waves, of a small weight, leave no room for that).
  constexpr int NT = WAVES <= 8 ? 2 : 1;
  if (M <= 48) return launch_stream<WAVES, NT, 3, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
  return launch_stream<WAVES, NT, 4, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
}

template <bool GATED>
static int pick_stream(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int splits,
                       hipStream_t stream) {
  // a slice of K is a multiple of 64 (whole groups) except the last
  const int k_split = splits == 1 ? K : ((K + splits - 1) / splits + 63) / 64 * 64;
  if ((size_t)k_split * (splits - 1) >= (size_t)K) return ERR_BAD_ARGUMENT;  // a slice would be empty
  // enough waves to cover the chip (about 2,048), but no more than there are groups of K
  const int tiles = (N + 15) / 16 * splits, groups = max(1, k_split / (16 * STREAM_GROUP));
  int waves = 4;
  while (waves < 16 && waves * tiles < 2048 && waves * 2 <= groups) waves *= 2;
  if (waves == 4) return pick_tiles<4, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
  if (waves == 8) return pick_tiles<8, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
  return pick_tiles<16, GATED>(x, w, bias, out, M, N, K, splits, k_split, stream);
}

// ---------------------------------------------------------------------------- many rows

#define TILE_K 16  // k a wave multiplies a step

// The tile (n, m) that a workgroup takes.  The chip hands workgroups to its eight chiplets in turn
// (workgroup i to chiplet i % 8), each with an L2 of its own: where the tiles divide by eight, chiplet c
// takes a contiguous run of them, counted down the rows of x first, so that what runs on a chiplet at
// one time shares its operands through that L2.
__device__ __forceinline__ int tile_of_workgroup(int id, int total) {
  return total % 8 == 0 ? (id % 8) * (total / 8) + id / 8 : id;
}

// WN x WM waves, each TN x TM tiles of 32 x 32, and WK of them to a tile, which take 16 k of a step each.
template <int WN, int WM, int WK, int TN, int TM, int AHEAD, bool GATED>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ out,
                                                             int M, int N, int K, int k_split, int tiles_m,
                                                             int tiles_n) {
  static_assert(WN * WM * WK == 4, "four waves");
  constexpr int TILE_N = WN * TN * 32, TILE_M = WM * TM * 32, ROWS = TILE_N + TILE_M;
  constexpr int STEP_K = TILE_K * WK, ROW_PIECES = STEP_K / 4, ROW_PAD = STEP_K + 4;  // floats a staged row takes, 4 of them padding
  constexpr int PIECES = ROWS * ROW_PIECES, MINE = (PIECES + 255) / 256;                // 16-byte pieces of a step; of one thread
  constexpr int SUMS = (WK - 1) * WN * WM * 64 * 16 * TN * TM;                          // floats that meet at the end
  constexpr int FLOATS = 2 * ROWS * ROW_PAD > SUMS ? 2 * ROWS * ROW_PAD : SUMS;
  __shared__ __attribute__((aligned(16))) float staged[FLOATS];
  const int tile = tile_of_workgroup(blockIdx.x, tiles_m * tiles_n);
  const int tile_m = tile % tiles_m, tile_n = tile / tiles_m;
  const int n0 = tile_n * TILE_N, m0 = tile_m * TILE_M;
  const int k_first = blockIdx.y * k_split;
  const int k_end = min(K, k_first + k_split);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wave_k = wave / (WN * WM);
  const int n_wave = (wave % WN) * TN * 32, m_wave = (wave / WN % WM) * TM * 32;
  const int i = lane & 31, half = lane >> 5;

  // what this thread brings of a step: pieces threadIdx.x + 256 h, the weights' rows before x's
  const float* from[MINE];
  int k_mine[MINE], to[MINE];
#pragma unroll
  for (int h = 0; h < MINE; ++h) {
    const int place = threadIdx.x + 256 * h, row = place / ROW_PIECES;
    k_mine[h] = place % ROW_PIECES * 4;
    to[h] = row * ROW_PAD + k_mine[h];
    from[h] = (row < TILE_N ? w + (size_t)min(n0 + row, N - 1) * K : x + (size_t)min(m0 + row - TILE_N, M - 1) * K) + k_mine[h];
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x16 acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  f32x4 in[AHEAD][MINE];
  auto fetch = [&](f32x4 (&to_here)[MINE], int k0) {
#pragma unroll
    for (int h = 0; h < MINE; ++h) to_here[h] = k0 + k_mine[h] < k_end ? load4(from[h] + k0) : zero;
  };
  auto stage = [&](const f32x4 (&here)[MINE], int buffer) {
#pragma unroll
    for (int h = 0; h < MINE; ++h)
      if (PIECES % 256 == 0 || threadIdx.x + 256 * h < PIECES) *(f32x4*)(staged + buffer * ROWS * ROW_PAD + to[h]) = here[h];
  };
  auto multiply = [&](int buffer) {
    // lane (i, half) holds k = 8 half .. + 7 of its wave's 16 of row i of each of its tiles; instruction s takes element s
    const float* at = staged + buffer * ROWS * ROW_PAD + wave_k * TILE_K + 8 * half;
    f32x4 a_low[TN], a_high[TN], b_low[TM], b_high[TM];
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      a_low[t] = *(const f32x4*)(at + (n_wave + 32 * t + i) * ROW_PAD);
      a_high[t] = *(const f32x4*)(at + (n_wave + 32 * t + i) * ROW_PAD + 4);
    }
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      b_low[t] = *(const f32x4*)(at + (TILE_N + m_wave + 32 * t + i) * ROW_PAD);
      b_high[t] = *(const f32x4*)(at + (TILE_N + m_wave + 32 * t + i) * ROW_PAD + 4);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(a_low[a][s], b_low[b][s], acc[a][b], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(a_high[a][s], b_high[b][s], acc[a][b], 0, 0, 0);
  };

  // AHEAD steps are asked for before they are multiplied (beyond the end: zeros, nothing is read), two are staged
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) fetch(in[u], k_first + u * STEP_K);
  stage(in[0], 0);
  __syncthreads();
  for (int k0 = k_first; k0 < k_end; k0 += AHEAD * STEP_K) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (k0 + u * STEP_K < k_end) {
        fetch(in[u], k0 + (u + AHEAD) * STEP_K);
        multiply(u & 1);
        stage(in[(u + 1) % AHEAD], (u + 1) & 1);
        __syncthreads();
      }
    }
  }
  if (WK > 1) {  // the waves of one tile add their sums, in the order of their k
    float* sums = staged + (size_t)((wave % (WN * WM)) * 64 + lane) * 16 * TN * TM;
    constexpr int OF_A_WAVE_K = WN * WM * 64 * 16 * TN * TM;
    if (wave_k > 0) {
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) *(f32x16*)(sums + (size_t)(wave_k - 1) * OF_A_WAVE_K + (a * TM + b) * 16) = acc[a][b];
    }
    __syncthreads();
    if (wave_k > 0) return;
#pragma unroll
    for (int v = 0; v < WK - 1; ++v)
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] += *(const f32x16*)(sums + (size_t)v * OF_A_WAVE_K + (a * TM + b) * 16);
  }

  // D[n][m] of a 32 x 32 tile: the lane holds column m = i and rows n = 8 q + 4 half + e, q = 0 .. 3, e = 0 .. 3
  const bool with_bias = bias && blockIdx.y == 0;
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int m = m0 + m_wave + 32 * b + i;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < TN; ++a) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + n_wave + 32 * a + 8 * q + 4 * half;
        if (n >= N) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[a][b][4 * q + e];
          if (with_bias) v[e] += bias[min(n + e, N - 1)];
        }
        if (GATED) {
          float* dst = out + (size_t)m * (N / 2) + n / 2;
          if (n + 1 < N) dst[0] = silu(v[0]) * v[1];
          if (n + 3 < N) dst[1] = silu(v[2]) * v[3];
        } else {
          float* dst = out + ((size_t)blockIdx.y * M + m) * N + n;
          if (n + 3 < N && (N & 3) == 0) {
            *(f32x4*)dst = (f32x4){v[0], v[1], v[2], v[3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < N) dst[e] = v[e];
          }
        }
      }
    }
  }
}

// gemm_f32_whole (65 to 512 rows, K in parts of whole stages of 64): a tile of 16 NT weight rows by 16 MT rows of x a workgroup, of which each of its four
// waves multiplies all with a quarter of every stage's k, in tiles of v_mfma_f32_16x16x4_f32, and whose sums meet through LDS at the end in the order of their
// k.  So a tile may be any number of sixteens (129 rows make 144, not 160) and have what it takes for one round of 256 workgroups, which is what bounds the kernel
// above.  Us, that kernel -> this, weights out of memory: N 17,920 K 1,536 gated: 65 rows 75 -> 54, 129 rows 105 -> 88, 160 rows (which a replayed step of 129 tokens has)
// 105 -> 99; N 2,048 K 1,536: 65 rows 17 -> 11, 129 rows 24 -> 15, 512 rows 43 -> 36; N 1,536 K 8,960 in parts: 129 rows 60 -> 44.  Both operands go from memory straight into LDS, as in gemm_blocks.hip: a stage is 64 k, 256 bytes a row, piece p of 16 of row r in slot
// p ^ (r % 16), so that the sixteen rows that LDS serves together hit all its banks; element j of each lane's piece goes to instruction j, so that an instruction
// takes k = 4 g + j of a wave's sixteen.  A wave holds all it needs of a stage when it begins to multiply it: behind one barrier the stage is asked for
// anew, and the next one's operands are read, between the products.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
constexpr int whole_stages(int rows) { return rows <= 64 ? 4 : 3; }

template <int NT, int MT, bool GATED>
__global__ __launch_bounds__(256, 1) void gemm_f32_whole_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                const float* __restrict__ bias, float* __restrict__ out, int M, int N, int K,
                                                                int k_split, int tiles_m, int tiles_n) {
  constexpr int PER = NT + MT, ROWS = PER * 16, STAGES = whole_stages(ROWS), STAGE_BYTES = ROWS * 256;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int tile = tile_of_workgroup(blockIdx.x, tiles_m * tiles_n);
  const int n0 = tile / tiles_m * (NT * 16), m0 = tile % tiles_m * (MT * 16);
  const int steps = k_split / 64, last = steps - 1;

  // what this thread brings of a stage: of row threadIdx.x / 16 of every sixteen the piece that its slot holds (rows beyond the operand are read as
  // its last one: their results are dropped)
  const float* src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = threadIdx.x >> 4, part = (threadIdx.x & 15) ^ row;
    src[i] = (i < NT ? w + (size_t)min(n0 + i * 16 + row, N - 1) * K : x + (size_t)min(m0 + (i - NT) * 16 + row, M - 1) * K) +
             (size_t)blockIdx.y * k_split + part * 4;
  }
  auto load_piece = [&](int i, int step, unsigned stage) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(src[i] + step * 64),
                                     (void __attribute__((address_space(3)))*)(lds + stage * STAGE_BYTES + i * 4096 + wave * 1024), 16, 0, 0);
  };
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds + (unsigned)(r * 256 + ((wave * 4 + g) ^ r) * 16);

  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < steps) {
#pragma unroll
      for (int i = 0; i < PER; ++i) load_piece(i, s, s);
    }
  // waits until the stage behind `step` has landed, of which `younger` are under way
  auto landed = [&](int younger) {
    if (STAGES > 3 && younger >= 3) wait_loads<(STAGES > 3 ? 3 : 0) * PER>();
    else if (STAGES > 2 && younger == 2) wait_loads<(STAGES > 2 ? 2 : 0) * PER>();
    else if (younger >= 1) wait_loads<PER>();
    else wait_loads<0>();
  };
  landed(min(last, STAGES - 1));
  __builtin_amdgcn_s_barrier();
  // (the reads of LDS as instructions with their waits, as in gemm_blocks.hip; a set of operands is used behind the wait that it passes through)
  f32x4 operand[2][PER];  // the weights' tiles, then x's
#define READ_TILE(set, o, at) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(operand[set][o]) : "v"(base + (at)), "n"((o) * 4096) : "memory")
#pragma unroll
  for (int o = 0; o < PER; ++o) READ_TILE(0, o, 0u);
  unsigned stage = 0;
  auto multiply = [&](auto which, int step) {
    constexpr int SET = decltype(which)::value;
    const unsigned next_stage = stage + 1 == STAGES ? 0 : stage + 1;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int o = 0; o < PER; ++o) asm volatile("" : "+v"(operand[SET][o]));
    landed(min(max(0, last - (step + 1)), STAGES - 2));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const bool more = step + STAGES < steps;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(operand[SET][i][e], operand[SET][NT + j][e], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int o = j * PER / MT; o < (j + 1) * PER / MT; ++o) {  // (behind the last stage these read one that holds nothing new, and nobody uses them)
        READ_TILE(SET ^ 1, o, next_stage * STAGE_BYTES);
        if (more) load_piece(o, step + STAGES, stage);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    stage = next_stage;
  };
  int step = 0;
  for (; step + 1 < steps; step += 2) {
    multiply(std::integral_constant<int, 0>{}, step);
    multiply(std::integral_constant<int, 1>{}, step + 1);
  }
  if (step < steps) multiply(std::integral_constant<int, 0>{}, step);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int o = 0; o < PER; ++o) {
    asm volatile("" ::"v"(operand[0][o]));
    asm volatile("" ::"v"(operand[1][o]));
  }
#undef READ_TILE

  // D[n][m] of a tile: a lane holds column m = r and rows n = 4 g .. + 3
  const bool with_bias = bias && blockIdx.y == 0;
  f32x4* sums = (f32x4*)lds;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT * MT; ++t) sums[(t * 4 + wave) * 64 + lane] = acc[t / MT][t % MT];
  __syncthreads();
  for (int t = wave; t < NT * MT; t += 4) {
    f32x4 total = sums[t * 4 * 64 + lane];
#pragma unroll
    for (int v = 1; v < 4; ++v) total += sums[(t * 4 + v) * 64 + lane];
    const int m = m0 + t % MT * 16 + r, n = n0 + t / MT * 16 + 4 * g;
    if (m >= M || n >= N) continue;
    if (with_bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) total[e] += bias[min(n + e, N - 1)];
    }
    if (GATED) {
      float* dst = out + (size_t)m * (N / 2) + n / 2;
      if (n + 1 < N) dst[0] = silu(total[0]) * total[1];
      if (n + 3 < N) dst[1] = silu(total[2]) * total[3];
    } else {
      float* dst = out + ((size_t)blockIdx.y * M + m) * N + n;
      if (n + 3 < N && (N & 3) == 0) {
        *(f32x4*)dst = total;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) dst[e] = total[e];
      }
    }
  }
}

template <int NT, int MT, bool GATED>
static int launch_whole(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int splits, hipStream_t stream) {
  constexpr int ROWS = (NT + MT) * 16, bytes = whole_stages(ROWS) * ROWS * 256;
  static_assert(bytes <= 160 * 1024 && NT * MT * 4096 <= bytes, "a CU's LDS, and in it the tiles' sums of four waves");
  static bool asked = false;
  if (!asked) {
    if (hipFuncSetAttribute((const void*)gemm_f32_whole_kernel<NT, MT, GATED>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
      return ERR_BAD_ARGUMENT;
    asked = true;
  }
  const int tiles_m = (M + 16 * MT - 1) / (16 * MT), tiles_n = (N + 16 * NT - 1) / (16 * NT);
  hipLaunchKernelGGL((gemm_f32_whole_kernel<NT, MT, GATED>), dim3(tiles_m * tiles_n, splits), dim3(256), bytes, stream, x, w, bias, out, M, N, K,
                     K / splits, tiles_m, tiles_n);
  return LAUNCH_STATUS();
}

template <int WN, int WM, int WK, int TN, int TM, int AHEAD, bool GATED>
static int launch_tiles(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int splits,
                        hipStream_t stream) {
  constexpr int TILE_N = WN * TN * 32, TILE_M = WM * TM * 32;
  const int k_split = splits == 1 ? K : ((K + splits - 1) / splits + TILE_K - 1) / TILE_K * TILE_K;
  if ((size_t)k_split * (splits - 1) >= (size_t)K) return ERR_BAD_ARGUMENT;
  const int tiles_m = (M + TILE_M - 1) / TILE_M, tiles_n = (N + TILE_N - 1) / TILE_N;
  hipLaunchKernelGGL((gemm_f32_tiled_kernel<WN, WM, WK, TN, TM, AHEAD, GATED>), dim3(tiles_m * tiles_n, splits), dim3(256), 0, stream, x, w,
                     bias, out, M, N, K, k_split, tiles_m, tiles_n);
  return LAUNCH_STATUS();
}

// The tiles, and what a workgroup of each takes over K = 1,536, us: the first on a CU, and every further one there
// (measured at 65 to 2,048 rows of the four weights named above; larger tiles read less from L2 a product, smaller
// ones leave fewer rows and fewer CUs idle).
struct TileCost {
  int n, m;
  float first, further;
};
static const TileCost TILE_COSTS[] = {{128, 128, 118.f, 100.f}, {128, 64, 68.f, 51.f}, {64, 64, 39.5f, 27.f},
                                      {64, 32, 27.f, 14.7f},    {32, 32, 17.f, 8.3f}};

// Us that the product takes with tile `t`: workgroups are spread over 256 CUs, and a part of K costs its partial
// sums' way to memory and back besides.
static float tiled_us(const TileCost& t, int M, int N, int K, int splits) {
  const long groups = (long)((N + t.n - 1) / t.n) * ((M + t.m - 1) / t.m) * splits;
  const float rounds = (float)((groups + 255) / 256);
  return (t.first + (rounds - 1.f) * t.further) * (float)K / (float)splits / 1536.f +
         (splits > 1 ? (float)splits * M * N * 8e-6f / 4.5f : 0.f);
}

// The tiles of the kernel of whole tiles, in sixteens.
#define WHOLE_TILES(X) X(1, 3) X(1, 5) X(2, 2) X(2, 3) X(3, 3) X(3, 5) X(5, 5)
constexpr int TILE_COUNT = 5, WHOLE_COUNT = 7, ALL_TILES = TILE_COUNT + WHOLE_COUNT;

// Which kernel takes a product of up to 512 rows goes by what their tiles take, us: a launch, a tile, a million bytes of the result, and a tile's 64 k where few CUs are
// busy, and where all are; of the whole ones of which a CU holds two also once a first CU holds two (`shared`) and once all do.  The other kernel's workgroups
// come to a CU as many as are left, so theirs (`a_cu` 0) are the first one's 64 k and every further one's.  Fitted to 965 products of 65 to 512 rows
// of 22 weights, in one to eight parts, every weight out of memory.  The choice by them is 18 percent faster than the other kernel alone and at none of 508 products in
// one piece or 107 in parts more than 3 percent slower, which AHEAD_FROM is for (0.97: one 17 percent).  Priced as if a round of 256 of the other kernel's workgroups took what
// one of many rounds does, that kernel kept products that were the whole tiles'.  Us, that kernel -> by that estimate -> by this: 128 rows of N 2,048 K 1,536
// 18.3 -> 18.3 -> 13.4, 512 rows of it 43.0 -> 43.0 -> 36.2, 160 rows of N 17,920 K 1,536 gated 105 -> 106 -> 99; 200 rows of it 124 each way, as whole tiles 131.
struct TileTimes {
  int n, m, a_cu;
  float launch, tile, alone, busy, a_million, shared, shared_all;
};
static const TileTimes TIMES[ALL_TILES] = {
    {128, 128, 0, 3.102f, 1.266f, 4.934f, 4.341f, 0.211f, 0.f, 0.f}, {128, 64, 0, 4.547f, 0.887f, 2.181f, 2.134f, 0.211f, 0.f, 0.f},
    {64, 64, 0, 2.093f, 0.972f, 1.454f, 1.064f, 0.264f, 0.f, 0.f}, {64, 32, 0, 2.252f, 0.568f, 1.220f, 0.531f, 0.304f, 0.f, 0.f},
    {32, 32, 0, 3.884f, 0.937f, 0.655f, 0.319f, 0.252f, 0.f, 0.f}, {16, 48, 2, 2.158f, 0.239f, 0.311f, 0.533f, 0.596f, 0.655f, 0.518f},
    {16, 80, 2, 1.828f, 0.123f, 0.515f, 0.819f, 0.440f, 0.791f, 0.812f}, {32, 32, 2, 2.935f, 0.042f, 0.359f, 0.637f, 0.483f, 0.586f, 0.685f},
    {32, 48, 2, 2.500f, 0.323f, 0.516f, 0.881f, 0.391f, 0.848f, 0.858f}, {48, 48, 2, 2.708f, 0.322f, 0.770f, 1.531f, 0.241f, 1.287f, 1.383f},
    {48, 80, 1, 1.836f, 1.291f, 1.202f, 1.073f, 0.272f, 0.f, 0.f}, {80, 80, 1, 1.915f, 2.209f, 1.853f, 1.708f, 0.174f, 0.f, 0.f}};
// (in parts, where two numbers of them are compared as well, from further ahead: with 0.95 224 rows of N 1,536 K 8,960 66 -> 71 us, 160 rows of N 3,584 K
// 3,584 in eight 50 -> 55)
constexpr float AHEAD_FROM = 0.95f, PARTS_AHEAD_FROM = 0.88f;

// Without what reads parts of K again.
static float measured_us(const TileTimes& t, int M, int N, int K, int splits) {
  const long groups = (long)((N + t.n - 1) / t.n) * ((M + t.m - 1) / t.m) * splits;
  const float steps = (float)K / (float)splits / 64.f;
  float us = t.launch + t.a_million * 4e-6f * (float)splits * M * N;  // (a gated result is half as large)
  if (t.a_cu == 0) {
    const float rounds = (float)((groups + 255) / 256);
    return us + rounds * t.tile + steps * (t.alone + (rounds - 1.f) * t.busy);
  }
  const long places = 256L * t.a_cu, full = groups / places, rest = groups % places;
  us += (float)full * (t.tile + steps * t.busy);
  if (rest > 256) us += t.tile + steps * (t.shared + (t.shared_all - t.shared) * (float)(rest - 256) / 256.f);
  else if (rest) us += t.tile + steps * fmaxf(t.alone, t.busy * (float)rest / (float)places);
  return us;
}

// The tile that a product takes (first those of the kernel above, then the whole ones), and what it is estimated to take: that kernel's by its own estimate, the whole
// ones by theirs.  `in_pieces`: both operands begin at a multiple of 16 bytes.  Whole tiles need that: their operands go into LDS by 16 bytes a lane without
// passing registers.  They take whole stages of 64 k; more rows than 512 have not been measured but for a few, of which half were behind.
static int pick_tile(int M, int N, int K, int splits, bool in_pieces, float* us = nullptr) {
  int best = 0;
  for (int t = 1; t < TILE_COUNT; ++t)
    if (tiled_us(TILE_COSTS[t], M, N, K, splits) < tiled_us(TILE_COSTS[best], M, N, K, splits)) best = t;
  if (in_pieces && M <= 512 && K % (64 * splits) == 0) {
    int whole = TILE_COUNT;
    for (int t = whole + 1; t < ALL_TILES; ++t)
      if (measured_us(TIMES[t], M, N, K, splits) < measured_us(TIMES[whole], M, N, K, splits)) whole = t;
    const float here = measured_us(TIMES[whole], M, N, K, splits);
    if (here < (splits == 1 ? AHEAD_FROM : PARTS_AHEAD_FROM) * measured_us(TIMES[best], M, N, K, splits)) {
      if (us) *us = here;
      return whole;
    }
  }
  if (us) *us = tiled_us(TILE_COSTS[best], M, N, K, splits);
  return best;
}

// Which tile a product of more than 64 rows takes whose operands begin at a multiple of 16 bytes (its place, the whole ones from TILE_COUNT on).
extern "C" int llmserve_gemm_f32_tile(int M, int N, int K, int splits) {
  return M <= 64 || N <= 0 || K <= 0 || splits < 1 ? -1 : pick_tile(M, N, K, splits, true);
}

// Into how many parts of K (at most 8, each at least 256 long) the product of these sizes is best cut where its
// result may stay in parts.  `in_pieces`: whether both operands begin at a multiple of 16 bytes.
// An error against 64 bits goes with the root of how many k one sum runs over (3.7e-8 of the result for 4 of them, in both kernels): a part of K over the
// waves that share a tile, four of them here and TILE_WAVES there.  So whole tiles are taken in no fewer parts than keep their sums as short as the
// other kernel's in its best number.  Relative errors, that kernel -> whole tiles in the parts that their time alone would have -> in
// these: 160 rows of N 1,536 K 1,536 2.1e-7 -> 3.5e-7 -> 1.8e-7, 224 rows of N 1,536 K 8,960 4.9e-7 -> 8.5e-7 -> 4.3e-7, 65 rows of N 3,584 K 3,584
// 3.2e-7 -> 5.4e-7 -> 2.0e-7.
static const int TILE_WAVES[TILE_COUNT] = {1, 1, 1, 2, 4};
extern "C" int llmserve_gemm_f32_parts(int M, int N, int K, int in_pieces) {
  int best = 1, tile = 0;
  float best_us = 0.f;
  for (int splits = 1; splits <= 8; ++splits) {
    if (splits > 1 && K / splits < 256) break;
    float us;
    const int picked = pick_tile(M, N, K, splits, false, &us);
    if (splits == 1 || us < best_us) best = splits, best_us = us, tile = picked;
  }
  if (!in_pieces || M > 512) return best;
  auto read_us = [&](int splits) { return splits > 1 ? (float)splits * M * N * 4e-6f / 4.5f : 0.f; };
  const int shortest = best * TILE_WAVES[tile];
  best_us = PARTS_AHEAD_FROM * (measured_us(TIMES[tile], M, N, K, best) + read_us(best));
  for (int splits = 1; splits <= 8; ++splits) {
    if (splits > 1 && K / splits < 256) break;
    float us;
    if (4 * splits < shortest || pick_tile(M, N, K, splits, true, &us) < TILE_COUNT) continue;
    if (us + read_us(splits) < best_us) best = splits, best_us = us + read_us(splits);
  }
  return best;
}

template <bool GATED>
static int launch_tiled(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int splits,
                        hipStream_t stream) {
  const int choice = pick_tile(M, N, K, splits, ((size_t)x | (size_t)w) % 16 == 0);
  int place = TILE_COUNT;
#define LAUNCH_WHOLE(NT, MT) \
  if (choice == place++) return launch_whole<NT, MT, GATED>(x, w, bias, out, M, N, K, splits, stream);
  WHOLE_TILES(LAUNCH_WHOLE)
#undef LAUNCH_WHOLE
  switch (choice) {
    case 0: return launch_tiles<2, 2, 1, 2, 2, 4, GATED>(x, w, bias, out, M, N, K, splits, stream);
    case 1: return launch_tiles<4, 1, 1, 1, 2, 4, GATED>(x, w, bias, out, M, N, K, splits, stream);
    case 2: return launch_tiles<2, 2, 1, 1, 1, 4, GATED>(x, w, bias, out, M, N, K, splits, stream);
    case 3: return launch_tiles<2, 1, 2, 1, 1, 4, GATED>(x, w, bias, out, M, N, K, splits, stream);
    default: return launch_tiles<1, 1, 4, 1, 1, 4, GATED>(x, w, bias, out, M, N, K, splits, stream);
  }
}

// out [M, N] (or [splits, M, N] partial sums) = x [M, K] . w [N, K]^T (+ bias [N]); all float32, K a multiple
// of 4.  gated: w's rows alternate gate and up (N even), out is [M, N / 2] = silu(gate) * up, no splits.
// Up to 64 rows of x go to the weight-streaming kernel, more to whole tiles or the tiled kernel (`pick_tile`).  (Us at 33 / 48 / 64 rows, in parts with what adds them
// up, one tile of weights against the tiled kernel against this: N 17,920 K 1,536 gated 56 / 61 / 74, 53 / 54 / 54, 52 / 55 / 63; N 1,536 K 8,960
// in parts 32 / 36 / 42, 30 / 30 / 31, 33 / 35 / 42; N 2,048 K 1,536 17 / 18 / 21, 18 / 18 / 18, 14 / 16 / 21; N 37,888 K 3,584 gated
// 221 / 266 / 316, 202 / 206 / 205, 175 / 189 / 211; N 3,584 K 18,944 in parts 138 / 148 / 176, 109 / 110 / 110, 94 / 100 / 119.)
extern "C" int llmserve_gemm_f32(const float* x, const float* w, const float* bias, float* out, int gated, int M, int N,
                                 int K, int splits, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 4 || splits < 1 || (gated && (splits != 1 || N % 2))) return ERR_BAD_ARGUMENT;
  if (M <= 64)
    return gated ? pick_stream<true>(x, w, bias, out, M, N, K, splits, stream)
                 : pick_stream<false>(x, w, bias, out, M, N, K, splits, stream);
  return gated ? launch_tiled<true>(x, w, bias, out, M, N, K, splits, stream)
               : launch_tiled<false>(x, w, bias, out, M, N, K, splits, stream);
}
