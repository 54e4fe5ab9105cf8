// bfloat16 products of many rows (prompt portions, mixed steps) on the matrix cores, float32 accumulation:
// out[M, N] = x[M, K] . w[N, K]^T (+ bias), or silu(gate) * up of weight rows that alternate gate_j, up_j, or partial sums
// over parts of K.
//
// A workgroup owns a tile of weight rows by rows of x; both operands of a stage of 64 k (32 where K is no multiple of 64)
// go from global memory straight into LDS (global_load_lds_dwordx4: a wave's 64 lanes fill 1 KB in lane order, no
// registers in between), two to six stages deep, and a wave multiplies TN x TM tiles of v_mfma_f32_32x32x16_bf16.  While
// the products of sixteen k run, the operands of the next sixteen are read from LDS into a second set of registers.  One
// barrier a stage, before its last products: by then every wave holds all it needs of the stage, so the stage is asked
// for anew at once, as many stages ahead as there are, and the next one is known to have landed for everybody.
// A staged row of 64 k is 128 bytes, eight pieces of 16; piece p of row r lies in slot p ^ (r / 2 % 8), so that the
// sixteen lanes that LDS serves together (the same piece of sixteen rows) hit all its banks (measured: no conflicts; with
// p ^ (r % 8), half of the reads' time).
//
// What bounds it: at 8,192 rows of 8,192 x 8,192 the matrix cores (0.85 ms, 1.29 PFLOP/s; the library 0.73); at the sizes a
// decoder has, how the tiles divide over 256 CUs, and what a tile costs besides its products: about 8 us for 256 x 256
// (first loads, the way out), 4 for 128 x 128.  Hence the shapes below and `pick_shape`.  Us, a captured chain over different weights,
// the library (with the kernel for silu(gate) * up behind it, 5 to 19 us) -> this: N 17,920 K 1,536 gated: 256 rows 35 -> 29, 384 rows 37 -> 30,
// 2,048 rows 133 -> 111 (256 x 320 tiles: 490 of them make two rounds where 256 x 256 make 2.2); N 1,536 K 8,960 in parts: 96 rows
// 18 -> 12, 256 rows 23 -> 15, 384 rows 25-33 -> 20, 1,024 rows 38 -> 36; K 1,536: 192 rows 8.1 -> 6.4, 384 rows 9.2 -> 7.8;
// N 3,584 K 18,944 in parts: 128 rows 51 -> 34, 256 rows 61 -> 47, 512 rows 85 -> 80; N 37,888 K 3,584 gated: 2,048 rows 546 -> 474.
#include "common.h"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Which tile a workgroup takes.  The chip hands workgroups to its eight chiplets (XCDs) in turn,
// workgroup i to chiplet i % 8, and every chiplet has an L2 of its own: tiles dealt out in launch
// order would make every chiplet read all of both operands.  So chiplet c takes a contiguous run
// of the tiles instead, counted through bands of eight tile rows of x, down the band first, then
// along the weight rows: what runs on a chiplet at one time is a few columns of one band, whose
// operand rows it fetches once and shares through its L2.
#define CHIPLETS 8
#define BAND 8
__device__ __forceinline__ void tile_of_workgroup(int index, int tiles_n, int tiles_m, int& tile_n, int& tile_m) {
  const int tiles = tiles_n * tiles_m;
  const int chiplet = index % CHIPLETS, turn = index / CHIPLETS;
  const int place = chiplet * (tiles / CHIPLETS) + min(chiplet, tiles % CHIPLETS) + turn;
  const int band = place / (BAND * tiles_n), within = place % (BAND * tiles_n);
  const int rows = min(BAND, tiles_m - band * BAND);
  tile_m = band * BAND + within % rows;
  tile_n = within / rows;
}

// What the way out does with the sums (and the bias).
#define OUT_PLAIN 0
#define OUT_GATED 1    // silu(gate) * up of columns that alternate gate_j, up_j
#define OUT_ROTATED 2  // rows of q, k and v heads: q and k rotated in neighbouring pairs, k and v stored in their pages too

// What OUT_ROTATED needs: cos and sin of [token][dim / 2], the layer's pages and each token's place there (negative: none; the
// layout of a page is common.h's).  `dim` is a multiple of 16.
struct Rotated {
  const float2* table;
  bf16_t *keys, *values;
  const int* slots;
  int heads, kv_heads, dim, page_size;
};

// What a wave of OUT_ROTATED asks for before its products, as their way from memory would be waited for at the end: lane l
// holds where row l % 32 of its row tile j goes (the place of a negative slot is not used), the bias of the columns that it will write, and,
// where one tile leaves the registers, their angles.
template <int TN, int TM>
struct Early {
  static constexpr int PASSES = TN * TM == 1 ? 32 / (64 / (4 * TN)) : 0;
  int slot[TM], page[TM], offset[TM], value_row[TM];
  float bias[8];
  f32x4 angles[PASSES ? PASSES : 1][2];
};

__device__ __forceinline__ const f32x4* angles_of(const Rotated& to, int m, int d) { return (const f32x4*)(to.table + ((size_t)m * to.dim + d) / 2); }

template <int TN, int TM>
__device__ __forceinline__ void ask_early(Early<TN, TM>& early, const Rotated& to, const void* bias, int bias_is_float, int M, int N,
                                          int n_wave, int m_wave, int lane) {
  constexpr int LANES_A_ROW = 4 * TN, ROWS_A_PASS = 64 / LANES_A_ROW;
  const int n = min(n_wave + lane % LANES_A_ROW * 8, N - 8), width = value_piece_width(to.page_size);
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m_wave + j * 32 + (lane & 31), slot = m < M ? to.slots[m] : -1;
    early.slot[j] = slot;
    early.page[j] = slot / to.page_size;
    early.offset[j] = slot % to.page_size;
    early.value_row[j] = early.offset[j] / width * width * to.dim + early.offset[j] % width;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) early.bias[e] = bias ? load_as_float(bias, bias_is_float, n + e) : 0.f;
#pragma unroll
  for (int pass = 0; pass < Early<TN, TM>::PASSES; ++pass) {
    const f32x4* angles = angles_of(to, min(m_wave + pass * ROWS_A_PASS + lane / LANES_A_ROW, M - 1), n % to.dim);
    early.angles[pass][0] = angles[0], early.angles[pass][1] = angles[1];
  }
}

// The values of 32 rows, which lie in `mine` with their bias (rows of `ROW` floats, a column each of the wave's 32 TN): a page keeps
// them transposed in pieces of eight keys, so a lane takes one column of eight rows, and where the rows are one piece (a prompt's
// portion) 64 lanes store 1 KB in a row.
template <int TN, int TM, int ROW>
__device__ __forceinline__ void store_values(const Rotated& to, const float* mine, const Early<TN, TM>& early, int j, int N, int n_wave, int lane) {
  const int v_first = (to.heads + to.kv_heads) * to.dim, width = value_piece_width(to.page_size);
  if (n_wave + 32 * TN <= v_first) return;
#pragma unroll 1
  for (int unit = 0; unit < 2 * TN; ++unit) {
    const int column = (unit * 64 + lane) % (32 * TN), octet = (unit * 64 + lane) / (32 * TN);
    const int n = n_wave + column;
    const bool mine_to_store = n >= v_first && n < N;
    const int head = (n - v_first) / to.dim, d = (n - v_first) % to.dim;
    const size_t a_page = (size_t)to.page_size * to.dim;
    bf16x8 run;
#pragma unroll
    for (int i = 0; i < 8; ++i) run[i] = (bf16_t)mine[(size_t)(octet * 8 + i) * ROW + column];
    const int slot = __shfl(early.slot[j], octet * 8);
    bool together = width == 8 && slot >= 0 && slot % 8 == 0;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      const int place = __shfl(early.slot[j], octet * 8 + i);
      together = together & (place == slot + i);
    }
    if (__all(together)) {
      const int page = __shfl(early.page[j], octet * 8), row = __shfl(early.value_row[j], octet * 8);
      if (mine_to_store) *(bf16x8*)(to.values + ((size_t)page * to.kv_heads + head) * a_page + row + d * 8) = run;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // (asked of other lanes by all lanes, before any is left out)
        const int place = __shfl(early.slot[j], octet * 8 + i), page = __shfl(early.page[j], octet * 8 + i);
        const int row = __shfl(early.value_row[j], octet * 8 + i);
        if (mine_to_store && place >= 0) to.values[((size_t)page * to.kv_heads + head) * a_page + row + d * width] = run[i];
      }
    }
  }
}

// The way out.  D[n][m] of a 32 x 32 tile: a lane holds column m = lane % 32 and rows n = 8 * (e / 4) +
// 4 * (lane / 32) + e % 4, so its values lie in 32 different rows of `out`.  They go through LDS (`mine`: 32 x
// (32 TN + 4) floats of this wave's own), 32 rows of x at a time, and leave as whole rows: 4 TN lanes write the
// 32 TN columns of a row, eight columns (16 bytes of bfloat16) a lane.  n_wave, m_wave: where the wave's tiles begin;
// `slice` the part of K (its own copy of `out`).  INSIDE: all of it lies inside the result, rows of which are a multiple of
// eight long, so nothing is asked row by row (such questions kept the reads of one row from running beside the next).
template <int TN, int TM, bool INSIDE, typename TO, int OUT>
__device__ __forceinline__ void store_tiles(const f32x16 (&acc)[TN][TM], float* mine, TO* __restrict__ out,
                                            const void* __restrict__ bias, int bias_is_float, int slice, int M, int N,
                                            int n_wave, int m_wave, int lane, const Rotated& rotated, const Early<TN, TM>& early) {
  static_assert(OUT == OUT_PLAIN || sizeof(TO) == 2, "a gated or rotated result is bfloat16");
  constexpr int ROW = 32 * TN + 4;  // floats of a transposed row, padded
  constexpr int LANES_A_ROW = 4 * TN, ROWS_A_PASS = 64 / LANES_A_ROW;
  const int r32 = lane & 31, half = lane >> 5;
  const int piece = lane % LANES_A_ROW, row_in_pass = lane / LANES_A_ROW;
  const int n_piece = n_wave + piece * 8;
  const bool with_bias = bias && slice == 0;
  float bias_here[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    bias_here[e] = OUT == OUT_ROTATED ? early.bias[e] : with_bias && (INSIDE || n_piece + e < N) ? load_as_float(bias, bias_is_float, n_piece + e) : 0.f;
  const int head = OUT == OUT_ROTATED ? n_piece / rotated.dim : 0, d = OUT == OUT_ROTATED ? n_piece % rotated.dim : 0;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int quad = 0; quad < 4; ++quad)
        *(f32x4*)(mine + (size_t)r32 * ROW + i * 32 + quad * 8 + half * 4) =
            (f32x4){acc[i][j][quad * 4], acc[i][j][quad * 4 + 1], acc[i][j][quad * 4 + 2], acc[i][j][quad * 4 + 3]};
    // (a wave reads only what it wrote itself: no barrier, the LDS operations of a wave complete in order)
#pragma unroll
    for (int pass = 0; pass < 32 / ROWS_A_PASS; ++pass) {
      const int row = pass * ROWS_A_PASS + row_in_pass;
      const int m = m_wave + j * 32 + row;
      const f32x4 lo = *(const f32x4*)(mine + (size_t)row * ROW + piece * 8);
      const f32x4 hi = *(const f32x4*)(mine + (size_t)row * ROW + piece * 8 + 4);
      float value[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int e = 0; e < 8; ++e) value[e] += bias_here[e];
      int slot = 0, page = 0, offset = 0;
      if constexpr (OUT == OUT_ROTATED) slot = __shfl(early.slot[j], row), page = __shfl(early.page[j], row), offset = __shfl(early.offset[j], row);
      if (!INSIDE && m >= M) continue;
      if constexpr (OUT == OUT_ROTATED) {
        if (!INSIDE && n_piece >= N) continue;  // (N is a multiple of 16)
        // rounded before they are rotated, as where a kernel of its own reads them from memory
        bf16_t packed[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) packed[e] = (bf16_t)value[e];
        if (head < rotated.heads + rotated.kv_heads) {
          constexpr bool HERE = Early<TN, TM>::PASSES > 0;
          const f32x4* angles = angles_of(rotated, m, d);
          const f32x4 first = HERE ? early.angles[HERE ? pass : 0][0] : angles[0], second = HERE ? early.angles[HERE ? pass : 0][1] : angles[1];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float c = e < 2 ? first[2 * e] : second[2 * e - 4], s = e < 2 ? first[2 * e + 1] : second[2 * e - 3];
            float x, y;
            turn_pair((float)packed[2 * e], (float)packed[2 * e + 1], c, s, e == 0 && d % 16 == 0, &x, &y);
            packed[2 * e] = (bf16_t)x, packed[2 * e + 1] = (bf16_t)y;
          }
        }
        *(uint4*)(out + (size_t)m * N + n_piece) = *(const uint4*)packed;
        if (head >= rotated.heads + rotated.kv_heads) {
          *(f32x4*)(mine + (size_t)row * ROW + piece * 8) = (f32x4){value[0], value[1], value[2], value[3]};  // (for store_values)
          *(f32x4*)(mine + (size_t)row * ROW + piece * 8 + 4) = (f32x4){value[4], value[5], value[6], value[7]};
        } else if (head >= rotated.heads && slot >= 0) {
          bf16_t* keys = rotated.keys + ((size_t)page * rotated.kv_heads + head - rotated.heads) * rotated.page_size * rotated.dim;
          *(uint4*)(keys + ((size_t)(d / KEY_PIECE) * rotated.page_size + offset) * KEY_PIECE) = *(const uint4*)packed;
        }
      } else if constexpr (OUT == OUT_GATED) {
        TO* dst = out + (size_t)m * (N / 2) + n_piece / 2;
        float gated[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // the hardware's 2^x and 1/x, as the result is bfloat16 (a tile has 128 of these a lane; the
          // library routines are some forty instructions each and took most of a tile's way out)
          const float gate = value[2 * e], up = value[2 * e + 1];
          gated[e] = gate * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gate * -1.44269504088896f)) * up;
        }
        if (INSIDE || (n_piece + 8 <= N && (N / 2) % 4 == 0)) {
          bf16_t packed[4] = {(bf16_t)gated[0], (bf16_t)gated[1], (bf16_t)gated[2], (bf16_t)gated[3]};
          *(uint2*)dst = *(const uint2*)packed;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n_piece + 2 * e + 1 < N) dst[e] = from_float<TO>(gated[e]);
        }
      } else {
        TO* dst = out + ((size_t)slice * M + m) * N + n_piece;
        if (INSIDE || (n_piece + 8 <= N && N % 8 == 0)) {
          if (sizeof(TO) == 2) {
            bf16_t packed[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) packed[e] = (bf16_t)value[e];
            *(uint4*)dst = *(const uint4*)packed;
          } else {
            *(f32x4*)dst = (f32x4){value[0], value[1], value[2], value[3]};
            *(f32x4*)((float*)dst + 4) = (f32x4){value[4], value[5], value[6], value[7]};
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n_piece + e < N) dst[e] = from_float<TO>(value[e]);
        }
      }
    }
    if constexpr (OUT == OUT_ROTATED) store_values<TN, TM, ROW>(rotated, mine, early, j, N, n_wave, lane);
  }
}

// The reads of LDS are written as instructions, with their waits: left to the compiler, every read of LDS waits for all
// loads into LDS that are under way, whichever stage they fill.  What a read brings is used only after `arrived`.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// waits until at most `younger` stages' loads of this wave (PER each) are under way; younger <= MOST or as if it were
template <int PER, int MOST>
__device__ __forceinline__ void wait_stages(int younger) {
  if constexpr (MOST > 0) {
    if (younger >= MOST) {
      wait_loads<PER * MOST>();
      return;
    }
    wait_stages<PER, MOST - 1>(younger);
  } else {
    wait_loads<0>();
  }
}

// WN x WM waves of TN x TM tiles; stages of BK k; A_SIMD: the waves a SIMD is to hold.
template <int WN, int WM, int TN, int TM, int BK, int STAGES, int A_SIMD, typename TO, int OUT>
__global__ __launch_bounds__(WN * WM * 64, A_SIMD) void gemm_block_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                          const void* __restrict__ bias, int bias_is_float,
                                                                          TO* __restrict__ out, int M, int N, int K, int k_split, Rotated rotated) {
  constexpr int THREADS = WN * WM * 64, BN = WN * TN * 32, BM = WM * TM * 32, SLOTS = BK / 8, HALVES = BK / 16;
  constexpr int ROW_BYTES = BK * 2, W_BYTES = BN * ROW_BYTES, STAGE_BYTES = W_BYTES + BM * ROW_BYTES;
  constexpr int PER_W = BN * SLOTS / THREADS, PER = PER_W + BM * SLOTS / THREADS;  // 16-byte pieces of a stage a lane asks for
  static_assert(BN * SLOTS % THREADS == 0 && BM * SLOTS % THREADS == 0 && HALVES % 2 == 0 && STAGES >= 2, "shape");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wave_n = wave % WN, wave_m = wave / WN;
  int tile_n, tile_m;
  tile_of_workgroup(blockIdx.x, (N + BN - 1) / BN, (M + BM - 1) / BM, tile_n, tile_m);
  const int n0 = tile_n * BN, m0 = tile_m * BM;
  const int k_first = blockIdx.z * k_split;
  const int r32 = lane & 31, half = lane >> 5;
  auto swizzle = [](int row) { return BK == 64 ? (row >> 1) & 7 : ((((row >> 1) ^ (row >> 3)) & 1) | (((row >> 2) & 1) << 1)); };

  // where this lane's pieces of a stage come from: piece -> (row, slot), the slot holds part slot ^ swizzle(row)
  // (rows beyond the operand are read as its last one: their results are dropped)
  const bf16_t* src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int piece = (i < PER_W ? i : i - PER_W) * THREADS + threadIdx.x;
    const int row = piece / SLOTS, part = (piece % SLOTS) ^ swizzle(row);
    src[i] = (i < PER_W ? w + (size_t)min(n0 + row, N - 1) * K : x + (size_t)min(m0 + row, M - 1) * K) + k_first + part * 8;
  }
  auto load_piece = [&](int i, int step, unsigned stage) {
    unsigned char* to = lds + stage * STAGE_BYTES + (i < PER_W ? i * THREADS * 16 : W_BYTES + (i - PER_W) * THREADS * 16) + wave * 1024;
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(src[i] + step * BK),
                                     (void __attribute__((address_space(3)))*)to, 16, 0, 0);
  };
  // where it reads its operands: rows r32 + 32 t of the wave's, part 2 * sixteen + half
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
  const int turned = swizzle(r32);
  const unsigned row_w = base + (unsigned)(wave_n * TN * 32 + r32) * ROW_BYTES;
  const unsigned row_x = base + W_BYTES + (unsigned)(wave_m * TM * 32 + r32) * ROW_BYTES;

  Early<TN, TM> early;
  if constexpr (OUT == OUT_ROTATED)
    ask_early(early, rotated, bias, bias_is_float, M, N, n0 + wave_n * TN * 32, m0 + wave_m * TM * 32, lane);

  f32x16 acc[TN][TM];  // [tile of weight rows][tile of x rows]
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int steps = k_split / BK, last = steps - 1;
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < steps) {
#pragma unroll
      for (int i = 0; i < PER; ++i) load_piece(i, s, s);
    }
  wait_stages<PER, STAGES - 1>(min(last, STAGES - 1));  // stage 0 has landed
  __builtin_amdgcn_s_barrier();
  bf16x8 a[2][TN], b[2][TM];  // two sets of operands
  // operand o of a set (the weight tiles', then x's) from `at` behind the wave's rows
#define READ_OPERAND(set, o, at)                                                                                            \
  do {                                                                                                                      \
    if ((o) < TN)                                                                                                           \
      asm volatile("ds_read_b128 %0, %1 offset:%2"                                                                          \
                   : "=v"(a[set][(o) < TN ? (o) : 0]) : "v"(row_w + (at)), "n"(((o) < TN ? (o) : 0) * 32 * ROW_BYTES) : "memory"); \
    else                                                                                                                    \
      asm volatile("ds_read_b128 %0, %1 offset:%2"                                                                          \
                   : "=v"(b[set][(o) < TN ? 0 : (o) - TN]) : "v"(row_x + (at)), "n"(((o) < TN ? 0 : (o) - TN) * 32 * ROW_BYTES) : "memory"); \
  } while (0)
  // The operands pass through the statements so that nothing that uses them is moved in front of the wait.
  auto arrived = [&](int set) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(a[set][i]));
#pragma unroll
    for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(b[set][j]));
  };
  auto slot_of = [&](int sixteen) { return (unsigned)(((sixteen * 2 + half) ^ turned) * 16); };
#pragma unroll
  for (int o = 0; o < TN + TM; ++o) READ_OPERAND(0, o, slot_of(0));
  unsigned stage = 0;
  // A stage with the loads of the one STAGES ahead dealt out between its last products (LOADS), or, at the end of K,
  // without: two bodies, so that neither has a branch inside.
  auto one_step = [&](int step, auto with_loads) {
    constexpr bool LOADS = decltype(with_loads)::value;
    const unsigned now = stage * STAGE_BYTES;
    const unsigned next_stage = stage + 1 == STAGES ? 0 : stage + 1;
    const unsigned then = next_stage * STAGE_BYTES;
#pragma unroll
    for (int sixteen = 0; sixteen < HALVES; ++sixteen) {
      constexpr int FINAL = HALVES - 1;
      const int set = sixteen & 1;
      arrived(set);
      if (sixteen == FINAL) {
        // this wave holds all it needs of the stage; the next one has to be there, for everybody
        if (LOADS) wait_loads<PER * (STAGES - 2)>();
        else wait_stages<PER, STAGES - 2>(max(0, last - (step + 1)));
        __builtin_amdgcn_s_barrier();
      }
      const unsigned slot = sixteen == FINAL ? then + slot_of(0) : now + slot_of(sixteen + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < TN * TM; ++p) {
        const int i = p / TM, j = p % TM;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[set][i], b[set][j], acc[i][j], 0, 0, 0);
        // two operands of the sixteen k to come behind each of the first products (after the last stage these read a
        // stage that holds nothing new: they stay inside LDS and nobody uses them)
#pragma unroll
        for (int o = 2 * p; o < (p + 1 == TN * TM ? TN + TM : min(2 * p + 2, TN + TM)); ++o) READ_OPERAND(set ^ 1, o, slot);
        if (LOADS && sixteen == FINAL) {
#pragma unroll
          for (int q = p; q < PER; q += TN * TM) load_piece(q, step + STAGES, stage);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    stage = next_stage;
  };
  int step = 0;
  for (; step + STAGES < steps; ++step) one_step(step, std::true_type{});
  for (; step < steps; ++step) one_step(step, std::false_type{});
  arrived(0);
  __syncthreads();  // every wave has read the last stage: LDS is free for the way out
  const int n_wave = n0 + wave_n * TN * 32, m_wave = m0 + wave_m * TM * 32;
  float* mine = (float*)lds + (size_t)wave * 32 * (32 * TN + 4);
  if (m_wave >= M || n_wave >= N) return;
  if (m_wave + 32 * TM <= M && n_wave + 32 * TN <= N && N % 8 == 0)
    store_tiles<TN, TM, true, TO, OUT>(acc, mine, out, bias, bias_is_float, blockIdx.z, M, N, n_wave, m_wave, lane, rotated, early);
  else
    store_tiles<TN, TM, false, TO, OUT>(acc, mine, out, bias, bias_is_float, blockIdx.z, M, N, n_wave, m_wave, lane, rotated, early);
}

template <int WN, int WM, int TN, int TM, int BK, int STAGES, int A_SIMD, typename TO, int OUT>
static int launch_block(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                        int splits, hipStream_t stream, const Rotated& rotated) {
  constexpr int BN = WN * TN * 32, BM = WM * TM * 32;
  constexpr size_t stages = (size_t)STAGES * (BN + BM) * BK * 2, way_out = (size_t)WN * WM * 32 * (32 * TN + 4) * sizeof(float);
  constexpr size_t bytes = stages > way_out ? stages : way_out;
  static_assert(bytes <= 160 * 1024, "a CU's LDS");
  static bool asked = false;
  if (!asked) {
    if (hipFuncSetAttribute((const void*)gemm_block_kernel<WN, WM, TN, TM, BK, STAGES, A_SIMD, TO, OUT>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
      return ERR_BAD_ARGUMENT;
    asked = true;
  }
  hipLaunchKernelGGL((gemm_block_kernel<WN, WM, TN, TM, BK, STAGES, A_SIMD, TO, OUT>),
                     dim3(((N + BN - 1) / BN) * ((M + BM - 1) / BM), 1, splits), dim3(WN * WM * 64), bytes, stream, (const bf16_t*)x,
                     (const bf16_t*)w, bias, bias_is_float, (TO*)out, M, N, K, K / splits, rotated);
  return LAUNCH_STATUS();
}

// The shapes: a tile's weight rows and rows of x, how many a CU holds at a time, and what a launch, a tile, and a tile's
// 64 k take, us (the last where few CUs are busy, and where all are: their clock is lower and they share L2).  Fitted to
// 88 products of 96 to 2,048 rows with the weights of the 1.5B and 7B sizes, whole and in parts, each shape within 9 to 14
// percent of what was measured; the shape picked by them is 4 percent slower than the best one on average.
struct BlockShape {
  int n, m, a_cu;
  float launch, tile, alone, busy;
};
static const BlockShape SHAPES[] = {{256, 256, 1, 0.95f, 7.25f, 1.195f, 2.156f}, {256, 320, 1, 1.99f, 8.13f, 1.347f, 2.404f},
                                    {256, 128, 1, 1.75f, 4.71f, 0.699f, 1.156f}, {128, 128, 1, 1.51f, 3.95f, 0.443f, 0.645f},
                                    {128, 64, 2, 3.98f, 0.74f, 0.336f, 0.866f},  {64, 64, 2, 3.68f, 1.08f, 0.235f, 0.492f}};
#define SHAPE_COUNT 6

static float shape_us(const BlockShape& t, int M, int N, int K, int splits) {
  const long groups = (long)((N + t.n - 1) / t.n) * ((M + t.m - 1) / t.m) * splits;
  const long places = 256L * t.a_cu, full = groups / places, rest = groups % places;
  const float steps = (float)(K / splits) / 64.f;
  float us = t.launch + (float)full * (t.tile + steps * t.busy);
  if (rest) us += t.tile + steps * fmaxf(t.alone, t.busy * (float)rest / (float)places);
  return us;
}

static int pick_shape(int M, int N, int K, int splits) {
  int best = 0;
  for (int s = 1; s < SHAPE_COUNT; ++s)
    if (shape_us(SHAPES[s], M, N, K, splits) < shape_us(SHAPES[best], M, N, K, splits)) best = s;
  return best;
}

// Into how many parts of K (at most 12, of whole stages) the product is best cut where its float32 result may stay partial
// sums: their way to the kernel that adds them up, at 4.5 TB/s, counts too.
extern "C" int llmserve_gemm_blocks_parts(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  const int stage = K % 64 ? 32 : 64;
  int best = 1;
  float best_us = 0.f;
  for (int splits = 1; splits <= 12; ++splits) {
    if (K % (splits * stage)) continue;
    const float us = shape_us(SHAPES[pick_shape(M, N, K, splits)], M, N, K, splits) + (float)splits * M * N * 4e-6f / 4.5f;
    if (splits == 1 || us < best_us) best = splits, best_us = us;
  }
  return best;
}

template <typename TO, int OUT>
static int launch_shape(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                        int splits, hipStream_t stream) {
#define BLOCK(...) return launch_block<__VA_ARGS__, TO, OUT>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, {})
  const int shape = pick_shape(M, N, K, splits);
  if ((K / splits) % 64) {  // a K that ends in half a stage: stages of 32
    if (shape < 3) BLOCK(2, 4, 4, 2, 32, 5, 2);
    BLOCK(2, 2, 2, 2, 32, 4, 2);
  }
  switch (shape) {
    case 0: BLOCK(2, 4, 4, 2, 64, 2, 2);
    case 1: BLOCK(4, 2, 2, 5, 64, 2, 2);
    case 2: BLOCK(4, 2, 2, 2, 64, 3, 2);
    case 3: BLOCK(2, 2, 2, 2, 64, 5, 1);
    case 4: BLOCK(2, 2, 2, 1, 64, 3, 2);
    default: BLOCK(2, 2, 1, 1, 64, 5, 2);
  }
#undef BLOCK
}

// x, w bfloat16; out bfloat16 or float32; any M and N, K a multiple of 32, an even N and a bfloat16 result with `gated` (silu).
// With splits > 1 (float32 out, not gated, K / splits a multiple of 32) `out` is [splits, M, N]
// partial sums, the bias in the first.
extern "C" int llmserve_gemm_blocks(const void* x, const void* w, const void* bias, int bias_is_float, void* out,
                                    int out_is_float, int gated, int M, int N, int K, int splits, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 32 || (gated && N % 2) || splits < 1 || gated > 1 || (gated && out_is_float)) return ERR_BAD_ARGUMENT;  // (this epilogue knows silu alone)
  if (splits > 1 && (gated || !out_is_float || K % splits || (K / splits) % 32)) return ERR_BAD_ARGUMENT;
  if (gated) return launch_shape<bf16_t, OUT_GATED>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  return out_is_float ? launch_shape<float, OUT_PLAIN>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)
                      : launch_shape<bf16_t, OUT_PLAIN>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
}

// A product whose heads are rotated on the way out, in the smallest tile of which one round of 256 workgroups holds the result, as
// more CUs then bring the operands.  Us at N 2,048 K 1,536, tiles of 64 x 32, 64 x 64, 128 x 64 and 128 x 128 (without the values' way to
// their pages): 96 rows 10.4 10.9 16.1 21.1, 256 rows 10.6 11.4 16.4 22.8, 512 rows 13.7 11.7 16.4 22.4, 1,024 rows 26.8 16.6 16.9 23.8,
// 2,048 rows 48.5 31.2 25.3 24.8; at N 4,608 K 3,584: 96 rows 19.2 19.9 30.0 37.6, 192 rows 26.6 21.3 30.7 36.0.  What it saves is a launch and
// the rows' way to memory and back: with the kernel that rotates and stores behind the library's product 15.5 us at 96 rows of N 2,048 K 1,536, here
// 11.6; 16.1 -> 11.7 at 256, 27.3 -> 26.0 at 2,048.  (Places, bias and angles asked for only on the way out: 13.4 at 96 rows.)
static int launch_rotated(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                          hipStream_t stream, const Rotated& rotated) {
#define BLOCK(...) return launch_block<__VA_ARGS__, bf16_t, OUT_ROTATED>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, rotated)
  auto one_round = [&](int n, int m) { return (long)((N + n - 1) / n) * ((M + m - 1) / m) <= 256; };
  if (K % 64) BLOCK(2, 2, 2, 2, 32, 4, 2);  // (a K that ends in half a stage, which the entry point takes; `_rotated_ahead` leaves it to the two kernels)
  if (one_round(64, 32)) BLOCK(2, 1, 1, 1, 64, 5, 2);
  if (one_round(64, 64)) BLOCK(2, 2, 1, 1, 64, 5, 2);
  if (one_round(128, 64)) BLOCK(2, 2, 2, 1, 64, 3, 2);
  BLOCK(2, 2, 2, 2, 64, 5, 1);
#undef BLOCK
}

// Rows of q, k and v heads: out [M, (heads + 2 kv_heads) dim] bfloat16 = x . w^T (+ bias), of which the q and k heads are rotated in
// neighbouring pairs by `table` (cos, sin of [M][dim / 2]), and k and v also stored in the pages.  `dim` a multiple of 16, K of 32.
extern "C" int llmserve_gemm_rotated(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int K,
                                     const float* table, int heads, int kv_heads, int dim, void* keys, void* values, const int* slots,
                                     int page_size, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K <= 0 || K % 32 || heads < 1 || kv_heads < 1 || dim < 16 || dim % 16 || page_size < 1 || !table || !keys || !values || !slots) return ERR_BAD_ARGUMENT;
  if ((size_t)table % 16 || (size_t)keys % 16 || (size_t)values % 16) return ERR_BAD_ARGUMENT;
  return launch_rotated(x, w, bias, bias_is_float, out, M, (heads + 2 * kv_heads) * dim, K, stream,
                        {(const float2*)table, (bf16_t*)keys, (bf16_t*)values, slots, heads, kv_heads, dim, page_size});
}
