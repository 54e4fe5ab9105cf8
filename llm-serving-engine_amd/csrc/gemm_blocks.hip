// bfloat16 products of many rows (prompt portions, mixed steps) on the matrix cores, float32 accumulation:
// out[M, N] = x[M, K] . w[N, K]^T (+ bias), or silu(gate) * up of weight rows that alternate gate_j, up_j, or partial sums
// over parts of K.
//
// A workgroup owns a tile of weight rows by rows of x; both operands of a stage of 64 k go from global memory straight into LDS
// (global_load_lds_dwordx4: a wave's 64 lanes fill 1 KB in lane order, no registers in between), two to five stages deep, and a wave
// multiplies TN x TM tiles of v_mfma_f32_16x16x32_bf16, whose operands it reads from LDS some tiles ahead of their products (Reads).  One
// barrier a stage, shortly before its last products: by then every wave has read all of the stage, and the next one is known to have landed for everybody;
// the stage is asked for anew, as many stages ahead as there are, piece by piece between the products that follow.
// A staged row of 64 k is 128 bytes, eight pieces of 16; piece p of row r lies in slot p ^ (r / 2 % 8), so that the
// sixteen lanes that LDS serves together (the same piece of sixteen rows) hit all its banks (measured: no conflicts; with
// p ^ (r % 8), half of the reads' time).
//
// What bounds it: at 8,192 rows of 8,192 x 8,192 the power that the matrix cores draw (shown for these sizes alone: gate/up of 2,048 rows is at 1.18 PFLOP/s; 0.78 ms, 1.41 PFLOP/s; the library 0.73): products alone, of random
// operands in registers, run at 2.0 PFLOP/s, of zeros at 2.4.  Tiles of 32 x 32 x 16, which move twice the sums in and out of the accumulators for a
// product, reach 1.81 there, and 0.83 ms here.  At the sizes a decoder has, how the tiles divide over 256 CUs, what a tile costs besides its
// products, and the way of the operands: a CU takes 64 bytes a clock from its caches, so what a stage brings (74 KB for 256 x 320) takes 1,150 clocks of the
// 2,560 of its products, and asked for all at once it stops the wave that asks.  Spread over the products, us before (asked for in the stage's last quarter) -> after:
// 2,048 rows of N 17,920 K 1,536 gated 110 -> 100, of N 2,048 K 1,536 20.4 -> 14.9, of N 1,536 K 1,536 16.9 -> 14.3, of N 1,536 K 8,960 in 128 x 128 77 -> 57;
// 320 rows of N 17,920 27.5 -> 25.7, and 8,960 as K in parts 20.1 -> 18.6.  There what bounds it is the weights' way from memory: three stages of all tiles are 7 MB,
// which take 2.4 us to come.  Bringing lines into L2 ahead of that gained nothing: what a wave asks for comes back in order, and waits for them.
// Against the library (with the kernel for silu(gate) * up behind it, 5 to 19 us), us: N 17,920 K 1,536 gated: 384 rows 37 -> 30, 2,048 rows 133 -> 100;
// N 1,536 K 8,960 in parts: 96 rows 18 -> 12, 384 rows 25-33 -> 19.
#include "common.h"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

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

// A result of more than so many bytes is stored past the caches: it does not fit the eight L2s (32 MB) beside the operands, and what lies there
// at a kernel's end is written back before the next one starts.  Us, kept -> past: 2,048 rows of N 17,920 K 1,536 gated (37 MB) 110.8 -> 102.8, a whole prompt of
// 2,048 tokens with it by 1 percent (7,138 -> 7,067 in one run).  Results that fit are read by the next kernel from there: a prompt of 77 1,798 -> 1,840.
#define STREAMED_FROM (16u << 20)

// What the way out does with the sums (and the bias).
#define OUT_PLAIN 0
#define OUT_GATED 1    // silu(gate) * up of columns that alternate gate_j, up_j
#define OUT_ROTATED 2  // rows of q, k and v heads: q and k rotated in neighbouring pairs, k and v stored in their pages too
#define OUT_NORM 3     // added to the residual stream; what the product behind the norm reads, and the squares it divides by (Link)
#define OUT_SCALED 4   // OUT_GATED of such rows: the sums are divided by the rows' root mean squares first
constexpr bool is_gated(int out) { return out == OUT_GATED || out == OUT_SCALED; }

// Two products with a norm between them, without a kernel for the norm (gemm_bf16.hip has the same for up to 64 rows).  The first (OUT_NORM) holds whole sums over
// K, adds them to the residual stream, and writes x * weight in bfloat16, not yet divided by the row's root mean square, with the sum of squares of each tile's
// columns a row.  The second (OUT_SCALED) adds those up and multiplies its float32 results by rsqrt(mean + eps): rounding
// x * weight loses what rounding the normed row loses.  A norm's kernel takes 5 us of a step of 96 to 320 rows and 11 of 2,048; against that the first needs whole sums (us in a
// step, before -> after: 96 rows of N 1,536 K 1,536 5.4 -> 6.4, 320 rows 6.5 -> 8.6, 2,048 rows 17.4 -> 21.2 with the stream's way) and the second the squares (17.9 -> 19.3,
// 24.6 -> 25.7, 98 -> 98).  A pass: prompt 77 1,714 -> 1,699 us, mixed 31 + 256 9,914 -> 9,790, prompt 2,048 by 1.5 percent.
struct Link {
  float* hidden;             // OUT_NORM: [M, N], added to in place
  const void* weight;        // OUT_NORM: the norm's [N]
  int weight_is_float;
  bf16_t* rows;              // OUT_NORM: [M, N]
  float* sums;               // [pieces, stride]: of a tile's columns of x each, row by row; `stride` is M up to a multiple of four
  float inverse_width, eps;  // OUT_SCALED
};
#define SUMS_MOST 48  // pieces of squares a row
__host__ __device__ __forceinline__ int sums_stride(int M) { return (M + 3) / 4 * 4; }

// What OUT_ROTATED needs: cos and sin of [token][dim / 2], the layer's pages and each token's place there (negative: none; the
// layout of a page is common.h's).  `dim` is a multiple of 16.
struct Rotated {
  const float2* table;
  bf16_t *keys, *values;
  const int* slots;
  int heads, kv_heads, dim, page_size;
};

// Which of a wave's weight rows row r of its tile i is.  A lane's sums of a tile are four rows of the product's result, 4 q .. 4 q + 3 for lanes
// 16 q .. 16 q + 15, all of one row of x.  So the rows are dealt to the tiles of a group (G of them) four at a time: over the group
// a lane then holds 4 G neighbours, which leave as one piece of 16 bytes (four float32, eight bfloat16, sixteen gates and ups).  Tiles that
// make no whole group hold their rows as they come.
template <int TN, int G>
__device__ __forceinline__ int weight_row(int i, int r) {
  return (i / G + 1) * G <= TN ? i / G * G * 16 + r / 4 * (4 * G) + i % G * 4 + r % 4 : i * 16 + r;
}
template <typename TO, int OUT, int TN>
constexpr int group_of() {
  int tiles = OUT == OUT_NORM ? 2 : sizeof(TO) == 4 ? 1 : is_gated(OUT) ? 4 : 2;
  while (tiles > TN) tiles /= 2;
  return tiles;
}

// What a wave of OUT_ROTATED asks for before its products, as their way from memory would be waited for at the end: where the rows of x that this
// lane will write go (the place of a negative slot is not used), the bias of its columns as it lies in memory (eight bfloat16, or eight float32 in two
// halves: nothing here may ask what it has brought, or it is waited for before the first stage is asked for), and their angles.
typedef unsigned u32x4_anywhere __attribute__((ext_vector_type(4), aligned(2)));
template <int TN, int TM>
struct Early {
  int slot[TM];
  u32x4 bias[TN / 2][2];
  f32x4 angles[TN / 2][TM][2];
};
template <int TN, int TM>
__device__ __forceinline__ float early_bias(const Early<TN, TM>& early, int i, int e, int bias_is_float) {
  const unsigned half = early.bias[i][0][e / 2];
  return __uint_as_float(bias_is_float ? early.bias[i][e / 4][e % 4] : e % 2 ? half & 0xffff0000u : half << 16);
}

__device__ __forceinline__ const f32x4* angles_of(const Rotated& to, int m, int d) { return (const f32x4*)(to.table + ((size_t)m * to.dim + d) / 2); }

template <int TN, int TM>
__device__ __forceinline__ void ask_early(Early<TN, TM>& early, const Rotated& to, const void* bias, int bias_is_float, int M, int N,
                                          int n_wave, int m_wave, int lane) {
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m_wave + j * 16 + (lane & 15);
    early.slot[j] = m < M ? to.slots[m] : -1;
  }
#pragma unroll
  for (int i = 0; i < TN / 2; ++i) {
    const int n = min(n_wave + i * 32 + (lane >> 4) * 8, N - 8);
    // (without a bias the same loads read the start of the angles, and nobody uses them)
    const char* from = bias ? (const char*)bias + (size_t)n * (bias_is_float ? 4 : 2) : (const char*)to.table;
    early.bias[i][0] = *(const u32x4_anywhere*)from;
    early.bias[i][1] = *(const u32x4_anywhere*)(from + (bias && bias_is_float ? 16 : 0));
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const f32x4* angles = angles_of(to, min(m_wave + j * 16 + (lane & 15), M - 1), n % to.dim);
      early.angles[i][j][0] = angles[0], early.angles[i][j][1] = angles[1];
    }
  }
}

// The values of 16 rows, which lie in `mine` with their bias (rows of `ROW` floats, a column each of the wave's 16 TN): a page keeps
// them transposed in pieces of eight keys, so a lane takes one column of eight rows, and where the rows are one piece (a prompt's
// portion) 64 lanes store 1 KB in a row.  `row_slot`, `row_page`, `row_offset`: where row lane % 16 goes.
template <int TN, int ROW>
__device__ __forceinline__ void store_values(const Rotated& to, const float* mine, int row_slot, int row_page, int row_offset, int N, int n_wave, int lane) {
  const int v_first = (to.heads + to.kv_heads) * to.dim, width = value_piece_width(to.page_size);
  const size_t a_page = (size_t)to.page_size * to.dim;
  // (divided once a row, not for every value.  Us at N 2,048 K 1,536, every seventh row kept nowhere: 160 rows 11.7 -> 9.7, 2,048 rows 30.7 -> 27.1; rows in pieces of
  // eight: 287 rows 10.5 -> 9.5)
  const int value_row = row_offset / width * width * to.dim + row_offset % width;
#pragma unroll 1
  for (int unit = 0; unit < TN / 2; ++unit) {
    const int column = (unit * 64 + lane) % (16 * TN), octet = (unit * 64 + lane) / (16 * TN);
    const int n = n_wave + column;
    const bool mine_to_store = n >= v_first && n < N;
    const int head = (n - v_first) / to.dim, d = (n - v_first) % to.dim;
    bf16x8 run;
#pragma unroll
    for (int i = 0; i < 8; ++i) run[i] = (bf16_t)mine[(size_t)(octet * 8 + i) * ROW + column];
    const int slot = __shfl(row_slot, octet * 8);
    bool together = width == 8 && slot >= 0 && slot % 8 == 0;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      const int place = __shfl(row_slot, octet * 8 + i);
      together = together & (place == slot + i);
    }
    auto row_of = [&](int page, int row) { return to.values + ((size_t)page * to.kv_heads + head) * a_page + row + d * width; };
    if (__all(together)) {
      const int page = __shfl(row_page, octet * 8), row = __shfl(value_row, octet * 8);
      if (mine_to_store) *(bf16x8*)row_of(page, row) = run;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // (asked of other lanes by all lanes, before any is left out)
        const int place = __shfl(row_slot, octet * 8 + i), page = __shfl(row_page, octet * 8 + i), row = __shfl(value_row, octet * 8 + i);
        if (mine_to_store && place >= 0) *row_of(page, row) = run[i];
      }
    }
  }
}

// The way out.  D[n][m] of a 16 x 16 tile: a lane holds column m = lane % 16 and four rows n (weight_row), and stores its run of a group's
// columns straight from its registers: four lanes write 64 bytes in a row, of sixteen rows.  n_wave, m_wave: where the wave's tiles begin;
// `slice` the part of K (its own copy of `out`).  INSIDE: all of it lies inside the result, rows of which are a multiple of
// eight long, so nothing is asked row by row.
template <int TN, int TM, bool INSIDE, typename TO, int OUT>
__device__ __forceinline__ void store_tiles(const f32x4 (&acc)[TN][TM], float* mine, TO* __restrict__ out,
                                            const void* __restrict__ bias, int bias_is_float, int slice, int M, int N,
                                            int n_wave, int m_wave, int lane, const Rotated& rotated, const Early<TN, TM>& early, bool streamed,
                                            const float* factor) {
  static_assert(OUT == OUT_PLAIN || OUT == OUT_NORM || sizeof(TO) == 2, "a gated or rotated result is bfloat16");
  constexpr int G = group_of<TO, OUT, TN>(), WHOLE = TN / G * G;
  const int r16 = lane & 15, q = lane >> 4;
  const bool with_bias = OUT != OUT_SCALED && bias && slice == 0;
  auto store_piece = [&](auto piece, TO* dst) {
    if (streamed) __builtin_nontemporal_store(piece, (decltype(piece)*)dst);
    else *(decltype(piece)*)dst = piece;
  };
  // a run of RUN neighbouring columns from n on, of row m: the sums of a group (or of one tile) and their bias
  auto store_run = [&](auto run_of, int m, int n, const float* sums) {
    constexpr int RUN = decltype(run_of)::value;
    if constexpr (is_gated(OUT)) {
      TO* dst = out + (size_t)m * (N / 2) + n / 2;
      bf16_t gated[RUN / 2];
#pragma unroll
      for (int e = 0; e < RUN / 2; ++e) {
        // the hardware's 2^x and 1/x, as the result is bfloat16 (a tile has 80 of these a lane; the
        // library routines are some forty instructions each and took most of a tile's way out)
        const float gate = sums[2 * e], up = sums[2 * e + 1];
        gated[e] = (bf16_t)(gate * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gate * -1.44269504088896f)) * up);
      }
      if (INSIDE || (n + RUN <= N && N % 8 == 0)) {
        if constexpr (RUN == 16) {
          // (of a width of 4 mod 8, N of 8 mod 16, every other row begins in the middle of 16 bytes: two halves.  Us by two bytes -> so: 2,048 rows of N 17,912
          // K 1,536 127 -> 103, of N 9,720 K 896 62 -> 46)
          if (N % 16 == 0) {
            store_piece(*(const u32x4*)gated, dst);
          } else {
            store_piece(*(const u32x2*)gated, dst);
            store_piece(*(const u32x2*)(gated + 4), dst + 4);
          }
        } else if constexpr (RUN == 8) *(uint2*)dst = *(const uint2*)gated;
        else *(unsigned*)dst = *(const unsigned*)gated;
      } else {
#pragma unroll
        for (int e = 0; e < RUN / 2; ++e)
          if (n + 2 * e + 1 < N) dst[e] = gated[e];
      }
    } else {
      TO* dst = out + ((size_t)slice * M + m) * N + n;
      if (INSIDE || (n + RUN <= N && N % 8 == 0)) {
        if constexpr (sizeof(TO) == 4) {
          store_piece((f32x4){sums[0], sums[1], sums[2], sums[3]}, dst);
        } else {
          bf16_t packed[RUN];
#pragma unroll
          for (int e = 0; e < RUN; ++e) packed[e] = (bf16_t)sums[e];
          if constexpr (RUN == 8) store_piece(*(const u32x4*)packed, dst);
          else *(uint2*)dst = *(const uint2*)packed;
        }
      } else {
#pragma unroll
        for (int e = 0; e < RUN; ++e)
          if (n + e < N) dst[e] = from_float<TO>(sums[e]);
      }
    }
  };
  if constexpr (OUT == OUT_ROTATED) {
    static_assert(G == 2 && WHOLE == TN, "runs of eight columns");
    constexpr int ROW = 16 * TN + 4;  // floats of a row of `mine`, padded
    const int v_first = (rotated.heads + rotated.kv_heads) * rotated.dim;
    const bool values_too = n_wave + 16 * TN > v_first;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int m = m_wave + j * 16 + r16;
      const int slot = early.slot[j], page = slot / rotated.page_size, offset = slot % rotated.page_size;
#pragma unroll
      for (int i = 0; i < TN / 2; ++i) {
        const int n = n_wave + i * 32 + q * 8;
        float value[8];
        bf16_t packed[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          value[e] = acc[2 * i + e / 4][j][e % 4] + (with_bias ? early_bias(early, i, e, bias_is_float) : 0.f);
          packed[e] = (bf16_t)value[e];  // rounded before they are rotated, as where a kernel of its own reads them from memory
        }
        const int head = n / rotated.dim, d = n % rotated.dim;
        if (n >= v_first) {
          *(f32x4*)(mine + (size_t)r16 * ROW + i * 32 + q * 8) = (f32x4){value[0], value[1], value[2], value[3]};  // (for store_values)
          *(f32x4*)(mine + (size_t)r16 * ROW + i * 32 + q * 8 + 4) = (f32x4){value[4], value[5], value[6], value[7]};
        } else {
          const f32x4 first = early.angles[i][j][0], second = early.angles[i][j][1];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float c = e < 2 ? first[2 * e] : second[2 * e - 4], s = e < 2 ? first[2 * e + 1] : second[2 * e - 3];
            float x, y;
            turn_pair((float)packed[2 * e], (float)packed[2 * e + 1], c, s, e == 0 && d % 16 == 0, &x, &y);
            packed[2 * e] = (bf16_t)x, packed[2 * e + 1] = (bf16_t)y;
          }
        }
        if (!INSIDE && (m >= M || n >= N)) continue;  // (N is a multiple of 16)
        *(uint4*)(out + (size_t)m * N + n) = *(const uint4*)packed;
        if (n < v_first && head >= rotated.heads && slot >= 0) {
          bf16_t* keys = rotated.keys + ((size_t)page * rotated.kv_heads + head - rotated.heads) * rotated.page_size * rotated.dim;
          *(uint4*)(keys + ((size_t)(d / KEY_PIECE) * rotated.page_size + offset) * KEY_PIECE) = *(const uint4*)packed;
        }
      }
      if (values_too) store_values<TN, ROW>(rotated, mine, slot, page, offset, N, n_wave, lane);  // (a wave reads only what it wrote itself: no barrier)
    }
  } else {
    float bias_here[TN][4];
    if (with_bias) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n_wave + weight_row<TN, G>(i, q * 4 + e);
          bias_here[i][e] = INSIDE || n < N ? load_as_float(bias, bias_is_float, n) : 0.f;
        }
    }
    auto sum_at = [&](int i, int j, int e, float row_factor) { return OUT == OUT_SCALED ? acc[i][j][e] * row_factor : with_bias ? acc[i][j][e] + bias_here[i][e] : acc[i][j][e]; };
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int m = m_wave + j * 16 + r16;
      if (!INSIDE && m >= M) continue;
      const float row_factor = OUT == OUT_SCALED ? factor[j * 16 + r16] : 1.f;
#pragma unroll
      for (int i = 0; i < WHOLE; i += G) {
        float sums[4 * G];
#pragma unroll
        for (int e = 0; e < 4 * G; ++e) sums[e] = sum_at(i + e / 4, j, e % 4, row_factor);
        store_run(std::integral_constant<int, 4 * G>{}, m, n_wave + i * 16 + q * 4 * G, sums);
      }
#pragma unroll
      for (int i = WHOLE; i < TN; ++i) {
        float sums[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[e] = sum_at(i, j, e, row_factor);
        store_run(std::integral_constant<int, 4>{}, m, n_wave + i * 16 + q * 4, sums);
      }
    }
  }
}

// What OUT_NORM adds to, and its norm's weight: asked for behind the first stages, used at the end.  A lane's columns of tile i: n_wave + weight_row(i, 4 q) .. + 3.
template <int TN, int TM>
struct Stream {
  f32x4 hidden[TN][TM];
  uint2 low[TN], high[TN];  // of the weight: four bfloat16 (twice) or the halves of four float32
};
template <int TN, int TM, int G>
__device__ __forceinline__ void ask_stream(Stream<TN, TM>& stream, const Link& link, int M, int N, int n_wave, int m_wave, int lane) {
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int n = min(n_wave + weight_row<TN, G>(i, (lane >> 4) * 4), N - 4);
    const char* weight = (const char*)link.weight + (size_t)n * (link.weight_is_float ? 4 : 2);
    stream.low[i] = *(const uint2*)weight;
    stream.high[i] = *(const uint2*)(weight + (link.weight_is_float ? 8 : 0));
#pragma unroll
    for (int j = 0; j < TM; ++j) stream.hidden[i][j] = *(const f32x4*)(link.hidden + (size_t)min(m_wave + j * 16 + (lane & 15), M - 1) * N + n);
  }
}
// The way out of OUT_NORM.  N is a multiple of eight: a run of four or eight columns lies inside it or beyond.
// `shares`: in LDS, where the squares of this wave's rows and columns go.
template <int TN, int TM, int G>
__device__ __forceinline__ void store_norm(const f32x4 (&acc)[TN][TM], const Stream<TN, TM>& stream, const Link& link, const void* bias, int bias_is_float, int M,
                                           int N, int n_wave, int m_wave, int lane, float* shares) {
  constexpr int WHOLE = TN / G * G;
  const int r16 = lane & 15, q = lane >> 4;
  f32x4 bias_here[TN];
  if (bias) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) bias_here[i][e] = load_as_float(bias, bias_is_float, min(n_wave + weight_row<TN, G>(i, q * 4) + e, N - 1));
  }
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m_wave + j * 16 + r16;
    float squares = 0.f;
    uint2 packed[TN];
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int n = n_wave + weight_row<TN, G>(i, q * 4);
      const bool inside = m < M && n < N;
      f32x4 x = acc[i][j];
      if (bias) x += bias_here[i];
      x += stream.hidden[i][j];
      const unsigned halves[4] = {stream.low[i].x << 16, stream.low[i].x & 0xffff0000u, stream.low[i].y << 16, stream.low[i].y & 0xffff0000u};
      const unsigned words[4] = {stream.low[i].x, stream.low[i].y, stream.high[i].x, stream.high[i].y};
      bf16_t row[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        row[e] = (bf16_t)(x[e] * __uint_as_float(link.weight_is_float ? words[e] : halves[e]));
        squares = inside ? fmaf(x[e], x[e], squares) : squares;
      }
      packed[i] = *(const uint2*)row;
      if (inside) *(f32x4*)(link.hidden + (size_t)m * N + n) = x;
    }
#pragma unroll
    for (int i = 0; i < TN; i += G) {
      const int n = n_wave + weight_row<TN, G>(i, q * 4);
      if (m >= M || n >= N) continue;
      bf16_t* to = link.rows + (size_t)m * N + n;
      if (G == 2 && i < WHOLE) {
        *(uint4*)to = make_uint4(packed[i].x, packed[i].y, packed[i + G - 1].x, packed[i + G - 1].y);
      } else {
        *(uint2*)to = packed[i];
      }
    }
    squares += __shfl_xor(squares, 16, WAVE);
    squares += __shfl_xor(squares, 32, WAVE);
    if (q == 0) shares[j * 16 + r16] = squares;
  }
}

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

// The order in which a wave reads its operands of 32 k from LDS.  The products of such a step go x tile by x tile (group j: x tile j with all the
// weight tiles), and the reads run AHEAD x tiles ahead of them, into SLOTS sets of registers in turn; the weight tiles have two sets, one a step.
// Behind the first product of group j come: of this step x tile j + AHEAD, while there is one (groups before FIRST); in group TURN the weight tiles of
// the next step and its x tiles that are due by then; later, one x tile of the next step a group.  At TURN nothing of this step is still to be read.
template <int TN, int TM, int AHEAD>
struct Reads {
  static constexpr int SLOTS = AHEAD < TM ? AHEAD + 1 : 2 * TM, FIRST = TM - AHEAD, TURN = FIRST == 0 ? 0 : FIRST + 1 < TM ? FIRST + 1 : TM - 1;
  static constexpr int AT_TURN = TURN - FIRST + 1;  // x tiles of the next step read in group TURN
  static_assert(AHEAD >= 1 && AHEAD <= TM && 2 * TM % SLOTS == 0, "two steps take whole turns of the registers");
  static constexpr int in_group(int j) { return j < FIRST ? 1 : j < TURN ? 0 : j == TURN ? TN + AT_TURN : 1; }
  // how many reads are younger than x tile j's when group j begins (the weight tiles' are older than x tile 0's)
  static constexpr int younger(int j) {
    int count = 0;
    if (j >= AHEAD) {
      for (int g = j - AHEAD + 1; g < j; ++g) count += in_group(g);
      return count;
    }
    for (int g = 0; g < j; ++g) count += in_group(g);
    const int asked = FIRST + j;  // in the step before, in this group or, all at once, in TURN
    for (int g = (asked > TURN ? asked : TURN) + 1; g < TM; ++g) count += in_group(g);
    return count + (asked < TURN ? TURN - asked : 0);
  }
};

// WN x WM waves of TN x TM tiles of 16 x 16; stages of 64 k, of which the last may be half full (HALF: K / splits % 64 == 32); A_SIMD: the waves a
// SIMD is to hold; AHEAD: see Reads.
// ONCE: no other workgroup reads these weights.  They then go past the caches: what a CU has under way of memory is limited (32 KB or so), a line that is kept
// nowhere takes less of it (measured with nothing but the loads: 112 CUs take 44 bytes a ns each, past the caches 47 to 53), and x keeps its place in
// L2.  Us, through them -> past them: 96 rows of N 17,920 K 1,536 17.7 -> 17.2, of N 37,888 K 3,584 56.8 -> 52.2; 160 rows 21.9 -> 21.2,
// of N 5,120 K 27,648 in parts 96 rows 63 -> 58.  (In parts shorter than 24 stages the product gains 1 to 5 percent and the norm that adds them up, alone behind it, loses more; whole
// prompts of 65 to 128 tokens are no longer for it, and at widths 1,536 to 2,560 up to 1 percent shorter.)  With a second tile of rows the other workgroup would find them gone: 320 rows of N 1,536 K 8,960 18.1 -> 21.1.
template <int WN, int WM, int TN, int TM, int AHEAD, int STAGES, int A_SIMD, bool HALF, typename TO, int OUT, bool ONCE>
__global__ __launch_bounds__(WN * WM * 64, A_SIMD) void gemm_block_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                          const void* __restrict__ bias, int bias_is_float,
                                                                          TO* __restrict__ out, int M, int N, int K, int k_split, Rotated rotated, Link link) {
  constexpr int BK = 64, THREADS = WN * WM * 64, BN = WN * TN * 16, BM = WM * TM * 16, SLOTS = BK / 8;
  constexpr int ROW_BYTES = BK * 2, W_BYTES = BN * ROW_BYTES, STAGE_BYTES = W_BYTES + BM * ROW_BYTES;
  constexpr int PER_W = BN * SLOTS / THREADS, PER = PER_W + BM * SLOTS / THREADS;  // 16-byte pieces of a stage a lane asks for
  static_assert(BN * SLOTS % THREADS == 0 && BM * SLOTS % THREADS == 0 && STAGES >= 2, "shape");
  using Order = Reads<TN, TM, AHEAD>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wave_n = wave % WN, wave_m = wave / WN;
  int tile_n, tile_m;
  tile_of_workgroup(blockIdx.x, (N + BN - 1) / BN, (M + BM - 1) / BM, tile_n, tile_m);
  const int n0 = tile_n * BN, m0 = tile_m * BM;
  const int k_first = blockIdx.z * k_split;
  const int r16 = lane & 15, q = lane >> 4;
  auto swizzle = [](int row) { return (row >> 1) & 7; };
  const int steps = (k_split + BK - 1) / BK, last = steps - 1;

  // where this lane's pieces of a stage come from: piece -> (row, slot), the slot holds part slot ^ swizzle(row)
  // (rows beyond the operand are read as its last one: their results are dropped; of a half stage the parts beyond it are read as the
  // parts before: nothing multiplies them)
  const bf16_t* src[PER];
  bool beyond[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int piece = (i < PER_W ? i : i - PER_W) * THREADS + threadIdx.x;
    const int row = piece / SLOTS, part = (piece % SLOTS) ^ swizzle(row);
    const int row_w = row / (TN * 16) * (TN * 16) + weight_row<TN, group_of<TO, OUT, TN>()>(row % (TN * 16) / 16, row % 16);
    src[i] = (i < PER_W ? w + (size_t)min(n0 + row_w, N - 1) * K : x + (size_t)min(m0 + row, M - 1) * K) + k_first + part * 8;
    beyond[i] = part >= SLOTS / 2;
  }
  auto load_piece = [&](int i, int step, unsigned stage) {
    unsigned char* to = lds + stage * STAGE_BYTES + (i < PER_W ? i * THREADS * 16 : W_BYTES + (i - PER_W) * THREADS * 16) + wave * 1024;
    const bf16_t* from = src[i] + step * BK - (HALF && step == last && beyond[i] ? BK / 2 : 0);
    if (ONCE && i < PER_W) __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)from, (void __attribute__((address_space(3)))*)to, 16, 0, 2);
    else __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)from, (void __attribute__((address_space(3)))*)to, 16, 0, 0);
  };
  // where it reads its operands: rows r16 + 16 t of the wave's, part 4 * step of 32 k + q.  Of that only `lane_at` differs by lane (a row is 128 bytes and
  // the second step's part the first one's with bit 2 turned, so 64 of it are turned): one register, as 256 x 320 has none to spare: with rows and parts
  // in four it kept two others in memory (READ_TILE says why none may lie there)
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
  const unsigned lane_at = (unsigned)(r16 * ROW_BYTES + (q ^ swizzle(r16)) * 16);
  const unsigned row_w = base + (unsigned)(wave_n * TN * 16) * ROW_BYTES, row_x = base + W_BYTES + (unsigned)(wave_m * TM * 16) * ROW_BYTES;

  Early<TN, TM> early;
  if constexpr (OUT == OUT_ROTATED)
    ask_early(early, rotated, bias, bias_is_float, M, N, n0 + wave_n * TN * 16, m0 + wave_m * TM * 16, lane);

  f32x4 acc[TN][TM];  // [tile of weight rows][tile of x rows]
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < steps) {
#pragma unroll
      for (int i = 0; i < PER; ++i) load_piece(i, s, s);
    }
  Stream<OUT == OUT_NORM ? TN : 1, OUT == OUT_NORM ? TM : 1> residual;
  if constexpr (OUT == OUT_NORM) {  // (the counts below do not know of these loads, and wait for as many of the stages' more until they have come)
    ask_stream<TN, TM, group_of<TO, OUT, TN>()>(residual, link, M, N, n0 + wave_n * TN * 16, m0 + wave_m * TM * 16, lane);
    asm volatile("" ::: "memory");
  }
  wait_stages<PER, STAGES - 1>(min(last, STAGES - 1));  // stage 0 has landed
  __builtin_amdgcn_s_barrier();
  // The reads of LDS are written as instructions, with their waits: left to the compiler, every read of LDS waits for all
  // loads into LDS that are under way, whichever stage they fill.  What a read brings is used only behind a wait that it passes through, so that
  // nothing that uses it is moved in front of the wait.  To the compiler a register is filled at its read: were it short of them, it could put one away that is
  // still to be filled.  So no shape may spill (`test_kernels_that_read_ahead_keep_their_registers`).
  bf16x8 a[2][TN], b[Order::SLOTS];
#define READ_TILE(into, row, tile, at) \
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(into) : "v"((row) + (at)), "n"((tile) * 16 * ROW_BYTES) : "memory")
  auto slot_of = [&](int chunk) { return lane_at ^ (unsigned)(chunk * 64); };
#pragma unroll
  for (int i = 0; i < TN; ++i) READ_TILE(a[0][i], row_w, i, slot_of(0));
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) READ_TILE(b[j], row_x, j, slot_of(0));
  unsigned stage = 0;
  // Half a stage (chunk 0 or 1).  In the second one's group TURN this wave holds all it needs of the stage: behind a barrier the next stage is read, and
  // this one is asked for anew (LOADS), a piece every PACE products, into the next stage's first half: a CU takes 64 bytes a clock from the caches, and
  // what is asked for faster than that holds up the products behind it.
  constexpr int LEFT = (TM - Order::TURN) * TN, PACE = LEFT + TM * TN < PER ? 1 : (LEFT + TM * TN) / PER;
  auto multiply = [&](auto which, auto with_loads, int step) {
    constexpr int CHUNK = decltype(which)::value;
    constexpr bool LOADS = decltype(with_loads)::value;
    const unsigned next_stage = stage + 1 == STAGES ? 0 : stage + 1, stage_before = stage == 0 ? STAGES - 1 : stage - 1;
    const unsigned here = stage * STAGE_BYTES + slot_of(CHUNK), then = CHUNK ? next_stage * STAGE_BYTES + slot_of(0) : stage * STAGE_BYTES + slot_of(1);
    constexpr int SET = CHUNK, B0 = CHUNK * TM;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      if (CHUNK && j == Order::TURN) {
        // (x tile j may still be on its way where TURN is the first group: the wait covers it)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (LOADS) wait_loads<PER * (STAGES - 2)>();
        else wait_stages<PER, STAGES - 2>(max(0, last - (step + 1)));
        __builtin_amdgcn_s_barrier();
      } else {
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(Order::younger(j) < 15 ? Order::younger(j) : 15) : "memory");
      }
      if (j == 0) {
#pragma unroll
        for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(a[SET][i]));
      }
      asm volatile("" : "+v"(b[(B0 + j) % Order::SLOTS]));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[SET][i], b[(B0 + j) % Order::SLOTS], acc[i][j], 0, 0, 0);
        if (j < Order::FIRST && i == 0) READ_TILE(b[(B0 + j + AHEAD) % Order::SLOTS], row_x, j + AHEAD, here);
        if (j == Order::TURN) {
          constexpr int COUNT = Order::in_group(Order::TURN), EACH = (COUNT + TN - 1) / TN;
#pragma unroll
          for (int r = i * EACH; r < min((i + 1) * EACH, COUNT); ++r) {
            if (r < TN) READ_TILE(a[SET ^ 1][r < TN ? r : 0], row_w, r < TN ? r : 0, then);
            else READ_TILE(b[(B0 + TM + (r < TN ? 0 : r - TN)) % Order::SLOTS], row_x, r < TN ? 0 : r - TN, then);
          }
        }
        if (j > Order::TURN && i == 0) READ_TILE(b[(B0 + j + AHEAD) % Order::SLOTS], row_x, j + AHEAD - TM, then);
        if (LOADS) {
          // (counted from TURN on; of the last product all that is left)
          const int place = CHUNK ? (j - Order::TURN) * TN + i : LEFT + j * TN + i;
          const bool end = CHUNK == 0 && j == TM - 1 && i == TN - 1;
          if (place >= 0) {
#pragma unroll
            for (int l = (place + PACE - 1) / PACE; l < PER && (end || l * PACE < place + 1); ++l) load_piece(l, CHUNK ? step + STAGES : step - 1 + STAGES, CHUNK ? stage : stage_before);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (CHUNK) stage = next_stage;
  };
  constexpr std::integral_constant<int, 0> first_half{};
  constexpr std::integral_constant<int, 1> second_half{};
  multiply(first_half, std::false_type{}, 0);
  int step = 0;
  for (; step + STAGES < steps; ++step) {
    multiply(second_half, std::true_type{}, step);
    multiply(first_half, std::true_type{}, step + 1);
  }
  // OUT_SCALED: the squares of this tile's rows, [pieces][BM], are brought into the first stage that is not asked for anew, some stages before they are used.  (The
  // waits below do not know of these loads, and wait for as many of the stages'.  The sums come as `bias`, their number, at most SUMS_MOST, as `bias_is_float`:
  // arguments that come with the wave.  As loads into registers before the stages they were waited for with all the stages behind them: 320 rows of N 17,920 K 1,536
  // 24.6 us without a norm, 26.1 so.)
  // (Not the largest tile, which has no registers to spare for it: it asks behind its last products.)
  constexpr bool SQUARES_EARLY = TN * TM <= 36;
  unsigned char* squares_at = lds;
  auto ask_squares = [&] {
    constexpr int QUADS = BM / 4;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // (nothing of this is to be made, and kept, before the products)
    for (int chunk = wave; chunk * 64 < bias_is_float * QUADS; chunk += WN * WM) {
      const int at = min(chunk * 64 + lane, bias_is_float * QUADS - 1), piece = at / QUADS, quad = at % QUADS;
      const float* from = (const float*)bias + (size_t)piece * sums_stride(M) + min(m0 + quad * 4, sums_stride(M) - 4);
      __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)from, (void __attribute__((address_space(3)))*)(squares_at + chunk * 1024), 16, 0, 0);
    }
  };
  [[maybe_unused]] const int first_free = step;
  for (; step < last; ++step) {
    multiply(second_half, std::false_type{}, step);
    if constexpr (OUT == OUT_SCALED && SQUARES_EARLY) {
      static_assert(SUMS_MOST * BM * 4 <= STAGE_BYTES, "in a stage's place");
      if (step == first_free) {
        squares_at = lds + (stage == 0 ? STAGES - 1 : stage - 1) * STAGE_BYTES;
        ask_squares();
      }
    }
    multiply(first_half, std::false_type{}, step + 1);
  }
  if (!HALF) multiply(second_half, std::false_type{}, last);
  // (what was read behind the last products stays inside LDS and nobody uses it, but its registers are not free before it has come)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    asm volatile("" ::"v"(a[0][i]));
    asm volatile("" ::"v"(a[1][i]));
  }
#pragma unroll
  for (int j = 0; j < Order::SLOTS; ++j) asm volatile("" ::"v"(b[j]));
#undef READ_TILE
  const int n_wave = n0 + wave_n * TN * 16, m_wave = m0 + wave_m * TM * 16;
  if constexpr (OUT == OUT_ROTATED) __syncthreads();  // every wave has read the last stage: LDS is free for the values
  const float* factor = nullptr;  // of the wave's rows, in LDS
  if constexpr (OUT == OUT_SCALED) {
    if constexpr (!SQUARES_EARLY) {
      __syncthreads();  // every wave has read the last stage
      ask_squares();
    }
    wait_loads<0>();
    __syncthreads();
    float* shares = (float*)squares_at;
    static_assert(BM <= THREADS, "a thread a row");
    int row = threadIdx.x;
    asm volatile("" : "+v"(row));
    if (row < BM) {  // (a row's squares are read, and the factor written in the place of the first, by one thread)
      float squares = 0.f;
#pragma unroll 8
      for (int c = 0; c < bias_is_float; ++c) squares += shares[c * BM + row];
      shares[row] = rsqrtf(squares * link.inverse_width + link.eps);
    }
    __syncthreads();
    factor = shares + wave_m * TM * 16;
  }
  float* mine = (float*)lds + (size_t)wave * 16 * (16 * TN + 4);
  const bool streamed = (size_t)gridDim.z * M * N * (is_gated(OUT) ? sizeof(TO) / 2 : sizeof(TO)) > STREAMED_FROM;
  if constexpr (OUT == OUT_NORM) {
    __syncthreads();  // every wave has read the last stage: LDS is free for the squares, [WN][BM]
    float* shares = (float*)lds;
    store_norm<TN, TM, group_of<TO, OUT, TN>()>(acc, residual, link, bias, bias_is_float, M, N, n_wave, m_wave, lane, shares + wave_n * BM + wave_m * TM * 16);
    __syncthreads();
    const int row = threadIdx.x;
    static_assert(BM <= THREADS, "a thread a row");
    if (row < BM && m0 + row < M) {
      float squares = shares[row];
#pragma unroll
      for (int c = 1; c < WN; ++c) squares += shares[c * BM + row];
      link.sums[(size_t)tile_n * sums_stride(M) + m0 + row] = squares;
    }
  } else {
    if (m_wave >= M || n_wave >= N) return;
  if (m_wave + 16 * TM <= M && n_wave + 16 * TN <= N && N % 8 == 0)
    store_tiles<TN, TM, true, TO, OUT>(acc, mine, out, bias, bias_is_float, blockIdx.z, M, N, n_wave, m_wave, lane, rotated, early, streamed, factor);
  else
    store_tiles<TN, TM, false, TO, OUT>(acc, mine, out, bias, bias_is_float, blockIdx.z, M, N, n_wave, m_wave, lane, rotated, early, streamed, factor);
  }
}

template <int WN, int WM, int TN, int TM, int AHEAD, int STAGES, int A_SIMD, bool HALF, typename TO, int OUT, bool ONCE>
static int launch_block_as(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                           int splits, hipStream_t stream, const Rotated& rotated, const Link& link) {
  constexpr int BN = WN * TN * 16, BM = WM * TM * 16;
  constexpr size_t stages = (size_t)STAGES * (BN + BM) * 128, values = OUT == OUT_ROTATED ? (size_t)WN * WM * 16 * (16 * TN + 4) * sizeof(float) : 0;
  constexpr size_t bytes = stages > values ? stages : values;
  static_assert(bytes <= 160 * 1024, "a CU's LDS");
  static bool asked = false;
  if (!asked) {
    if (hipFuncSetAttribute((const void*)gemm_block_kernel<WN, WM, TN, TM, AHEAD, STAGES, A_SIMD, HALF, TO, OUT, ONCE>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
      return ERR_BAD_ARGUMENT;
    asked = true;
  }
  hipLaunchKernelGGL((gemm_block_kernel<WN, WM, TN, TM, AHEAD, STAGES, A_SIMD, HALF, TO, OUT, ONCE>),
                     dim3(((N + BN - 1) / BN) * ((M + BM - 1) / BM), 1, splits), dim3(WN * WM * 64), bytes, stream, (const bf16_t*)x,
                     (const bf16_t*)w, bias, bias_is_float, (TO*)out, M, N, K, K / splits, rotated, link);
  return LAUNCH_STATUS();
}
// (a weight of up to 8 MB may have been brought into the caches, or live there with the rest of a small model: it is kept)
template <int WN, int WM, int TN, int TM, int AHEAD, int STAGES, int A_SIMD, bool HALF, typename TO, int OUT>
static int launch_block(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                        int splits, hipStream_t stream, const Rotated& rotated, const Link& link = {}) {
  if constexpr (OUT != OUT_ROTATED && !HALF)
    if (M <= WM * TM * 16 && (long)N * K > (1L << 22))
      return launch_block_as<WN, WM, TN, TM, AHEAD, STAGES, A_SIMD, HALF, TO, OUT, true>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, rotated, link);
  return launch_block_as<WN, WM, TN, TM, AHEAD, STAGES, A_SIMD, HALF, TO, OUT, false>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, rotated, link);
}

// The shapes: a tile's weight rows and rows of x, how many a CU holds at a time, and what a launch, a tile, a tile's
// 64 k (where few CUs are busy, and where all are: their clock is lower and they share L2) and a million bytes of the result take, us; where a CU holds two,
// also what 64 k take once a first CU holds two (`shared`) and once all do (`shared_all`): a workgroup that shares its CU takes up to twice as long, and the product ends
// with it.  Fitted to 1,764 products of 65 to 3,000 rows with 36 weights (K of 448 to 18,944), whole and in parts, every weight out of memory; the shape
// picked is 0.7 percent slower than the best one on average.  Two workgroups to a CU priced as one each as long as they were fewer than 512, and
// without 128 x 128 and 256 x 128, it was 5 percent, and one product in eleven was more than 3 percent slower than with the shapes that this kernel had before
// it spread its loads; of 936 others timed since it is one in eighty-five.  Us, those shapes -> ten under that estimate -> these: 400 rows of N 4,608 K 3,584 gated
// 27.9 -> 37.0 -> 24.1, 640 rows of N 11,008 K 2,048 33.9 -> 47.3 -> 32.4; in parts 160 rows of N 1,536 K 8,960 14.4 -> 15.6 -> 13.8, 513 rows of N 896 K 4,864
// 11.8 -> 15.1 -> 13.0.
struct BlockShape {
  int n, m, a_cu;
  float launch, tile, alone, busy, a_million, shared, shared_all;
};
static const BlockShape SHAPES[] = {
    {256, 256, 1, 3.208f, 0.501f, 1.248f, 1.421f, 0.166f, 0.f, 0.f}, {256, 320, 1, 4.907f, 0.205f, 1.570f, 1.513f, 0.137f, 0.f, 0.f},
    {128, 256, 1, 4.192f, 0.239f, 0.685f, 0.849f, 0.173f, 0.f, 0.f}, {192, 128, 1, 4.432f, 0.351f, 0.612f, 0.617f, 0.165f, 0.f, 0.f},
    {160, 160, 1, 4.840f, 0.430f, 0.549f, 0.674f, 0.164f, 0.f, 0.f}, {128, 160, 1, 5.356f, 0.222f, 0.503f, 0.512f, 0.169f, 0.f, 0.f},
    {96, 128, 1, 2.454f, 0.693f, 0.384f, 0.415f, 0.297f, 0.f, 0.f}, {128, 96, 1, 2.827f, 0.103f, 0.406f, 0.430f, 0.288f, 0.f, 0.f},
    {64, 128, 2, 2.135f, 0.025f, 0.369f, 0.592f, 0.232f, 0.648f, 0.732f}, {64, 64, 2, 2.180f, 0.100f, 0.187f, 0.426f, 0.281f, 0.348f, 0.506f},
    {128, 128, 1, 2.997f, 0.460f, 0.497f, 0.473f, 0.290f, 0.f, 0.f}, {256, 128, 1, 4.363f, 0.161f, 0.795f, 0.812f, 0.167f, 0.f, 0.f}};
#define SHAPE_COUNT 12

static float shape_us(const BlockShape& t, int M, int N, int K, int splits, int bytes) {  // (`bytes` of a column of the product in the result)
  const long groups = (long)((N + t.n - 1) / t.n) * ((M + t.m - 1) / t.m) * splits;
  const long places = 256L * t.a_cu, full = groups / places, rest = groups % places;
  const float steps = (float)((K / splits + 63) / 64);
  float us = t.launch + t.a_million * 1e-6f * (float)bytes * splits * M * N + (float)full * (t.tile + steps * t.busy);
  if (full == 0 && rest > 256) us += t.tile + steps * (t.shared + (t.shared_all - t.shared) * (float)(rest - 256) / 256.f);
  else if (rest) us += t.tile + steps * fmaxf(t.alone, t.busy * (float)rest / (float)places);
  return us;
}

// The shapes that take a K which ends in half a stage: five, as each is a kernel of its own in every kind of result.  A half stage costs what a whole one does.
// Us, in stages of 32 and tiles of 256 x 256 or 128 x 128 -> in those two tiles, picked by other shapes' estimates, and stages of 64 -> now: in three parts 160 rows
// of N 1,536 K 480 5.4 -> 6.3 -> 3.6; 513 rows of N 512 K 96 4.3 -> 4.8 -> 2.9; 160 rows of N 4,096 K 1,568 18.2 -> 19.0 -> 10.3; 513 rows of it 16.3 -> 16.1 -> 17.6.
static bool takes_half(int shape) { return shape == 0 || (shape >= 7 && shape <= 10); }

static int pick_shape(int M, int N, int K, int splits, int bytes) {
  int best = 0;
  for (int s = 1; s < SHAPE_COUNT; ++s)
    if ((K / splits % 64 == 0 || takes_half(s)) && shape_us(SHAPES[s], M, N, K, splits, bytes) < shape_us(SHAPES[best], M, N, K, splits, bytes)) best = s;
  return best;
}

// Which of the shapes a product takes (its place in SHAPES): `kind` 0 plain bfloat16, 1 float32, 2 gated.
extern "C" int llmserve_gemm_blocks_shape(int M, int N, int K, int splits, int kind) {
  if (M <= 0 || N <= 0 || K <= 0 || splits < 1 || kind < 0 || kind > 2) return -1;
  return pick_shape(M, N, K, splits, kind == 0 ? 2 : kind == 1 ? 4 : 1);
}

// Into how many parts of K (at most 12, of whole stages) the product is best cut where its float32 result may stay partial
// sums: their way to the kernel that adds them up, at 4.5 TB/s, counts too.  The number of parts decides in which order a result's sums meet, so
// it goes by an estimate of its own, over six tiles (weight rows, rows of x, how many a CU holds, what a launch, a tile and its 64 k take), which a shape added
// above, or timed anew, does not move: the same product gives the same bits.  Parts counted by the shapes' own estimate differ at half of the sizes and were no gain
// (us, those parts -> these: N 1,536 K 8,960 at 192 rows 22.8 -> 17.3, 960 rows 38.9 -> 38.7, 256 rows 18.5 -> 19.1; K 6,144 at 80 rows 9.8 -> 7.6).
static const struct { int n, m, a_cu; float launch, tile, alone, busy; } PART_TILES[] = {
    {256, 256, 1, 0.95f, 7.25f, 1.195f, 2.156f}, {256, 320, 1, 1.99f, 8.13f, 1.347f, 2.404f}, {256, 128, 1, 1.75f, 4.71f, 0.699f, 1.156f},
    {128, 128, 1, 1.51f, 3.95f, 0.443f, 0.645f}, {128, 64, 2, 3.98f, 0.74f, 0.336f, 0.866f},  {64, 64, 2, 3.68f, 1.08f, 0.235f, 0.492f}};

static float parts_us(int M, int N, int K, int splits) {
  float best = 0.f;
  for (const auto& t : PART_TILES) {
    const long groups = (long)((N + t.n - 1) / t.n) * ((M + t.m - 1) / t.m) * splits;
    const long places = 256L * t.a_cu, full = groups / places, rest = groups % places;
    const float steps = (float)(K / splits) / 64.f;
    float us = t.launch + (float)full * (t.tile + steps * t.busy);
    if (rest) us += t.tile + steps * fmaxf(t.alone, t.busy * (float)rest / (float)places);
    if (&t == PART_TILES || us < best) best = us;
  }
  return best + (float)splits * M * N * 4e-6f / 4.5f;
}

extern "C" int llmserve_gemm_blocks_parts(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  const int stage = K % 64 ? 32 : 64;
  int best = 1;
  float best_us = 0.f;
  for (int splits = 1; splits <= 12; ++splits) {
    if (K % (splits * stage)) continue;
    const float us = parts_us(M, N, K, splits);
    if (splits == 1 || us < best_us) best = splits, best_us = us;
  }
  return best;
}

template <typename TO, int OUT>
static int launch_shape(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                        int splits, hipStream_t stream, const Link& link = {}) {
#define BLOCK(...) return launch_block<__VA_ARGS__, TO, OUT>(x, w, bias, bias_is_float, out, M, N, K, splits, stream, {}, link)
  // Few rows of a weight that makes more than a round of such tiles (a head): a stream of the weight, for which what counts is 128 or 256 weight
  // rows to a row of tiles that holds all of x, with 72 to 132 KB of LDS asked for at a time.  Us, the library -> the shape that the estimate would pick -> this one: N 151,936 K 1,536 at
  // 17 rows 110 -> 81 -> 82, 32 rows 108 -> 93 -> 88, 48 rows 125 -> 104 -> 94, 64 rows 118 -> 113 -> 99 (5.1 TB/s, the result's way among it), 80 rows 133 -> 113 -> 105,
  // 96 rows 128 -> 117 -> 108; N 152,064 K 3,584 at 32 rows 257 -> 201 -> 189, 64 rows 217 -> 241 -> 210, 96 rows 234 -> 239 -> 219.  128 x 32 at 32 rows 88 and 188, 256 x 64 at 64 rows 101 and 210.
  if constexpr (OUT == OUT_PLAIN) {
    if (K % 64 == 0 && splits == 1 && M <= 64 && N > 256 * 128) BLOCK(4, 1, 2, 4, 3, 3, 2, false);
    if (K % 64 == 0 && splits == 1 && M > 64 && M <= 96 && N > 256 * 256) BLOCK(4, 1, 4, 6, 5, 3, 2, false);
  }
  const int shape = pick_shape(M, N, K, splits, is_gated(OUT) ? sizeof(TO) / 2 : sizeof(TO));
  if constexpr (OUT != OUT_SCALED) if ((K / splits) % 64) {  // a K that ends in half a stage
    switch (shape) {
      case 0: BLOCK(4, 2, 4, 8, 3, 2, 2, true);
      case 7: BLOCK(2, 2, 4, 3, 3, 5, 2, true);
      case 8: BLOCK(2, 2, 2, 4, 4, 3, 2, true);
      case 9: BLOCK(2, 2, 2, 2, 2, 5, 2, true);
      default: BLOCK(2, 2, 4, 4, 4, 5, 2, true);
    }
  }
  switch (shape) {
    case 0: BLOCK(4, 2, 4, 8, 3, 2, 2, false);
    case 1: BLOCK(4, 2, 4, 10, 4, 2, 2, false);
    case 2: BLOCK(2, 4, 4, 4, 4, 3, 2, false);
    case 3: BLOCK(2, 2, 6, 4, 4, 4, 2, false);
    case 4: BLOCK(2, 2, 5, 5, 4, 4, 2, false);
    case 5: BLOCK(2, 2, 4, 5, 4, 4, 2, false);
    case 6: BLOCK(2, 2, 3, 4, 4, 5, 2, false);
    case 7: BLOCK(2, 2, 4, 3, 3, 5, 2, false);
    case 8: BLOCK(2, 2, 2, 4, 4, 3, 2, false);
    case 9: BLOCK(2, 2, 2, 2, 2, 5, 2, false);
    case 10: BLOCK(2, 2, 4, 4, 4, 5, 2, false);
    default: BLOCK(4, 2, 4, 4, 4, 3, 2, false);
  }
#undef BLOCK
}

// x, w bfloat16, both from a multiple of 16 bytes on; out bfloat16 or float32; any M and N, K a multiple of 32, an even N and a bfloat16 result with `gated` (silu).
// With splits > 1 (float32 out, not gated, K / splits a multiple of 32) `out` is [splits, M, N]
// partial sums, the bias in the first.
extern "C" int llmserve_gemm_blocks(const void* x, const void* w, const void* bias, int bias_is_float, void* out,
                                    int out_is_float, int gated, int M, int N, int K, int splits, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 32 || (gated && N % 2) || splits < 1 || gated > 1 || (gated && out_is_float)) return ERR_BAD_ARGUMENT;  // (this epilogue knows silu alone)
  if (splits > 1 && (gated || !out_is_float || K % splits || (K / splits) % 32)) return ERR_BAD_ARGUMENT;
  if (((size_t)x | (size_t)w) & 15) return ERR_BAD_ARGUMENT;
  if (gated) return launch_shape<bf16_t, OUT_GATED>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
  return out_is_float ? launch_shape<float, OUT_PLAIN>(x, w, bias, bias_is_float, out, M, N, K, splits, stream)
                      : launch_shape<bf16_t, OUT_PLAIN>(x, w, bias, bias_is_float, out, M, N, K, 1, stream);
}

// The shape of OUT_NORM, which holds whole sums and a part of the stream beside them: tiles as small as one round of 256 workgroups allows, as more CUs then bring the
// operands, and what a CU brings (44 bytes a ns) is what they take; beyond a round, the estimate's; no more than SUMS_MOST tiles a row.  0: 32 x 32, 1: 64 x 32, else of SHAPES.
static int pick_norm_shape(int M, int N, int K) {
  auto workgroups = [&](int n, int m) { return (long)((N + n - 1) / n) * ((M + m - 1) / m); };
  if (workgroups(32, 32) <= 256 && N <= 32 * SUMS_MOST) return 0;
  if (workgroups(64, 32) <= 256 && N <= 64 * SUMS_MOST) return 1;
  int best = N <= 64 * SUMS_MOST ? 9 : 10;
  for (int s : {8, 6, 10})
    if (N <= SHAPES[s].n * SUMS_MOST && shape_us(SHAPES[s], M, N, K, 1, 10) < shape_us(SHAPES[best], M, N, K, 1, 10)) best = s;
  return best;
}

// How many pieces of squares the product into a norm leaves a row.
extern "C" int llmserve_gemm_blocks_norm_pieces(int M, int N, int K) {
  const int shape = pick_norm_shape(M, N, K), columns = shape == 0 ? 32 : shape == 1 ? 64 : SHAPES[shape].n;
  return (N + columns - 1) / columns;
}

// What the whole sums cost it, in thousandths of a us: its own time (of the two smallest tiles by K alone: 6.6 and 8.8 us at K 1,536, where 96 and 320 rows of N 1,536 take 6.4 and 8.6)
// over that in as many parts as `llmserve_gemm_blocks_parts` says.
extern "C" int llmserve_gemm_blocks_norm_cost(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 64 || N > 128 * SUMS_MOST) return 1 << 30;
  const int splits = llmserve_gemm_blocks_parts(M, N, K);
  const int shape = pick_norm_shape(M, N, K);
  const float whole = shape < 2 ? 2.3f + (float)(K / 64) * (shape == 0 ? 0.18f : 0.27f) : shape_us(SHAPES[shape], M, N, K, 1, 4), parts = shape_us(SHAPES[pick_shape(M, N, K, splits, 4)], M, N, K, splits, 4);
  return (int)(1000.f * (whole - parts));
}

// hidden [M, N] float32 += x . w^T (+ bias); rows [M, N] bfloat16 = hidden * weight; sums float32 [pieces, M up to a multiple of four], as above.  N a multiple
// of 16 up to 6,144, K of 64; x, w, hidden, weight and rows begin at a multiple of 16 bytes.
extern "C" int llmserve_gemm_blocks_into_norm(const void* x, const void* w, const void* bias, int bias_is_float, float* hidden, const void* weight,
                                              int weight_is_float, void* rows, float* sums, int M, int N, int K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 64 || N % 16 || N > 128 * SUMS_MOST || (((size_t)x | (size_t)w | (size_t)hidden | (size_t)weight | (size_t)rows) & 15)) return ERR_BAD_ARGUMENT;
  const Link link{hidden, weight, weight_is_float, (bf16_t*)rows, sums, 0.f, 0.f};
#define BLOCK(...) return launch_block<__VA_ARGS__, float, OUT_NORM>(x, w, bias, bias_is_float, nullptr, M, N, K, 1, stream, {}, link)
  switch (pick_norm_shape(M, N, K)) {
    case 0: BLOCK(2, 2, 1, 1, 1, 8, 1, false);  // (in four waves: in two 6.6 us at 96 rows of N 1,536 K 1,536 for 6.4, the next 8.8 at 320 rows for 8.6)
    case 1: BLOCK(2, 2, 2, 1, 1, 8, 1, false);
    case 6: BLOCK(2, 2, 3, 4, 4, 5, 2, false);
    case 8: BLOCK(2, 2, 2, 4, 4, 3, 2, false);
    case 9: BLOCK(2, 2, 2, 2, 2, 5, 2, false);
    default: BLOCK(2, 2, 4, 4, 4, 5, 2, false);
  }
#undef BLOCK
}

// silu(gate) * up of the rows that it leaves (K wide, a multiple of 64 from 128 on; w [N, K] alternates gate_j, up_j): out [M, N / 2] bfloat16.
extern "C" int llmserve_gemm_blocks_scaled(const void* rows, const float* sums, int pieces, float eps, const void* w, void* out, int M, int N, int K,
                                           hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 128 || K % 64 || N % 2 || pieces < 1 || pieces > SUMS_MOST || (((size_t)rows | (size_t)sums | (size_t)w) & 15)) return ERR_BAD_ARGUMENT;
  Link link{};
  link.inverse_width = 1.f / (float)K, link.eps = eps;
  return launch_shape<bf16_t, OUT_SCALED>(rows, w, sums, pieces, out, M, N, K, 1, stream, link);
}

// A product whose heads are rotated on the way out, in the smallest tile of which one round of 256 workgroups holds the result, as
// more CUs then bring the operands.  Us at N 2,048 K 1,536: 96 rows 6.8, 287 rows 9.9, 512 rows 9.0, 1,024 rows 13.4, 2,048 rows 21.6 (before the loads were
// spread over the products, the smallest tiles had as many waves as they have now, and with bias and places waited for before the first stage 10.6, 11.7, 11.9, 15.3, 22.5); in the smallest tile that does not
// make one round, measured then: 512 rows of 64 x 32 13.7, of 64 x 64 11.7, 1,024 rows of 64 x 64 26.8, of 128 x 64 16.6.  What it saves is a launch and
// the rows' way to memory and back: with the kernel that rotates and stores behind the library's product 15.5 us at 96 rows, 27.3 at 2,048.
static int launch_rotated(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int N, int K,
                          hipStream_t stream, const Rotated& rotated) {
#define BLOCK(...) return launch_block<__VA_ARGS__, bf16_t, OUT_ROTATED>(x, w, bias, bias_is_float, out, M, N, K, 1, stream, rotated)
  // Of the smallest, with as many waves as a tile has: 64 x 32 in four waves for two, us at N 2,048 K 1,536: 160 rows 8.9 -> 8.3, 256 rows 9.1 -> 8.4; 32 x 64 where that makes more
  // workgroups: 160 rows 7.6 (256 rows 8.6, as many); 32 x 32: 65 to 128 rows 8.3 -> 6.8, N 1,152 K 896 65 to 224 rows 6.8 -> 5.6; 64 x 64 in eight waves for four gains nothing.  A
  // prompt of 77 tokens with 32 x 32 1,699 -> 1,639.
  auto workgroups = [&](int n, int m) { return (long)((N + n - 1) / n) * ((M + m - 1) / m); };
  auto one_round = [&](int n, int m) { return workgroups(n, m) <= 256; };
  if (K % 64) BLOCK(2, 2, 4, 4, 4, 5, 2, true);  // (a K that ends in half a stage, which the entry point takes; `_rotated_ahead` leaves it to the two kernels)
  if (one_round(32, 32)) BLOCK(1, 2, 2, 1, 1, 8, 2, false);
  if (one_round(32, 64) && workgroups(32, 64) > workgroups(64, 32)) BLOCK(1, 4, 2, 1, 1, 8, 2, false);
  if (one_round(64, 32)) BLOCK(2, 2, 2, 1, 1, 6, 2, false);
  if (one_round(64, 64)) BLOCK(2, 2, 2, 2, 2, 5, 2, false);
  if (one_round(128, 64)) BLOCK(2, 2, 4, 2, 2, 3, 2, false);
  BLOCK(2, 2, 4, 4, 4, 5, 2, false);
#undef BLOCK
}

// Rows of q, k and v heads: out [M, (heads + 2 kv_heads) dim] bfloat16 = x . w^T (+ bias), of which the q and k heads are rotated in
// neighbouring pairs by `table` (cos, sin of [M][dim / 2]), and k and v also stored in the pages.  `dim` a multiple of 16, K of 32; x,
// w, the table and the pages begin at a multiple of 16 bytes.
extern "C" int llmserve_gemm_rotated(const void* x, const void* w, const void* bias, int bias_is_float, void* out, int M, int K,
                                     const float* table, int heads, int kv_heads, int dim, void* keys, void* values, const int* slots,
                                     int page_size, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K <= 0 || K % 32 || heads < 1 || kv_heads < 1 || dim < 16 || dim % 16 || page_size < 1 || !table || !keys || !values || !slots) return ERR_BAD_ARGUMENT;
  if (((size_t)x | (size_t)w | (size_t)table | (size_t)keys | (size_t)values) & 15) return ERR_BAD_ARGUMENT;
  return launch_rotated(x, w, bias, bias_is_float, out, M, (heads + 2 * kv_heads) * dim, K, stream,
                        {(const float2*)table, (bf16_t*)keys, (bf16_t*)values, slots, heads, kv_heads, dim, page_size});
}
