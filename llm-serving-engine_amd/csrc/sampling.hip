// Choosing the next token from float32 logits: argmax, temperature sampling, top-p.
//
// The reference samples with torch.multinomial from a per-request generator
// (engine.py:29-72).  A generator's stream cannot be reproduced here, so the engine defines
// its own rule, the same in its plain implementation: the host passes one uniform u in
// [0, 1) per row (a counter-based draw from the request's seed and its number of sampled
// tokens) and the kernel inverts the distribution's CDF at u:
//   top_p >= 1: p = softmax(logits / T); token = first index whose running sum of p, in
//               index order, exceeds u * sum(p);
//   top_p <  1: entries are ranked by descending p (ties by ascending index); an entry is
//               kept if the mass ranked before it is < top_p (engine.py:34-37); token =
//               first kept entry, in rank order, whose running sum exceeds u * (kept mass).
// p is exp((logit - max) / T), never divided by its sum Z: bounds are multiplied by Z instead.  Sums of
// p are float64 in an order that the sizes fix, or exact integers (see below): a call gives the same
// token on every run.
#include "common.h"
#include "no_alloc.h"

#include <mutex>
#include <stdio.h>

#define SAMPLE_THREADS 1024

__device__ __forceinline__ double block_sum_f64(double v, double* shared /* >= 17 */) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, waves = blockDim.x / WAVE;
#pragma unroll
  for (int offset = WAVE / 2; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, WAVE);
  __syncthreads();
  if (lane == 0) shared[wave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double total = 0.0;
    for (int i = 0; i < waves; ++i) total += shared[i];
    shared[16] = total;
  }
  __syncthreads();
  return shared[16];
}

// (value, index) of the first maximum of a row; every thread gets it.
__device__ __forceinline__ void block_argmax(const float* row, int n, float* best_value, int* best_index,
                                             float* shared_v, int* shared_i) {
  float value = -INFINITY;
  int index = 0x7fffffff;  // no entry seen yet
  for (int first = threadIdx.x; first < n; first += 4 * blockDim.x) {  // four loads under way together
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = first + u * blockDim.x;
      v[u] = i < n ? row[i] : -INFINITY;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = first + u * blockDim.x;
      if (i < n && (v[u] > value || index == 0x7fffffff)) {  // strided indices ascend, so ties keep the first
        value = v[u];
        index = i;
      }
    }
  }
#pragma unroll
  for (int offset = WAVE / 2; offset > 0; offset >>= 1) {
    const float ov = __shfl_xor(value, offset, WAVE);
    const int oi = __shfl_xor(index, offset, WAVE);
    if (ov > value || (ov == value && oi < index)) {
      value = ov;
      index = oi;
    }
  }
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, waves = blockDim.x / WAVE;
  __syncthreads();
  if (lane == 0) {
    shared_v[wave] = value;
    shared_i[wave] = index;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float bv = shared_v[0];
    int bi = shared_i[0];
    for (int i = 1; i < waves; ++i)
      if (shared_v[i] > bv || (shared_v[i] == bv && shared_i[i] < bi)) {
        bv = shared_v[i];
        bi = shared_i[i];
      }
    shared_v[16] = bv;
    shared_i[16] = bi;
  }
  __syncthreads();
  *best_value = shared_v[16];
  *best_index = shared_i[16];
}

// Two stages, so that a few rows still fill the chip: each row is cut into `pieces` pieces,
// a block finds the first maximum of its piece, and one more block per row picks among them.
// `zero` (may be null): for every row, `zero_words` words that the launch clears, `zero_stride` apart, for whoever runs after it.
__global__ __launch_bounds__(SAMPLE_THREADS) void argmax_pieces_kernel(const float* __restrict__ logits,
                                                                       float* __restrict__ piece_values,
                                                                       int* __restrict__ piece_indices, int vocab,
                                                                       int pieces, unsigned* __restrict__ zero,
                                                                       size_t zero_stride, int zero_words) {
  __shared__ float sv[17];
  __shared__ int si[17];
  if (zero != nullptr) {
    unsigned* mine = zero + blockIdx.x * zero_stride;
    for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < zero_words; i += gridDim.y * blockDim.x) mine[i] = 0u;
  }
  const int per = (vocab + pieces - 1) / pieces;
  const int begin = min(vocab, (int)blockIdx.y * per), count = min(vocab, begin + per) - begin;
  float value;
  int index;
  block_argmax(logits + (size_t)blockIdx.x * vocab + begin, count, &value, &index, sv, si);
  if (threadIdx.x == 0) {
    piece_values[blockIdx.x * pieces + blockIdx.y] = count > 0 ? value : -INFINITY;
    piece_indices[blockIdx.x * pieces + blockIdx.y] = count > 0 ? begin + index : 0x7fffffff;
  }
}

// One wave picks among a row's pieces, which ascend in index, so the first maximum among them is the
// row's; every lane gets its index (0 for a row without entries).
__device__ __forceinline__ int wave_pick_argmax(const float* __restrict__ piece_values,
                                                const int* __restrict__ piece_indices, int pieces) {
  const int lane = threadIdx.x % WAVE;
  float value = -INFINITY;
  int index = 0x7fffffff;
  for (int i = lane; i < pieces; i += WAVE) {
    const float v = piece_values[i];
    const int at = piece_indices[i];
    if (at != 0x7fffffff && (v > value || index == 0x7fffffff)) {
      value = v;
      index = at;
    }
  }
#pragma unroll
  for (int offset = WAVE / 2; offset > 0; offset >>= 1) {
    const float ov = __shfl_xor(value, offset, WAVE);
    const int oi = __shfl_xor(index, offset, WAVE);
    if (oi != 0x7fffffff && (index == 0x7fffffff || ov > value || (ov == value && oi < index))) {
      value = ov;
      index = oi;
    }
  }
  return index == 0x7fffffff ? 0 : index;
}

__global__ void argmax_pick_kernel(const float* __restrict__ piece_values, const int* __restrict__ piece_indices,
                                   int* __restrict__ out, int pieces) {
  const int index = wave_pick_argmax(piece_values + blockIdx.x * pieces, piece_indices + blockIdx.x * pieces, pieces);
  if (threadIdx.x == 0) out[blockIdx.x] = index;
}

#define ARGMAX_PIECES 64

// Into how many pieces a row is cut: 64 for a few rows (so that they fill the chip), fewer for many (a piece
// of 2,400 logits leaves a thread of its block two or three of them and the block's reduction dominates:
// 64 rows of 151,936 took 33 us in 64 pieces each).  About a thousand blocks in all, at least 8 pieces a row.
static int argmax_pieces(int rows) {
  int pieces = ARGMAX_PIECES;
  while (pieces > 8 && rows * pieces > 1024) pieces /= 2;
  return pieces;
}

// scratch: at least rows * 64 floats and rows * 64 ints
extern "C" int llmserve_argmax(const float* logits, float* piece_values, int* piece_indices, int* out, int rows,
                               int vocab, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (vocab <= 0) return ERR_BAD_ARGUMENT;
  const int pieces = argmax_pieces(rows);
  hipLaunchKernelGGL(argmax_pieces_kernel, dim3(rows, pieces), dim3(SAMPLE_THREADS), 0, stream, logits,
                     piece_values, piece_indices, vocab, pieces, (unsigned*)nullptr, (size_t)0, 0);
  hipLaunchKernelGGL(argmax_pick_kernel, dim3(rows), dim3(WAVE), 0, stream, piece_values, piece_indices, out, pieces);
  return LAUNCH_STATUS();
}

// The pieces' (value, index) pairs of `llmserve_argmax_static`: values first, then indices.  Each GPU
// holds its own copy of the array at its own address; host code reaches it only through the address
// that hipGetSymbolAddress gave for that device, never through the array's name.
#define ARGMAX_STATIC_SLOTS (LLMSERVE_ARGMAX_STATIC_MAX_ROWS * ARGMAX_PIECES)
static __device__ __align__(256) unsigned char argmax_static_scratch[ARGMAX_STATIC_SLOTS * (sizeof(float) + sizeof(int))];

#define ARGMAX_STATIC_MAX_DEVICES 64
static void* argmax_static_address[ARGMAX_STATIC_MAX_DEVICES];  // by device; null until that device's first call
static std::mutex argmax_static_lock;

extern "C" int llmserve_argmax_static(const float* logits, int* out, int rows, int vocab, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (vocab <= 0) return ERR_BAD_ARGUMENT;
  if (rows > LLMSERVE_ARGMAX_STATIC_MAX_ROWS) {
    fprintf(stderr, "llmserve_argmax_static: %d rows are more than the %d its fixed scratch buffer holds\n", rows,
            LLMSERVE_ARGMAX_STATIC_MAX_ROWS);
    return LLMSERVE_ERR_TOO_LARGE;
  }
  int device = -1;
  hipError_t status = hipGetDevice(&device);
  if (status != hipSuccess) return (int)status;
  if (device < 0 || device >= ARGMAX_STATIC_MAX_DEVICES) return ERR_BAD_ARGUMENT;
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> guard(argmax_static_lock);
    base = argmax_static_address[device];
    if (base == nullptr) {  // once per device, with that device current
      status = hipGetSymbolAddress(&base, HIP_SYMBOL(argmax_static_scratch));
      if (status != hipSuccess || base == nullptr) return status != hipSuccess ? (int)status : ERR_BAD_ARGUMENT;
      argmax_static_address[device] = base;
    }
  }
  // Nothing has to start at zero: the first kernel writes every slot that the second one reads.
  float* piece_values = (float*)base;
  int* piece_indices = (int*)((unsigned char*)base + ARGMAX_STATIC_SLOTS * sizeof(float));
  const int pieces = argmax_pieces(rows);
  hipLaunchKernelGGL(argmax_pieces_kernel, dim3(rows, pieces), dim3(SAMPLE_THREADS), 0, stream, logits,
                     piece_values, piece_indices, vocab, pieces, (unsigned*)nullptr, (size_t)0, 0);
  hipLaunchKernelGGL(argmax_pick_kernel, dim3(rows), dim3(WAVE), 0, stream, piece_values, piece_indices, out, pieces);
  return LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------------------
// Sampling with a temperature and top-p.
//
// Every launch but the last cuts a row into `pieces` contiguous pieces, a block a (row, piece), so that a few rows of a large
// vocabulary use the whole chip: the row's argmax; p and its sums; with top-p, the entries that the choice is among.  In the last one
// a block a row chooses the token, or a few blocks where a row leaves many to choose among.
//
// Top-p needs, twice, the smallest float t with mass_above(t) below a bound, where mass_above(t) is the
// sum of the entries of p greater than t: first the value at which the kept set ends (bound top_p * Z,
// strict), then the value in which u falls (bound u * kept mass).  p >= 0, so float order is the order
// of the bit patterns, and p <= 1 = exp(0), so a pattern has 30 bits.  A search fixes them ten at a
// time: it adds up the mass and the number of the entries in each of the 1,024 bins that the next
// ten bits cut the present bucket into, takes the lowest bin at whose end the bound is met and goes on inside it.
// After three levels the bucket is one value.  Both searches start from the same first histogram, which the
// blocks of the second launch make together.  What the later levels look at are the entries of a few of its bins, an eighth
// of an octave each: the one in which the kept set ends, and those in which u can fall, as the kept mass lies between the
// first bound and the end of that bin beyond it.  The third launch lists those entries (of a row of 151,936 whose logits have a spread of three
// some hundreds) and the row's block has them in registers and does all levels by itself.  Where they are more than 8,192 (small spreads,
// high temperatures, equal entries), the third launch adds up their second level instead, of up to three bins, and of the last launch up to
// sixteen blocks a row gather what lies in the one or two of its 1,024 runs that are left and add up the third level; the one that is done last
// goes on with the block's part.  So one block never goes through all of a row but for the place of one among a thousand equal entries.
// Us a call in a captured chain, 1 / 8 / 16 / 32 / 64 / 256 rows of 151,936: a launch a level, of many blocks a row | lists of any length,
// searched by one block | this:
//   spread 3, temperature 0.8, top-p 0.9   43 54 61 73 99 317   | 30 38 45 50 65 376     | 31 37 42 47 60 156
//   spread 1, temperature 1.5 (20,000)     44 54 63 77 104      | 46 59 66 70 89         | 40 48 55 67 87
//   spread 0.01 (nearly all)               49 62 76 104 155 523 | 162 195 218 263 324 977 | 45 56 68 92 137 394
//   equal entries                          62 86 130 215 383    | 129 141 144 160 221    | 61 66 81 111 170
//   two values                             52 65 90 137 229     | 244 254 262 300 353    | 62 64 76 102 152
// What is left is four launches that wait for one another.
//
// The entries of a bin share their exponent (it lies in the ten bits that are fixed first), so their
// sum is 2^exponent times the sum of their 24-bit significands, an integer below 2^42: a bin's mass is
// kept as that integer.  Integer sums do not depend on their order, so threads and blocks add into
// one histogram with atomic additions and the result is the same on every run.

#define SAMPLE_BLOCK 512  // threads of a block that works on a piece of a row
#define SAMPLE_BINS 1024
#define SAMPLE_LEVEL_BITS 10
#define SAMPLE_PIECES_MAX 64  // a wave looks at a row's pieces, a lane at each
#define SAMPLE_KEPT 8         // listed entries that a thread of the row's block keeps in registers
#define SAMPLE_LIST (SAMPLE_KEPT * SAMPLE_THREADS)

// About 512 blocks of 512 threads in all for top-p, where every piece adds its bins to the row's with atomic additions of
// its own (64 rows: 98 us, 110 with twice as many; 16 rows 61 and 81; 256 threads and 2,048 blocks 121 and 69), and twice as
// many without, where more blocks only hide more of the trips to memory (64 rows: 38 us and 43).
static int sample_pieces(int rows, bool with_top_p) {
  int pieces = SAMPLE_PIECES_MAX;
  while (pieces > 4 && rows * pieces > (with_top_p ? 512 : 1024)) pieces /= 2;
  return pieces;
}

// How many blocks of the last launch a row with many candidates has: what fills the chip once, as further ones only wait (spread 0.01, 16 / 64
// rows: 256 blocks in all 69.4 / 137 us, one a row 77.5 / 138; two values 77 / 153 and 165 / 219).  A row with few leaves all but the first at once.
static int pick_parts(int rows) { return rows >= 256 ? 1 : rows > 16 ? 256 / rows : 16; }

__device__ __forceinline__ int level_shift(int level) { return (2 - level) * SAMPLE_LEVEL_BITS; }

// value = significand * 2^(binary_exponent): what a float's pattern says, also for the subnormal ones
__device__ __forceinline__ unsigned long long significand_of(unsigned pattern) {
  return (pattern & 0x7fffffu) | ((pattern >> 23) != 0u ? 0x800000u : 0u);
}
__device__ __forceinline__ int binary_exponent_of(unsigned pattern) {
  const int exponent = (int)(pattern >> 23);
  return (exponent != 0 ? exponent : 1) - 150;
}

// The mass above the end of each of the 1,024 bins of one level, to `above` (LDS): that of the bucket, `start`, and of the bins
// after it.  `sums`: the histogram; `base`: the bucket's first pattern.  THREADS threads, a run of bins each; waves: a double of LDS a wave.
template <int THREADS>
__device__ __forceinline__ void masses_above(const unsigned long long* sums, unsigned base, int level, double start, double* above, double* waves) {
  constexpr int EACH = SAMPLE_BINS / THREADS;
  const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
  double mass[EACH], inclusive = 0.0;
#pragma unroll
  for (int j = EACH - 1; j >= 0; --j) {
    const int bin = t * EACH + j;
    mass[j] = ldexp((double)sums[bin], binary_exponent_of(base + ((unsigned)bin << level_shift(level))));
    inclusive += mass[j];
  }
#pragma unroll
  for (int offset = 1; offset < WAVE; offset <<= 1) {
    const double other = __shfl_down(inclusive, offset, WAVE);
    if (lane + offset < WAVE) inclusive += other;
  }
  const double after_in_wave = __shfl_down(inclusive, 1, WAVE);
  __syncthreads();  // whoever read the LDS arrays before is done
  if (lane == 0) waves[wave] = inclusive;
  __syncthreads();
  double later = lane == WAVE - 1 ? 0.0 : after_in_wave;
  for (int w = THREADS / WAVE - 1; w > wave; --w) later += waves[w];
#pragma unroll
  for (int j = EACH - 1; j >= 0; --j) {
    above[t * EACH + j] = start + later;
    later += mass[j];
  }
}

// The lowest bin at whose end the bound is met (mass above < limit if strict, else <= limit); the last one if it is nowhere (it
// cannot be: nothing lies above the maximum).  Every thread asks for its own run of `above`; *lowest is LDS, and nobody reads it any more.
template <int THREADS>
__device__ __forceinline__ int lowest_bin(const double* above, double limit, bool strict, int* lowest) {
  constexpr int EACH = SAMPLE_BINS / THREADS;
  if (threadIdx.x == 0) *lowest = SAMPLE_BINS - 1;
  __syncthreads();
  int mine = SAMPLE_BINS;
#pragma unroll
  for (int j = EACH - 1; j >= 0; --j) {
    const double m = above[threadIdx.x * EACH + j];
    if (strict ? m < limit : m <= limit) mine = (int)threadIdx.x * EACH + j;
  }
  const unsigned long long met = __ballot(mine < SAMPLE_BINS);  // (the first lane of a wave that meets it has the wave's lowest bin)
  if (met != 0ull && (int)threadIdx.x % WAVE == __ffsll((long long)met) - 1) atomicMin(lowest, mine);
  __syncthreads();
  return *lowest;
}

// The same for two bounds that are not strict, together; lowest: two of LDS.
template <int THREADS>
__device__ __forceinline__ void lowest_two_bins(const double* above, double limit0, double limit1, int* lowest) {
  constexpr int EACH = SAMPLE_BINS / THREADS;
  if (threadIdx.x < 2) lowest[threadIdx.x] = SAMPLE_BINS - 1;
  __syncthreads();
  int mine0 = SAMPLE_BINS, mine1 = SAMPLE_BINS;
#pragma unroll
  for (int j = EACH - 1; j >= 0; --j) {
    const double m = above[threadIdx.x * EACH + j];
    if (m <= limit0) mine0 = (int)threadIdx.x * EACH + j;
    if (m <= limit1) mine1 = (int)threadIdx.x * EACH + j;
  }
  const unsigned long long met0 = __ballot(mine0 < SAMPLE_BINS), met1 = __ballot(mine1 < SAMPLE_BINS);
  if (met0 != 0ull && (int)threadIdx.x % WAVE == __ffsll((long long)met0) - 1) atomicMin(lowest, mine0);
  if (met1 != 0ull && (int)threadIdx.x % WAVE == __ffsll((long long)met1) - 1) atomicMin(lowest + 1, mine1);
  __syncthreads();
}

// Which bins of the first histogram a row's choice is among, and the bound at which its kept set ends.
struct Candidates {
  double limit;                     // top_p * Z
  double above_cut;                 // the mass above `cut_bin`, as it met the bound: a search inside the bin begins from it
  int cut_bin, first_bin, last_bin;  // the kept set ends in the first of them, u falls in one of the run between the others
  int many;                         // whether they hold more entries than a list: then their second level is made instead
  __device__ __forceinline__ bool has(unsigned bin) const {
    return bin == (unsigned)cut_bin || (bin >= (unsigned)first_bin && bin <= (unsigned)last_bin);
  }
  // which second-level histogram is the bin's; -1 for the bins inside the run, which hold an entry at most: they begin above the cut, and u's
  // two bounds lie less than a value of the cut bin apart
  __device__ __forceinline__ int slot(int bin) const { return bin == cut_bin ? 0 : bin == first_bin ? 1 : bin == last_bin ? 2 : -1; }
};

// What the launches share of a row with top-p.  The first launch clears it up to the list, the second the second level, the third, where it
// makes that one, the third level.
#define SAMPLE_SLOTS 3
#define SAMPLE_FEW 1024
struct SampleRow {
  unsigned listed;  // how many entries are listed
  unsigned found, done;  // of a row with many candidates: how many entries are in `few` or would be, parts of the row that are done
  unsigned unused[61];
  unsigned long long sums[SAMPLE_BINS];  // the first histogram
  unsigned counts[SAMPLE_BINS];
  union {
    uint2 list[SAMPLE_LIST];  // pattern and index of the candidates, in no order
    struct {
      unsigned long long fine_sums[SAMPLE_SLOTS][SAMPLE_BINS];  // or the second level of their bins,
      unsigned fine_counts[SAMPLE_SLOTS][SAMPLE_BINS];
      unsigned long long run_sums[2][SAMPLE_BINS];  // the third of one or two runs of a second one,
      unsigned run_counts[2][SAMPLE_BINS];
      uint2 few[SAMPLE_FEW];  // and the entries of those runs
    };
  };
  Candidates candidates;
};
#define SAMPLE_CLEARED offsetof(SampleRow, list)

__device__ __forceinline__ void clear_histogram(unsigned long long* lds_sums, unsigned* lds_counts) {
  for (int i = threadIdx.x; i < SAMPLE_BINS; i += blockDim.x) {
    lds_sums[i] = 0ull;
    lds_counts[i] = 0u;
  }
}

// A piece's entries are taken in batches, all loads of a batch under way together: a thread of 256 had ten entries of a row of
// 151,936 in 64 pieces, and a loop that asks for one, waits, and adds it paid ten trips to memory one after the other.
#define SAMPLE_BATCH 6
struct Batch {
  float v[SAMPLE_BATCH];
};
// entries first, first + SAMPLE_BLOCK, ... below end; beyond it zeros, which nobody uses
__device__ __forceinline__ Batch load_batch(const float* __restrict__ p, int first, int end) {
  Batch batch;
#pragma unroll
  for (int u = 0; u < SAMPLE_BATCH; ++u) {
    const int i = first + u * SAMPLE_BLOCK;
    batch.v[u] = i < end ? p[i] : 0.f;
  }
  return batch;
}

// adds an entry to the first histogram (a pattern of more than 30 bits is that of no probability: of NaN)
__device__ __forceinline__ void add_entry(float value, unsigned long long* lds_sums, unsigned* lds_counts) {
  const unsigned pattern = __float_as_uint(value), bin = pattern >> level_shift(0);
  if (bin < SAMPLE_BINS) {
    atomicAdd(lds_sums + bin, significand_of(pattern));
    atomicAdd(lds_counts + bin, 1u);
  }
}

// Adds a lane's entry to a histogram in LDS, where `mine`; all lanes of the wave that are here together.  Additions to one place wait for one
// another, so entries that are equal in many lanes (a row of equal entries, or of a few values) go together, two values a time.
__device__ __forceinline__ void add_equal_together(bool mine, unsigned pattern, unsigned bin, unsigned long long* sums, unsigned* counts) {
  const int lane = threadIdx.x % WAVE;
#pragma unroll
  for (int turn = 0; turn < 2; ++turn) {
    const unsigned long long left = __ballot(mine);
    if (left == 0ull) return;
    const int leader = __ffsll((long long)left) - 1;
    const unsigned long long same = __ballot(mine && pattern == (unsigned)__builtin_amdgcn_readlane((int)pattern, leader));
    const int equal = __popcll(same);
    if (equal < 4) break;
    if (lane == leader) {
      atomicAdd(sums + bin, significand_of(pattern) * (unsigned long long)equal);
      atomicAdd(counts + bin, (unsigned)equal);
    }
    if ((same >> lane) & 1ull) mine = false;
  }
  if (mine) {
    atomicAdd(sums + bin, significand_of(pattern));
    atomicAdd(counts + bin, 1u);
  }
}

// Adds what the block has gathered of its piece to the row's histogram of `bins` bins (a barrier before).
__device__ __forceinline__ void give_histogram(const unsigned long long* lds_sums, const unsigned* lds_counts, int bins,
                                               unsigned long long* __restrict__ sums, unsigned* __restrict__ counts) {
  for (int bin = threadIdx.x; bin < bins; bin += blockDim.x) {
    const unsigned count = lds_counts[bin];
    if (count != 0u) {
      atomicAdd(sums + bin, lds_sums[bin]);
      atomicAdd(counts + bin, count);
    }
  }
}

// What the launches share: p, whose rows begin `stride` entries apart (a multiple of four), its pieces' sums, and what rows with top-p need.
struct SampleBuffers {
  float* p;
  size_t stride;
  double* piece_sums;         // [rows, pieces]
  SampleRow* rows;            // null where no row has top-p
  const float* piece_values;  // [rows, argmax_pieces]
  const int* piece_indices;
};

// The row's argmax (to out), p = exp((logit - max) / T) of one piece, not yet divided by its sum Z
// (engine.py:32), the piece's sum, and for a row with top-p the first histogram, which depends on no bucket.
__global__ __launch_bounds__(SAMPLE_BLOCK) void sample_exp_kernel(const float* __restrict__ logits,
                                                                  const float* __restrict__ temperatures,
                                                                  const float* __restrict__ top_ps, SampleBuffers buffers,
                                                                  int* __restrict__ out, int rows, int vocab, int pieces,
                                                                  int argmax_pieces, int with_top_p) {
  __shared__ double sd[17];
  __shared__ int best_index;
  __shared__ unsigned long long lds_sums[SAMPLE_BINS];
  __shared__ unsigned lds_counts[SAMPLE_BINS];
  const int r = blockIdx.x, piece = blockIdx.y;
  clear_histogram(lds_sums, lds_counts);
  if (threadIdx.x < WAVE) {
    const int index = wave_pick_argmax(buffers.piece_values + r * argmax_pieces,
                                       buffers.piece_indices + r * argmax_pieces, argmax_pieces);
    if (threadIdx.x == 0) {
      best_index = index;
      if (piece == 0) out[r] = index;
    }
  }
  __syncthreads();
  const float temperature = temperatures[r];
  if (temperature <= 0.f) return;  // engine.py:30-31: the argmax stands
  const float* row = logits + (size_t)r * vocab;
  float* p = buffers.p + r * buffers.stride;
  const int per = (vocab + pieces - 1) / pieces;
  const int begin = min(vocab, piece * per), end = min(vocab, begin + per);
  const bool with_histogram = with_top_p && top_ps[r] < 1.f;
  const float top_logit = row[best_index] / temperature;
  double partial = 0.0;
  if (with_histogram) {
    unsigned* fine = (unsigned*)buffers.rows[r].fine_sums;
    for (int i = piece * SAMPLE_BLOCK + threadIdx.x; i < SAMPLE_SLOTS * SAMPLE_BINS * 3; i += pieces * SAMPLE_BLOCK) fine[i] = 0u;
  }
  for (int first = begin + threadIdx.x; first < end; first += SAMPLE_BATCH * SAMPLE_BLOCK) {
    const Batch batch = load_batch(row, first, end);
#pragma unroll
    for (int u = 0; u < SAMPLE_BATCH; ++u) {
      const int i = first + u * SAMPLE_BLOCK;
      if (i >= end) break;
      const float v = expf(batch.v[u] / temperature - top_logit);
      p[i] = v;
      partial += (double)v;
      if (with_histogram) add_entry(v, lds_sums, lds_counts);
    }
  }
  const double sum = block_sum_f64(partial, sd);  // (its barriers stand between the additions and what reads them)
  if (threadIdx.x == 0) buffers.piece_sums[r * pieces + piece] = sum;
  if (!with_histogram) return;
  give_histogram(lds_sums, lds_counts, SAMPLE_BINS, buffers.rows[r].sums, buffers.rows[r].counts);
}

// Sums of v over the threads before this one, in thread order.  shared: at least 16 of its kind.
__device__ __forceinline__ double block_sum_before_f64(double v, double* shared) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  double inclusive = v;
#pragma unroll
  for (int offset = 1; offset < WAVE; offset <<= 1) {
    const double other = __shfl_up(inclusive, offset, WAVE);
    if (lane >= offset) inclusive += other;
  }
  __syncthreads();
  if (lane == WAVE - 1) shared[wave] = inclusive;
  __syncthreads();
  double before = 0.0;
  for (int w = 0; w < wave; ++w) before += shared[w];
  const double in_wave = __shfl_up(inclusive, 1, WAVE);
  return lane == 0 ? before : before + in_wave;
}

__device__ __forceinline__ int block_sum_before_int(int v, int* shared) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  int inclusive = v;
#pragma unroll
  for (int offset = 1; offset < WAVE; offset <<= 1) {
    const int other = __shfl_up(inclusive, offset, WAVE);
    if (lane >= offset) inclusive += other;
  }
  __syncthreads();
  if (lane == WAVE - 1) shared[wave] = inclusive;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < wave; ++w) before += shared[w];
  return before + inclusive - v;
}

// Lists the entries that the choice of a row with top-p is among, or, where they are more than a list holds, adds them up by the second
// ten bits: a block takes its piece's.
__global__ __launch_bounds__(SAMPLE_BLOCK) void sample_list_kernel(const float* __restrict__ temperatures, const float* __restrict__ top_ps,
                                                                   const float* __restrict__ uniforms, SampleBuffers buffers, int vocab,
                                                                   int pieces) {
  __shared__ double above[SAMPLE_BINS], waves[SAMPLE_BLOCK / WAVE], sums_here[SAMPLE_PIECES_MAX];
  __shared__ unsigned long long fine_sums[SAMPLE_SLOTS * SAMPLE_BINS];
  __shared__ unsigned fine_counts[SAMPLE_SLOTS * SAMPLE_BINS];
  __shared__ int lowest, lowest_two[2];
  __shared__ unsigned candidates, found, place;
  constexpr unsigned STAGE = SAMPLE_SLOTS * SAMPLE_BINS;
  uint2* stage = (uint2*)fine_sums;  // (a row has a list or the second level)
  const int r = blockIdx.x, piece = blockIdx.y, t = threadIdx.x;
  const float top_p = top_ps[r];
  if (temperatures[r] <= 0.f || top_p >= 1.f) return;
  SampleRow& row = buffers.rows[r];
  const int per = (vocab + pieces - 1) / pieces;
  const int begin = min(vocab, piece * per), end = min(vocab, begin + per);
  const float* p = buffers.p + r * buffers.stride;
  Batch batch = load_batch(p, begin + t, end);  // under way while the histogram is looked at
  if (t < pieces) sums_here[t] = buffers.piece_sums[r * pieces + t];  // a thread a piece asks, then everybody adds them in order
  if (t == 0) candidates = found = 0u;
  unsigned in_bin[SAMPLE_BINS / SAMPLE_BLOCK];
#pragma unroll
  for (int j = 0; j < SAMPLE_BINS / SAMPLE_BLOCK; ++j) in_bin[j] = row.counts[t + j * SAMPLE_BLOCK];
  masses_above<SAMPLE_BLOCK>(row.sums, 0u, 0, 0.0, above, waves);
  double total = 0.0;
  for (int q = 0; q < pieces; ++q) total += sums_here[q];
  Candidates c;
  // the bound is strict, so a bound of 0 would be met nowhere: the least positive one keeps the maximum alone
  c.limit = fmax((double)top_p * total, 2.2250738585072014e-308);
  c.cut_bin = lowest_bin<SAMPLE_BLOCK>(above, c.limit, true, &lowest);
  c.above_cut = above[c.cut_bin];
  // the kept mass is at least the bound, and beyond it by less than a value of that bin (up to rounding, which the row's block sees to);
  // and what is chosen is not below the cut
  const double end_of_bin = (double)__uint_as_float((unsigned)(c.cut_bin + 1) << level_shift(0)), u = (double)uniforms[r];
  lowest_two_bins<SAMPLE_BLOCK>(above, u * (c.limit + end_of_bin), u * c.limit, lowest_two);
  c.first_bin = max(c.cut_bin, lowest_two[0]);
  c.last_bin = max(c.cut_bin, lowest_two[1]);
#pragma unroll
  for (int j = 0; j < SAMPLE_BINS / SAMPLE_BLOCK; ++j)
    if (c.has(t + j * SAMPLE_BLOCK) && in_bin[j] != 0u) atomicAdd(&candidates, in_bin[j]);
  __syncthreads();
  c.many = candidates > SAMPLE_LIST ? 1 : 0;
  if (piece == 0 && t == 0) row.candidates = c;

  if (c.many) {
    for (int i = t; i < SAMPLE_SLOTS * SAMPLE_BINS; i += SAMPLE_BLOCK) fine_sums[i] = 0ull, fine_counts[i] = 0u;
    unsigned* runs = (unsigned*)row.run_sums;
    for (int i = piece * SAMPLE_BLOCK + t; i < 2 * SAMPLE_BINS * 3; i += pieces * SAMPLE_BLOCK) runs[i] = 0u;
    __syncthreads();
    for (int first = begin + t; first < end; first += SAMPLE_BATCH * SAMPLE_BLOCK) {
      if (first != begin + t) batch = load_batch(p, first, end);
#pragma unroll
      for (int k = 0; k < SAMPLE_BATCH; ++k) {
        const unsigned pattern = __float_as_uint(batch.v[k]);
        const int slot = first + k * SAMPLE_BLOCK < end ? c.slot((int)(pattern >> level_shift(0))) : -1;
        const int bin = max(slot, 0) * SAMPLE_BINS + (int)((pattern >> level_shift(1)) & (SAMPLE_BINS - 1));
        add_equal_together(slot >= 0, pattern, bin, fine_sums, fine_counts);
      }
    }
    __syncthreads();
    give_histogram(fine_sums, fine_counts, SAMPLE_SLOTS * SAMPLE_BINS, row.fine_sums[0], row.fine_counts[0]);
    return;
  }
  // They are gathered here, and go to a run of the row's list together; what does not fit here (a piece that holds most of them) is gone through
  // again.  The list holds them all, as the first histogram has counted them.
  auto gather = [&](auto f) {
    for (int first = begin + t; first < end; first += SAMPLE_BATCH * SAMPLE_BLOCK) {
#pragma unroll
      for (int k = 0; k < SAMPLE_BATCH; ++k) {
        const int i = first + k * SAMPLE_BLOCK;
        if (i < end && c.has(__float_as_uint(batch.v[k]) >> level_shift(0))) f(atomicAdd(&found, 1u), make_uint2(__float_as_uint(batch.v[k]), (unsigned)i));
      }
      batch = load_batch(p, first + SAMPLE_BATCH * SAMPLE_BLOCK, end);
    }
  };
  gather([&](unsigned at, uint2 entry) {
    if (at < STAGE) stage[at] = entry;
  });
  __syncthreads();
  const unsigned here = found;
  if (here == 0u) return;
  if (t == 0) place = atomicAdd(&row.listed, here);
  __syncthreads();
  if (here <= STAGE) {
    for (unsigned i = t; i < here; i += SAMPLE_BLOCK)
      if (place + i < SAMPLE_LIST) row.list[place + i] = stage[i];
    return;
  }
  if (t == 0) found = 0u;
  batch = load_batch(p, begin + t, end);
  __syncthreads();
  gather([&](unsigned at, uint2 entry) {
    if (place + at < SAMPLE_LIST) row.list[place + at] = entry;
  });
}

// The token of a row with top-p (out holds the argmax already), by the row's block or blocks; see the head of this section.  Bound by trips to memory, barriers
// and code that is fetched for the first time, one after the other: a row of 151,936 with a short list 14 us, with a long one 24.
__device__ __forceinline__ void sample_top_p(const SampleBuffers& buffers, int r, float uniform, int vocab, int* __restrict__ out) {
  constexpr int T = SAMPLE_THREADS;
  __shared__ double above[SAMPLE_BINS], first_above[SAMPLE_BINS], fine_above[SAMPLE_BINS], waves[T / WAVE];
  __shared__ unsigned long long sums[2 * SAMPLE_BINS];
  __shared__ unsigned counts[2 * SAMPLE_BINS];
  __shared__ uint2 stage[SAMPLE_FEW];
  __shared__ unsigned found, place;
  __shared__ int lowest, before_lowest, scan[17];
  const int t = threadIdx.x, lane = t % WAVE;
  const float* p = buffers.p + r * buffers.stride;
  SampleRow& row = buffers.rows[r];
  const Candidates c = row.candidates;
  const unsigned listed = row.listed;
  const double u = (double)uniform;
  uint2 kept[SAMPLE_KEPT];  // (the pattern ~0u: no entry)
  int n = 0;  // how many of the block's
  auto keep = [&](const uint2* list, int entries) __attribute__((always_inline)) {
    n = entries;
#pragma unroll
    for (int k = 0; k < SAMPLE_KEPT; ++k) kept[k] = t + k * T < n ? list[t + k * T] : make_uint2(~0u, 0u);
  };
  keep(row.list, (int)min(listed, (unsigned)SAMPLE_LIST));  // (none of a row with many candidates)
  if (blockIdx.y > 0 && !c.many) return;
  masses_above<T>(row.sums, 0u, 0, 0.0, first_above, waves);
  // calls f(pattern, index) for the entries that are kept or, where what is looked for may be none of them, for the whole row, a part at a time
  bool from_row = false;
  auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll 1
    for (unsigned first = t; first < (unsigned)(from_row ? vocab : T); first += SAMPLE_KEPT * T) {
      if (from_row) {
#pragma unroll
        for (int k = 0; k < SAMPLE_KEPT; ++k)
          kept[k] = first + k * T < (unsigned)vocab ? make_uint2(__float_as_uint(p[first + k * T]), first + k * T) : make_uint2(~0u, 0u);
      }
      const int here = from_row ? SAMPLE_KEPT * T : n;
#pragma unroll
      for (int k = 0; k < SAMPLE_KEPT; ++k) {
        if (k * T >= here) break;  // (most lists are short, and code that is not reached is not waited for)
        f(kept[k].x, (int)kept[k].y);
      }
    }
  };
  // one level of a search: the bin of a histogram at whose end the bound is met, inside the bucket that begins at `base`, `mass` above it
  // (a barrier before the next)
  auto level_of = [&](const unsigned long long* of, unsigned& base, int level, double& mass, double bound, bool strict) __attribute__((always_inline)) {
    masses_above<T>(of, base, level, mass, above, waves);
    const int bin = lowest_bin<T>(above, bound, strict, &lowest);
    mass = above[bin];
    base += (unsigned)bin << level_shift(level);
  };
  // the levels from `level` on: the value's pattern to `base`, and the mass above it
  auto searched = [&](unsigned& base, int level, double& mass, double bound, bool strict) __attribute__((always_inline)) {
#pragma unroll 1
    for (; level <= 2; ++level) {
      sums[t] = 0ull, counts[t] = 0u;
      __syncthreads();
      const int shift = level_shift(level);
      const unsigned bucket = base >> (shift + SAMPLE_LEVEL_BITS);
      each([&](unsigned pattern, int) {
        add_equal_together((pattern >> (shift + SAMPLE_LEVEL_BITS)) == bucket, pattern, (pattern >> shift) & (SAMPLE_BINS - 1), sums, counts);
      });
      __syncthreads();
      level_of(sums, base, level, mass, bound, strict);
      if (level < 2) __syncthreads();
    }
  };
  // of a row with many candidates: the run of 1,024 patterns of a bin at whose end the bound is met, and the mass above it
  int held = -1;  // whose masses fine_above holds
  auto fine_run = [&](int bin, int slot, double bound, double& mass) __attribute__((always_inline)) -> unsigned {
    if (held != slot) masses_above<T>(row.fine_sums[slot], (unsigned)bin << level_shift(0), 1, first_above[bin], fine_above, waves);
    held = slot;
    const int run = lowest_bin<T>(fine_above, bound, false, &lowest);
    mass = fine_above[run];
    __syncthreads();
    return ((unsigned)bin << SAMPLE_LEVEL_BITS) + (unsigned)run;
  };
  unsigned cut_run = 0u, first_run = 0u, last_run = 0u;  // of 1,024 patterns: the one of the cut, those in one of which u falls
  double above_run = c.above_cut;
  __syncthreads();
  if (c.many) {
    cut_run = (unsigned)c.cut_bin << level_shift(0);
    level_of(row.fine_sums[0], cut_run, 1, above_run, c.limit, true);
    cut_run >>= level_shift(1);
    __syncthreads();
    auto run_of = [&](double bound, unsigned whole) __attribute__((always_inline)) -> unsigned {
      const int bin = lowest_bin<T>(first_above, bound, false, &lowest), slot = c.slot(bin);
      __syncthreads();
      if (bin < c.cut_bin) return cut_run;
      if (slot < 0) return ((unsigned)bin << SAMPLE_LEVEL_BITS) | whole;
      double mass;
      const unsigned run = fine_run(bin, slot, bound, mass);
      return run > cut_run ? run : cut_run;
    };
    first_run = run_of(u * (c.limit + (double)__uint_as_float((cut_run + 1u) << level_shift(1))), 0u);
    last_run = run_of(u * c.limit, SAMPLE_BINS - 1);
    // Every part of the row gathers the entries of those runs and adds up the third level of the cut's and, if it is one alone, u's.  (One block
    // for the whole row is bound by its instructions, about a microsecond for each that it spends on an entry of 151,936.)
    const bool second = first_run == last_run && first_run != cut_run;
    const unsigned from_cut = cut_run << level_shift(1), from_u = first_run << level_shift(1), span_u = (last_run - first_run + 1u) << level_shift(1);
    const int quads = (vocab + 3) / 4, a_part = (quads + (int)gridDim.y - 1) / (int)gridDim.y;
    const int begin = min(quads, (int)blockIdx.y * a_part), end = min(quads, begin + a_part);
    auto of_part = [&](auto f) __attribute__((always_inline)) {  // f(quad, its number, whether it is there), a quad a lane; all lanes
      constexpr int TOGETHER = 4;
#pragma unroll 1
      for (int first = begin; first < end; first += TOGETHER * T) {
        float4 v[TOGETHER];
#pragma unroll
        for (int k = 0; k < TOGETHER; ++k) v[k] = ((const float4*)p)[min(first + k * T + t, end - 1)];
#pragma unroll
        for (int k = 0; k < TOGETHER; ++k) f(v[k], first + k * T + t, first + k * T + t < end);
      }
    };
    auto at_cut = [&](unsigned pattern) { return pattern - from_cut < (unsigned)SAMPLE_BINS; };
    auto at_u = [&](unsigned pattern) { return pattern - from_u < span_u; };
    auto patterns_of = [&](const float4& v, unsigned* patterns) __attribute__((always_inline)) {
      patterns[0] = __float_as_uint(v.x), patterns[1] = __float_as_uint(v.y), patterns[2] = __float_as_uint(v.z), patterns[3] = __float_as_uint(v.w);
    };
    auto add = [&](bool there, unsigned pattern) __attribute__((always_inline)) {
      const bool cuts = at_cut(pattern);
      add_equal_together(there && (cuts || (second && at_u(pattern))), pattern, (cuts ? 0u : SAMPLE_BINS) + (pattern & (SAMPLE_BINS - 1)), sums, counts);
    };
    for (int i = t; i < 2 * SAMPLE_BINS; i += T) sums[i] = 0ull, counts[i] = 0u;
    if (t == 0) found = 0u;
    __syncthreads();
    of_part([&](const float4& v, int quad, bool there) __attribute__((always_inline)) {
      unsigned patterns[4];
      patterns_of(v, patterns);
      bool any = false;
#pragma unroll
      for (int j = 0; j < 4; ++j) any |= at_cut(patterns[j]) || at_u(patterns[j]);
      if (__ballot(there && any) == 0ull || !there) return;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (quad * 4 + j >= vocab || !(at_cut(patterns[j]) || at_u(patterns[j]))) continue;
        const unsigned at = atomicAdd(&found, 1u);
        if (at < SAMPLE_FEW) stage[at] = make_uint2(patterns[j], (unsigned)(quad * 4 + j));
      }
    });
    __syncthreads();
    const unsigned here = found;
    if (here <= SAMPLE_FEW) {
      for (unsigned i = t; i < SAMPLE_FEW; i += T) add(i < here, i < here ? stage[i].x : 0u);
    } else {  // (equal entries, a thousand of them)
      of_part([&](const float4& v, int quad, bool there) __attribute__((always_inline)) {
        unsigned patterns[4];
        patterns_of(v, patterns);
#pragma unroll
        for (int j = 0; j < 4; ++j) add(there && quad * 4 + j < vocab, patterns[j]);
      });
    }
    unsigned all = here;
    const uint2* few = stage;
    if (gridDim.y > 1) {
      if (t == 0 && here > 0u) place = atomicAdd(&row.found, min(here, SAMPLE_FEW + 1u));
      __syncthreads();
      if (here <= SAMPLE_FEW)
        for (unsigned i = t; i < here; i += T)
          if (place + i < SAMPLE_FEW) row.few[place + i] = stage[i];
      give_histogram(sums, counts, 2 * SAMPLE_BINS, row.run_sums[0], row.run_counts[0]);
      // The part that is done last goes on, with what all have left: every wave's writes have ended and are out of its chiplet's cache before the
      // part counts itself done, and nothing of it is read before the last one is.  Nobody waits for another part.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (t == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        place = atomicAdd(&row.done, 1u);
      }
      __syncthreads();
      if (place != gridDim.y - 1) return;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      for (int i = t; i < 2 * SAMPLE_BINS; i += T) sums[i] = row.run_sums[0][i], counts[i] = row.run_counts[0][i];
      all = row.found;
      few = row.few;
    }
    from_row = all > SAMPLE_FEW;
    __syncthreads();
    keep(few, from_row ? 0 : (int)all);
  }
  // The cut value: everything above it is kept, and of the entries equal to it as many as still
  // start below the bound (engine.py:34-37).  Then the chosen value: the smallest one whose preceding mass is <= target.
  // (one copy of the searches' code for both, which the second finds in the instruction cache)
  unsigned cut = 0u, equal_at_cut = 0u, chosen = 0u, equal = 0u;
  double above_cut = 0.0, above_chosen = 0.0, kept_at_cut = 0.0, target = 0.0;
#pragma unroll 1
  for (int search = 0; search < 2; ++search) {
    int level = 1, made = -1;  // where the last level is made already
    if (search == 0) {
      chosen = (unsigned)c.cut_bin << level_shift(0), above_chosen = c.above_cut;
      if (c.many) chosen = cut_run << level_shift(1), above_chosen = above_run, made = 0;
    } else {
      const int bin = lowest_bin<T>(first_above, target, false, &before_lowest);
      if (bin < c.cut_bin) break;
      chosen = (unsigned)bin << level_shift(0), above_chosen = first_above[bin];
      const int slot = c.many ? c.slot(bin) : -1;
      if (slot >= 0) {
        const unsigned run = fine_run(bin, slot, target, above_chosen);
        chosen = run << level_shift(1), level = 2;
        made = run == cut_run ? 0 : run == first_run && run == last_run ? SAMPLE_BINS : -1;
      }
      // (rounding may put the target outside what was listed)
      const unsigned run = chosen >> level_shift(1);
      if (c.many ? made < 0 && (run < first_run || (slot >= 0 ? run : run | (SAMPLE_BINS - 1)) > last_run) : !c.has((unsigned)bin)) from_row = true;
    }
    __syncthreads();
    if (made >= 0) level_of(sums + made, chosen, 2, above_chosen, search == 0 ? c.limit : target, search == 0);
    else searched(chosen, level, above_chosen, search == 0 ? c.limit : target, search == 0);
    equal = counts[max(made, 0) + (int)(chosen & (SAMPLE_BINS - 1))];
    if (search == 0) {
      cut = chosen, above_cut = above_chosen, equal_at_cut = equal;
      const double cut_value = (double)__uint_as_float(cut), count_at_cut = (double)equal_at_cut;
      kept_at_cut = count_at_cut;
      if (cut_value > 0.0) kept_at_cut = fmin(count_at_cut, ceil((c.limit - above_cut) / cut_value));
      if (kept_at_cut < 1.0) kept_at_cut = 1.0;
      target = u * (above_cut + kept_at_cut * cut_value);
    }
  }
  if (chosen < cut) {  // never below the cut
    chosen = cut;
    above_chosen = above_cut;
    equal = equal_at_cut;
  }
  if (equal == 0u) return;  // no entry has the chosen value: the argmax stands
  const double chosen_value = (double)__uint_as_float(chosen);
  double which = chosen_value > 0.0 ? floor((target - above_chosen) / chosen_value) : 0.0;
  if (which < 0.0) which = 0.0;
  if (chosen == cut && which > kept_at_cut - 1.0) which = kept_at_cut - 1.0;
  // rounding may put the target past the last equal entry: then that one
  int rank = which > (double)(equal - 1) ? (int)equal - 1 : (int)which;
  if (equal == 1u) {
    each([&](unsigned pattern, int index) {
      if (pattern == chosen) *out = index;
    });
    return;
  }
  // the entry of that rank among the equal ones in index order
  if (from_row) {
    // thousands of them: how many a wave's contiguous share of the row holds, then in the share of the one with the entry how many a thread's
    const int wave = t / WAVE, quads = (vocab + 3) / 4, a_wave = (quads + T / WAVE - 1) / (T / WAVE);
    int begin = min(quads, wave * a_wave), end = min(quads, begin + a_wave), mine = 0;
#pragma unroll 1
    for (int first = begin; first < end; first += 8 * WAVE) {
      float4 v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = ((const float4*)p)[min(first + k * WAVE + lane, end - 1)];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int quad = first + k * WAVE + lane;
        const int equal_here = (__float_as_uint(v[k].x) == chosen) + (quad * 4 + 1 < vocab && __float_as_uint(v[k].y) == chosen) +
                               (quad * 4 + 2 < vocab && __float_as_uint(v[k].z) == chosen) + (quad * 4 + 3 < vocab && __float_as_uint(v[k].w) == chosen);
        mine += quad < end ? equal_here : 0;
      }
    }
    int before = block_sum_before_int(mine, scan);  // (of all lanes of the waves before, and of this wave's lanes before)
    before = __shfl(before, 0, WAVE);
#pragma unroll
    for (int offset = WAVE / 2; offset > 0; offset >>= 1) mine += __shfl_xor(mine, offset, WAVE);
    if (lane == 0 && before <= rank && rank < before + mine) lowest = wave, before_lowest = before;
    __syncthreads();
    begin = (int)min((long)vocab, (long)lowest * a_wave * 4), end = (int)min((long)vocab, (long)begin + (long)a_wave * 4), rank -= before_lowest;
    const int a_thread = (end - begin + T - 1) / T, from = min(end, begin + t * a_thread), to = min(end, from + a_thread);
    mine = 0;
    for (int i = from; i < to; ++i) mine += __float_as_uint(p[i]) == chosen ? 1 : 0;
    before = block_sum_before_int(mine, scan);
    if (before <= rank && rank < before + mine)
      for (int i = from, seen = before; i < to; ++i)
        if (__float_as_uint(p[i]) == chosen && seen++ == rank) *out = i;
    return;
  }
  // their indices ten bits at a time, from the highest
  int shift = 0, prefix = 0;
  while (shift + SAMPLE_LEVEL_BITS < 31 && (vocab - 1) >> (shift + SAMPLE_LEVEL_BITS) != 0) shift += SAMPLE_LEVEL_BITS;
#pragma unroll 1
  for (; shift >= 0; shift -= SAMPLE_LEVEL_BITS) {
    __syncthreads();
    counts[t] = 0u;
    __syncthreads();
    each([&](unsigned pattern, int index) {
      if (pattern != chosen || (shift + SAMPLE_LEVEL_BITS < 31 && index >> (shift + SAMPLE_LEVEL_BITS) != prefix)) return;
      const int bin = (index >> shift) & (SAMPLE_BINS - 1);
      const unsigned long long here = __ballot(1), same = __ballot(bin == __builtin_amdgcn_readfirstlane(bin));
      if (same != here) atomicAdd(counts + bin, 1u);
      else if (lane == __ffsll((long long)here) - 1) atomicAdd(counts + bin, (unsigned)__popcll(here));
    });
    __syncthreads();
    const int here = (int)counts[t], before = block_sum_before_int(here, scan);
    if (before <= rank && rank < before + here) {  // one thread
      lowest = t;
      before_lowest = before;
    }
    __syncthreads();
    prefix = (prefix << SAMPLE_LEVEL_BITS) | lowest;
    rank -= before_lowest;
  }
  if (t == 0) *out = prefix;
}

// The token of every row with a temperature.  `out` holds the argmax already.  A block a row, and WITH_TOP_P (rows may have top_p < 1) as many
// parts of a row as the grid has, of which a row with many candidates needs more than the first.
template <bool WITH_TOP_P>
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_pick_kernel(const float* __restrict__ temperatures,
                                                                     const float* __restrict__ top_ps,
                                                                     const float* __restrict__ uniforms,
                                                                     SampleBuffers buffers, int* __restrict__ out,
                                                                     int vocab, int pieces) {
  __shared__ double sd[17];
  __shared__ int owner_piece, owner_thread;
  __shared__ double before_piece, shared_target;
  const int r = blockIdx.x;
  if (temperatures[r] <= 0.f) return;  // engine.py:30-31
  const float* p = buffers.p + r * buffers.stride;
  const float top_p = top_ps[r];
  const int per_piece = (vocab + pieces - 1) / pieces;
  const int lane = threadIdx.x % WAVE;

  if (WITH_TOP_P && !(top_p >= 1.f)) {
    sample_top_p(buffers, r, uniforms[r], vocab, out + r);
    return;
  }
  if (blockIdx.y > 0) return;
  // inverse CDF in index order: the piece first, from the pieces' sums, then inside it
  if (threadIdx.x == 0) owner_thread = 0x7fffffff;
  if (threadIdx.x < WAVE) {  // a lane per piece
    const double sum = lane < pieces ? buffers.piece_sums[r * pieces + lane] : 0.0;
    double inclusive = sum;
#pragma unroll
    for (int offset = 1; offset < WAVE; offset <<= 1) {
      const double other = __shfl_up(inclusive, offset, WAVE);
      if (lane >= offset) inclusive += other;
    }
    const double total = __shfl(inclusive, WAVE - 1, WAVE);
    const double target = (double)uniforms[r] * total;
    const double from_below = __shfl_up(inclusive, 1, WAVE);  // every lane takes part in it
    const double before = lane == 0 ? 0.0 : from_below;
    const unsigned long long holds = __ballot(lane < pieces && before + sum > target);
    const int owner = holds != 0ull ? __ffsll((long long)holds) - 1 : -1;
    if (lane == (owner < 0 ? 0 : owner)) {
      owner_piece = owner;
      before_piece = before;
      shared_target = target;
    }
  }
  __syncthreads();
  if (owner_piece < 0) {
    if (threadIdx.x == 0) out[r] = vocab - 1;
    return;
  }
  const double target = shared_target;
  const int begin = min(vocab, owner_piece * per_piece), end = min(vocab, begin + per_piece);
  const int per = (end - begin + blockDim.x - 1) / blockDim.x;  // each thread owns a contiguous run
  const int b = min(end, begin + (int)threadIdx.x * per), e = min(end, b + per);
  double mine = 0.0;
  for (int i = b; i < e; ++i) mine += (double)p[i];
  const double before = before_piece + block_sum_before_f64(mine, sd);
  if (before + mine > target) atomicMin(&owner_thread, (int)threadIdx.x);
  __syncthreads();
  if (owner_thread == 0x7fffffff) {  // rounding put the target past the piece's end
    if (threadIdx.x == 0) out[r] = end - 1;
  } else if ((int)threadIdx.x == owner_thread) {
    double running = before;
    int found = e - 1;
    for (int i = b; i < e; ++i) {
      running += (double)p[i];
      if (running > target) { found = i; break; }
    }
    out[r] = found;
  }
}

static size_t rounded(size_t bytes) { return (bytes + 255) / 256 * 256; }

struct SampleWorkspace {
  size_t stride, p, piece_sums, piece_values, piece_indices, plain_bytes, rows, bytes;  // (what only rows with top-p need comes last)
};

static SampleWorkspace sample_workspace(int rows, int vocab) {
  const size_t pieces = sample_pieces(rows, false);
  SampleWorkspace w;
  size_t at = 0;
  w.stride = ((size_t)vocab + 3) / 4 * 4;
  w.p = at, at += rounded((size_t)rows * w.stride * sizeof(float));
  w.piece_sums = at, at += rounded((size_t)rows * pieces * sizeof(double));
  w.piece_values = at, at += rounded((size_t)rows * ARGMAX_PIECES * sizeof(float));
  w.piece_indices = at, at += rounded((size_t)rows * ARGMAX_PIECES * sizeof(int));
  w.plain_bytes = at;
  w.rows = at, at += rounded((size_t)rows * sizeof(SampleRow));
  w.bytes = at;
  return w;
}

// The size, in KiB, of the workspace that llmserve_sample needs for these sizes; -1 if they are not positive.
extern "C" int llmserve_sample_workspace_kib(int rows, int vocab) {
  if (rows <= 0 || vocab <= 0) return -1;
  return (int)((sample_workspace(rows, vocab).bytes + 1023) / 1024);
}

// The same with with_top_p = 0: 0.6 MB a row of 151,936, with top-p 0.08 more.
extern "C" int llmserve_sample_plain_workspace_kib(int rows, int vocab) {
  if (rows <= 0 || vocab <= 0) return -1;
  return (int)((sample_workspace(rows, vocab).plain_bytes + 1023) / 1024);
}

// out[r]: the token of row r.  workspace: 256-byte aligned device memory of llmserve_sample_workspace_kib
// KiB, overwritten.  with_top_p = 0 promises that no row with a temperature has top_p < 1, leaves the
// searches out, and needs llmserve_sample_plain_workspace_kib KiB alone.
extern "C" int llmserve_sample(const float* logits, const float* temperatures, const float* top_ps,
                               const float* uniforms, void* workspace, int workspace_kib, int* out, int rows,
                               int vocab, int with_top_p, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (vocab <= 0 || workspace == nullptr || ((size_t)workspace & 255) != 0) return ERR_BAD_ARGUMENT;
  const SampleWorkspace w = sample_workspace(rows, vocab);
  if ((size_t)workspace_kib * 1024 < (with_top_p ? w.bytes : w.plain_bytes)) return ERR_BAD_ARGUMENT;
  unsigned char* base = (unsigned char*)workspace;
  float* piece_values = (float*)(base + w.piece_values);
  int* piece_indices = (int*)(base + w.piece_indices);
  SampleRow* of_rows = with_top_p ? (SampleRow*)(base + w.rows) : nullptr;
  const SampleBuffers buffers = {(float*)(base + w.p), w.stride, (double*)(base + w.piece_sums), of_rows, piece_values, piece_indices};
  const int first_pieces = argmax_pieces(rows), pieces = sample_pieces(rows, with_top_p != 0);
  static_assert(sizeof(SampleRow) % 8 == 0 && SAMPLE_CLEARED % sizeof(unsigned) == 0, "rows lie side by side");
  hipLaunchKernelGGL(argmax_pieces_kernel, dim3(rows, first_pieces), dim3(SAMPLE_THREADS), 0, stream, logits,
                     piece_values, piece_indices, vocab, first_pieces, (unsigned*)of_rows, sizeof(SampleRow) / sizeof(unsigned),
                     (int)(SAMPLE_CLEARED / sizeof(unsigned)));
  hipLaunchKernelGGL(sample_exp_kernel, dim3(rows, pieces), dim3(SAMPLE_BLOCK), 0, stream, logits, temperatures, top_ps,
                     buffers, out, rows, vocab, pieces, first_pieces, with_top_p);
  if (with_top_p) {
    hipLaunchKernelGGL(sample_list_kernel, dim3(rows, pieces), dim3(SAMPLE_BLOCK), 0, stream, temperatures, top_ps, uniforms, buffers, vocab, pieces);
    hipLaunchKernelGGL(sample_pick_kernel<true>, dim3(rows, pick_parts(rows)), dim3(SAMPLE_THREADS), 0, stream, temperatures, top_ps, uniforms,
                       buffers, out, vocab, pieces);
  } else {
    hipLaunchKernelGGL(sample_pick_kernel<false>, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, temperatures, top_ps, uniforms, buffers, out, vocab,
                       pieces);
  }
  return LAUNCH_STATUS();
}
