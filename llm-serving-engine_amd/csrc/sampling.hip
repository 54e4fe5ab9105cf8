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
// `zero` (may be null): `zero_words` words that the launch clears, for whoever runs after it.
__global__ __launch_bounds__(SAMPLE_THREADS) void argmax_pieces_kernel(const float* __restrict__ logits,
                                                                       float* __restrict__ piece_values,
                                                                       int* __restrict__ piece_indices, int vocab,
                                                                       int pieces, unsigned* __restrict__ zero,
                                                                       size_t zero_words) {
  __shared__ float sv[17];
  __shared__ int si[17];
  if (zero != nullptr) {
    const size_t block = (size_t)blockIdx.y * gridDim.x + blockIdx.x, blocks = (size_t)gridDim.x * gridDim.y;
    for (size_t i = block * blockDim.x + threadIdx.x; i < zero_words; i += blocks * blockDim.x) zero[i] = 0u;
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
                     piece_values, piece_indices, vocab, pieces, (unsigned*)nullptr, (size_t)0);
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
                     piece_values, piece_indices, vocab, pieces, (unsigned*)nullptr, (size_t)0);
  hipLaunchKernelGGL(argmax_pick_kernel, dim3(rows), dim3(WAVE), 0, stream, piece_values, piece_indices, out, pieces);
  return LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------------------
// Sampling with a temperature and top-p.
//
// Every launch but the last cuts a row into `pieces` contiguous pieces, a block a (row, piece), so that a few rows of a large
// vocabulary use the whole chip: the row's argmax; p and its sums; with top-p, the entries that the choice is among.  In the last one
// a block a row chooses the token.
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
// first bound and the end of that bin beyond it.  The third launch lists those entries (of a row of 151,936 some
// thousands), the row's block has them in registers and does all levels by itself.  A launch a level, of many blocks a row, took 8.6 us for
// each of the four levels behind the first, most of it launch, trips to memory and atomic additions: 1 / 8 / 16 / 32 / 64
// rows of 151,936 with top-p 45.1 / 54.4 / 62.0 / 71.7 / 97.6 -> 30.1 / 38.1 / 45.0 / 48.6 / 64.4 us; logits of a third of the spread at
// temperature 1.5, which list some twenty thousand, 46.8 / 55.2 / 63.7 / 76.4 / 102.8 -> 46.3 / 53.6 / 63.1 / 68.3 / 83.2; rows of
// nothing but equal entries, which list all, 63 / 87 / 131 / 215 / 381 -> 130 / 141 / 143 / 159 / 220.  What is left is four launches that wait for one another.
//
// The entries of a bin share their exponent (it lies in the ten bits that are fixed first), so their
// sum is 2^exponent times the sum of their 24-bit significands, an integer below 2^42: a bin's mass is
// kept as that integer.  Integer sums do not depend on their order, so threads and blocks add into
// one histogram with atomic additions and the result is the same on every run.

#define SAMPLE_BLOCK 512  // threads of a block that works on a piece of a row
#define SAMPLE_BINS 1024
#define SAMPLE_LEVEL_BITS 10
#define SAMPLE_PIECES_MAX 64  // a wave looks at a row's pieces, a lane at each
#define SAMPLE_KEPT 8         // listed entries that a thread of the row's block keeps in registers; further ones are read again at every level

// About 512 blocks of 512 threads in all for top-p, where every piece adds its bins to the row's with atomic additions of
// its own (64 rows: 98 us, 110 with twice as many; 16 rows 61 and 81; 256 threads and 2,048 blocks 121 and 69), and twice as
// many without, where more blocks only hide more of the trips to memory (64 rows: 38 us and 43).
static int sample_pieces(int rows, bool with_top_p) {
  int pieces = SAMPLE_PIECES_MAX;
  while (pieces > 4 && rows * pieces > (with_top_p ? 512 : 1024)) pieces /= 2;
  return pieces;
}

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
__device__ void masses_above(const unsigned long long* sums, unsigned base, int level, double start, double* above, double* waves) {
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

// Which bins of the first histogram a row's choice is among, and the bound at which its kept set ends.
struct Candidates {
  double limit;                     // top_p * Z
  int cut_bin, first_bin, last_bin;  // the kept set ends in the first of them, u falls in one of the run between the others
  __device__ __forceinline__ bool has(unsigned bin) const {
    return bin == (unsigned)cut_bin || (bin >= (unsigned)first_bin && bin <= (unsigned)last_bin);
  }
};

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

__device__ __forceinline__ void add_entry(float value, unsigned bucket, int shift, unsigned long long* lds_sums, unsigned* lds_counts) {
  const unsigned pattern = __float_as_uint(value);
  if ((pattern >> (shift + SAMPLE_LEVEL_BITS)) == bucket) {
    const unsigned bin = (pattern >> shift) & (SAMPLE_BINS - 1);
    atomicAdd(lds_sums + bin, significand_of(pattern));
    atomicAdd(lds_counts + bin, 1u);
  }
}

// Adds what the block has gathered of its piece to the row's histogram (a barrier before).
__device__ __forceinline__ void give_histogram(const unsigned long long* lds_sums, const unsigned* lds_counts,
                                               unsigned long long* __restrict__ sums, unsigned* __restrict__ counts) {
  for (int bin = threadIdx.x; bin < SAMPLE_BINS; bin += blockDim.x) {
    const unsigned count = lds_counts[bin];
    if (count != 0u) {
      atomicAdd(sums + bin, lds_sums[bin]);
      atomicAdd(counts + bin, count);
    }
  }
}

// The layout of what the launches share, per row: the first histogram (cleared by the first launch), p and its pieces' sums.
struct SampleBuffers {
  float* p;                     // [rows, vocab]
  double* piece_sums;           // [rows, pieces]
  unsigned long long* sums;     // [rows, SAMPLE_BINS]
  unsigned* counts;             // [rows, SAMPLE_BINS]
  unsigned* listed;             // [rows]: how many entries are listed (cleared by the first launch)
  uint2* list;                  // [rows, vocab]: pattern and index of each, in no order
  Candidates* candidates;       // [rows]
  const float* piece_values;    // [rows, argmax_pieces]
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
  float* p = buffers.p + (size_t)r * vocab;
  const int per = (vocab + pieces - 1) / pieces;
  const int begin = min(vocab, piece * per), end = min(vocab, begin + per);
  const bool with_histogram = with_top_p && top_ps[r] < 1.f;
  const float top_logit = row[best_index] / temperature;
  double partial = 0.0;
  for (int first = begin + threadIdx.x; first < end; first += SAMPLE_BATCH * SAMPLE_BLOCK) {
    const Batch batch = load_batch(row, first, end);
#pragma unroll
    for (int u = 0; u < SAMPLE_BATCH; ++u) {
      const int i = first + u * SAMPLE_BLOCK;
      if (i >= end) break;
      const float v = expf(batch.v[u] / temperature - top_logit);
      p[i] = v;
      partial += (double)v;
      if (with_histogram) add_entry(v, 0u, level_shift(0), lds_sums, lds_counts);
    }
  }
  const double sum = block_sum_f64(partial, sd);  // (its barriers stand between the additions and what reads them)
  if (threadIdx.x == 0) buffers.piece_sums[r * pieces + piece] = sum;
  if (!with_histogram) return;
  give_histogram(lds_sums, lds_counts, buffers.sums + (size_t)r * SAMPLE_BINS, buffers.counts + (size_t)r * SAMPLE_BINS);
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

// Lists the entries that the choice of a row with top-p is among: a block takes its piece's.
__global__ __launch_bounds__(SAMPLE_BLOCK) void sample_list_kernel(const float* __restrict__ temperatures, const float* __restrict__ top_ps,
                                                                   const float* __restrict__ uniforms, SampleBuffers buffers, int vocab,
                                                                   int pieces) {
  __shared__ double above[SAMPLE_BINS], waves[SAMPLE_BLOCK / WAVE], sums_here[SAMPLE_PIECES_MAX];
  __shared__ int lowest;
  __shared__ unsigned found, place;
  const int r = blockIdx.x, piece = blockIdx.y, t = threadIdx.x;
  const float top_p = top_ps[r];
  if (temperatures[r] <= 0.f || top_p >= 1.f) return;
  const int per = (vocab + pieces - 1) / pieces;
  const int begin = min(vocab, piece * per), end = min(vocab, begin + per);
  const float* p = buffers.p + (size_t)r * vocab;
  Batch batch = load_batch(p, begin + t, end);  // under way while the histogram is looked at
  if (t < pieces) sums_here[t] = buffers.piece_sums[r * pieces + t];  // a thread a piece asks, then everybody adds them in order
  if (t == 0) found = 0u;
  masses_above<SAMPLE_BLOCK>(buffers.sums + (size_t)r * SAMPLE_BINS, 0u, 0, 0.0, above, waves);
  double total = 0.0;
  for (int q = 0; q < pieces; ++q) total += sums_here[q];
  Candidates c;
  // the bound is strict, so a bound of 0 would be met nowhere: the least positive one keeps the maximum alone
  c.limit = fmax((double)top_p * total, 2.2250738585072014e-308);
  c.cut_bin = lowest_bin<SAMPLE_BLOCK>(above, c.limit, true, &lowest);
  // the kept mass is at least the bound, and beyond it by less than a value of that bin (up to rounding, which the row's block sees to)
  const double end_of_bin = (double)__uint_as_float((unsigned)(c.cut_bin + 1) << level_shift(0)), u = (double)uniforms[r];
  __syncthreads();
  c.first_bin = lowest_bin<SAMPLE_BLOCK>(above, u * (c.limit + end_of_bin), false, &lowest);
  __syncthreads();
  c.last_bin = lowest_bin<SAMPLE_BLOCK>(above, u * c.limit, false, &lowest);
  if (piece == 0 && t == 0) buffers.candidates[r] = c;
  // count them, ask for a place in the row's list, and write them there
  auto taken = [&](int i, float v) { return i < end && c.has(__float_as_uint(v) >> level_shift(0)); };
  unsigned mine = 0u;
  for (int first = begin + t; first < end; first += SAMPLE_BATCH * SAMPLE_BLOCK) {
    if (first != begin + t) batch = load_batch(p, first, end);
#pragma unroll
    for (int k = 0; k < SAMPLE_BATCH; ++k) mine += taken(first + k * SAMPLE_BLOCK, batch.v[k]) ? 1u : 0u;
  }
  if (mine != 0u) mine = atomicAdd(&found, mine);  // (where this thread's begin)
  __syncthreads();
  if (found == 0u) return;
  if (t == 0) place = atomicAdd(buffers.listed + r, found);
  __syncthreads();
  uint2* list = buffers.list + (size_t)r * vocab + place;
  const bool again = begin + SAMPLE_BATCH * SAMPLE_BLOCK < end;  // more than one batch: the first is not here any more
  for (int first = begin + t; first < end; first += SAMPLE_BATCH * SAMPLE_BLOCK) {
    if (again) batch = load_batch(p, first, end);
#pragma unroll
    for (int k = 0; k < SAMPLE_BATCH; ++k) {
      const int i = first + k * SAMPLE_BLOCK;
      if (taken(i, batch.v[k])) list[mine++] = make_uint2(__float_as_uint(batch.v[k]), (unsigned)i);
    }
  }
}

// The token of a row with top-p (out holds the argmax already), by the row's block; see the head of this section.
__device__ void sample_top_p(const SampleBuffers& buffers, int r, float uniform, int vocab, int* __restrict__ out) {
  __shared__ double above[SAMPLE_BINS], first_above[SAMPLE_BINS], waves[SAMPLE_THREADS / WAVE];
  __shared__ unsigned long long sums[SAMPLE_BINS];
  __shared__ unsigned counts[SAMPLE_BINS];
  __shared__ int lowest, before_lowest, scan[17];
  const int t = threadIdx.x, lane = t % WAVE;
  const float* p = buffers.p + (size_t)r * vocab;
  const uint2* list = buffers.list + (size_t)r * vocab;
  const int n = (int)buffers.listed[r];
  const Candidates c = buffers.candidates[r];
  uint2 kept[SAMPLE_KEPT];
#pragma unroll
  for (int k = 0; k < SAMPLE_KEPT; ++k) kept[k] = t + k * SAMPLE_THREADS < n ? list[t + k * SAMPLE_THREADS] : make_uint2(~0u, 0u);
  masses_above<SAMPLE_THREADS>(buffers.sums + (size_t)r * SAMPLE_BINS, 0u, 0, 0.0, first_above, waves);
  bool listed = true;  // whether the entries that a search looks at are in the list
  // calls f(pattern, index) for every entry, of the list (and for none, whose pattern is no entry's) or of the row
  auto each = [&](auto f) {
    if (listed) {
#pragma unroll
      for (int k = 0; k < SAMPLE_KEPT; ++k) f(kept[k].x, (int)kept[k].y);
      for (int first = t + SAMPLE_KEPT * SAMPLE_THREADS; first < n; first += SAMPLE_KEPT * SAMPLE_THREADS) {
        uint2 more[SAMPLE_KEPT];
#pragma unroll
        for (int k = 0; k < SAMPLE_KEPT; ++k) more[k] = list[min(first + k * SAMPLE_THREADS, n - 1)];
#pragma unroll
        for (int k = 0; k < SAMPLE_KEPT; ++k) f(first + k * SAMPLE_THREADS < n ? more[k].x : ~0u, (int)more[k].y);
      }
    } else {
      for (int first = t; first < vocab; first += SAMPLE_KEPT * SAMPLE_THREADS) {
        float more[SAMPLE_KEPT];
#pragma unroll
        for (int k = 0; k < SAMPLE_KEPT; ++k) more[k] = p[min(first + k * SAMPLE_THREADS, vocab - 1)];
#pragma unroll
        for (int k = 0; k < SAMPLE_KEPT; ++k)
          f(first + k * SAMPLE_THREADS < vocab ? __float_as_uint(more[k]) : ~0u, first + k * SAMPLE_THREADS);
      }
    }
  };
  // levels 1 and 2 of a search, inside the bucket of the first level that begins at `base`, `mass` above it: the value's pattern, and the mass above it
  auto searched = [&](unsigned base, double& mass, double bound, bool strict) {
    for (int level = 1; level <= 2; ++level) {
      __syncthreads();
      sums[t] = 0ull;
      counts[t] = 0u;
      __syncthreads();
      const int shift = level_shift(level);
      const unsigned bucket = base >> (shift + SAMPLE_LEVEL_BITS);
      each([&](unsigned pattern, int) {
        if ((pattern >> (shift + SAMPLE_LEVEL_BITS)) != bucket) return;
        const unsigned bin = (pattern >> shift) & (SAMPLE_BINS - 1);
        // (equal entries of a wave go together: additions to one place wait for one another)
        const unsigned long long here = __ballot(1), same = __ballot(pattern == (unsigned)__builtin_amdgcn_readfirstlane((int)pattern));
        if (same == here) {
          if (lane == __ffsll((long long)here) - 1) {
            atomicAdd(sums + bin, significand_of(pattern) * (unsigned long long)__popcll(here));
            atomicAdd(counts + bin, (unsigned)__popcll(here));
          }
          return;
        }
        atomicAdd(sums + bin, significand_of(pattern));
        atomicAdd(counts + bin, 1u);
      });
      __syncthreads();
      masses_above<SAMPLE_THREADS>(sums, base, level, mass, above, waves);
      const int bin = lowest_bin<SAMPLE_THREADS>(above, bound, strict, &lowest);
      mass = above[bin];
      base += (unsigned)bin << shift;
    }
    return base;
  };
  // the cut value: everything above it is kept, and of the entries equal to it as many as still
  // start below the bound (engine.py:34-37)
  __syncthreads();
  double above_cut = first_above[c.cut_bin];
  // (a long list may be of one value over and over, as of a row of equal entries: nothing is left to search then)
  bool one_value = n > SAMPLE_KEPT * SAMPLE_THREADS;
  if (one_value) {
    unsigned least = ~0u, most = 0u;
    each([&](unsigned pattern, int) {
      least = min(least, pattern);
      most = max(most, pattern == ~0u ? 0u : pattern);
    });
    if (t < 2) counts[t] = t == 0 ? ~0u : 0u;
    __syncthreads();
    atomicMin(counts, least);
    atomicMax(counts + 1, most);
    __syncthreads();
    one_value = counts[0] == counts[1] && (counts[0] >> level_shift(0)) == (unsigned)c.cut_bin;
  }
  const unsigned cut = one_value ? counts[0] : searched((unsigned)c.cut_bin << level_shift(0), above_cut, c.limit, true);
  const unsigned equal_at_cut = one_value ? (unsigned)n : counts[cut & (SAMPLE_BINS - 1)];
  const double cut_value = (double)__uint_as_float(cut), count_at_cut = (double)equal_at_cut;
  double kept_at_cut = count_at_cut;
  if (cut_value > 0.0) kept_at_cut = fmin(count_at_cut, ceil((c.limit - above_cut) / cut_value));
  if (kept_at_cut < 1.0) kept_at_cut = 1.0;
  const double target = (double)uniform * (above_cut + kept_at_cut * cut_value);
  // the chosen value: the smallest one whose preceding mass is <= target
  __syncthreads();
  const int chosen_bin = lowest_bin<SAMPLE_THREADS>(first_above, target, false, &lowest);
  listed = c.has((unsigned)chosen_bin);
  double above_chosen = first_above[chosen_bin];
  const bool at_cut = one_value && chosen_bin == c.cut_bin;
  unsigned chosen = at_cut ? cut : searched((unsigned)chosen_bin << level_shift(0), above_chosen, target, false);
  unsigned equal = at_cut ? equal_at_cut : counts[chosen & (SAMPLE_BINS - 1)];
  if (chosen < cut) {  // never below the cut
    chosen = cut;
    above_chosen = above_cut;
    equal = equal_at_cut;
    listed = true;
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
  // the entry of that rank among the equal ones in index order: their indices ten bits at a time, from the highest
  int shift = 0, prefix = 0;
  while (shift + SAMPLE_LEVEL_BITS < 31 && (vocab - 1) >> (shift + SAMPLE_LEVEL_BITS) != 0) shift += SAMPLE_LEVEL_BITS;
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

// The token of every row with a temperature: one block per row.  `out` holds the argmax already.  WITH_TOP_P: rows may have top_p < 1.
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
  const float* p = buffers.p + (size_t)r * vocab;
  const float top_p = top_ps[r];
  const int per_piece = (vocab + pieces - 1) / pieces;
  const int lane = threadIdx.x % WAVE;

  if (WITH_TOP_P && !(top_p >= 1.f)) {
    sample_top_p(buffers, r, uniforms[r], vocab, out + r);
    return;
  }
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
  size_t sums, counts, listed, cleared_words;  // these come first: the first launch clears them
  size_t p, piece_sums, list, candidates, piece_values, piece_indices, bytes;
};

static SampleWorkspace sample_workspace(int rows, int vocab) {
  const size_t pieces = sample_pieces(rows, false), bins = (size_t)rows * SAMPLE_BINS;
  SampleWorkspace w;
  size_t at = 0;
  w.sums = at, at += rounded(bins * sizeof(unsigned long long));
  w.counts = at, at += rounded(bins * sizeof(unsigned));
  w.listed = at, at += rounded((size_t)rows * sizeof(unsigned));
  w.cleared_words = at / sizeof(unsigned);
  w.p = at, at += rounded((size_t)rows * vocab * sizeof(float));
  w.piece_sums = at, at += rounded((size_t)rows * pieces * sizeof(double));
  w.list = at, at += rounded((size_t)rows * vocab * sizeof(uint2));
  w.candidates = at, at += rounded((size_t)rows * sizeof(Candidates));
  w.piece_values = at, at += rounded((size_t)rows * ARGMAX_PIECES * sizeof(float));
  w.piece_indices = at, at += rounded((size_t)rows * ARGMAX_PIECES * sizeof(int));
  w.bytes = at;
  return w;
}

// The size, in KiB, of the workspace that llmserve_sample needs for these sizes; -1 if they are not positive.
extern "C" int llmserve_sample_workspace_kib(int rows, int vocab) {
  if (rows <= 0 || vocab <= 0) return -1;
  return (int)((sample_workspace(rows, vocab).bytes + 1023) / 1024);
}

// out[r]: the token of row r.  workspace: 256-byte aligned device memory of llmserve_sample_workspace_kib
// KiB, overwritten.  with_top_p = 0 promises that no row with a temperature has top_p < 1, and leaves the
// searches out.
extern "C" int llmserve_sample(const float* logits, const float* temperatures, const float* top_ps,
                               const float* uniforms, void* workspace, int workspace_kib, int* out, int rows,
                               int vocab, int with_top_p, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (vocab <= 0 || workspace == nullptr || ((size_t)workspace & 255) != 0) return ERR_BAD_ARGUMENT;
  const SampleWorkspace w = sample_workspace(rows, vocab);
  if ((size_t)workspace_kib * 1024 < w.bytes) return ERR_BAD_ARGUMENT;
  unsigned char* base = (unsigned char*)workspace;
  float* piece_values = (float*)(base + w.piece_values);
  int* piece_indices = (int*)(base + w.piece_indices);
  SampleBuffers buffers;
  buffers.p = (float*)(base + w.p);
  buffers.piece_sums = (double*)(base + w.piece_sums);
  buffers.sums = (unsigned long long*)(base + w.sums);
  buffers.counts = (unsigned*)(base + w.counts);
  buffers.listed = (unsigned*)(base + w.listed);
  buffers.list = (uint2*)(base + w.list);
  buffers.candidates = (Candidates*)(base + w.candidates);
  buffers.piece_values = piece_values;
  buffers.piece_indices = piece_indices;
  const int first_pieces = argmax_pieces(rows), pieces = sample_pieces(rows, with_top_p != 0);
  hipLaunchKernelGGL(argmax_pieces_kernel, dim3(rows, first_pieces), dim3(SAMPLE_THREADS), 0, stream, logits,
                     piece_values, piece_indices, vocab, first_pieces, with_top_p ? (unsigned*)base : (unsigned*)nullptr,
                     with_top_p ? w.cleared_words : (size_t)0);
  hipLaunchKernelGGL(sample_exp_kernel, dim3(rows, pieces), dim3(SAMPLE_BLOCK), 0, stream, logits, temperatures, top_ps,
                     buffers, out, rows, vocab, pieces, first_pieces, with_top_p);
  if (with_top_p) {
    hipLaunchKernelGGL(sample_list_kernel, dim3(rows, pieces), dim3(SAMPLE_BLOCK), 0, stream, temperatures, top_ps, uniforms, buffers, vocab, pieces);
    hipLaunchKernelGGL(sample_pick_kernel<true>, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, temperatures, top_ps, uniforms, buffers, out, vocab,
                       pieces);
  } else {
    hipLaunchKernelGGL(sample_pick_kernel<false>, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, temperatures, top_ps, uniforms, buffers, out, vocab,
                       pieces);
  }
  return LAUNCH_STATUS();
}
