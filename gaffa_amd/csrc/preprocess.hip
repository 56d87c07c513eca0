// Batched in-place preprocessing of a DM x time plane on gfx950: uint32 ->
// float conversion, riptide's fast running-median detrend and normalisation
// (preprocessing.cpp:53-145, 212-231; time_series.cpp:50-104).
//
// Kernels (one launch each, all series at once, grid.y = series):
//   scrunch   - low[k] = float(sum_j double(x[k*f + j]) / f), serial FP64 sum
//               per output so the rounding equals the CPU loop
//   median    - exact centred median of an edge-padded window: a workgroup
//               bitonic-sorts (value, padded position) pairs of its tile's
//               union window in LDS, then each output counts members of its
//               own window in sorted order
//   detrend   - FP64 linear interpolation of the low-resolution median back to
//               full resolution (same operation order as the CPU), subtract,
//               write float
//   stats     - the FP64 sum and sum of squares with exactly the roundings of
//               the CPU loop, which adds in sample order, then mean and
//               1/stddev (time_series.cpp:50-77): in parallel from maps of
//               short runs, or, where the sum itself can round, a lane per
//               series
//   normalise - (x - mean) * (1/stddev) in FP64, rounded to float
// Integer-valued inputs (dedispersed sums) make the scrunch sums exact, and
// every other FP operation runs in the CPU's order, so the output is the
// CPU's bit for bit.
#include "common.hpp"

#include <mutex>

#include <cmath>
#include <type_traits>

namespace gaffa_hip {
namespace {

constexpr int kThreads = 256;
constexpr int kDetrendItems = 8;  // samples per thread in detrend/normalise
constexpr int kBlockSamples = kThreads * kDetrendItems;

template <typename T>
__device__ inline float load_as_float(const T* p, uint64_t i) {
  return static_cast<float>(p[i]);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
scrunch_kernel(const T* __restrict__ data, uint64_t stride, uint64_t factor,
               uint64_t m, float* __restrict__ low) {
  const uint64_t k = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const uint64_t series = blockIdx.y;
  if (k >= m) return;
  const T* x = data + series * stride + k * factor;
  double sum = 0.0;
  for (uint64_t j = 0; j < factor; ++j) sum += static_cast<double>(load_as_float(x, j));
  low[series * m + k] = static_cast<float>(sum / static_cast<double>(factor));
}

// uint32 input: each sample is rounded to float (as gaffa converts a uint32
// DM series), which leaves an integer of at most 2^32; the sum of f of them
// is exact in a 64-bit integer, hence equal to the CPU's serial FP64 sum.  A
// workgroup loads whole outputs' samples, kScrunchSpan at most, with coalesced
// loads into LDS, and `lanes` (a power of two) neighbouring lanes sum one
// output.  The read of the plane bounds it: a wave per output left lanes idle
// at f = 38 and had one load in flight each.  128 series x 400k samples, f = 38
// (205 MB): 226 us before, 57 us now, 3.6 TB/s.  Fewer outputs a workgroup where
// kScrunchGroups of them would not be reached: detrending one series of 16384
// samples at f = 2 takes 39 us so, 44 us with 4 full workgroups.
constexpr uint32_t kScrunchSpan = 4096;
constexpr uint32_t kScrunchGroups = 1024;
// Past some factor a wave per output keeps all lanes busy and is the faster one
// where its waves fill the chip: past 256 (whose outputs divide a span), or past 400
// where the plane is large and the spans' longer bursts count.  Detrending, wave per
// output against spans, us: 64 series of 131072 samples at f = 256 66, 65; 309 66, 69;
// 16 of 2^20 at 309 91, 94; 700 86, 92; 64 of 2^20 at 309 305, 302; 512 of 2^22 at 257
// 10770, 10170; 309 10230, 10040; 400 10070, 9960; 600 9700, 9870; one of 2^20 at 309
// (3393 outputs) 43, 44; 1000 (1048 outputs) 42, 41; 3000 (349) 55, 47.
constexpr uint32_t kScrunchWave = 256, kScrunchWaveLarge = 400;
constexpr uint64_t kScrunchLarge = 1ull << 25;  // samples of all series
constexpr uint32_t kScrunchWaveOutputs = 2048;

__global__ void __launch_bounds__(kThreads)
scrunch_u32_kernel(const uint32_t* __restrict__ data, uint64_t stride, uint32_t factor,
                   uint64_t m, uint32_t outputs, uint32_t lanes, float* __restrict__ low) {
  __shared__ uint32_t x[kScrunchSpan];
  const uint64_t k0 = static_cast<uint64_t>(blockIdx.x) * outputs;
  const uint64_t series = blockIdx.y;
  const uint32_t count = static_cast<uint32_t>(min<uint64_t>(outputs, m - k0));
  const uint32_t total = count * factor;
  const uint32_t* src = data + series * stride + k0 * factor;
#pragma unroll
  for (uint32_t e = 0; e < kScrunchSpan; e += kThreads)
    if (e + threadIdx.x < total) x[e + threadIdx.x] = src[e + threadIdx.x];
  __syncthreads();
  const uint32_t part = threadIdx.x & (lanes - 1);
  const uint32_t groups = kThreads / lanes;
  for (uint32_t k1 = 0; k1 < count; k1 += groups) {
    const uint32_t k = k1 + threadIdx.x / lanes;
    uint64_t sum = 0;
    if (k < count)
      for (uint32_t j = part; j < factor; j += lanes)
        sum += static_cast<uint64_t>(static_cast<float>(x[k * factor + j]));
    for (uint32_t off = lanes / 2; off > 0; off /= 2) sum += __shfl_xor(sum, off, 64);
    if (part == 0 && k < count)
      low[series * m + k0 + k] =
          static_cast<float>(static_cast<double>(sum) / static_cast<double>(factor));
  }
}

// The same with one wave per output and a shuffle reduction.
__global__ void __launch_bounds__(kThreads)
scrunch_u32_wide_kernel(const uint32_t* __restrict__ data, uint64_t stride, uint64_t factor,
                        uint64_t m, float* __restrict__ low) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t k = static_cast<uint64_t>(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
  const uint64_t series = blockIdx.y;
  if (k >= m) return;  // wave-uniform
  const uint32_t* x = data + series * stride + k * factor;
  uint64_t sum = 0;
  for (uint64_t j = lane; j < factor; j += 64)
    sum += static_cast<uint64_t>(static_cast<float>(x[j]));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (lane == 0)
    low[series * m + k] = static_cast<float>(static_cast<double>(sum) / static_cast<double>(factor));
}

// Median of every centred window of `window` (odd) points over an
// edge-padded sequence of length m.  SORT >= kThreads + window - 1.
template <int SORT, typename T>
__global__ void __launch_bounds__(kThreads)
median_kernel(const T* __restrict__ src, uint64_t src_stride, uint64_t m,
              uint32_t window, float* __restrict__ med, uint64_t med_stride) {
  __shared__ float key[SORT];
  __shared__ int32_t pos[SORT];
  const uint32_t tid = threadIdx.x;
  const uint64_t series = blockIdx.y;
  const int64_t k0 = static_cast<int64_t>(blockIdx.x) * kThreads;
  const int32_t half = static_cast<int32_t>(window / 2);
  const int32_t span = kThreads + static_cast<int32_t>(window) - 1;
  const T* s = src + series * src_stride;
  for (int32_t e = tid; e < SORT; e += kThreads) {
    if (e < span) {
      const int64_t p = k0 - half + e;  // padded position
      const int64_t idx = p < 0 ? 0 : (p >= static_cast<int64_t>(m) ? static_cast<int64_t>(m) - 1 : p);
      key[e] = load_as_float(s, static_cast<uint64_t>(idx));
      pos[e] = e;
    } else {
      key[e] = INFINITY;
      pos[e] = 0x7fffffff;
    }
  }
  __syncthreads();
  // bitonic sort ascending by key
  for (int32_t size = 2; size <= SORT; size <<= 1) {
    for (int32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (int32_t e = tid; e < SORT / 2; e += kThreads) {
        const int32_t lo = 2 * e - (e & (stride - 1));
        const int32_t hi = lo + stride;
        const bool ascending = (lo & size) == 0;
        const float a = key[lo], b = key[hi];
        if ((a > b) == ascending) {
          key[lo] = b;
          key[hi] = a;
          const int32_t t = pos[lo];
          pos[lo] = pos[hi];
          pos[hi] = t;
        }
      }
      __syncthreads();
    }
  }
  const int64_t k = k0 + tid;
  if (k >= static_cast<int64_t>(m)) return;
  // window of output tid covers padded offsets [tid, tid + window)
  const uint32_t lo = tid;
  int32_t count = 0;
  float value = 0.0f;
  for (int32_t e = 0; e < span; ++e) {
    const uint32_t off = static_cast<uint32_t>(pos[e]) - lo;
    if (off < window) {
      if (count == half) {
        value = key[e];
        break;
      }
      ++count;
    }
  }
  med[series * med_stride + static_cast<uint64_t>(k)] = value;
}

// What the statistics need of one block of samples (see the statistics below).
struct BlockSums {
  double sum;        // of the samples, in any order
  float squares;     // about the sum of squares
  float magnitude;   // no less than the sum of |x|; inf or NaN where a sample is not finite
  int32_t quantum;   // every sample is a multiple of 2^(quantum - 150)
  int32_t exponent;  // block_exponent_kernel: the running sum of squares' exponent
};

// quantum of one sample: the exponent of its lowest set bit.
__device__ __forceinline__ int32_t sample_quantum(float v) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, v) & 0x7FFFFFFFu;
  const int32_t q = static_cast<int32_t>(max(bits >> 23, 1u)) + __builtin_ctz(bits | 0x800000u);
  return bits == 0 ? 4096 : q;
}

// x - interpolated median, written in place as float; a workgroup runs
// kDetrendItems x 256 samples or, for statistics in blocks (kSums), `items` x 256
// and leaves their sums in sums[block].  The sums and the loop over items cost 8 %
// (128 series of 400k uint32 samples converted in 75 us, 81 with them), so callers
// without such statistics have a kernel without.
template <typename T, bool kSums>
__global__ void __launch_bounds__(kThreads)
detrend_kernel(T* __restrict__ data, uint64_t stride, uint64_t n,
               int32_t detrend, uint64_t factor, const float* __restrict__ med,
               uint64_t m, int32_t* __restrict__ status, uint32_t items,
               BlockSums* __restrict__ sums) {
  const uint32_t tid = threadIdx.x;
  const uint64_t series = blockIdx.y;
  T* x = data + series * stride;
  float* out = reinterpret_cast<float*>(x);
  const float* md = med + series * (factor == 1 ? n : m);
  const double offset = 0.5 * static_cast<double>(factor - 1);
  const double fd = static_cast<double>(factor);
  bool bad = false;
  double sum = 0.0;
  float squares = 0.0f, magnitude = 0.0f;
  int32_t quantum = 4096;
  if constexpr (!kSums) items = kDetrendItems;
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * items * kThreads;
  for (uint32_t r0 = 0; r0 < items; r0 += kDetrendItems) {
#pragma unroll
    for (int r = 0; r < kDetrendItems; ++r) {
      const uint64_t i = base + static_cast<uint64_t>(r0 + r) * kThreads + tid;
      if (i >= n) break;
      const float v = load_as_float(x, i);
      bad |= !isfinite(v);
      float d = v;
      if (detrend) {
        float baseline;
        if (factor == 1) {
          baseline = md[i];
        } else {
          const double p = (static_cast<double>(i) - offset) / fd;
          if (p <= 0.0) {
            baseline = md[0];
          } else {
            const uint64_t lo = static_cast<uint64_t>(floor(p));
            if (lo >= m - 1) {
              baseline = md[m - 1];
            } else {
              const double fr = p - static_cast<double>(lo);
              const double w0 = (1.0 - fr) * static_cast<double>(md[lo]);
              const double w1 = fr * static_cast<double>(md[lo + 1]);
              baseline = static_cast<float>(w0 + w1);
            }
          }
        }
        d = v - baseline;
      }
      out[i] = d;
      if constexpr (kSums) {
        sum += static_cast<double>(d);
        squares += d * d;
        magnitude += fabsf(d);
        quantum = min(quantum, sample_quantum(d));
      }
    }
  }
  if (bad) atomicExch(&status[series], 1);
  if constexpr (!kSums) return;
  __shared__ BlockSums part[kThreads / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
    squares += __shfl_xor(squares, off, 64);
    magnitude += __shfl_xor(magnitude, off, 64);
    quantum = min(quantum, __shfl_xor(quantum, off, 64));
  }
  if ((tid & 63u) == 0) part[tid >> 6] = BlockSums{sum, squares, magnitude, quantum, 0};
  __syncthreads();
  if (tid == 0) {
    BlockSums t = part[0];
    for (int w = 1; w < kThreads / 64; ++w) {
      t.sum += part[w].sum;
      t.squares += part[w].squares;
      t.magnitude += part[w].magnitude;
      t.quantum = min(t.quantum, part[w].quantum);
    }
    t.magnitude *= 1.01f;  // past the rounding of its float sum
    sums[series * gridDim.x + blockIdx.x] = t;
  }
}

// Statistics: the sum and sum of squares of each series in FP64 in sample order,
// as time_series_stats_cpu does (time_series.cpp:55-60), so every rounding is the
// CPU's; then mean, 1/stddev and a status flag.
//
// One FP64 add per sample and chain is a chain of n dependent adds, whatever the
// batch: 12 ns a sample in stats_kernel, 12.7 ms at 2^20 samples.  Both sums can
// be had in parallel with the same bits:
//   sum      where every sample is a multiple of some 2^q and the sum of |x| is
//            below 2^53 2^q, no partial sum rounds, in any order.  Detrended
//            integer series are such: x is a difference of multiples of the
//            baseline's last place.
//   squares  the running sum S never falls.  While it stays in one binade
//            [2^k, 2^(k+1)), with last place u, adding q rounds to S + m u where m
//            depends on q and, in a tie, on the parity of S / u alone.  So a run
//            of samples maps a parity to an increment, and such maps compose in
//            any grouping.  Each thread measures its run's two increments by
//            adding it to 2^k and to 2^k + u, with the real FP64 adds.
// detrend_kernel leaves each block's sums, block_exponent_kernel predicts k for
// every block from their prefix sums, square_map_kernel composes each block's
// map, and combine_stats_kernel walks the blocks of a series: it applies a map
// only where S really starts and ends in the map's binade, and else runs the
// block in finer pieces, down to sample by sample around a binade's end.  A batch
// with a series whose sum can round (or a sample that is not finite) is left to
// stats_kernel, whose time hardly depends on the number of series:
// block_exponent_kernel finds it, and neither maps nor walks follow.  Ordinary
// float series round: 64 of 16384 samples take 211 us in the chain alone, took 291
// us with the maps and walks before it, and take 219 us without them.
// The read of the plane bounds square_map_kernel.  Measured, statistics with
// their part of detrend_kernel: 256 series of 2^20 samples 12.7 -> 0.5 ms, 512
// of 2^21 25.1 -> 1.2 ms, 128 of 400k 4.8 -> 0.2 ms.
constexpr uint32_t kMapThreads = 512;
constexpr uint32_t kMapRun = 8;                           // samples per thread and step
constexpr uint32_t kMapBlock = kMapThreads * kMapRun;     // smallest block: 4096 samples
constexpr uint32_t kMapMaxShift = 4;                      // blocks of up to 65536 samples
constexpr int32_t kNoExponent = -1;                       // a block that holds a binade's end
constexpr int32_t kZeroBlock = -2;                        // a block of zeros
constexpr int32_t kSerialStats = INT32_MIN;  // quantum of the batch's first block: left to
                                             // stats_kernel

// The biased exponent of x >= 0 (zero for a zero).
__device__ __forceinline__ int32_t exponent_of(double x) {
  return static_cast<int32_t>(__builtin_bit_cast(uint64_t, x) >> 52);
}
__device__ __forceinline__ double binade(int32_t exponent) {
  return __builtin_bit_cast(double, static_cast<uint64_t>(exponent) << 52);
}
__device__ __forceinline__ bool is_odd(double x) {
  return (__builtin_bit_cast(uint64_t, x) & 1u) != 0;
}
// The exponent that a running sum from `from` to `to` (both about right) keeps.
__device__ __forceinline__ int32_t kept_exponent(double from, double to, double margin) {
  const int32_t lo = exponent_of(from * (1.0 - margin)), hi = exponent_of(to * (1.0 + margin));
  return lo == hi && lo > 53 && hi < 0x7FE ? lo : kNoExponent;
}

// A run's increments of a sum in binade k that starts even (x) or odd (y).
__device__ __forceinline__ double2 compose(double2 f, double2 g, double base) {
  return make_double2(f.x + (is_odd(base + f.x) ? g.y : g.x),
                      f.y + (is_odd(base + f.y) ? g.x : g.y));
}

__device__ __forceinline__ double read_lane(double x, uint32_t lane) {
  const uint64_t bits = __builtin_bit_cast(uint64_t, x);
  const uint64_t lo = static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(bits), static_cast<int>(lane)));
  const uint64_t hi = static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(bits >> 32), static_cast<int>(lane)));
  return __builtin_bit_cast(double, lo | (hi << 32));
}

// sums[b].exponent of every block of a series, and whether its sum can round, a
// wave per series.
__global__ void __launch_bounds__(64)
block_exponent_kernel(BlockSums* sums, uint32_t nblocks) {
  BlockSums* const s = sums + static_cast<uint64_t>(blockIdx.x) * nblocks;
  const uint32_t lane = threadIdx.x;
  double before = 0.0, magnitude = 0.0;
  int32_t quantum = 4096;
  for (uint32_t b0 = 0; b0 < nblocks; b0 += 64) {
    const uint32_t b = b0 + lane;
    const double q = b < nblocks ? static_cast<double>(s[b].squares) : 0.0;
    double upto = q;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double x = __shfl_up(upto, off, 64);
      if (lane >= static_cast<uint32_t>(off)) upto += x;
    }
    if (b < nblocks) {
      s[b].exponent = kept_exponent(before + (upto - q), before + upto, 1e-5);
      magnitude += static_cast<double>(s[b].magnitude);
      quantum = min(quantum, s[b].quantum);
    }
    before += read_lane(upto, 63);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    magnitude += __shfl_xor(magnitude, off, 64);
    quantum = min(quantum, __shfl_xor(quantum, off, 64));
  }
  // multiples of 2^(quantum - 150) that add up to less than 2^53 of them do not
  // round; a magnitude that is not finite fails.  Where another wave's kSerialStats
  // is read as the first series' quantum, that series fails too, to the same end.
  if (lane == 0 && !(magnitude < ldexp(1.0, min(quantum, 400) - 150 + 52)))
    sums->quantum = kSerialStats;
}

// maps[series][block]: the block's increments of the sum of squares.
__global__ void __launch_bounds__(kMapThreads)
square_map_kernel(const float* __restrict__ data, uint64_t stride, uint64_t n, uint32_t run,
                  const BlockSums* __restrict__ sums, double2* __restrict__ maps) {
  const uint64_t block = static_cast<uint64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
  const int32_t k = sums[block].exponent;
  if (k < 0 || sums->quantum == kSerialStats) return;
  const float* x = data + blockIdx.y * stride;
  const uint32_t tid = threadIdx.x;
  const uint64_t i0 = (static_cast<uint64_t>(blockIdx.x) * kMapThreads + tid) * run;
  const double base = binade(k);
  const double odd = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, base) | 1u);
  double a = base, c = odd;
  struct Run {
    float x[kMapRun];
  };
  for (uint32_t r = 0; r < run; r += kMapRun) {
    const uint64_t i = i0 + r;
    if (i + kMapRun <= n) {
      const Run v = *reinterpret_cast<const Run*>(x + i);
#pragma unroll
      for (uint32_t u = 0; u < kMapRun; ++u) {
        const double d = static_cast<double>(v.x[u]);
        const double q = d * d;
        a = a + q;
        c = c + q;
      }
    } else {
      for (uint64_t e = i; e < n; ++e) {
        const double d = static_cast<double>(x[e]);
        const double q = d * d;
        a = a + q;
        c = c + q;
      }
    }
  }
  double2 f = make_double2(a - base, c - odd);
  // runs in order: lane l joins lane l + off, for growing off
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double2 g = make_double2(__shfl_down(f.x, off, 64), __shfl_down(f.y, off, 64));
    f = compose(f, g, base);  // lanes that are not a multiple of 2 off are not read again
  }
  __shared__ double2 part[kMapThreads / 64];
  if ((tid & 63u) == 0) part[tid >> 6] = f;
  __syncthreads();
  if (tid == 0) {
    for (uint32_t w = 1; w < kMapThreads / 64; ++w) f = compose(f, part[w], base);
    maps[block] = f;
  }
}

// A two-wave workgroup owns 64 series, a lane of each wave per series: wave 0
// runs the chain of sums, wave 1 the chain of squares (the two are
// independent, so each wave has one serial chain instead of two and the
// launch twice the waves).  The workgroup loads chunks of 64 series x 128
// samples with coalesced 16-byte loads (two 512-byte row segments per
// instruction) into registers, stores them to LDS, and while each lane adds
// its own row of the chunk in order, the next chunk's loads are already in
// flight.  Rows must be 16-byte aligned (the pipeline's plane is); other
// layouts take the per-lane path, which reads each row directly.
// a native 4-float vector: HIP's float4 struct is copied through memory,
// which would keep a register array of them in scratch
typedef float vf4 __attribute__((ext_vector_type(4)));
constexpr int kStatsLanes = 64;                // series per workgroup
constexpr int kStatsThreads = 2 * kStatsLanes; // one wave per chain
constexpr int kStatsChunk = 128;               // samples per series per chunk
constexpr int kStatsPitch = kStatsChunk + 4;   // LDS floats per row (bank spread)
constexpr int kStatsLoads = kStatsLanes * kStatsChunk / 4 / kStatsThreads;  // float4 per thread
constexpr uint32_t kStatsVecs = kStatsChunk / 4;  // float4 per row of a chunk
constexpr uint32_t kStatsLdsBytes = 2u * kStatsLanes * kStatsPitch * 4u;

struct SerialSums {
  double sum = 0.0, squares = 0.0;
  __device__ __forceinline__ void add(float v) {
    const double x = static_cast<double>(v);
    sum = sum + x;
    squares = squares + x * x;  // separately rounded: the code is built without contraction
  }
  __device__ __forceinline__ void add4(float4 v) {
    add(v.x);
    add(v.y);
    add(v.z);
    add(v.w);
  }
};

// Whether S plus a map's increment is what the adds give: it starts and ends in
// binade k.  Then S becomes it.
__device__ __forceinline__ bool apply_map(double& S, int32_t k, double even, double odd) {
  if (k < 0 || exponent_of(S) != k) return false;
  const double to = S + (is_odd(S) ? odd : even);
  if (exponent_of(to) != k) return false;
  S = to;
  return true;
}

__device__ __forceinline__ void finish_stats(const SerialSums& acc, uint64_t n, uint32_t series,
                                             int32_t reject_constant, double2* stats,
                                             int32_t* flags, int32_t* status) {
  const double count = static_cast<double>(n);
  const double mean = acc.sum / count;
  double var = acc.squares / count - mean * mean;
  if (var < 0.0 && var > -1.0e-12) var = 0.0;
  int32_t flag = 0;
  if (var < 0.0 || !isfinite(var)) flag = 3;
  const double sd = sqrt(var);
  if (flag == 0 && (!(sd > 0.0) || !isfinite(sd))) flag = reject_constant ? 2 : 4;
  stats[series] = make_double2(mean, flag == 0 ? 1.0 / sd : 0.0);
  flags[series] = flag;
  if (flag == 2 || flag == 3) atomicCAS(&status[series], 0, flag);
}

// One wave per series: S over the blocks' maps, finer where a map does not hold.
__global__ void __launch_bounds__(64)
combine_stats_kernel(const float* __restrict__ data, uint64_t stride, uint64_t n,
                     uint32_t nblocks, uint32_t block, const BlockSums* __restrict__ sums,
                     const double2* __restrict__ maps, int32_t reject_constant,
                     double2* __restrict__ stats, int32_t* __restrict__ flags,
                     int32_t* __restrict__ status) {
  const uint32_t series = blockIdx.x;
  const uint32_t lane = threadIdx.x;
  if (sums->quantum == kSerialStats) return;
  const float* x = data + series * stride;
  const BlockSums* const s = sums + static_cast<uint64_t>(series) * nblocks;
  const double2* const f = maps + static_cast<uint64_t>(series) * nblocks;
  SerialSums acc;
  for (uint32_t b = lane; b < nblocks; b += 64) acc.sum += s[b].sum;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc.sum += __shfl_xor(acc.sum, off, 64);
  constexpr uint32_t kRun = 32;  // samples per lane in a block run in finer pieces
  double S = 0.0;
  for (uint32_t b0 = 0; b0 < nblocks; b0 += 64) {
    const uint32_t b = b0 + lane;
    int32_t k = kZeroBlock;
    double2 map = make_double2(0.0, 0.0);
    if (b < nblocks) {
      k = s[b].magnitude == 0.0f ? kZeroBlock : s[b].exponent;
      if (k >= 0) map = f[b];
    }
    const uint32_t count = min(64u, nblocks - b0);
    for (uint32_t l = 0; l < count; ++l) {
      const int32_t kl = __builtin_amdgcn_readlane(k, l);
      if (kl == kZeroBlock) continue;  // adding zeros leaves S as it is
      if (apply_map(S, kl, read_lane(map.x, l), read_lane(map.y, l))) continue;
      const uint64_t first = static_cast<uint64_t>(b0 + l) * block;
      const uint64_t last = min(n, first + block);
      for (uint64_t p = first; p < last; p += 64 * kRun) {
        float v[kRun];
        double own = 0.0;
#pragma unroll
        for (uint32_t j = 0; j < kRun; ++j) {
          const uint64_t i = p + lane * kRun + j;
          v[j] = i < last ? x[i] : 0.0f;
          own += static_cast<double>(v[j]) * static_cast<double>(v[j]);
        }
        double upto = own;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const double y = __shfl_up(upto, off, 64);
          if (lane >= static_cast<uint32_t>(off)) upto += y;
        }
        const int32_t kr = kept_exponent(S + (upto - own), S + upto, 1e-9);
        const double base = binade(max(kr, 0));
        const double odd = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, base) | 1u);
        double a = base, c = odd;
#pragma unroll
        for (uint32_t j = 0; j < kRun; ++j) {
          const double q = static_cast<double>(v[j]) * static_cast<double>(v[j]);
          a = a + q;
          c = c + q;
        }
        a -= base;
        c -= odd;
        for (uint32_t w = 0; w < 64; ++w) {
          if (apply_map(S, __builtin_amdgcn_readlane(kr, w), read_lane(a, w), read_lane(c, w)))
            continue;
#pragma unroll
          for (uint32_t j = 0; j < kRun; ++j) {
            const double d = static_cast<double>(__builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[j]), w)));
            S = S + d * d;
          }
        }
      }
    }
  }
  acc.squares = S;
  if (lane == 0) finish_stats(acc, n, series, reject_constant, stats, flags, status);
}

__global__ void __launch_bounds__(kStatsThreads) __attribute__((amdgpu_waves_per_eu(1, 2)))
stats_kernel(const float* __restrict__ data, uint64_t stride, uint64_t n, uint32_t nseries,
             int32_t reject_constant, double2* __restrict__ stats,
             int32_t* __restrict__ flags, int32_t* __restrict__ status,
             const BlockSums* __restrict__ blocks) {
  if (blocks != nullptr && blocks->quantum != kSerialStats) return;  // combine_stats_kernel's
  extern __shared__ __align__(16) float stage[];  // [2][kStatsLanes][kStatsPitch]
  __shared__ double squares_of[kStatsLanes];
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u;
  const bool squares = tid >= 64u;  // wave-uniform: wave 1 runs the squares
  const uint32_t first = blockIdx.x * kStatsLanes;
  const uint32_t rows = min(static_cast<uint32_t>(kStatsLanes), nseries - first);
  const uint64_t nchunks = n / kStatsChunk;
  const float* base = data + static_cast<uint64_t>(first) * stride;
  // load k of a chunk: element e = k * 128 + tid is row e / kStatsVecs,
  // float4 e % kStatsVecs
  // (rows past the batch re-read the last row); every index is a constant
  // after unrolling, so the chunk stays in registers
  vf4 reg[kStatsLoads];
  double acc = 0.0;
  if (nchunks > 0) {
#pragma unroll
    for (int k = 0; k < kStatsLoads; ++k) {
      const uint32_t e = static_cast<uint32_t>(k) * kStatsThreads + tid;
      const uint32_t r = min(e / kStatsVecs, rows - 1);
      reg[k] = *reinterpret_cast<const vf4*>(base + static_cast<uint64_t>(r) * stride +
                                                4u * (e % kStatsVecs));
    }
  }
  for (uint64_t c = 0; c < nchunks; ++c) {
    const uint32_t buf = static_cast<uint32_t>(c & 1u);
#pragma unroll
    for (int k = 0; k < kStatsLoads; ++k) {
      const uint32_t e = static_cast<uint32_t>(k) * kStatsThreads + tid;
      *reinterpret_cast<vf4*>(stage + (buf * kStatsLanes + e / kStatsVecs) * kStatsPitch +
                                 4u * (e % kStatsVecs)) = reg[k];
    }
    __syncthreads();
    if (c + 1 < nchunks) {  // in flight while this chunk is summed
      const uint64_t col = (c + 1) * kStatsChunk;
#pragma unroll
      for (int k = 0; k < kStatsLoads; ++k) {
        const uint32_t e = static_cast<uint32_t>(k) * kStatsThreads + tid;
        const uint32_t r = min(e / kStatsVecs, rows - 1);
        reg[k] = *reinterpret_cast<const vf4*>(base + static_cast<uint64_t>(r) * stride + col +
                                                  4u * (e % kStatsVecs));
      }
    }
    const vf4* row = reinterpret_cast<const vf4*>(stage + (buf * kStatsLanes + lane) *
                                                  kStatsPitch);
    // eight samples at a time: the conversions (and squares) first,
    // independent of each other, then the in-order add chain, which is all
    // that remains on the critical path
    if (!squares) {
#pragma unroll 2
      for (int j = 0; j < kStatsChunk / 4; j += 2) {
        const vf4 v0 = row[j], v1 = row[j + 1];
        const float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        double d[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) d[u] = static_cast<double>(f[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = acc + d[u];
      }
    } else {
#pragma unroll 2
      for (int j = 0; j < kStatsChunk / 4; j += 2) {
        const vf4 v0 = row[j], v1 = row[j + 1];
        const float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        double q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const double d = static_cast<double>(f[u]);
          q[u] = d * d;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = acc + q[u];
      }
    }
    // the other buffer is rewritten after the next barrier, once both waves
    // are done with it
  }
  // the tail (< 128 samples) of each row, then the squares join the sums
  if (lane < rows) {
    const float* x = base + static_cast<uint64_t>(lane) * stride;
    for (uint64_t i = nchunks * kStatsChunk; i < n; ++i) {
      const double d = static_cast<double>(x[i]);
      acc = squares ? acc + d * d : acc + d;
    }
    if (squares) squares_of[lane] = acc;
  }
  __syncthreads();
  if (squares || lane >= rows) return;
  SerialSums sums;
  sums.sum = acc;
  sums.squares = squares_of[lane];
  finish_stats(sums, n, first + lane, reject_constant, stats, flags, status);
}

// Rows that are not 16-byte aligned: each lane reads its row directly.
__global__ void __launch_bounds__(kStatsLanes)
stats_rowwise_kernel(const float* __restrict__ data, uint64_t stride, uint64_t n,
                     uint32_t nseries, int32_t reject_constant, double2* __restrict__ stats,
                     int32_t* __restrict__ flags, int32_t* __restrict__ status,
                     const BlockSums* __restrict__ blocks) {
  if (blocks != nullptr && blocks->quantum != kSerialStats) return;  // combine_stats_kernel's
  const uint32_t series = blockIdx.x * kStatsLanes + threadIdx.x;
  if (series >= nseries) return;
  const float* x = data + static_cast<uint64_t>(series) * stride;
  SerialSums acc;
  for (uint64_t i = 0; i < n; ++i) acc.add(x[i]);
  finish_stats(acc, n, series, reject_constant, stats, flags, status);
}

__global__ void __launch_bounds__(kThreads)
normalise_kernel(float* __restrict__ data, uint64_t stride, uint64_t n,
                 const double2* __restrict__ stats, const int32_t* __restrict__ flags) {
  const uint32_t tid = threadIdx.x;
  const uint64_t series = blockIdx.y;
  const int32_t flag = flags[series];
  if (flag == 2 || flag == 3) return;  // rejected: data left detrended, status set
  const double mean = stats[series].x, scale = stats[series].y;
  float* x = data + series * stride;
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kBlockSamples;
#pragma unroll
  for (int r = 0; r < kDetrendItems; ++r) {
    const uint64_t i = base + static_cast<uint64_t>(r) * kThreads + tid;
    if (i >= n) break;
    // flag 4: constant input accepted -> zeros (time_series.cpp:90-93)
    x[i] = flag == 4 ? 0.0f
                     : static_cast<float>((static_cast<double>(x[i]) - mean) * scale);
  }
}

uint64_t median_points(uint64_t n, uint64_t factor) { return factor == 1 ? n : n / factor; }

template <typename T>
void launch_median(const T* src, uint64_t src_stride, uint64_t m, uint32_t window,
                   float* med, uint64_t med_stride, uint64_t nseries, hipStream_t st) {
  const dim3 grid(static_cast<uint32_t>(ceil_div(m, kThreads)), static_cast<uint32_t>(nseries));
  const uint32_t span = kThreads + window - 1;
  if (span <= 512) {
    hipLaunchKernelGGL((median_kernel<512, T>), grid, dim3(kThreads), 0, st, src, src_stride, m,
                       window, med, med_stride);
  } else if (span <= 1024) {
    hipLaunchKernelGGL((median_kernel<1024, T>), grid, dim3(kThreads), 0, st, src, src_stride, m,
                       window, med, med_stride);
  } else if (span <= 2048) {
    hipLaunchKernelGGL((median_kernel<2048, T>), grid, dim3(kThreads), 0, st, src, src_stride, m,
                       window, med, med_stride);
  } else {
    hipLaunchKernelGGL((median_kernel<4096, T>), grid, dim3(kThreads), 0, st, src, src_stride, m,
                       window, med, med_stride);
  }
  launch_check("median_kernel");
}

struct Layout {
  uint64_t m, low_floats, med_floats, nblocks, stats_offset,
      flags_offset, total;
};

Layout layout(uint64_t nseries, uint64_t n, uint64_t factor) {
  Layout l{};
  l.m = median_points(n, factor);
  l.low_floats = factor == 1 ? 0 : nseries * l.m;
  l.med_floats = nseries * l.m;
  l.nblocks = ceil_div(n, kBlockSamples);
  l.stats_offset = ((l.low_floats + l.med_floats) * 4 + 255) / 256 * 256;
  l.flags_offset = l.stats_offset + (nseries * sizeof(double2) + 255) / 256 * 256;
  l.total = l.flags_offset + nseries * sizeof(int32_t);
  return l;
}

// Where the parallel statistics keep their blocks: the low-resolution series is
// free once its medians are taken, and the medians once they are subtracted, so
// blocks of kMapBlock << shift samples live there and need no room of their own.
// Off where they do not fit (scrunch factors past 10^4, an exact running median,
// which leaves no low-resolution series) and for short series: stats_kernel then
// runs every series.
struct StatsBlocks {
  bool on = false;
  uint32_t shift = 0;
  uint64_t nblocks = 0;
  BlockSums* sums = nullptr;
  double2* maps = nullptr;
};

StatsBlocks stats_blocks(const gaffa_hip_preprocess_args* a, const Layout& l, void* workspace) {
  StatsBlocks s;
  if (!a->normalise || (a->detrend && a->scrunch_factor == 1)) return s;
  // Three launches more than the chain, which takes 12 ns a sample: chain -> blocks,
  // us, of whole numbers 1 x 1024 samples 21 -> 30, 1024 x 1024 26 -> 35, 1 x 2048
  // 35 -> 32, 1024 x 2048 42 -> 41.  Floats, whose batch may end in the chain: 1024 x
  // 2048 42 -> 55 (there), 1 x 2048 35 -> 35, 1 x 4096 59 -> 44, 1024 x 4096 73 -> 85
  // (there).
  if (a->nsamples < (a->input_is_u32 ? 2048u : 4096u)) return s;
  auto align = [](uint64_t v) { return (v + 15) / 16 * 16; };
  const uint64_t end = (l.low_floats + l.med_floats) * 4;
  for (uint32_t shift = 0; shift <= kMapMaxShift; ++shift) {
    const uint64_t nblocks = ceil_div(a->nsamples, static_cast<uint64_t>(kMapBlock) << shift);
    const uint64_t sums = a->nseries * nblocks * sizeof(BlockSums);
    // the detrend pass reads the medians while it writes the sums
    const uint64_t maps = align(a->detrend ? l.low_floats * 4 : sums);
    if ((a->detrend && sums > l.low_floats * 4) ||
        maps + a->nseries * nblocks * sizeof(double2) > end)
      continue;
    s.on = true;
    s.shift = shift;
    s.nblocks = nblocks;
    s.sums = static_cast<BlockSums*>(workspace);
    s.maps = reinterpret_cast<double2*>(static_cast<char*>(workspace) + maps);
    return s;
  }
  return s;
}

template <typename T>
void run(const gaffa_hip_preprocess_args* a, void* workspace, hipStream_t st) {
  const Layout l = layout(a->nseries, a->nsamples, a->detrend ? a->scrunch_factor : 1);
  float* low = static_cast<float*>(workspace);
  float* med = low + l.low_floats;
  char* ws = static_cast<char*>(workspace);
  double2* stats = reinterpret_cast<double2*>(ws + l.stats_offset);
  int32_t* flags = reinterpret_cast<int32_t*>(ws + l.flags_offset);
  T* data = static_cast<T*>(a->data);
  const uint64_t f = a->scrunch_factor;
  if (a->detrend) {
    if (f > 1) {
      if constexpr (std::is_same_v<T, uint32_t>) {
        const uint64_t all = a->nseries * l.m;
        const uint32_t wave =
            a->nseries * a->nsamples < kScrunchLarge ? kScrunchWave : kScrunchWaveLarge;
        if (f <= kScrunchSpan && (f <= wave || all < kScrunchWaveOutputs)) {
          const uint32_t outputs = static_cast<uint32_t>(std::min<uint64_t>(
              kScrunchSpan / f, std::max<uint64_t>(1, all / kScrunchGroups)));
          uint32_t lanes = 1;  // about one output per group of lanes
          while (lanes < 64 && 2 * lanes * outputs <= kThreads) lanes *= 2;
          const dim3 g(static_cast<uint32_t>(ceil_div(l.m, outputs)),
                       static_cast<uint32_t>(a->nseries));
          hipLaunchKernelGGL(scrunch_u32_kernel, g, dim3(kThreads), 0, st, data, a->stride,
                             static_cast<uint32_t>(f), l.m, outputs, lanes, low);
        } else {
          const dim3 g(static_cast<uint32_t>(ceil_div(l.m, kThreads / 64)),
                       static_cast<uint32_t>(a->nseries));
          hipLaunchKernelGGL(scrunch_u32_wide_kernel, g, dim3(kThreads), 0, st, data, a->stride, f,
                             l.m, low);
        }
      } else {
        const dim3 g(static_cast<uint32_t>(ceil_div(l.m, kThreads)),
                     static_cast<uint32_t>(a->nseries));
        hipLaunchKernelGGL((scrunch_kernel<T>), g, dim3(kThreads), 0, st, data, a->stride, f,
                           l.m, low);
      }
      launch_check("scrunch_kernel");
      launch_median<float>(low, l.m, l.m, static_cast<uint32_t>(a->median_window), med, l.m,
                           a->nseries, st);
    } else {
      launch_median<T>(data, a->stride, a->nsamples, static_cast<uint32_t>(a->median_window), med,
                       a->nsamples, a->nseries, st);
    }
  }
  const dim3 g(static_cast<uint32_t>(l.nblocks), static_cast<uint32_t>(a->nseries));
  const StatsBlocks sb = stats_blocks(a, l, workspace);
  const uint32_t block = kMapBlock << sb.shift;
  const dim3 dg(static_cast<uint32_t>(sb.on ? sb.nblocks : l.nblocks),
                static_cast<uint32_t>(a->nseries));
  auto* detrend = sb.on ? detrend_kernel<T, true> : detrend_kernel<T, false>;
  hipLaunchKernelGGL(detrend, dg, dim3(kThreads), 0, st, data, a->stride, a->nsamples, a->detrend,
                     a->detrend ? f : 1, med, l.m, a->status, block / kThreads, sb.sums);
  launch_check("detrend_kernel");
  if (a->normalise) {
    const dim3 sg(static_cast<uint32_t>(ceil_div(a->nseries, kStatsLanes)));
    const float* fdata = reinterpret_cast<const float*>(data);
    if (sb.on) {
      const uint32_t ns = static_cast<uint32_t>(a->nseries);
      const uint32_t nblocks = static_cast<uint32_t>(sb.nblocks);
      hipLaunchKernelGGL(block_exponent_kernel, dim3(ns), dim3(64), 0, st, sb.sums, nblocks);
      launch_check("block_exponent_kernel");
      hipLaunchKernelGGL(square_map_kernel, dim3(nblocks, ns), dim3(kMapThreads), 0, st, fdata,
                         a->stride, a->nsamples, block / kMapThreads, sb.sums, sb.maps);
      launch_check("square_map_kernel");
      hipLaunchKernelGGL(combine_stats_kernel, dim3(ns), dim3(64), 0, st, fdata, a->stride,
                         a->nsamples, nblocks, block, sb.sums, sb.maps, a->reject_constant, stats,
                         flags, a->status);
      launch_check("combine_stats_kernel");
    }
    if ((reinterpret_cast<uintptr_t>(fdata) & 15u) == 0 && a->stride % 4 == 0) {
      // two chunk buffers exceed the default 64 KiB of dynamic LDS
      hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(stats_kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(kStatsLdsBytes)),
                "hipFuncSetAttribute");
      hipLaunchKernelGGL(stats_kernel, sg, dim3(kStatsThreads), kStatsLdsBytes, st, fdata,
                         a->stride, a->nsamples, static_cast<uint32_t>(a->nseries),
                         a->reject_constant, stats, flags, a->status, sb.sums);
      launch_check("stats_kernel");
    } else {
      hipLaunchKernelGGL(stats_rowwise_kernel, sg, dim3(kStatsLanes), 0, st, fdata, a->stride,
                         a->nsamples, static_cast<uint32_t>(a->nseries), a->reject_constant,
                         stats, flags, a->status, sb.sums);
      launch_check("stats_rowwise_kernel");
    }
    hipLaunchKernelGGL(normalise_kernel, g, dim3(kThreads), 0, st,
                       reinterpret_cast<float*>(data), a->stride, a->nsamples, stats, flags);
    launch_check("normalise_kernel");
  }
}

}  // namespace
}  // namespace gaffa_hip

namespace gaffa_hip {
namespace {

// Checks shared by both preprocess entry points; returns the scratch layout.
Layout validate(const gaffa_hip_preprocess_args* a) {
  check(a != nullptr, "preprocess arguments must not be null");
  check(a->data != nullptr && a->status != nullptr, "preprocess pointers must not be null");
  check(a->nseries > 0 && a->nsamples > 0, "preprocess batch must not be empty");
  check(a->stride >= a->nsamples, "preprocess stride must be >= nsamples");
  check(a->detrend || a->normalise || a->input_is_u32,
        "preprocess plan must contain at least one step");
  check(a->nseries < 65536, "preprocess batch has too many series for one launch");
  const uint64_t f = a->detrend ? a->scrunch_factor : 1;
  if (a->detrend) {
    check(a->median_window > 0 && a->median_window % 2 == 1,
          "running median detrend window must be odd and > 0");
    check(f >= 1, "scrunch factor must be >= 1");
    check(a->median_window + kThreads - 1 <= 4096,
          "GPU running median supports windows up to 3841 points");
    const uint64_t m = median_points(a->nsamples, f);
    if (f == 1) {
      check(a->median_window < a->nsamples,
            "running median detrend window_samples must be < input size");
    } else {
      check(m > a->median_window,
            "running median detrend low-resolution sample count must be > min_points");
    }
  }
  const Layout l = layout(a->nseries, a->nsamples, f);
  check_overflow(l.nblocks < 0x7FFFFFFFull, "preprocess series too long");
  return l;
}

// Scratch of the no-allocation entry point: the low-resolution series,
// medians, statistics and flags of one call.  Every kernel
// writes each element before reading it, so nothing needs clearing between
// calls.  Each device holds its own copy for the life of the process; calls
// that overlap on one device share it and race.
constexpr uint64_t kNoAllocScratchBytes = GAFFA_HIP_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// Device address of `scratch` on the current device, looked up with the
// device current on the first call there and kept per device (host code
// never passes the symbol itself to a kernel).
void* noalloc_scratch() {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* ptr[kMaxDevices] = {};
  int dev = 0;
  hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices)
    throw status_error(GAFFA_HIP_RUNTIME, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (ptr[dev] == nullptr) {
    void* p = nullptr;
    hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress");
    if (p == nullptr) throw status_error(GAFFA_HIP_RUNTIME, "scratch symbol has no address");
    ptr[dev] = p;
  }
  return ptr[dev];
}

}  // namespace
}  // namespace gaffa_hip

using namespace gaffa_hip;

extern "C" {

uint64_t gaffa_hip_preprocess_workspace_bytes(uint64_t nseries, uint64_t nsamples,
                                              uint64_t scrunch_factor) {
  if (nseries == 0 || nsamples == 0 || scrunch_factor == 0) return 0;
  return layout(nseries, nsamples, scrunch_factor).total;
}

int gaffa_hip_detrend_normalise_batch(const gaffa_hip_preprocess_args* a,
                                      gaffa_hip_stream stream) {
  return guarded([&] {
    const Layout l = validate(a);
    check(a->workspace != nullptr && a->workspace_bytes >= l.total,
          "preprocess workspace is too small");
    if (a->input_is_u32) {
      run<uint32_t>(a, a->workspace, as_stream(stream));
    } else {
      run<float>(a, a->workspace, as_stream(stream));
    }
  });
}

int gaffa_hip_detrend_normalise_batch_noalloc(const gaffa_hip_preprocess_args* a,
                                              gaffa_hip_stream stream) {
  return guarded([&] {
    const Layout l = validate(a);
    check(a->workspace == nullptr && a->workspace_bytes == 0,
          "the no-allocation preprocess entry point uses its own scratch: workspace must be "
          "null and workspace_bytes 0");
    check_overflow(l.total <= kNoAllocScratchBytes,
                   "preprocess batch needs more scratch than the no-allocation entry point "
                   "holds (GAFFA_HIP_NOALLOC_SCRATCH_BYTES); split the batch");
    void* ws = noalloc_scratch();
    if (a->input_is_u32) {
      run<uint32_t>(a, ws, as_stream(stream));
    } else {
      run<float>(a, ws, as_stream(stream));
    }
  });
}

uint64_t gaffa_hip_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes; }

}  // extern "C"
