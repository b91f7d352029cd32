// The distribution a batch's tokens are drawn from: temperature, softmax, top-k, top-p
// and renormalisation per row (reference mini_vllm/sampler.py:71-124), greedy rows
// one-hot, without sorting the vocabulary.
//
// A row keeps the n first tokens of the descending order (equal values in vocabulary
// order), n the largest count whose last token has fewer than top_k tokens and less than
// top_p of the mass strictly before it (and at least one). So a row needs only its last
// kept token, which is a weighted selection, not a sort: one histogram over the distance
// from the row's maximum finds the bin it lies in, and an exact selection among that
// bin's few tokens finds the token.
//
// Four launches, a workgroup per (row, segment of 4096 to 16384 logits, see segment_of) in
// each, so a single row already runs on nineteen CUs of a 151936-entry vocabulary:
//   max      the segment's largest logit and its index (argmax_key order: NaN highest)
//   mass     exp(x - max) of every token summed into 512 bins of 1/32 nat (LDS atomics)
//            with, for top-k rows, the bins' token counts; rows that do not truncate
//            only sum. The last bin, all tokens 16 nats and more below the maximum and so
//            most of a language model's vocabulary, is summed in registers, and the
//            others are held eight times, by lane, so that a wave's atomics to a popular
//            bin do not queue (32 x 151936: 56 us as one histogram, 16 us so)
//   gather   the row's bins added up and scanned, the boundary bin found, and the
//            segment's tokens in it listed
//   write    the last kept token selected among the listed ones (every workgroup of the
//            row does it again, cheaper than a launch: they are mostly a handful; see
//            select_last for rows where they are not), and the probabilities written in
//            vocabulary order
// Bounds: the logits are read four times (10 MB at 32 x 151936 bf16, from L2 and the
// last-level cache after the first) and the probabilities written once (19 MB); each
// launch is a few microseconds of latency and of vector work (an IEEE division by the
// temperature and an expf per token; the last two kernels first drop the tokens that an
// approximate quotient already rules out). 32 rows of 151936 with mixed parameters: 48 us
// of kernels, where the sort, scan and scatter of torch's path took 1000 us.
//
// Masses are fixed-point 64-bit integers (2^44 for a maximal token at this vocabulary: the
// sum cannot overflow), so every sum is exact whatever the order and the result
// deterministic. The order of tokens is one 64-bit integer: the complement of the
// value's monotone key, then the index.

#include <algorithm>

#include "common.hpp"
#include "sampling.hpp"

namespace mvllm {

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / kWave;
constexpr int kLongestSegment = 16384;
constexpr int kMaxSegments = 64;
constexpr int kBins = kThreads;      // one per thread in the scans
constexpr float kBinsPerNat = 32.0f;
constexpr int kCopies = 8;           // of the histogram in LDS, a lane's by its number

enum Mode : int { kGreedy = 0, kSoftmax = 1, kTruncate = 2 };

struct Rows {
  SamplingRow row[kSamplingRows];
};

// Workspace of one launch set: [row][segment] keys and softmax sums, [row][segment][bin]
// masses and counts, [row][segment] list lengths, [row][segment][kSegment] list entries.
struct Work {
  uint64_t* keys;
  uint64_t* sums;
  uint64_t* masses;
  uint32_t* counts;
  uint32_t* listed;
  uint16_t* list;
};

__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t bits = __float_as_uint(f);
  if (f == 0.0f) bits = 0;  // -0 orders as +0
  return (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? key & 0x7fffffffu : ~key);
}

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src) {
  const int lo = __shfl(static_cast<int>(v), src, kWave);
  const int hi = __shfl(static_cast<int>(v >> 32), src, kWave);
  return (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo);
}

// Reductions over the workgroup; every thread calls and gets the result. `lds` holds
// kWaves words and may be reused after the next barrier.
template <typename Op>
__device__ __forceinline__ uint64_t block_reduce64(uint64_t v, uint64_t* lds, Op op) {
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int mask = 1; mask < kWave; mask <<= 1) v = op(v, shfl64(v, lane ^ mask));
  __syncthreads();
  if (lane == 0) lds[threadIdx.x / kWave] = v;
  __syncthreads();
  v = lds[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) v = op(v, lds[w]);
  return v;
}
__device__ __forceinline__ uint64_t block_max64(uint64_t v, uint64_t* lds) {
  return block_reduce64(v, lds, [](uint64_t a, uint64_t b) { return a > b ? a : b; });
}
__device__ __forceinline__ uint64_t block_sum64(uint64_t v, uint64_t* lds) {
  return block_reduce64(v, lds, [](uint64_t a, uint64_t b) { return a + b; });
}

// Sum of the threads before this one; `total` gets the workgroup's.
__device__ __forceinline__ uint64_t block_exclusive_scan64(uint64_t v, uint64_t* lds,
                                                           uint64_t& total) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  uint64_t incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t other = shfl64(incl, max(lane - off, 0));
    if (lane >= off) incl += other;
  }
  __syncthreads();
  if (lane == kWave - 1) lds[wave] = incl;
  __syncthreads();
  uint64_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) before += lds[w];
    total += lds[w];
  }
  return before + incl - v;
}

// f(index, logit) over this thread's elements of the segment [lo, hi) of a row. kVec: 16-byte
// chunks (rows 16-byte aligned; a segment is a whole number of chunks), a thread's loads
// issued together; the elements past the last whole chunk, and every element otherwise,
// one by one.
template <typename T, bool kVec, int kSegment, typename F>
__device__ __forceinline__ void for_each(const T* row, int64_t lo, int64_t hi, F f) {
  constexpr int kPer = 16 / sizeof(T);
  int64_t done = lo;
  if constexpr (kVec) {
    constexpr int kAhead = kSegment / kPer / kThreads;
    const int64_t c_lo = lo / kPer, c_hi = hi / kPer;
    if (c_hi > c_lo) {
      u32x4 w[kAhead];
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int64_t c = min(c_lo + threadIdx.x + a * kThreads, c_hi - 1);
        w[a] = load16(reinterpret_cast<const char*>(row) + c * 16);
      }
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int64_t c = c_lo + threadIdx.x + a * kThreads;
        if (c < c_hi) {
          float x[kPer];
          Chunk<T>::unpack(w[a], x);
#pragma unroll
          for (int i = 0; i < kPer; ++i) f(c * kPer + i, x[i]);
        }
      }
    }
    done = max(done, c_hi * kPer);
  }
  for (int64_t i = done + threadIdx.x; i < hi; i += kThreads) f(i, Elem<T>::load(row, i));
}

// An approximate quotient below it errs by more than its own few 2^-23: subnormals (one of
// temperatures near the largest float) by up to their spacing.
constexpr float kTinyQuotient = 1e-37f;

// What a workgroup knows of its row before it looks at a logit.
struct RowState {
  float t, p, max;   // temperature, top_p, the scaled maximum
  float inv_t;       // 1 / t, for approximate quotients
  bool approx;       // they are within a few 2^-23 of the exact ones (no overflow)
  int k, mode;
  uint32_t best;     // the maximum's index
  bool finite;       // every probability is a number
};

__device__ __forceinline__ RowState row_state(const SamplingRow& r, const Work& w, int row,
                                              int segments, int64_t v, uint64_t* lds) {
  RowState s;
  uint64_t key = 0;
  for (int i = threadIdx.x; i < segments; i += kThreads) key = w.keys[row * segments + i];
  key = block_max64(key, lds);
  const uint32_t hi = static_cast<uint32_t>(key >> 32);
  s.best = 0xffffffffu - static_cast<uint32_t>(key);
  s.t = r.temperature;
  s.p = r.top_p;
  s.k = r.top_k > 0 && r.top_k < v ? r.top_k : INT32_MAX;
  s.mode = r.temperature == 0.0f ? kGreedy
           : s.k != INT32_MAX || r.top_p < 1.0f ? kTruncate
                                                : kSoftmax;
  s.max = key_value(hi) / s.t;
  s.inv_t = 1.0f / s.t;
  s.approx = fabsf(s.max) < 1e30f;
  // NaN sorts highest, so a row holding one has it as its maximum
  s.finite = hi != 0xffffffffu && __builtin_isfinite(s.max);
  return s;
}

__device__ __forceinline__ int bin_of(float max, float x) {
  return static_cast<int>(fminf((max - x) * kBinsPerNat, static_cast<float>(kBins - 1)));
}
__device__ __forceinline__ uint64_t mass_of(float e, float unit) {
  return static_cast<uint64_t>(e * unit);
}
__device__ __forceinline__ uint64_t rank_of(float x, uint32_t index) {
  return (static_cast<uint64_t>(~order_key(x)) << 32) | index;
}

// Whether the token (or bin) with these tokens and this mass before it is kept.
__device__ __forceinline__ bool keeps(uint64_t count_before, uint64_t mass_before, int k,
                                      double limit) {
  return count_before < static_cast<uint64_t>(k) && static_cast<double>(mass_before) < limit;
}

template <typename T, bool kVec, int kSegment>
__global__ __launch_bounds__(kThreads) void sampling_max_kernel(const Work w, const T* logits,
                                                               int64_t v, int64_t row_stride) {
  __shared__ uint64_t lds[kWaves];
  const T* row = logits + static_cast<int64_t>(blockIdx.x) * row_stride;
  const int64_t lo = static_cast<int64_t>(blockIdx.y) * kSegment, hi = min(v, lo + kSegment);
  uint64_t best = 0;
  for_each<T, kVec, kSegment>(row, lo, hi, [&](int64_t i, float x) __attribute__((always_inline)) {
    const uint64_t key = x != x ? 0xffffffffu : order_key(x);
    const uint64_t mine = (key << 32) | (0xffffffffu - static_cast<uint32_t>(i));
    best = best > mine ? best : mine;
  });
  best = block_max64(best, lds);
  if (threadIdx.x == 0) w.keys[blockIdx.x * gridDim.y + blockIdx.y] = best;
}

template <typename T, bool kVec, int kSegment>
__global__ __launch_bounds__(kThreads) void sampling_mass_kernel(const Rows rows, const Work w,
                                                                const T* logits, int64_t v,
                                                                int64_t row_stride, float unit) {
  __shared__ uint64_t lds[kWaves];
  __shared__ unsigned long long mass[kBins][kCopies];
  __shared__ uint32_t count[kBins][kCopies];
  const int r = blockIdx.x, seg = blockIdx.y, segments = gridDim.y;
#pragma unroll
  for (int c = 0; c < kCopies; ++c) {
    mass[threadIdx.x][c] = 0;
    count[threadIdx.x][c] = 0;
  }
  const RowState s = row_state(rows.row[r], w, r, segments, v, lds);  // (has barriers)
  if (s.mode == kGreedy || !s.finite) return;
  const T* row = logits + static_cast<int64_t>(r) * row_stride;
  const int64_t lo = static_cast<int64_t>(seg) * kSegment, hi = min(v, lo + kSegment);
  const int64_t cell = static_cast<int64_t>(r) * segments + seg;
  if (s.mode == kSoftmax) {
    uint64_t sum = 0;
    for_each<T, kVec, kSegment>(row, lo, hi, [&](int64_t, float l) __attribute__((always_inline)) {
      sum += mass_of(expf(l / s.t - s.max), unit);
    });
    sum = block_sum64(sum, lds);
    if (threadIdx.x == 0) w.sums[cell] = sum;
    return;
  }
  const bool counted = s.k != INT32_MAX;
  const int copy = threadIdx.x % kCopies;
  uint64_t tail = 0, tail_count = 0;
  for_each<T, kVec, kSegment>(row, lo, hi, [&](int64_t, float l) __attribute__((always_inline)) {
    const float x = l / s.t;
    const int bin = bin_of(s.max, x);
    const uint64_t m = mass_of(expf(x - s.max), unit);
    if (bin == kBins - 1) {
      tail += m;
      ++tail_count;
    } else {
      atomicAdd(&mass[bin][copy], static_cast<unsigned long long>(m));
      if (counted) atomicAdd(&count[bin][copy], 1u);
    }
  });
  tail = block_sum64(tail, lds);  // (its barriers close the atomics)
  if (counted) tail_count = block_sum64(tail_count, lds);
  uint64_t m = threadIdx.x == kBins - 1 ? tail : 0;
  uint64_t n = threadIdx.x == kBins - 1 ? tail_count : 0;
#pragma unroll
  for (int c = 0; c < kCopies; ++c) {
    m += mass[threadIdx.x][c];
    n += count[threadIdx.x][c];
  }
  w.masses[cell * kBins + threadIdx.x] = m;
  if (counted) w.counts[cell * kBins + threadIdx.x] = static_cast<uint32_t>(n);
}

// The boundary bin of a truncated row with the tokens and the mass before it, and the
// mass below which a token is kept. Every thread of every workgroup of the row gets
// the same.
struct Boundary {
  int bin;
  uint64_t count, mass;
  double limit;
};

__device__ __forceinline__ Boundary find_boundary(const RowState& s, const Work& w, int r,
                                                  int segments, uint64_t* lds) {
  const bool counted = s.k != INT32_MAX;
  uint64_t mass = 0, count = 0;
  const int64_t first = static_cast<int64_t>(r) * segments * kBins + threadIdx.x;
#pragma unroll 8
  for (int g = 0; g < segments; ++g) mass += w.masses[first + g * kBins];
  if (counted) {
#pragma unroll 8
    for (int g = 0; g < segments; ++g) count += w.counts[first + g * kBins];
  }
  uint64_t total = 0, tokens = 0;
  const uint64_t mass_before = block_exclusive_scan64(mass, lds, total);
  const uint64_t count_before = counted ? block_exclusive_scan64(count, lds, tokens) : 0;
  Boundary b;
  b.limit = s.p < 1.0f ? static_cast<double>(s.p) * static_cast<double>(total)
                       : __builtin_huge_val();
  // the last bin holding tokens whose first one is kept (bin 0 holds the maximum); a bin
  // of tokens that all round to no mass changes nothing by being passed over, unless
  // tokens are counted
  const bool holds = counted ? count > 0 : mass > 0;
  const bool mine = holds && (threadIdx.x == 0 || keeps(count_before, mass_before, s.k, b.limit));
  b.bin = static_cast<int>(block_max64(mine ? threadIdx.x : 0, lds));
  __syncthreads();
  if (static_cast<int>(threadIdx.x) == b.bin) {
    lds[0] = mass_before;
    lds[1] = count_before;
  }
  __syncthreads();
  b.mass = lds[0];
  b.count = lds[1];
  return b;
}

template <typename T, bool kVec, int kSegment>
__global__ __launch_bounds__(kThreads) void sampling_gather_kernel(const Rows rows, const Work w,
                                                                  const T* logits, int64_t v,
                                                                  int64_t row_stride) {
  __shared__ uint64_t lds[kWaves];
  __shared__ uint32_t n;
  const int r = blockIdx.x, seg = blockIdx.y, segments = gridDim.y;
  if (threadIdx.x == 0) n = 0;
  const RowState s = row_state(rows.row[r], w, r, segments, v, lds);
  if (s.mode != kTruncate || !s.finite) return;
  const Boundary b = find_boundary(s, w, r, segments, lds);
  const T* row = logits + static_cast<int64_t>(r) * row_stride;
  const int64_t lo = static_cast<int64_t>(seg) * kSegment, hi = min(v, lo + kSegment);
  const int64_t cell = static_cast<int64_t>(r) * segments + seg;
  uint16_t* list = w.list + cell * kSegment;
  // The approximate distance d' = max - l * inv_t is within slack + d' * 1e-6 of the exact
  // one, so a token whose d' misses the bin by more is not in it.
  const float slack = fabsf(s.max) * 1e-6f + kTinyQuotient;
  const float near = static_cast<float>(b.bin) / kBinsPerNat * (1.0f - 1e-5f) - slack;
  const float far = b.bin == kBins - 1 ? INFINITY
                                       : static_cast<float>(b.bin + 1) / kBinsPerNat * (1.0f + 1e-5f) + slack;
  for_each<T, kVec, kSegment>(row, lo, hi, [&](int64_t i, float l) __attribute__((always_inline)) {
    const float d = s.max - l * s.inv_t;
    if (s.approx && !(d >= near && d <= far)) return;
    if (bin_of(s.max, l / s.t) == b.bin) {
      list[atomicAdd(&n, 1u)] = static_cast<uint16_t>(i - lo);
    }
  });
  __syncthreads();
  if (threadIdx.x == 0) w.listed[cell] = n;
}

// The last kept token's rank and the mass of all kept ones: an exact selection among
// the boundary bin's listed tokens. While more than kThreads remain, passes narrow them by the
// rule of the bins; then each thread takes one and compares it with all.
//   They are a handful, or the whole vocabulary: flat rows, and rows of which one token stands
// out or all but a few are masked while top_k asks for more. The passes:
//   - the listed values' range; none of them with a probability ends here (masked tokens:
//     which are kept changes nothing)
//   - 1024 bins of equal width over that range, where it is a usual one
//   - digits of ten bits of the value, from the first that can differ
//   - of one value left, the segments, then ten bits of the index within one
// What bounds them is one CU's vector work and LDS atomics, 25 to 60 us a pass over 151936
// tokens. us a call for 1 and 32 rows of 151936 bf16 logits, sorted by torch, with 8-bit digits
// of the rank from its first on, now: one value everywhere 198, 908; 2970, 4280; 129, 192; N(0,
// 1e-3) with top-p 201, 964; 703, 744; 192, 288; N(0, 2) and one 25 with top-k 50 202, 968; 701,
// 757; 165, 244; all but 30 masked, top-k 50 198, 906; 2952, 4246; 76, 118.
constexpr int kDigit = 10;
constexpr int kDigitBins = 1 << kDigit;
constexpr int kDigitCopies = 2;
constexpr int kPerThread = kDigitBins / kThreads;
static_assert(kMaxSegments <= kDigitBins && kLongestSegment <= 1 << 14, "");

template <typename T, bool kVec, int kSegment>
__device__ __forceinline__ uint64_t select_last(const RowState& s, const Boundary& b,
                                                const Work& w, const T* row, int64_t v, int r,
                                                int segments, float unit, uint64_t* lds, uint64_t& kept_mass) {
  __shared__ uint32_t start[kMaxSegments + 1];
  __shared__ unsigned long long mass[kDigitCopies][kDigitBins];
  __shared__ uint32_t count[kDigitCopies][kDigitBins];
  __shared__ uint64_t c_rank[kThreads], c_mass[kThreads];
  __shared__ uint32_t taken;
  const int lane = threadIdx.x % kWave;
  const int64_t cell = static_cast<int64_t>(r) * segments;
  uint64_t total = 0;
  {
    const uint64_t mine = threadIdx.x < segments ? w.listed[cell + threadIdx.x] : 0;
    const uint64_t before = block_exclusive_scan64(mine, lds, total);
    if (threadIdx.x <= segments && threadIdx.x <= kMaxSegments) {
      start[threadIdx.x] = static_cast<uint32_t>(before);
    }
  }
  __syncthreads();
  const uint32_t listed = static_cast<uint32_t>(total);
  // f(x, index in the row) for segment a's listed tokens; from the list, a thread's loads kAhead
  // at a time, or where it holds a good part of the segment from the row itself (its chunks
  // in order, no load waiting for another: 151936 tokens 90 us by the list, 30 so).
  constexpr int kAhead = 4;
  auto for_segment = [&](int a, auto f) __attribute__((always_inline)) {
    const uint32_t n = start[a + 1] - start[a];
    const int64_t lo = static_cast<int64_t>(a) * kSegment, hi = min(v, lo + kSegment);
    if (8 * n >= hi - lo) {
      for_each<T, kVec, kSegment>(row, lo, hi, [&](int64_t i, float l) __attribute__((always_inline)) {
        const float x = l / s.t;
        if (bin_of(s.max, x) == b.bin) f(x, static_cast<uint32_t>(i));
      });
      return;
    }
    const uint16_t* list = w.list + (cell + a) * kSegment;
    for (uint32_t j0 = 0; j0 < n; j0 += kAhead * kThreads) {
      uint32_t index[kAhead];
      float x[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        index[u] = a * kSegment + list[min(j0 + u * kThreads + threadIdx.x, n - 1)];
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) x[u] = Elem<T>::load(row, index[u]);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (j0 + u * kThreads + threadIdx.x < n) f(x[u] / s.t, index[u]);
      }
    }
  };
  uint64_t count_before = b.count, mass_before = b.mass;
  uint32_t left = listed;
  float top = 0.0f, per_unit = 0.0f;
  int bin_chosen = -1;   // equal-width bin
  uint64_t prefix = 0;   // of the rank
  int known = 0;         // its bits
  int first = 0, last = segments;  // the segments left
  auto width_bin = [&](float x) __attribute__((always_inline)) -> int {
    return static_cast<int>(fminf((top - x) * per_unit, static_cast<float>(kDigitBins - 1)));
  };
  auto matches = [&](float x, uint64_t rank) __attribute__((always_inline)) -> bool {
    return (bin_chosen < 0 || width_bin(x) == bin_chosen) &&
           (known == 0 || rank >> (64 - known) == prefix);
  };
  // One pass: bin_of_token over the tokens left, the last bin whose first token is kept (the
  // first non-empty one's is: it was chosen for it), and what comes before it.
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
#pragma unroll
      for (int c = 0; c < kDigitCopies; ++c) {
        mass[c][i * kThreads + threadIdx.x] = 0;
        count[c][i * kThreads + threadIdx.x] = 0;
      }
    }
    __syncthreads();
  };
  auto choose = [&]() __attribute__((always_inline)) -> int {
    __syncthreads();
    uint64_t bm[kPerThread], bc[kPerThread], m = 0, c = 0, unused;
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {  // thread t owns bins kPerThread t and on
      bm[i] = bc[i] = 0;
#pragma unroll
      for (int k = 0; k < kDigitCopies; ++k) {
        bm[i] += mass[k][kPerThread * threadIdx.x + i];
        bc[i] += count[k][kPerThread * threadIdx.x + i];
      }
      m += bm[i];
      c += bc[i];
    }
    uint64_t mb = mass_before + block_exclusive_scan64(m, lds, unused);
    uint64_t cb = count_before + block_exclusive_scan64(c, lds, unused);
    uint64_t my_bin = 0, my_mb = 0, my_cb = 0, my_c = 0;
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      if (bc[i] > 0 && (cb == count_before || keeps(cb, mb, s.k, b.limit))) {
        my_bin = kPerThread * threadIdx.x + i;
        my_mb = mb;
        my_cb = cb;
        my_c = bc[i];
      }
      mb += bm[i];
      cb += bc[i];
    }
    const uint64_t bin = block_max64(my_c > 0 ? my_bin : 0, lds);
    __syncthreads();
    if (my_c > 0 && my_bin == bin) {
      lds[0] = my_mb;
      lds[1] = my_cb;
      lds[2] = my_c;
    }
    __syncthreads();
    mass_before = lds[0];
    count_before = lds[1];
    left = static_cast<uint32_t>(lds[2]);
    __syncthreads();
    return static_cast<int>(bin);
  };
  auto pass = [&](auto bin_of_token) __attribute__((always_inline)) -> int {
    clear();
    for (int a = first; a < last; ++a) {
      for_segment(a, [&](float x, uint32_t index) __attribute__((always_inline)) {
        const uint64_t rank = rank_of(x, index);
        if (matches(x, rank)) {
          const int bin = bin_of_token(x, rank);
          atomicAdd(&mass[lane % kDigitCopies][bin],
                    static_cast<unsigned long long>(mass_of(expf(x - s.max), unit)));
          atomicAdd(&count[lane % kDigitCopies][bin], 1u);
        }
      });
    }
    return choose();
  };
  if (left > kThreads) {
    uint64_t low = ~uint64_t{0}, high = 0;  // of the values' halves of the ranks
    for (int a = 0; a < segments; ++a) {
      for_segment(a, [&](float x, uint32_t) __attribute__((always_inline)) {
        const uint64_t value = rank_of(x, 0) >> 32;
        low = min(low, value);
        high = max(high, value);
      });
    }
    low = ~block_max64(~low, lds);
    high = block_max64(high, lds);
    top = key_value(~static_cast<uint32_t>(low));
    if (expf(top - s.max) == 0.0f) {
      kept_mass = b.mass;
      return ~uint64_t{0};
    }
    const float range = top - key_value(~static_cast<uint32_t>(high));
    if (range > 0.0f && range < 1024.0f) {
      per_unit = static_cast<float>(kDigitBins) / range;
      if (per_unit < 1e30f) bin_chosen = pass([&](float x, uint64_t) { return width_bin(x); });
    }
    known = low == high ? 32 : __builtin_clzll(low ^ high) - 32;
    prefix = low >> (32 - known);
  }
  while (left > kThreads && known < 64) {  // (all 64 bits known leave one)
    if (known == 32) {
      // One value: its count in each segment.
      clear();
      const uint64_t m = mass_of(expf(key_value(~static_cast<uint32_t>(prefix)) - s.max), unit);
      for (int a = 0; a < segments; ++a) {
        int mine = 0;
        for_segment(a, [&](float x, uint32_t index) __attribute__((always_inline)) {
          mine += matches(x, rank_of(x, index)) ? 1 : 0;
        });
        const uint32_t n = __builtin_amdgcn_readlane(wave_inclusive_scan(mine), kWave - 1);
        if (lane == 0) {
          atomicAdd(&mass[0][a], static_cast<unsigned long long>(m * n));
          atomicAdd(&count[0][a], n);
        }
      }
      first = choose();
      last = first + 1;
      constexpr int kIndexBits = __builtin_ctz(kSegment);
      prefix = (prefix << (32 - kIndexBits)) | static_cast<uint64_t>(first);
      known = 64 - kIndexBits;
      continue;
    }
    const int width = min(kDigit, (known < 32 ? 32 : 64) - known);
    const int shift = 64 - known - width;
    const int bin = pass([&](float, uint64_t rank) __attribute__((always_inline)) {
      return static_cast<int>(rank >> shift) & ((1 << width) - 1);
    });
    prefix = (prefix << width) | static_cast<uint64_t>(bin);
    known += width;
  }
  if (threadIdx.x == 0) taken = 0;
  __syncthreads();
  auto take = [&](float x, uint32_t index) __attribute__((always_inline)) {
    const uint64_t rank = rank_of(x, index);
    if (!matches(x, rank)) return;
    const uint32_t at = atomicAdd(&taken, 1u);
    if (at >= kThreads) return;  // (`left` of them)
    c_rank[at] = rank;
    c_mass[at] = mass_of(expf(x - s.max), unit);
  };
  if (listed <= kThreads) {
    const uint32_t j = threadIdx.x;
    if (j < listed) {
      int a = 0, e = segments;  // start[a] <= j < start[e]
      while (e - a > 1) {
        const int mid = (a + e) >> 1;
        if (start[mid] <= j) a = mid; else e = mid;
      }
      const uint32_t index = a * kSegment + w.list[(cell + a) * kSegment + (j - start[a])];
      take(Elem<T>::load(row, index) / s.t, index);
    }
  } else {
    for (int a = first; a < last; ++a) {
      for_segment(a, take);
    }
  }
  __syncthreads();
  // Each thread's token against all: what comes before it, and whether it is kept.
  uint64_t kept = 0, upto = 0;
  if (threadIdx.x < left) {
    const uint64_t rank = c_rank[threadIdx.x];
    uint64_t before_mass = 0, before_count = 0;
    for (uint32_t j = 0; j < left; ++j) {
      const bool before = c_rank[j] < rank;
      before_mass += before ? c_mass[j] : 0;
      before_count += before ? 1 : 0;
    }
    if (before_count == 0 ||
        keeps(count_before + before_count, mass_before + before_mass, s.k, b.limit)) {
      kept = rank;
      upto = mass_before + before_mass + c_mass[threadIdx.x];
    }
  }
  // Ranks grow with the masses up to them, so both maxima are the last kept token's.
  kept = block_max64(kept, lds);
  kept_mass = block_max64(upto, lds);
  return kept;
}

template <typename T, bool kVec, int kSegment>
__global__ __launch_bounds__(kThreads) void sampling_write_kernel(const Rows rows, const Work w,
                                                                 float* __restrict__ probs,
                                                                 const T* logits, int64_t v,
                                                                 int64_t row_stride, float unit,
                                                                 float inv_unit) {
  __shared__ uint64_t lds[kWaves];
  const int r = blockIdx.x, seg = blockIdx.y, segments = gridDim.y;
  const RowState s = row_state(rows.row[r], w, r, segments, v, lds);
  const T* row = logits + static_cast<int64_t>(r) * row_stride;
  float* out = probs + static_cast<int64_t>(r) * v;
  const int64_t lo = static_cast<int64_t>(seg) * kSegment, hi = min(v, lo + kSegment);
  uint64_t last = ~uint64_t{0};  // rank of the last kept token
  float sum = 1.0f;
  if (s.mode == kGreedy) {
    sum = 0.0f;
  } else if (!s.finite) {
    sum = __int_as_float(0x7fc00000);
  } else if (s.mode == kSoftmax) {
    uint64_t z = 0;
    for (int i = threadIdx.x; i < segments; i += kThreads) {
      z += w.sums[static_cast<int64_t>(r) * segments + i];
    }
    sum = static_cast<float>(block_sum64(z, lds)) * inv_unit;
  } else {
    const Boundary b = find_boundary(s, w, r, segments, lds);
    uint64_t kept_mass = 0;
    last = select_last<T, kVec, kSegment>(s, b, w, row, v, r, segments, unit, lds, kept_mass);
    sum = static_cast<float>(kept_mass) * inv_unit;
  }
  // Tokens whose approximate quotient is below the last kept value by more than the two can
  // differ are not kept.
  const float value = key_value(~static_cast<uint32_t>(last >> 32));
  const float below = s.mode == kTruncate && s.finite && s.approx
                          ? value - ((fabsf(value) + fabsf(s.max)) * 1e-6f + kTinyQuotient)
                          : -INFINITY;
  auto prob = [&](int64_t i, float l) __attribute__((always_inline)) -> float {
    if (s.mode == kGreedy) return static_cast<uint32_t>(i) == s.best ? 1.0f : 0.0f;
    if (!s.finite) return sum;
    if (l * s.inv_t < below) return 0.0f;
    const float x = l / s.t;
    if (rank_of(x, static_cast<uint32_t>(i)) > last) return 0.0f;
    return expf(x - s.max) / sum;
  };
  if constexpr (kVec) {
    // chunks of 16 bytes of logits, written as whole 16-byte stores
    constexpr int kPer = 16 / sizeof(T);
    constexpr int kAhead = kSegment / kPer / kThreads;
    const int64_t c_lo = lo / kPer, c_hi = hi / kPer;
    if (c_hi > c_lo) {
      u32x4 raw[kAhead];
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int64_t c = min(c_lo + threadIdx.x + a * kThreads, c_hi - 1);
        raw[a] = load16(reinterpret_cast<const char*>(row) + c * 16);
      }
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int64_t c = c_lo + threadIdx.x + a * kThreads;
        if (c < c_hi) {
          float x[kPer], y[kPer];
          Chunk<T>::unpack(raw[a], x);
#pragma unroll
          for (int i = 0; i < kPer; ++i) y[i] = prob(c * kPer + i, x[i]);
#pragma unroll
          for (int i = 0; i < kPer; i += 4) {
            nt_store16(out + c * kPer + i,
                       u32x4{__float_as_uint(y[i]), __float_as_uint(y[i + 1]),
                             __float_as_uint(y[i + 2]), __float_as_uint(y[i + 3])});
          }
        }
      }
    }
    for (int64_t i = max(lo, c_hi * kPer) + threadIdx.x; i < hi; i += kThreads) {
      out[i] = prob(i, Elem<T>::load(row, i));
    }
  } else {
    for (int64_t i = lo + threadIdx.x; i < hi; i += kThreads) {
      out[i] = prob(i, Elem<T>::load(row, i));
    }
  }
}

int segments_of(int64_t v, int segment) { return static_cast<int>((v + segment - 1) / segment); }

// A row's segment length: shorter ones spread few rows over more CUs, but every workgroup
// of a truncated row adds up the histograms of all its segments, so they pay only while all
// workgroups run at once (256 CUs), and the shortest only for rows of up to eight of them.
// Graph-replayed calls with 16384, 8192 and 4096: 8 rows of 151936 34.1, 31.4 and 43.7 us,
// 16 rows 34.6, 39.7 and 53.2; 32 rows of 32000 32.0, 27.1 and 25.0, 64 rows 32.9, 28.1 and
// 31.8, 128 rows 34.7, 35.3 and 50.5.
int segment_of(int64_t rows, int64_t v) {
  if (segments_of(v, 4096) <= 8 && rows * segments_of(v, 4096) <= 256) return 4096;
  if (segments_of(v, 8192) <= kMaxSegments && rows * segments_of(v, 8192) <= 256) return 8192;
  return kLongestSegment;
}

uint64_t align256(uint64_t n) { return (n + 255) / 256 * 256; }

// The workspace's parts for `rows` rows; returns its size.
uint64_t layout(int64_t rows, int64_t v, int segment, char* base, Work& w) {
  const uint64_t cells = static_cast<uint64_t>(rows) * segments_of(v, segment);
  uint64_t at = 0;
  auto part = [&](uint64_t bytes) {
    char* p = base == nullptr ? nullptr : base + at;
    at += align256(bytes);
    return p;
  };
  w.keys = reinterpret_cast<uint64_t*>(part(cells * 8));
  w.sums = reinterpret_cast<uint64_t*>(part(cells * 8));
  w.masses = reinterpret_cast<uint64_t*>(part(cells * kBins * 8));
  w.counts = reinterpret_cast<uint32_t*>(part(cells * kBins * 4));
  w.listed = reinterpret_cast<uint32_t*>(part(cells * 4));
  w.list = reinterpret_cast<uint16_t*>(part(cells * segment * 2));
  return at;
}

template <typename T, bool kVec, int kSegment>
hipError_t launch(float* probs, const void* logits, int64_t v, int64_t row_stride,
                  const Rows& rows, int n, const Work& w, bool truncates, bool softmax,
                  hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(n), segments_of(v, kSegment));
  const T* l = static_cast<const T*>(logits);
  int bits = 0;  // the least with 2^bits >= v: v maximal masses of 2^(62 - bits) sum to at most 2^62
  while ((int64_t{1} << bits) < v) ++bits;
  const float unit = static_cast<float>(uint64_t{1} << (62 - bits));
  sampling_max_kernel<T, kVec, kSegment><<<grid, kThreads, 0, stream>>>(w, l, v, row_stride);
  if (truncates || softmax) {
    sampling_mass_kernel<T, kVec, kSegment><<<grid, kThreads, 0, stream>>>(rows, w, l, v, row_stride, unit);
  }
  if (truncates) {
    sampling_gather_kernel<T, kVec, kSegment><<<grid, kThreads, 0, stream>>>(rows, w, l, v, row_stride);
  }
  sampling_write_kernel<T, kVec, kSegment><<<grid, kThreads, 0, stream>>>(rows, w, probs, l, v, row_stride,
                                                               unit, 1.0f / unit);
  return hipGetLastError();
}

template <typename T, int kSegment>
hipError_t launch_rows(float* probs, const void* logits, int64_t rows, int64_t v,
                       int64_t row_stride, const SamplingRow* params, void* workspace,
                       hipStream_t stream) {
  Work w;
  layout(std::min<int64_t>(rows, kSamplingRows), v, kSegment, static_cast<char*>(workspace), w);
  const bool vec = reinterpret_cast<uintptr_t>(logits) % 16 == 0 &&
                   (row_stride * static_cast<int64_t>(sizeof(T))) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(probs) % 16 == 0 && v % 4 == 0;
  for (int64_t r0 = 0; r0 < rows; r0 += kSamplingRows) {
    const int n = static_cast<int>(std::min<int64_t>(rows - r0, kSamplingRows));
    Rows part{};
    bool truncates = false, softmax = false;
    for (int i = 0; i < n; ++i) {
      const SamplingRow& p = params[r0 + i];
      part.row[i] = p;
      if (p.temperature == 0.0f) continue;
      const bool cut = p.top_p < 1.0f || (p.top_k > 0 && p.top_k < v);
      truncates = truncates || cut;
      softmax = softmax || !cut;
    }
    const T* l = static_cast<const T*>(logits) + r0 * row_stride;
    float* out = probs + r0 * v;
    const hipError_t e =
        vec ? launch<T, true, kSegment>(out, l, v, row_stride, part, n, w, truncates, softmax, stream)
            : launch<T, false, kSegment>(out, l, v, row_stride, part, n, w, truncates, softmax, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <typename T>
hipError_t launch_segments(float* probs, const void* logits, int64_t rows, int64_t v,
                           int64_t row_stride, const SamplingRow* params, void* workspace,
                           hipStream_t stream) {
  switch (segment_of(rows, v)) {
    case 4096:
      return launch_rows<T, 4096>(probs, logits, rows, v, row_stride, params, workspace, stream);
    case 8192:
      return launch_rows<T, 8192>(probs, logits, rows, v, row_stride, params, workspace, stream);
    default:
      return launch_rows<T, kLongestSegment>(probs, logits, rows, v, row_stride, params, workspace,
                                             stream);
  }
}

}  // namespace

uint64_t sampling_workspace_bytes(int64_t rows, int64_t v) {
  Work w;
  return layout(std::min<int64_t>(rows, kSamplingRows), v, segment_of(rows, v), nullptr, w);
}

int64_t sampling_max_vocab() { return int64_t{kLongestSegment} * kMaxSegments; }

hipError_t launch_sampling_probabilities(float* probs, const void* logits, int64_t rows,
                                         int64_t v, int64_t row_stride, int dtype,
                                         const SamplingRow* params, void* workspace,
                                         hipStream_t stream) {
  switch (dtype) {
    case kF32:
      return launch_segments<float>(probs, logits, rows, v, row_stride, params, workspace, stream);
    case kF16:
      return launch_segments<f16_t>(probs, logits, rows, v, row_stride, params, workspace, stream);
    case kBF16:
      return launch_segments<bf16_t>(probs, logits, rows, v, row_stride, params, workspace, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mvllm
