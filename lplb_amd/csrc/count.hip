// Per-expert token histogram with an inclusive prefix over slices.
//
// Slices of up to 4096 indices, up to 256 of them and not too few for the experts: one launch on the caller's stream (count_and_scan,
// below).  Else, and in a capture, two:
//   1. slice_histogram: one workgroup per slice, LDS histogram (eight copies, chosen by lane)
//      fed by coalesced 16-byte index loads, row p of the output = counts of slice p;
//   2. prefix_over_slices: turns the rows into running sums down the slice axis,
//      16 experts per workgroup and 16 row bands per expert, instead of the serial
//      walk over all slices the reference does after its grid barrier
//      (minilp.cu:439-442).
// (Doing the scan inside the first kernel, by the last workgroup to finish, was
// measured and rejected: one CU sustains too few outstanding misses to pull the
// 256 KB table, 20 us against 3 us for this kernel.)
// HBM-bound: 8 bytes read per index; the [n_blocks, n_experts] table is small.  The indices are read with ordinary
// loads because the redirect reads them again: with non-temporal ones, as the redirect's own last read is, that second
// read came from HBM ([1048576 x 8], 67 MB, whole plan as four kernels: 48.7 us, with ordinary loads 44.7; with the next
// batch of loads under way while one is counted 44.2; walking a slice backwards, so that its beginning is the
// part read last, gains nothing).  The price is a count that no redirect follows.  Histogram, scan and redirect / histogram
// and scan alone, non-temporal -> ordinary, us: [262144 x 8] 15.6 -> 15.1 / 8.3 -> 8.3, [1048576 x 8] 42.0 -> 37.5 / 16.3 -> 17.0,
// [3145728 x 8] 121 -> 97.5 / 35.8 -> 38.3, [8388608 x 8] (537 MB, twice the last-level cache) 290 -> 272 / 91 -> 100; shorter batches
// the same both ways.
// Callers that need only the totals of a short batch get them in one launch: slice_histogram with
// TOTALS (slices add their counts to one vector) or expert_totals (every workgroup owns four experts).
#include "map_kernel.h"
#include "plan_sync.h"
#include "scan.h"

namespace lplb {

constexpr int kLoadsInFlight = 4;   // 16-byte loads a thread issues before it consumes them

// COPIES histograms side by side, lane l counts into copy l % COPIES: lanes of one instruction that
// hold the same expert are served one after the other by the LDS, and at Zipf(1.0) the hottest expert
// has ten of a wave's 64 tokens.  The copies start 4 banks apart (a stride of 4 modulo the 32 banks),
// so that the counters of one expert sit in eight different banks.  (Measured at [262144 x 8] in 256
// slices, kernel alone: one copy 5.3 us, two 5.1, four 4.9, eight 4.8, eight in different banks 4.6;
// a copy per wave instead of per lane: no gain.)
constexpr int kHistogramCopies = 8;
__host__ __device__ constexpr int histogram_stride(int n_experts, int copies) {
  return copies > 1 ? ((n_experts + 31) & ~31) + 4 : n_experts;
}

// The tokens of slice p into the histograms `hist` (LDS), by nt threads; ends with a workgroup barrier.  `meanwhile` is called while the first loads
// are on their way.
template <int COPIES, typename Meanwhile>
__device__ __forceinline__ void count_slice(const int64_t *__restrict__ idx, int64_t n, int n_experts, int64_t per, int p, int nt, int32_t *hist,
                                            Meanwhile meanwhile) {
  const int tid = threadIdx.x;
  const int stride = histogram_stride(n_experts, COPIES);
  int32_t *mine = hist + (tid % COPIES) * stride;
  auto count = [&](int64_t v) {
    if ((uint64_t)v < (uint64_t)n_experts)
      atomicAdd(&mine[(int)v], 1);
  };
  const int64_t begin = slice_begin(n, per, p);
  const int64_t end = slice_begin(n, per, p + 1);
  // Pairs are loaded 16 bytes at a time.  Slices start on multiples of 256 indices,
  // so a slice starts on a 16-byte boundary unless the array itself sits at an odd
  // multiple of 8 bytes (a view that starts inside a tensor); then its first index
  // is counted alone.
  const int64_t head = (begin < end && (reinterpret_cast<uintptr_t>(idx + begin) & 8)) ? 1 : 0;
  const int64_t n_pairs = (end - begin - head) >> 1;
  typedef long long i64x2 __attribute__((ext_vector_type(2)));
  const i64x2 *pairs = reinterpret_cast<const i64x2 *>(idx + begin + head);
  // the first batch of loads is on its way while the histogram is cleared, every later one while the batch before it
  // is counted
  auto load_batch = [&](i64x2 (&v)[kLoadsInFlight], int64_t i0) {
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      const int64_t i = i0 + tid + (int64_t)u * nt;
      v[u] = i < n_pairs ? pairs[i] : i64x2{-1, -1};
    }
  };
  auto count_batch = [&](const i64x2 (&v)[kLoadsInFlight]) {
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      count(v[u].x);
      count(v[u].y);
    }
  };
  const int64_t batch = (int64_t)nt * kLoadsInFlight;
  i64x2 even[kLoadsInFlight], odd[kLoadsInFlight];
  load_batch(even, 0);
  for (int e = tid; e < COPIES * stride; e += nt)
    hist[e] = 0;
  meanwhile();
  __syncthreads();
  for (int64_t i0 = 0; i0 < n_pairs; i0 += 2 * batch) {
    load_batch(odd, i0 + batch);
    count_batch(even);
    if (i0 + batch >= n_pairs)
      break;
    load_batch(even, i0 + 2 * batch);
    count_batch(odd);
  }
  if (tid == 0 && head)
    count(idx[begin]);
  if (tid == 0 && ((end - begin - head) & 1))
    count(idx[end - 1]);
  __syncthreads();
}

// TOTALS: instead of writing its row, a slice adds its counts to the one vector `counts` [n_experts]
// (device-wide atomic adds, none for an expert the slice has no token of).  The launch sets the vector `clear` [n_experts]
// (if given) to zero -- a caller that takes two vectors in turn never has to zero one --, or without TOTALS to kNoTotal,
// for scan_and_solve.
template <int COPIES, bool TOTALS>
__global__ __launch_bounds__(1024) void slice_histogram(
    const int64_t *__restrict__ idx, int64_t n, int n_experts, int64_t per,
    int32_t *__restrict__ counts, int32_t *__restrict__ clear) {
  extern __shared__ int32_t hist[];
  fetch_arguments_now(idx, n, n_experts, per, counts, clear);
  const int tid = threadIdx.x, nt = blockDim.x;
  const int p = blockIdx.x;
  const int stride = histogram_stride(n_experts, COPIES);
  count_slice<COPIES>(idx, n, n_experts, per, p, nt, hist, [&]() {
    if (clear)
      for (int64_t e = (int64_t)p * nt + tid; e < n_experts; e += (int64_t)gridDim.x * nt)
        clear[e] = TOTALS ? 0 : kNoTotal;
  });
  int32_t *row = TOTALS ? counts : counts + (int64_t)p * n_experts;
  if constexpr (!TOTALS) {
    for (int e = tid; e < n_experts; e += nt) {
      int32_t sum = 0;
#pragma unroll
      for (int k = 0; k < COPIES; ++k)
        sum += hist[k * stride + e];
      row[e] = sum;
    }
  } else {
    // Two counters per atomic add: updates of one 64-byte line of memory are served one after the other
    // (about 14 ns each), and every slice updates every line, so the number of updates is what this
    // costs.  A counter stays below 2^31, so the low half never carries into the high one.
    unsigned long long *both = reinterpret_cast<unsigned long long *>(row);
    for (int e2 = tid; 2 * e2 < n_experts; e2 += nt) {
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int k = 0; k < COPIES; ++k) {
        lo += (uint32_t)hist[k * stride + 2 * e2];
        hi += 2 * e2 + 1 < n_experts ? (uint32_t)hist[k * stride + 2 * e2 + 1] : 0u;
      }
      if (2 * e2 + 1 < n_experts) {
        if ((lo | hi) != 0)
          __hip_atomic_fetch_add(both + e2, ((unsigned long long)hi << 32) | lo, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      } else if (lo != 0) {
        __hip_atomic_fetch_add(row + 2 * e2, (int32_t)lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

// The launch all callers share: eight copies while they fit the 64 KiB of LDS a kernel gets unasked
// (up to 2016 experts), else one.  TOTALS as in the kernel.
template <bool TOTALS>
static int launch_slice_histogram(const int64_t *idx, int64_t n_elements, int n_experts, int n_blocks, int32_t *counts,
                                  int32_t *clear, hipStream_t s, unsigned flags) {
  const size_t one = sizeof(int32_t) * (size_t)n_experts;
  LPLB_REQUIRE(one <= 64 * 1024, LPLB_EUNSUPPORTED, "n_experts=%d does not fit the LDS histogram", n_experts);
  const int64_t per = slice_len(n_elements, n_blocks);
  // one 16-byte load per thread covers 2 indices; a thread has kLoadsInFlight of them under
  // way, so a slice gets as many threads as cover it in one such batch, up to 1024
  const int64_t batches = (per / 2 + kLoadsInFlight - 1) / kLoadsInFlight;
  const int threads = batches <= 256 ? 256 : batches <= 512 ? 512 : 1024;
  const size_t copies = sizeof(int32_t) * (size_t)kHistogramCopies * histogram_stride(n_experts, kHistogramCopies);
  if (copies <= 64 * 1024)
    launch_with_flags(slice_histogram<kHistogramCopies, TOTALS>, dim3(n_blocks), dim3(threads), copies, s, flags, idx,
                      n_elements, n_experts, per, counts, clear);
  else
    launch_with_flags(slice_histogram<1, TOTALS>, dim3(n_blocks), dim3(threads), one, s, flags, idx, n_elements,
                      n_experts, per, counts, clear);
  LPLB_HIP_TRY(hipGetLastError());
  return LPLB_OK;
}

__global__ __launch_bounds__(kScanThreads) void prefix_over_slices(int32_t *__restrict__ counts, int n_blocks, int n_experts) {
  __shared__ ScanLds lds;
  fetch_arguments_now(counts, n_blocks, n_experts);
  scan_columns(counts, n_blocks, n_experts, blockIdx.x, lds, [](int, int32_t) {});
}

// ---- histogram and running sums in one launch ----
// Up to kCountMaxSlices slices: a slice publishes its counts as soon as it has them, and the first of them turn a few columns of the
// published rows into running sums each: a trip from CU to CU instead of a launch and a trip of the table through memory and back.
// [32768 x 8] in 256 slices 6.2 -> 4.8 us, and one launch (2.1 us of the calling thread) less, which is what the three calls waited for.
// What bounds it: the launch, the indices'
// and the words' trip, instructions.  One copy of the histogram: a slice is 16 or 32 of a wave's instructions here, and eight copies
// to clear and to add up cost more than lanes that wait for each other (eight 5.45 us, four 5.1, two 4.95, one 4.8).
// What crosses workgroups are words as in the one-launch plan (plan_sync.h): the launch's tag in the high half, two counts of 16
// bits in the low half, so that nothing has to be cleared and words may arrive in any order.  The host gives every launch
// of a device a number; it is the tag, and one of kCountRegions parts of the array in turn is the launch's.
// Nothing has to be resident at once: the workgroups with columns wait (the first of the grid, as many as there are fours of columns or,
// with 512 threads, eights; with 1024 experts or few slices that is all of them), but not for long: should their words not come within
// kCountPolls polls (a launch that is kept off the GPU for long, or that finds its region in use by one kCountRegions launches later), they
// count those columns of all slices themselves, every waiting workgroup the whole batch once a round.  So every wait ends and the rows are
// right in any case.  (1024 polls are 0.5 ms and more, a few times what that counting takes.)
// A call that is captured takes two launches: a replay would carry the same tag.
constexpr int kCountMaxSlices = 256, kCountMaxExperts = 1024, kCountRegions = 8, kCountPolls = 1 << 10;
// Up to 4096 indices a slice.  Longer ones keep the adding workgroups' loads waiting behind the indices', and the calling thread is not what
// the three calls wait for any more: [131072 x 8] (4096) 18.1 -> 16.6 us, [262144 x 8] (8192) 19.6 in two launches, 20.1 in one, at 32 ranks
// 32.1 and 32.7.
constexpr int64_t kCountMaxSlice = 4096;
static_assert(kCountMaxSlice < 65536, "two counts to a word");
// The slices take the columns four at a time and in turn, by 256 or 512 threads one or two of those fours.  A round is a chain of a load past the
// caches, sums over the wave and four barriers, 0.7 us with 256 threads and 0.9 with 512, where a second launch takes all columns at once: 256
// experts in one slice are 64 rounds, 48 us instead of 6, 1024 experts 256 rounds and 188 us.  us a call in two launches / in one, call behind call:
//   256 threads, slices of 2048:  two rounds, 256 experts in 32 slices 6.6 / 5.1, 1024 in 128 6.9 / 5.9; three, 256 in 22 6.6 / 5.9, 512 in 43 6.5 / 6.1,
//     1024 in 86 6.8 / 6.4; four, 64 in 4 6.5 / 5.8, 256 in 16 6.6 / 6.8, 512 in 32 6.6 / 6.9, 1024 in 64 6.8 / 7.2
//   512 threads, slices of 4096:  two rounds, 256 in 16 6.7 / 5.5, 1024 in 64 6.6 / 5.7; three, 256 in 11 6.6 / 6.4, 1024 in 43 6.6 / 6.6 (each waited
//     for, 17.4 / 17.4 and 17.5 / 17.6); four, 256 in 8 6.6 / 7.3, 1024 in 32 6.6 / 7.5
constexpr int most_count_rounds(int groups) { return groups == 1 ? 3 : 2; }
constexpr int kCountRegionWords = kCountMaxSlices * kCountMaxExperts / 2;
static __device__ __attribute__((aligned(4096))) unsigned long long g_count_words[kCountRegions * kCountRegionWords];
static __device__ int g_count_recounts;   // columns' turns that workgroups counted for themselves, since the library was loaded

// A pair of words, 16-byte aligned, with one load past the caches (see agent_load_pairs), polled until both have the tag.  By whole
// waves; false: they did not come, or a later launch has the region.
__device__ inline bool poll_pair(u32x4 &v, const unsigned long long *p, uint32_t tag, int max_polls) {
  bool in = false, later = false;
  for (int polls = 0; polls < max_polls; ++polls) {
    if (!in) {
      asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v) : "v"(p) : "memory");
      in = ((v.y ^ tag) | (v.w ^ tag)) == 0;
      later = (int32_t)(v.y - tag) > 0 || (int32_t)(v.w - tag) > 0;
    }
    if (__all(in))
      return true;
    if (__any(later))
      return false;
    __builtin_amdgcn_s_sleep(2);
  }
  return false;
}
// Sum over the lanes up to this one.
__device__ inline int32_t wave_inclusive_scan(int32_t v) {
  v += row_shr<1>(v);
  v += row_shr<2>(v);
  v += row_shr<4>(v);
  v += row_shr<8>(v);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142 /* row_bcast:15 */, 0xa, 0xf, false);
  return v + __builtin_amdgcn_update_dpp(0, v, 0x143 /* row_bcast:31 */, 0xc, 0xf, false);
}

__host__ __device__ constexpr int padded_experts(int n) { return (n + 3) / 4 * 4; }
// GROUPS of kCountMaxSlices threads; thread = (four columns, slice).
template <int GROUPS>
__global__ __launch_bounds__(GROUPS *kCountMaxSlices) void count_and_scan(const int64_t *__restrict__ idx, int64_t n, int n_experts, int64_t per,
                                                                          int n_slices, int32_t *__restrict__ counts, unsigned long long *rows,
                                                                          uint32_t tag, int max_polls) {
  constexpr int nt = GROUPS * kCountMaxSlices, kGroupWaves = kCountMaxSlices / kWave;
  extern __shared__ int32_t hist[];
  __shared__ int32_t of_wave[GROUPS][kGroupWaves][4];
  __shared__ int missing;
  fetch_arguments_now(idx, n, n_experts, per, n_slices, counts, rows, tag, max_polls);
  const int tid = threadIdx.x, lane = tid % kWave, wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int p = blockIdx.x, group = wave_s / kGroupWaves, slice = tid % kCountMaxSlices;
  const int words = padded_experts(n_experts) / 2, quads = words / 2;
  count_slice<1>(idx, n, n_experts, per, p, nt, hist, [&]() {
    if (tid == 0)
      missing = 0;
  });
  auto counted = [&](int e) { return e < n_experts ? (uint32_t)hist[e] : 0u; };
  for (int w = tid; w < words; w += nt)
    agent_store(rows + p * words + w, (unsigned long long)tag << 32 | counted(2 * w) | counted(2 * w + 1) << 16);
  for (int q0 = p * GROUPS; q0 < quads; q0 += n_slices * GROUPS) {
    const int q = q0 + group;
    int32_t c[4] = {};
    if (q < quads) {
      u32x4 v{};
      if (!poll_pair(v, rows + min(slice, n_slices - 1) * words + 2 * q, tag, max_polls))
        missing = 1;
      if (slice < n_slices) {
        c[0] = (int32_t)(v.x & 0xffffu), c[1] = (int32_t)(v.x >> 16);
        c[2] = (int32_t)(v.z & 0xffffu), c[3] = (int32_t)(v.z >> 16);
      }
    }
    __syncthreads();
    if (missing) {   // words did not come: the columns are counted here, slice by slice
      if (tid == 0)
        atomicAdd(&g_count_recounts, 1);
      for (int i = tid; i < 4 * nt; i += nt)
        hist[i] = 0;
      __syncthreads();
      for (int64_t i = tid; i < n; i += nt) {
        const int64_t e = idx[i] - 4 * q0;
        if ((uint64_t)e < 4 * GROUPS && e + 4 * q0 < n_experts)
          atomicAdd(&hist[((int)e / 4 * kCountMaxSlices + (int)(i / per)) * 4 + (int)e % 4], 1);
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < 4; ++j)
        c[j] = hist[4 * tid + j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      c[j] = wave_inclusive_scan(c[j]);
    if (lane == kWave - 1)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        of_wave[group][wave_s % kGroupWaves][j] = c[j];
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kGroupWaves - 1; ++w)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        c[j] += w < wave_s % kGroupWaves ? of_wave[group][w][j] : 0;
    if (q < quads && slice < n_slices) {
      int32_t *to = counts + (int64_t)slice * n_experts + 4 * q;
      if (n_experts % 4 == 0 && (reinterpret_cast<uintptr_t>(counts) & 15) == 0) {
        *reinterpret_cast<int4 *>(to) = int4{c[0], c[1], c[2], c[3]};
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (4 * q + j < n_experts)
            to[j] = c[j];
      }
    }
    __syncthreads();
  }
}

// Test hook (lplb_count_inject_fault): if the next histogram with running sums is one launch, it waits for nothing, every slice counts for itself.
static std::atomic<bool> g_count_fault{false};
static std::atomic<long long> g_one_launch_counts{0};
// *done = false: not a case for one launch; nothing was enqueued.  (A launch that is captured would carry its tag again when it is replayed.)
static int try_count_and_scan(const int64_t *idx, int64_t n, int n_experts, int n_blocks, int32_t *counts, hipStream_t s, unsigned flags, int max_polls,
                              bool *done) {
  const int64_t per = slice_len(n, n_blocks);
  if (n_blocks > kCountMaxSlices || n_experts > kCountMaxExperts || per > kCountMaxSlice)
    return LPLB_OK;
  const int64_t batches = (per / 2 + kLoadsInFlight - 1) / kLoadsInFlight;   // (threads as for launch_slice_histogram)
  const int groups = batches <= kCountMaxSlices ? 1 : 2, quads_of_a_round = n_blocks * groups;
  if ((padded_experts(n_experts) / 4 + quads_of_a_round - 1) / quads_of_a_round > most_count_rounds(groups))
    return LPLB_OK;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess) {
    (void)hipGetLastError();   // (the launch behind this looks at it)
    return LPLB_OK;
  }
  if (capture != hipStreamCaptureStatusNone)
    return LPLB_OK;
  static std::atomic<unsigned long long *> known[64];
  static std::atomic<uint32_t> launches[64];
  int dev = -1;
  LPLB_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64)
    return LPLB_OK;
  unsigned long long *words = known[dev].load(std::memory_order_acquire);
  if (!words) {
    if (hipGetSymbolAddress(reinterpret_cast<void **>(&words), HIP_SYMBOL(g_count_words)) != hipSuccess) {
      (void)hipGetLastError();
      return LPLB_OK;
    }
    known[dev].store(words, std::memory_order_release);
  }
  // (a word's tag is told from a later one's by its sign: after 2^31 launches the two-launch form takes over for good)
  uint32_t number = launches[dev].load(std::memory_order_relaxed);
  do {
    if (number >= (uint32_t)INT32_MAX)
      return LPLB_OK;
  } while (!launches[dev].compare_exchange_weak(number, number + 1, std::memory_order_relaxed));
  words += (size_t)(number % kCountRegions) * kCountRegionWords;
  const auto go = [&](auto kernel) {
    const int threads = groups * kCountMaxSlices;
    const size_t ints = std::max(n_experts, 4 * threads);
    launch_with_flags(kernel, dim3(n_blocks), dim3(threads), ints * sizeof(int32_t), s, flags, idx, n, n_experts, per, n_blocks, counts, words,
                      number + 1, max_polls);
  };
  if (groups == 1)
    go(count_and_scan<1>);
  else
    go(count_and_scan<2>);
  LPLB_HIP_TRY(hipGetLastError());
  g_one_launch_counts.fetch_add(1, std::memory_order_relaxed);
  *done = true;
  return LPLB_OK;
}

// ---- totals only, for short batches: one launch, nothing shared between workgroups ----
// A workgroup owns kOwned experts and reads the whole batch; what it counts is final, so there is no
// second kernel, no atomic between workgroups and nothing to clear.  Every workgroup pulls all n indices
// through its CU (64 bytes per clock), which bounds the batch this pays for: 65536 indices take about as
// long as the launch itself, against two launches for histogram and scan.  A lane keeps four counters;
// the values of a batch of loads are first added up in one register, a byte per owned expert.
constexpr int kOwned = 4;
constexpr int64_t kTotalsMaxIndices = LPLB_COUNT_TOTALS_MAX_INDICES;   // per call; beyond, the two-kernel form is faster
constexpr int kTotalsMaxExperts = LPLB_COUNT_TOTALS_MAX_EXPERTS;

__global__ __launch_bounds__(1024) void expert_totals(const int64_t *__restrict__ idx, int64_t n, int n_experts,
                                                      int32_t *__restrict__ totals) {
  __shared__ int32_t per_wave[16][kOwned];
  fetch_arguments_now(idx, n, n_experts, totals);
  typedef long long i64x2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x, nt = blockDim.x;
  const int64_t base = (int64_t)blockIdx.x * kOwned;
  // one byte per owned expert: 1 << (8 * (v - base)) for a value this workgroup owns, else 0
  auto key = [&](int64_t v) -> uint32_t {
    const uint64_t rel = (uint64_t)(v - base);
    return rel < (uint64_t)kOwned && v < n_experts ? 1u << (8 * (uint32_t)rel) : 0u;
  };
  const int64_t head = (n > 0 && (reinterpret_cast<uintptr_t>(idx) & 8)) ? 1 : 0;   // (see slice_histogram)
  const int64_t n_pairs = (n - head) >> 1;
  const i64x2 *pairs = reinterpret_cast<const i64x2 *>(idx + head);
  uint32_t mine[kOwned] = {};
  for (int64_t i0 = tid; i0 < n_pairs; i0 += (int64_t)nt * kLoadsInFlight) {
    i64x2 v[kLoadsInFlight];
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      const int64_t i = i0 + (int64_t)u * nt;
      v[u] = i < n_pairs ? pairs[i] : i64x2{-1, -1};
    }
    uint32_t packed = 0;   // at most 2 * kLoadsInFlight per byte
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u)
      packed += key(v[u].x) + key(v[u].y);
#pragma unroll
    for (int k = 0; k < kOwned; ++k)
      mine[k] += (packed >> (8 * k)) & 0xffu;
  }
  if (tid == 0) {
    uint32_t packed = head ? key(idx[0]) : 0u;
    if ((n - head) & 1)
      packed += key(idx[n - 1]);
#pragma unroll
    for (int k = 0; k < kOwned; ++k)
      mine[k] += (packed >> (8 * k)) & 0xffu;
  }
  // butterfly over the wave, the four counters side by side
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    uint32_t other[kOwned];
#pragma unroll
    for (int k = 0; k < kOwned; ++k)
      other[k] = bpermute(mine[k], lane_id() ^ off);
#pragma unroll
    for (int k = 0; k < kOwned; ++k)
      mine[k] += other[k];
  }
  if (tid % kWave == 0)
#pragma unroll
    for (int k = 0; k < kOwned; ++k)
      per_wave[tid / kWave][k] = (int32_t)mine[k];
  __syncthreads();
  if (tid < kOwned && base + tid < n_experts) {
    int32_t sum = 0;
    for (int w = 0; w < nt / kWave; ++w)
      sum += per_wave[w][tid];
    totals[base + tid] = sum;
  }
}

// Enqueues the histogram alone: rows of counts that are not summed over the slices yet, and kNoTotal into no_totals.
int enqueue_histogram(const int64_t *idx, int64_t n_elements, int n_experts, int n_blocks, int32_t *counts_by_block,
                      int32_t *no_totals, hipStream_t s) {
  return launch_slice_histogram<false>(idx, n_elements, n_experts, n_blocks, counts_by_block, no_totals, s, 0u);
}
// Enqueues histogram and prefix.  any_order: the histogram launch does not wait for
// the kernel enqueued just before it on the stream (it still starts after everything
// that kernel waited for); the prefix launch is ordered after both.
int enqueue_count(const int64_t *idx, int64_t n_elements, int n_experts, int n_blocks,
                  int32_t *counts_by_block, hipStream_t s, bool any_order) {
  bool done = false;
  const int max_polls = g_count_fault.load(std::memory_order_relaxed) && g_count_fault.exchange(false) ? 0 : kCountPolls;
  int rc = try_count_and_scan(idx, n_elements, n_experts, n_blocks, counts_by_block, s, any_order ? hipExtAnyOrderLaunch : 0u, max_polls, &done);
  if (rc != LPLB_OK || done)
    return rc;
  rc = launch_slice_histogram<false>(idx, n_elements, n_experts, n_blocks, counts_by_block, nullptr, s,
                                               any_order ? hipExtAnyOrderLaunch : 0u);
  if (rc != LPLB_OK)
    return rc;
  launch(prefix_over_slices, dim3((n_experts + kScanCols - 1) / kScanCols), dim3(kScanThreads), 0, s,
         counts_by_block, n_blocks, n_experts);
  LPLB_HIP_TRY(hipGetLastError());
  return LPLB_OK;
}

} // namespace lplb

extern "C" int lplb_count_idx(const int64_t *idx, int64_t n_elements,
                              int n_experts, int n_blocks,
                              int32_t *counts_by_block, lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(n_elements >= 0 && n_elements <= INT32_MAX, LPLB_EINVAL,
               "count_idx: n_elements=%lld out of range", (long long)n_elements);
  LPLB_REQUIRE(n_experts > 0 && n_blocks > 0, LPLB_EINVAL,
               "count_idx: n_experts=%d n_blocks=%d must be positive", n_experts, n_blocks);
  LPLB_REQUIRE(counts_by_block != nullptr && (idx != nullptr || n_elements == 0), LPLB_EINVAL,
               "count_idx: null pointer");
  LPLB_REQUIRE((reinterpret_cast<uintptr_t>(idx) & 7) == 0, LPLB_EINVAL,
               "count_idx: idx must be 8-byte aligned");
  return enqueue_count(idx, n_elements, n_experts, n_blocks, counts_by_block,
                       static_cast<hipStream_t>(stream), /*any_order=*/false);
}

extern "C" int lplb_count_totals(const int64_t *idx, int64_t n_elements, int n_experts, int32_t *totals,
                                 lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(n_elements >= 0 && n_experts > 0, LPLB_EINVAL, "count_totals: n_elements=%lld n_experts=%d",
               (long long)n_elements, n_experts);
  LPLB_REQUIRE(totals != nullptr && (idx != nullptr || n_elements == 0), LPLB_EINVAL, "count_totals: null pointer");
  LPLB_REQUIRE((reinterpret_cast<uintptr_t>(idx) & 7) == 0, LPLB_EINVAL, "count_totals: idx must be 8-byte aligned");
  LPLB_REQUIRE(n_elements <= kTotalsMaxIndices && n_experts <= kTotalsMaxExperts, LPLB_EUNSUPPORTED,
               "count_totals: serves up to %lld indices and %d experts (use lplb_count_idx beyond)",
               (long long)kTotalsMaxIndices, kTotalsMaxExperts);
  launch(expert_totals, dim3((n_experts + kOwned - 1) / kOwned), dim3(1024), 0, static_cast<hipStream_t>(stream), idx,
         n_elements, n_experts, totals);
  LPLB_HIP_TRY(hipGetLastError());
  return LPLB_OK;
}

extern "C" int lplb_count_totals_add(const int64_t *idx, int64_t n_elements, int n_experts, int32_t *totals,
                                     int32_t *clear, lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(n_elements >= 0 && n_elements <= INT32_MAX && n_experts > 0, LPLB_EINVAL,
               "count_totals_add: n_elements=%lld n_experts=%d", (long long)n_elements, n_experts);
  LPLB_REQUIRE(totals != nullptr && (idx != nullptr || n_elements == 0), LPLB_EINVAL, "count_totals_add: null pointer");
  LPLB_REQUIRE(totals != clear, LPLB_EINVAL, "count_totals_add: totals and clear are the same vector");
  LPLB_REQUIRE(((reinterpret_cast<uintptr_t>(idx) | reinterpret_cast<uintptr_t>(totals)) & 7) == 0, LPLB_EINVAL,
               "count_totals_add: idx and totals must be 8-byte aligned");
  LPLB_REQUIRE(n_elements <= kTotalsMaxIndices, LPLB_EUNSUPPORTED,
               "count_totals_add: serves up to %lld indices (use lplb_count_idx beyond)", (long long)kTotalsMaxIndices);
  // Slices of 8192 indices (1024 threads with four 16-byte loads each): at most 16 of them, because every
  // slice updates every line of the totals and those updates queue up.
  const int64_t wanted = (n_elements + 8191) / 8192;
  const int n_blocks = (int)(wanted < 1 ? 1 : wanted);
  return launch_slice_histogram<true>(idx, n_elements, n_experts, n_blocks, totals, clear,
                                      static_cast<hipStream_t>(stream), 0u);
}

// Measurement aid: the histogram kernel alone (no scan behind it), n_launches times, launch r on idx[r] and
// counts_by_block[r], each recording its own begin and end into start_events[r] / stop_events[r].
extern "C" int lplb_slice_histogram_series(const int64_t *const *idx, int64_t n_elements, int n_experts, int n_blocks,
                                           int32_t *const *counts_by_block, int n_launches, void *const *start_events,
                                           void *const *stop_events, lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(idx && counts_by_block && n_launches >= 0, LPLB_EINVAL, "slice_histogram_series: null pointer or negative count");
  LPLB_REQUIRE(n_elements > 0 && n_elements <= INT32_MAX && n_experts > 0 && n_blocks > 0 &&
                   sizeof(int32_t) * (size_t)n_experts <= 64 * 1024,
               LPLB_EINVAL, "slice_histogram_series: n_elements=%lld n_experts=%d n_blocks=%d", (long long)n_elements,
               n_experts, n_blocks);
  for (int r = 0; r < n_launches; ++r) {
    LPLB_REQUIRE(idx[r] && counts_by_block[r] && (reinterpret_cast<uintptr_t>(idx[r]) & 7) == 0, LPLB_EINVAL,
                 "slice_histogram_series: bad pointer in launch %d", r);
    lplb_time_next_launch(start_events ? start_events[r] : nullptr, stop_events ? stop_events[r] : nullptr);
    const int rc = launch_slice_histogram<false>(idx[r], n_elements, n_experts, n_blocks, counts_by_block[r], nullptr,
                                                 static_cast<hipStream_t>(stream), 0u);
    if (rc != LPLB_OK) {
      lplb_time_next_launch(nullptr, nullptr);
      return rc;
    }
  }
  return LPLB_OK;
}

extern "C" int lplb_count_one_launch_count(long long *count) {
  LPLB_REQUIRE(count != nullptr, LPLB_EINVAL, "count_one_launch_count: null pointer");
  *count = lplb::g_one_launch_counts.load(std::memory_order_relaxed);
  return LPLB_OK;
}

extern "C" int lplb_count_recounts(int *count) {
  LPLB_REQUIRE(count != nullptr, LPLB_EINVAL, "count_recounts: null pointer");
  void *at = nullptr;
  LPLB_HIP_TRY(hipGetSymbolAddress(&at, HIP_SYMBOL(lplb::g_count_recounts)));
  LPLB_HIP_TRY(hipDeviceSynchronize());
  LPLB_HIP_TRY(hipMemcpy(count, at, sizeof(int), hipMemcpyDeviceToHost));
  return LPLB_OK;
}

extern "C" int lplb_count_inject_fault(void) {
  lplb::g_count_fault = true;
  return LPLB_OK;
}
