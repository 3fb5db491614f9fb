// Running sums down the slices of a table of counts, for prefix_over_slices (count.hip) and scan_and_solve (plan_kernel.h).
#pragma once
#include "common.h"

namespace lplb {

constexpr int kScanBands = 16;      // bands of rows, one per group of kScanCols lanes
constexpr int kScanRows = 16;       // rows of a band a thread keeps in registers
constexpr int kScanCols = 16;       // experts per workgroup: many small workgroups pull the
                                    // table through many CUs (one CU sustains few misses)
constexpr int kScanThreads = kScanBands * kScanCols;
constexpr int32_t kNoTotal = -1;    // in a vector of totals: not there yet

struct ScanLds {
  int32_t part[kScanBands][kScanCols];
  int32_t carry[kScanCols];
};

// counts[p][e] <- sum_{p' <= p} counts[p'][e] for the experts of workgroup `block` of kScanThreads threads; total(e, sum) is
// called with each expert's sum over all slices.  Thread = (band of rows, expert).  All loads of a band are in flight at
// once (clamped addresses, masked values); band sums meet in LDS; tables with more than 256 slices take several
// sweeps with a running carry.
template <typename Total>
__device__ inline void scan_columns(int32_t *__restrict__ counts, int n_blocks, int n_experts, int block, ScanLds &lds,
                                    Total total) {
  const int col = threadIdx.x % kScanCols, band = threadIdx.x / kScanCols;
  const int e = block * kScanCols + col;
  const bool live = e < n_experts;
  int32_t *column = counts + (live ? e : 0);
  if (band == 0)
    lds.carry[col] = 0;
  __syncthreads();
  for (int row0 = 0; row0 < n_blocks; row0 += kScanBands * kScanRows) {
    const int r0 = row0 + band * kScanRows;
    int32_t v[kScanRows];
#pragma unroll
    for (int k = 0; k < kScanRows; ++k)
      v[k] = column[(int64_t)min(r0 + k, n_blocks - 1) * n_experts];
#pragma unroll
    for (int k = 0; k < kScanRows; ++k)
      v[k] = (live && r0 + k < n_blocks) ? v[k] : 0;
#pragma unroll
    for (int k = 1; k < kScanRows; ++k)
      v[k] += v[k - 1];
    lds.part[band][col] = v[kScanRows - 1];
    __syncthreads();
    int32_t offset = lds.carry[col];
#pragma unroll
    for (int b = 0; b < kScanBands; ++b)
      offset += b < band ? lds.part[b][col] : 0;
    // (rows past the end count nothing, so the last band has the sum over all rows so far)
    if (live && band == kScanBands - 1 && row0 + kScanBands * kScanRows >= n_blocks)
      total(e, v[kScanRows - 1] + offset);
#pragma unroll
    for (int k = 0; k < kScanRows; ++k)
      if (live && r0 + k < n_blocks)
        column[(int64_t)(r0 + k) * n_experts] = v[k] + offset;
    __syncthreads();
    if (band == kScanBands - 1)
      lds.carry[col] = offset + v[kScanRows - 1];
    __syncthreads();
  }
}

} // namespace lplb
