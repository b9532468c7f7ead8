// Device-memory helpers shared by the op files (defined in util.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace mccnn {

// Zeroes `bytes` bytes (a multiple of 4) at `ptr` (4-byte aligned) with a fill
// kernel rather than hipMemsetAsync, so that callers may capture the stream
// into a graph.
int fill_zero(hipStream_t stream, void *ptr, size_t bytes);

// In-place scan of counts[0..n): on return counts[i] holds the INCLUSIVE prefix
// sum (the end offset of segment i) and *total_dev the grand total (int64).
// block_sums is scratch for scan_scratch_ints(n) ints.  The total is one atomic store of system
// scope, so that it may go to pinned memory that the host looks at while the kernel runs; with
// `flag` (device or pinned memory that kernels before have written) it carries kScanFlag where
// *flag is not zero: what the host then needs to know is in the one word that it looks at.
constexpr int64_t kScanFlag = (int64_t)1 << 62;        // (totals of int32 counts are smaller)
size_t scan_scratch_ints(int64_t n);
int inclusive_scan_i32(hipStream_t stream, int64_t n, int *counts, int *block_sums,
                       int64_t *total_dev, const int64_t *flag = nullptr);

}  // namespace mccnn
