// Error reporting, fill and prefix-sum helpers of libmccnn_hip.so.
#include <stdarg.h>

#include <chrono>

#include "common.h"
#include "fill.h"

namespace mccnn {

static thread_local char g_error[512] = "";

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

__global__ void __launch_bounds__(256) fill_zero_kernel(uint32_t *p, size_t words) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < words;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

int fill_zero(hipStream_t stream, void *ptr, size_t bytes) {
  if (bytes == 0) return MCCNN_OK;
  size_t words = bytes / 4;
  unsigned grid = (unsigned)((words + 1023) / 1024);
  if (grid > 65535u * 4) grid = 65535u * 4;
  if (grid < 1) grid = 1;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(grid), dim3(256), 0, stream, (uint32_t *)ptr, words);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

// ------------------------------------------------------------ prefix sum ----
// Up to kScanSingleMax values: one launch, one block.  Up to 4 M values: two launches, no
// inter-block waiting: (1) each block writes the sum of its tile, (2) each block adds up the
// tile sums in front of its own (at most 2048 values, from L2) and rescans its tile.  Beyond
// that a launch in between scans the tile sums.  A launch costs 2 to 4 us, as much as the
// bytes of a million values, so the number of launches is what the short forms save (16 384
// values: 9.1 us in rounds of 8 scalar loads per thread, 4 us with 16-byte loads; 100 000
// values 11 us with three launches, 7 us with two).
// The scanned values are int32 (pair counts are int32 in the op contract); tile sums and the
// grand total are formed in 64 bits and a sum that does not fit saturates, so that a total of
// 2^31 - 1 or more is always reported as at least 2^31 - 1 and the callers can refuse it
// instead of working on wrapped offsets.

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;
constexpr int kScanMaxOwnPrefix = 2048;        // tile sums a block adds up by itself

size_t scan_scratch_ints(int64_t n) { return (size_t)((n + kScanTile - 1) / kScanTile) + 1; }

constexpr long long kScanMax = 0x7fffffffLL;

__device__ __forceinline__ int saturate_i32(long long v) {
  return (int)(v > kScanMax ? kScanMax : v);
}

template <int kThreads>
__device__ __forceinline__ long long block_exclusive_scan_i64(long long v, long long *total) {
  __shared__ long long wave_sums[kThreads / kWave];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  long long incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const long long t = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += t;
  }
  if (lane == kWave - 1) wave_sums[wave] = incl;
  __syncthreads();
  long long carry = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < kThreads / kWave; ++w) {
    if (w < wave) carry += wave_sums[w];
    sum += wave_sums[w];
  }
  __syncthreads();
  *total = sum;
  return carry + incl - v;
}

// kItems values from `base` on, 0 past n; 16-byte loads where all of them exist and the array
// is aligned to 16 bytes (`vec`).
template <int kItems>
__device__ __forceinline__ void load_items(const int *__restrict__ src, int64_t base, int64_t n,
                                           bool vec, int *v) {
  if (vec && base + kItems <= n) {
#pragma unroll
    for (int k = 0; k < kItems / 4; ++k) {
      const int4 q = reinterpret_cast<const int4 *>(src + base)[k];
      v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < kItems; ++k) v[k] = base + k < n ? src[base + k] : 0;
  }
}

template <int kItems>
__device__ __forceinline__ void store_items(int *__restrict__ dst, int64_t base, int64_t n,
                                            bool vec, const int *v) {
  if (vec && base + kItems <= n) {
#pragma unroll
    for (int k = 0; k < kItems / 4; ++k)
      reinterpret_cast<int4 *>(dst + base)[k] =
          make_int4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
  } else {
#pragma unroll
    for (int k = 0; k < kItems; ++k)
      if (base + k < n) dst[base + k] = v[k];
  }
}

__global__ void __launch_bounds__(kScanThreads) scan_tile_sums_kernel(
    int64_t n, bool vec, const int *__restrict__ counts, int *__restrict__ block_sums) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int v[kScanItems];
  load_items<kScanItems>(counts, base, n, vec, v);
  long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) s += v[k];
  long long total;
  block_exclusive_scan_i64<kScanThreads>(s, &total);
  if (threadIdx.x == 0) block_sums[blockIdx.x] = saturate_i32(total);
}

__device__ __forceinline__ void store_total(int64_t *total_dev, long long total,
                                            const int64_t *flag) {
  if (flag && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0)
    total |= kScanFlag;
  __hip_atomic_store(total_dev, (int64_t)total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Single block: exclusive scan of block_sums[0..nb) in place, total to *total_dev.
__global__ void __launch_bounds__(kScanThreads) scan_block_sums_kernel(int nb, int *block_sums,
                                                                       int64_t *total_dev,
                                                                       const int64_t *flag) {
  long long carry = 0;
  for (int base = 0; base < nb; base += kScanThreads) {
    const int i = base + threadIdx.x;
    const long long v = i < nb ? block_sums[i] : 0;
    long long total;
    const long long ex = block_exclusive_scan_i64<kScanThreads>(v, &total);
    if (i < nb) block_sums[i] = saturate_i32(carry + ex);
    carry += total;
  }
  if (threadIdx.x == 0) store_total(total_dev, carry, flag);
}

// kOwnPrefix: block_sums are the tile sums themselves and the block adds up those in front of
// it (the last block also writes the total); otherwise they have been scanned.
template <bool kOwnPrefix>
__global__ void __launch_bounds__(kScanThreads) scan_apply_kernel(
    int64_t n, bool vec, int *__restrict__ counts, const int *__restrict__ block_sums,
    int64_t *total_dev, const int64_t *flag) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int v[kScanItems];
  load_items<kScanItems>(counts, base, n, vec, v);
  long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) s += v[k];
  long long total, carry;
  if (kOwnPrefix) {
    long long before = 0;
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kScanThreads) before += block_sums[i];
    block_exclusive_scan_i64<kScanThreads>(before, &carry);
  } else {
    carry = block_sums[blockIdx.x];
  }
  long long run = carry + block_exclusive_scan_i64<kScanThreads>(s, &total);
  if (kOwnPrefix && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
    store_total(total_dev, carry + total, flag);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    run += v[k];
    v[k] = saturate_i32(run);
  }
  store_items<kScanItems>(counts, base, n, vec, v);
}

// Short inputs: one block walks tiles of 16 values per thread and carries the running total.
constexpr int kScanSingleThreads = 1024;
constexpr int kScanSingleItems = 16;
constexpr int kScanSingleTile = kScanSingleThreads * kScanSingleItems;
constexpr int64_t kScanSingleMax = 2 * kScanSingleTile;

__global__ void __launch_bounds__(kScanSingleThreads) scan_single_block_kernel(
    int64_t n, bool vec, int *counts, int64_t *total_dev, const int64_t *flag) {
  long long carry = 0;
  for (int64_t tile = 0; tile < n; tile += kScanSingleTile) {
    const int64_t base = tile + (int64_t)threadIdx.x * kScanSingleItems;
    int v[kScanSingleItems];
    load_items<kScanSingleItems>(counts, base, n, vec, v);
    long long s = 0;
#pragma unroll
    for (int k = 0; k < kScanSingleItems; ++k) s += v[k];
    long long total;
    long long run = carry + block_exclusive_scan_i64<kScanSingleThreads>(s, &total);
#pragma unroll
    for (int k = 0; k < kScanSingleItems; ++k) {
      run += v[k];
      v[k] = saturate_i32(run);
    }
    store_items<kScanSingleItems>(counts, base, n, vec, v);
    carry += total;
  }
  if (threadIdx.x == 0) store_total(total_dev, carry, flag);
}

int inclusive_scan_i32(hipStream_t stream, int64_t n, int *counts, int *block_sums,
                       int64_t *total_dev, const int64_t *flag) {
  const int nb = (int)((n + kScanTile - 1) / kScanTile);
  if (nb == 0) {
    return fill_zero(stream, total_dev, sizeof(int64_t));
  }
  const bool vec = reinterpret_cast<uintptr_t>(counts) % 16 == 0;
  if (n <= kScanSingleMax) {
    hipLaunchKernelGGL(scan_single_block_kernel, dim3(1), dim3(kScanSingleThreads), 0, stream, n,
                       vec, counts, total_dev, flag);
    MCCNN_LAUNCH_CHECK();
    return MCCNN_OK;
  }
  hipLaunchKernelGGL(scan_tile_sums_kernel, dim3(nb), dim3(kScanThreads), 0, stream, n, vec,
                     counts, block_sums);
  MCCNN_LAUNCH_CHECK();
  if (nb <= kScanMaxOwnPrefix) {
    hipLaunchKernelGGL(scan_apply_kernel<true>, dim3(nb), dim3(kScanThreads), 0, stream, n, vec,
                       counts, block_sums, total_dev, flag);
    MCCNN_LAUNCH_CHECK();
    return MCCNN_OK;
  }
  hipLaunchKernelGGL(scan_block_sums_kernel, dim3(1), dim3(kScanThreads), 0, stream, nb,
                     block_sums, total_dev, flag);
  MCCNN_LAUNCH_CHECK();
  hipLaunchKernelGGL(scan_apply_kernel<false>, dim3(nb), dim3(kScanThreads), 0, stream, n, vec,
                     counts, block_sums, total_dev, (const int64_t *)nullptr);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

template <class T>
static int wait_for_values(hipStream_t s, const T *values, int n) {
  const auto start = std::chrono::steady_clock::now();
  for (int i = 0; i < n;) {
    if (__atomic_load_n(&values[i], __ATOMIC_ACQUIRE) != (T)-1) {
      ++i;
      continue;
    }
    __builtin_ia32_pause();
    if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(20)) {
      MCCNN_HIP_CHECK(hipStreamSynchronize(s));
      return MCCNN_OK;
    }
  }
  return MCCNN_OK;
}

int wait_for_host_values(hipStream_t s, const int64_t *values, int n) {
  return wait_for_values(s, values, n);
}
int wait_for_host_values(hipStream_t s, const int32_t *values, int n) {
  return wait_for_values(s, values, n);
}

}  // namespace mccnn

extern "C" const char *mccnn_last_error(void) { return mccnn::g_error; }
extern "C" int mccnn_abi_version(void) { return 1; }
