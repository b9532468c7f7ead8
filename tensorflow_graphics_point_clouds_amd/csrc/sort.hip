// Stable descending radix sort of (cell key, point index) pairs: the sort step
// of the reference's grid construction (pylib/pc/Grid.py:56-64,
// tf.argsort(keys, 'DESCENDING'): equal keys keep ascending original index).
//
// LSD radix sort, 8-bit digits, on the complemented digit so that ascending
// digit order is descending key order while stability keeps equal keys in input
// order.  Three launches per pass: (1) per-tile digit histogram in LDS, written
// digit-major, (2) one block per digit scans its row over the tiles, (3) stable scatter:
// every block adds up the 256 row totals in front of its digits, ranks the tile's items --
// wavefront w owns the w-th quarter of the tile, the rank among lanes with the same digit
// comes from ballots, never from atomics, so the order is deterministic --, orders the tile
// by digit in LDS and writes it out in runs (a tile of 2048 items has runs of about eight;
// written in input order every lane is a memory transaction of its own).
// The grid's keys travel as 32-bit words where they fit (they nearly always do), its
// histogram of the first pass comes with the keys, and its last pass also gathers the points:
// 763 k keys of 21 bits took 90 us with 64-bit keys, a scan of three launches per pass and a
// separate gather.
#include "common.h"
#include "fill.h"
#include "small_sort.h"
#include "sort.h"

namespace mccnn {

template <class K>
__device__ __forceinline__ int digit_of(K key, int shift) {
  return (int)((~key >> shift) & (K)(kSortRadix - 1));
}

template <class K>
__global__ void __launch_bounds__(kSortThreads) sort_hist_kernel(int64_t n, int shift, int nb,
                                                                 const K *__restrict__ keys,
                                                                 int *__restrict__ hist) {
  __shared__ int bins[kSortRadix];
  bins[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k) {
    const int64_t i = base + k * kSortThreads + threadIdx.x;
    if (i < n) atomicAdd(&bins[digit_of(keys[i], shift)], 1);
  }
  __syncthreads();
  hist[(int64_t)threadIdx.x * nb + blockIdx.x] = bins[threadIdx.x];
}

// Exclusive scan of 256 per-thread values over the block.
__device__ __forceinline__ int block_exclusive_256(int v, int *wave_sums, int *total) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int incl = wave_inclusive_scan(v);
  if (lane == kWave - 1) wave_sums[wave] = incl;
  __syncthreads();
  int carry = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < kSortThreads / kWave; ++w) {
    carry += w < wave ? wave_sums[w] : 0;
    sum += wave_sums[w];
  }
  __syncthreads();
  *total = sum;
  return carry + incl - v;
}

// Block d: row d of the histogram becomes its exclusive prefix over the tiles, its total goes
// to totals[d].
__global__ void __launch_bounds__(kSortThreads) sort_row_scan_kernel(int nb, int *__restrict__ hist,
                                                                     int *__restrict__ totals) {
  __shared__ int wave_sums[kSortThreads / kWave];
  int *row = hist + (int64_t)blockIdx.x * nb;
  int carry = 0;
  for (int base = 0; base < nb; base += kSortThreads) {
    const int i = base + threadIdx.x;
    const int v = i < nb ? row[i] : 0;
    int total;
    const int ex = block_exclusive_256(v, wave_sums, &total);
    if (i < nb) row[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// kFirst: the index of an item is its position.  KO: type of the keys written.  D > 0: also
// out_pts[rank] = pts[index], out_bids[rank] = bids[index] (the last pass of a grid).
template <class KI, class KO, bool kFirst, int D>
__global__ void __launch_bounds__(kSortThreads) sort_scatter_kernel(
    int64_t n, int shift, int nb, const KI *__restrict__ keys_in, const int *__restrict__ idx_in,
    const int *__restrict__ hist, const int *__restrict__ totals, KO *__restrict__ keys_out,
    int *__restrict__ idx_out, const float *__restrict__ pts, const int *__restrict__ bids,
    float *__restrict__ out_pts, int *__restrict__ out_bids) {
  __shared__ int start[kSortWaves][kSortRadix];    // counts, then next free position in the tile
  __shared__ int to_global[kSortRadix];            // position in the tile -> in the output
  __shared__ int wave_sums[kSortThreads / kWave];
  __shared__ KI tile_key[kSortTile];
  __shared__ int tile_idx[kSortTile];
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
  const int live_items = n - base < kSortTile ? (int)(n - base) : kSortTile;
  const int first = wave * (kSortTile / kSortWaves);
  KI key[kSortItems];
  int idx[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int i = first + r * kWave + lane;
    key[r] = i < live_items ? keys_in[base + i] : (KI)0;
    idx[r] = kFirst ? (int)(base + i) : (i < live_items ? idx_in[base + i] : 0);
  }
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) start[w][t] = 0;
  const int row_prefix = hist[(int64_t)t * nb + blockIdx.x];
  const int row_total = totals[t];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r)
    if (first + r * kWave + lane < live_items) atomicAdd(&start[wave][digit_of(key[r], shift)], 1);
  __syncthreads();
  int unused;
  const int digit_base = block_exclusive_256(row_total, wave_sums, &unused) + row_prefix;
  int count = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) count += start[w][t];
  int run = block_exclusive_256(count, wave_sums, &unused);
  to_global[t] = digit_base - run;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    const int c = start[w][t];
    start[w][t] = run;
    run += c;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    if (first + r * kWave < live_items) {                // uniform in the wavefront
      const bool live = first + r * kWave + lane < live_items;
      const int d = digit_of(key[r], shift);
      uint64_t same = __ballot(live);                    // lanes with this digit
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        const uint64_t b = __ballot((d >> bit) & 1);
        same &= ((d >> bit) & 1) ? b : ~b;
      }
      const int below = __popcll(same & ((1ull << lane) - 1ull));
      int pos = 0;
      if (live) pos = start[wave][d] + below;
      wave_lds_sync();                                   // every lane has read its position
      if (live && below == 0) start[wave][d] = pos + __popcll(same);
      wave_lds_sync();
      if (live) {
        tile_key[pos] = key[r];
        tile_idx[pos] = idx[r];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int i = r * kSortThreads + t;
    if (i < live_items) {
      const KI k = tile_key[i];
      const int id = tile_idx[i];
      const int64_t dst = (int64_t)to_global[digit_of(k, shift)] + i;
      keys_out[dst] = (KO)k;
      idx_out[dst] = id;
      if constexpr (D > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d) out_pts[dst * D + d] = pts[(int64_t)id * D + d];
        out_bids[dst] = bids[id];
      }
    }
  }
}

// The whole sort in one launch for up to 16 384 keys (small_sort.h).
__global__ void __launch_bounds__(kSmallThreads) sort_small_kernel(
    int n, int bits, const int64_t *__restrict__ keys, int64_t *__restrict__ keys_out,
    int *__restrict__ idx_out) {
  extern __shared__ __align__(16) char lds_raw[];
  SmallSortLds &s = *reinterpret_cast<SmallSortLds *>(lds_raw);
  const int first = small_first(n), last = small_last(n), lane = lane_id();
  int item[kSmallRounds];
  small_sort_any(n, bits, keys, 0, item, s);
#pragma unroll
  for (int r = 0; r < kSmallRounds; ++r) {
    const int i = first + r * kWave + lane;
    if (i < last) {
      keys_out[i] = keys[item[r]];
      idx_out[i] = item[r];
    }
  }
}

// keys[m] = num_pts - 1 - neighbour id (descending key order = ascending id), and
// the number of pairs of each point.
__global__ void __launch_bounds__(256) transpose_keys_kernel(int64_t m_total, int64_t num_pts,
                                                             const int2 *__restrict__ nbrs,
                                                             int64_t *__restrict__ keys,
                                                             int *__restrict__ counts) {
  for (int64_t m = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; m < m_total;
       m += (int64_t)gridDim.x * blockDim.x) {
    const int n = nbrs[m].x;
    keys[m] = num_pts - 1 - n;
    atomicAdd(&counts[n], 1);
  }
}

SortWorkspace carve_sort_workspace(void *ws, int64_t n) {
  const int64_t nb = (n + kSortTile - 1) / kSortTile;
  char *p = (char *)ws;
  SortWorkspace w;
  size_t off = 0;
  w.keys_tmp = (int64_t *)(p + off);
  off += align256(sizeof(int64_t) * (size_t)n);
  w.idx_tmp = (int *)(p + off);
  off += align256(sizeof(int) * (size_t)n);
  w.hist = (int *)(p + off);
  off += align256(sizeof(int) * (size_t)(kSortRadix * nb));
  w.totals = (int *)(p + off);
  off += align256(sizeof(int) * kSortRadix);
  w.bytes = off;
  return w;
}

// One pass over 64-bit or 32-bit keys; the histogram of a first pass may be there already.
template <class KI, class KO, bool kFirst, int D>
static int sort_pass(hipStream_t s, int64_t n, int shift, bool have_hist, const KI *kin,
                     const int *iin, KO *kout, int *iout, const SortWorkspace &w,
                     const SortedPoints &g) {
  const int nb = (int)((n + kSortTile - 1) / kSortTile);
  if (!have_hist) {
    hipLaunchKernelGGL((sort_hist_kernel<KI>), dim3(nb), dim3(kSortThreads), 0, s, n, shift, nb,
                       kin, w.hist);
    MCCNN_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(sort_row_scan_kernel, dim3(kSortRadix), dim3(kSortThreads), 0, s, nb, w.hist,
                     w.totals);
  MCCNN_LAUNCH_CHECK();
  hipLaunchKernelGGL((sort_scatter_kernel<KI, KO, kFirst, D>), dim3(nb), dim3(kSortThreads), 0, s,
                     n, shift, nb, kin, iin, w.hist, w.totals, kout, iout, g.points, g.batch_ids,
                     g.points_out, g.batch_ids_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

template <int D>
static int sort_grid_keys_d(hipStream_t s, int64_t n, int bits, unsigned *keys32,
                            const SortWorkspace &w, int64_t *keys_out, int *idx_out,
                            const SortedPoints &g) {
  const int passes = (bits + 7) / 8;
  // the 32-bit keys ping-pong between keys32 and the workspace, the indices between the
  // workspace and the output so that the last pass lands there
  unsigned *kbuf[2] = {(unsigned *)w.keys_tmp, keys32};
  int *ibuf[2] = {passes % 2 ? idx_out : w.idx_tmp, passes % 2 ? w.idx_tmp : idx_out};
  const unsigned *kin = keys32;
  const int *iin = nullptr;
  for (int p = 0; p < passes; ++p) {
    const bool last = p == passes - 1;
    unsigned *ko = kbuf[p & 1];
    int *io = ibuf[p & 1];
    int rc;
    if (p == 0)
      rc = last ? sort_pass<unsigned, int64_t, true, D>(s, n, 0, true, kin, iin, keys_out, io, w, g)
                : sort_pass<unsigned, unsigned, true, 0>(s, n, 0, true, kin, iin, ko, io, w, g);
    else
      rc = last ? sort_pass<unsigned, int64_t, false, D>(s, n, 8 * p, false, kin, iin, keys_out,
                                                         io, w, g)
                : sort_pass<unsigned, unsigned, false, 0>(s, n, 8 * p, false, kin, iin, ko, io, w,
                                                          g);
    if (rc != MCCNN_OK) return rc;
    kin = ko;
    iin = io;
  }
  return MCCNN_OK;
}

int sort_grid_keys(hipStream_t s, int num_dims, int64_t n, int bits, unsigned *keys32,
                   const SortWorkspace &w, int64_t *keys_out, int *idx_out,
                   const SortedPoints &g) {
  int rc = MCCNN_OK;
  MCCNN_DIM_SWITCH(num_dims, rc = sort_grid_keys_d<D>(s, n, bits, keys32, w, keys_out, idx_out, g));
  return rc;
}

int sort_order32(hipStream_t s, int64_t n, unsigned *keys32, const SortWorkspace &w,
                 int *idx_out) {
  unsigned *kbuf[2] = {(unsigned *)w.keys_tmp, keys32};
  int *ibuf[2] = {w.idx_tmp, idx_out};              // four passes: the last lands in idx_out
  const unsigned *kin = keys32;
  const int *iin = nullptr;
  const SortedPoints none = {};
  for (int p = 0; p < 4; ++p) {
    unsigned *ko = kbuf[p & 1];
    int *io = ibuf[p & 1];
    int rc = p == 0 ? sort_pass<unsigned, unsigned, true, 0>(s, n, 0, false, kin, iin, ko, io, w,
                                                             none)
                    : sort_pass<unsigned, unsigned, false, 0>(s, n, 8 * p, false, kin, iin, ko, io,
                                                              w, none);
    if (rc != MCCNN_OK) return rc;
    kin = ko;
    iin = io;
  }
  return MCCNN_OK;
}

}  // namespace mccnn

using namespace mccnn;

extern "C" size_t mccnn_sort_keys_workspace_bytes(int64_t num_pts) {
  if (num_pts < 0) num_pts = 0;
  return carve_sort_workspace(nullptr, num_pts).bytes;
}

extern "C" int mccnn_sort_keys_descending(mccnn_stream_t stream, int64_t num_pts, int key_bits,
                                          const int64_t *keys, int64_t *sorted_keys_out,
                                          int32_t *sorted_indices_out, void *workspace,
                                          size_t workspace_bytes) {
  MCCNN_REQUIRE(num_pts >= 0 && num_pts < ((int64_t)1 << 31),
                "sort_keys expects 0 <= num_pts < 2^31");
  MCCNN_REQUIRE(key_bits >= 1 && key_bits <= 64, "sort_keys expects key_bits in [1, 64]");
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(keys && sorted_keys_out && sorted_indices_out && workspace,
                "sort_keys received a null tensor");
  MCCNN_REQUIRE((const void *)keys != (const void *)sorted_keys_out,
                "sort_keys output must not alias the input");
  const SortWorkspace w = carve_sort_workspace(workspace, num_pts);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "sort_keys workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  hipStream_t s = as_stream(stream);
  const int passes = (key_bits + 7) / 8;
  // Ping-pong so that the last pass lands in the caller's buffers.
  int64_t *kbuf[2];
  int *ibuf[2];
  if (passes % 2 == 1) {
    kbuf[0] = (int64_t *)sorted_keys_out; ibuf[0] = sorted_indices_out;
    kbuf[1] = w.keys_tmp;                 ibuf[1] = w.idx_tmp;
  } else {
    kbuf[0] = w.keys_tmp;                 ibuf[0] = w.idx_tmp;
    kbuf[1] = (int64_t *)sorted_keys_out; ibuf[1] = sorted_indices_out;
  }
  if (num_pts <= kSmallMax) {
    MCCNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(sort_small_kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)sizeof(SmallSortLds)));
    hipLaunchKernelGGL(sort_small_kernel, dim3(1), dim3(kSmallThreads), sizeof(SmallSortLds), s,
                       (int)num_pts, key_bits, (const int64_t *)keys, (int64_t *)sorted_keys_out,
                       sorted_indices_out);
    MCCNN_LAUNCH_CHECK();
    return MCCNN_OK;
  }
  const int64_t *kin = (const int64_t *)keys;
  const int *iin = nullptr;
  const SortedPoints none = {};
  for (int p = 0; p < passes; ++p) {
    int64_t *kout = kbuf[p & 1];
    int *iout = ibuf[p & 1];
    int rc = p == 0 ? sort_pass<int64_t, int64_t, true, 0>(s, num_pts, 0, false, kin, iin, kout,
                                                           iout, w, none)
                    : sort_pass<int64_t, int64_t, false, 0>(s, num_pts, 8 * p, false, kin, iin,
                                                            kout, iout, w, none);
    if (rc != MCCNN_OK) return rc;
    kin = kout;
    iin = iout;
  }
  return MCCNN_OK;
}

// ------------------------------------------------- transposed pair lists ----

namespace mccnn {
struct TransposeWorkspace {
  int64_t *keys;
  int64_t *sorted_keys;
  void *sort_ws;
  size_t sort_ws_bytes;
  int *scan_scratch;
  int64_t *total;
  size_t bytes;
};

static TransposeWorkspace carve_transpose_workspace(void *ws, int64_t m, int64_t n) {
  char *p = (char *)ws;
  TransposeWorkspace w;
  size_t off = 0;
  w.keys = (int64_t *)(p + off); off += align256(sizeof(int64_t) * (size_t)m);
  w.sorted_keys = (int64_t *)(p + off); off += align256(sizeof(int64_t) * (size_t)m);
  w.sort_ws = p + off;
  w.sort_ws_bytes = carve_sort_workspace(nullptr, m).bytes;
  off += align256(w.sort_ws_bytes);
  w.scan_scratch = (int *)(p + off); off += align256(sizeof(int) * scan_scratch_ints(n));
  w.total = (int64_t *)(p + off); off += 256;
  w.bytes = off;
  return w;
}
}  // namespace mccnn

extern "C" size_t mccnn_transpose_neighbors_workspace_bytes(int64_t num_neighbors,
                                                            int64_t num_pts) {
  if (num_neighbors < 0) num_neighbors = 0;
  if (num_pts < 0) num_pts = 0;
  return carve_transpose_workspace(nullptr, num_neighbors, num_pts).bytes;
}

extern "C" int mccnn_transpose_neighbors(mccnn_stream_t stream, int64_t num_neighbors,
                                         const int32_t *neighbors, int64_t num_pts,
                                         void *workspace, size_t workspace_bytes,
                                         int32_t *point_ranges_out, int32_t *pair_order_out) {
  MCCNN_REQUIRE(num_neighbors >= 0 && num_neighbors < ((int64_t)1 << 31) && num_pts >= 0 &&
                    num_pts < ((int64_t)1 << 31),
                "transpose_neighbors expects sizes in [0, 2^31)");
  hipStream_t s = as_stream(stream);
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(point_ranges_out, "transpose_neighbors received a null tensor");
  int rc = fill_zero(s, point_ranges_out, sizeof(int32_t) * (size_t)num_pts);
  if (rc != MCCNN_OK) return rc;
  if (num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(neighbors && workspace && pair_order_out,
                "transpose_neighbors received a null tensor");
  const TransposeWorkspace w = carve_transpose_workspace(workspace, num_neighbors, num_pts);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "transpose_neighbors workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  int64_t work = num_neighbors > ((int64_t)1 << 26) ? ((int64_t)1 << 26) : num_neighbors;
  hipLaunchKernelGGL(transpose_keys_kernel, dim3(blocks_for(work, 256)), dim3(256), 0, s,
                     num_neighbors, num_pts, (const int2 *)neighbors, w.keys, point_ranges_out);
  MCCNN_LAUNCH_CHECK();
  int bits = 1;
  while (((int64_t)1 << bits) < num_pts) ++bits;
  rc = mccnn_sort_keys_descending(stream, num_neighbors, bits, w.keys, w.sorted_keys,
                                  pair_order_out, w.sort_ws, w.sort_ws_bytes);
  if (rc != MCCNN_OK) return rc;
  return inclusive_scan_i32(s, num_pts, point_ranges_out, w.scan_scratch, w.total);
}
