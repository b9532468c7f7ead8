// Regular-grid stage: bounding boxes and grid shape, cell keys, gathers and the
// 2-D column table.  Integer results must equal the reference's bit for bit, so
// this file is compiled with -ffp-contract=off: every float operation that
// decides a cell index is rounded once, as the op contract states it
// (custom_ops/tfg_custom_ops/shared/cc/kernels/grid_utils.h:63-100).
#include <float.h>

#include "common.h"
#include "fill.h"
#include "small_sort.h"
#include "sort.h"

namespace mccnn {

// ------------------------------------------------------------------ keys ----

template <int D>
__global__ void __launch_bounds__(256) compute_keys_kernel(
    int64_t n, const float *__restrict__ pts, const int *__restrict__ bids,
    const float *__restrict__ smin, const int *__restrict__ num_cells,
    const float *__restrict__ inv_cell, int64_t *__restrict__ keys) {
  const GridShape<D> g = load_shape<D>(num_cells);
  float ic[D];
#pragma unroll
  for (int d = 0; d < D; ++d) ic[d] = inv_cell[d];
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int b = bids[i];
    float p[D], m[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      p[d] = pts[i * D + d];
      m[d] = smin[(int64_t)b * D + d];
    }
    int cell[D];
    cell_of_point<D>(p, m, ic, g, cell);
    keys[i] = key_of_cell<D>(cell, g, b);
  }
}

// --------------------------------------------------------------- gathers ----

template <int D>
__global__ void __launch_bounds__(256) gather_points_kernel(
    int64_t n, const float *__restrict__ pts, const int *__restrict__ bids,
    const int *__restrict__ idx, float *__restrict__ pts_out, int *__restrict__ bids_out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = idx[i];
#pragma unroll
    for (int d = 0; d < D; ++d) pts_out[i * D + d] = pts[j * D + d];
    bids_out[i] = bids[j];
  }
}

__global__ void __launch_bounds__(256) original_ids_kernel(int64_t m,
                                                           const int2 *__restrict__ nbrs,
                                                           const int *__restrict__ sorted_idx,
                                                           int2 *__restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int2 p = nbrs[i];
    out[i] = make_int2(sorted_idx[p.x], p.y);
  }
}

// Rows of the transposed pair table: out[i] = (centre, point) of pair order[i].
__global__ void __launch_bounds__(256) swapped_pairs_kernel(int64_t m,
                                                            const int2 *__restrict__ nbrs,
                                                            const int *__restrict__ order,
                                                            int2 *__restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int2 p = nbrs[order[i]];
    out[i] = make_int2(p.y, p.x);
  }
}

__global__ void __launch_bounds__(256) gather_pdf_kernel(int64_t m, const int2 *__restrict__ nbrs,
                                                         int column, const float *__restrict__ pdf,
                                                         float *__restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int2 p = nbrs[i];
    out[i] = pdf[column == 0 ? p.x : p.y];
  }
}

// Both tables of a neighbourhood at once, column 0 of one and column 1 of the other: small clouds pay for
// launches (three levels of 16 x 1024 points 15.2 us and the gaps of six, 8.7 and those of three;
// 61 k points x 28 pairs 13.0 -> 9.1, 763 k x 37 168 -> 139).
__global__ void __launch_bounds__(256) gather_pdf_both_kernel(
    int64_t m, const int2 *__restrict__ nbrs, const int2 *__restrict__ transposed,
    const float *__restrict__ pdf, float *__restrict__ out, float *__restrict__ out_transposed) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int p = nbrs[i].x, q = transposed[i].y;
    out[i] = pdf[p];
    out_transposed[i] = pdf[q];
  }
}

__global__ void __launch_bounds__(256) gather_i32_kernel(int64_t n, const int *__restrict__ src,
                                                         const int *__restrict__ idx,
                                                         int *__restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = src[idx[i]];
}

// out[i, :] = src[idx[i], :] for rows of 4 * row_vecs floats, 16 bytes per lane.
__global__ void __launch_bounds__(256) gather_rows_kernel(int64_t total, int row_vecs,
                                                          const float4 *__restrict__ src,
                                                          const int *__restrict__ idx,
                                                          float4 *__restrict__ out) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = t / row_vecs;
    const int v = (int)(t - row * row_vecs);
    out[t] = src[(int64_t)idx[row] * row_vecs + v];
  }
}

// ------------------------------------------------------------ grid table ----

// Column of a key in the [B, n0, n1] table: key / prod(n[2:]).
template <int D>
__global__ void __launch_bounds__(256) build_grid_ds_kernel(
    int64_t n, const int64_t *__restrict__ keys, const int *__restrict__ num_cells,
    int2 *__restrict__ ds) {
  int64_t div = 1;
#pragma unroll
  for (int d = 2; d < D; ++d) div *= num_cells[d];
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t col = keys[i] / div;
    if (i > 0 && keys[i - 1] / div != col) ds[col].x = (int)i;
    if (i + 1 == n || keys[i + 1] / div != col) ds[col].y = (int)(i + 1);
  }
}

// ------------------------------------------------ bounding box and shape ----

// Order-preserving map float -> uint32 so that min/max can be taken with
// integer atomics.
__device__ __forceinline__ unsigned enc_float(float f) {
  unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float dec_float(unsigned u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

__global__ void aabb_init_kernel(int count, unsigned *mn, unsigned *mx) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) {
    mn[i] = enc_float(FLT_MAX);
    mx[i] = enc_float(-FLT_MAX);
  }
}

// Running minima / maxima of one cloud over the lanes of a wavefront.
template <int D>
struct Bounds {
  float lo[D], hi[D];
  __device__ __forceinline__ Bounds() { reset(); }
  __device__ __forceinline__ void reset() {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = FLT_MAX;
      hi[d] = -FLT_MAX;
    }
  }
  __device__ __forceinline__ void add(const float *p) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = fminf(lo[d], p[d]);
      hi[d] = fmaxf(hi[d], p[d]);
    }
  }
  // The wavefront's bounds into mn[0..D), mx[0..D) (encoded), then start over.  Inside a row of
  // sixteen lanes by rotations of the row (vector instructions), between the four rows through the
  // lane exchange, whose latency six steps in a row would pay six times.
  template <int kCtrl>
  static __device__ __forceinline__ float rotated(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kCtrl, 0xf, 0xf, false));
  }
  __device__ __forceinline__ void flush(unsigned *mn, unsigned *mx) {
    constexpr int kRor = 0x120;                    // row_ror:n is 0x120 + n
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = fminf(lo[d], rotated<kRor + 8>(lo[d]));
      hi[d] = fmaxf(hi[d], rotated<kRor + 8>(hi[d]));
      lo[d] = fminf(lo[d], rotated<kRor + 4>(lo[d]));
      hi[d] = fmaxf(hi[d], rotated<kRor + 4>(hi[d]));
      lo[d] = fminf(lo[d], rotated<kRor + 2>(lo[d]));
      hi[d] = fmaxf(hi[d], rotated<kRor + 2>(hi[d]));
      lo[d] = fminf(lo[d], rotated<kRor + 1>(lo[d]));
      hi[d] = fmaxf(hi[d], rotated<kRor + 1>(hi[d]));
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int off = kWave / 2; off >= 16; off >>= 1) {
        lo[d] = fminf(lo[d], __shfl_xor(lo[d], off, kWave));
        hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], off, kWave));
      }
      if (lane_id() == 0) {
        atomicMin(&mn[d], enc_float(lo[d]));
        atomicMax(&mx[d], enc_float(hi[d]));
      }
    }
    reset();
  }
};

// 64 more points into the running bounds of cloud `cur`.  Where clouds meet inside the 64 the
// wavefront goes on from one to the next like between iterations; ids that change more often than
// that (clouds not stored one after another) send their points on their own.  (Point by point the
// one iteration at a boundary is 64 atomics on each of the same few addresses: 15 us for the
// boxes of 61 k points in 5 clouds, 7 us now.)  Where ids change more than `together` times in the 64 all
// points go on their own at once.  That pays where they go to LDS (from the second change on: grid of
// 8000 points in 5 shuffled clouds 52 us, 91 with four clouds taken together first, in strips of 23 points 64
// and 77) or to as many clouds as there are lanes (from the fourth on: 600 points in 300 clouds 40 and
// 54 us, 30 k in 64 113 and 117); fewer addresses in memory are worth sparing (100 k points in 5
// shuffled clouds 1460 and 733).  How long a stretch is hardly matters there: the boxes of 763 k points in
// 8 shuffled clouds take 5.67 ms with 256 blocks and 5.70 with 745, those of 300 k points in 20 000
// clouds one after another 77 and 89 us.
template <int D, class Flush, class Direct>
__device__ __forceinline__ void add_points(bool live, int b, const float *p, int together,
                                           Bounds<D> &box, int &cur, Flush &&flush,
                                           Direct &&direct) {
  uint64_t todo = __ballot(live);
  if (todo == __ballot(live && b == cur)) {       // the usual case: all of the cloud at hand
    if (live) box.add(p);
    return;
  }
  const int before = __shfl_up(b, 1, kWave);      // (live lanes are the first ones)
  if (__popcll(__ballot(live && lane_id() > 0 && b != before)) > together) {
    if (live) direct(b, p);
    return;
  }
  for (int runs = 0; todo != 0; ++runs) {
    if (runs == 4) {
      if ((todo >> lane_id()) & 1) direct(b, p);
      return;
    }
    const int b0 = __builtin_amdgcn_readlane(b, __ffsll((unsigned long long)todo) - 1);
    if (b0 != cur) {
      if (cur >= 0) flush(cur, box);
      cur = b0;
    }
    const bool mine = live && b == b0;
    if (mine) box.add(p);
    todo &= ~__ballot(mine);
  }
}

// Bounding boxes of all clouds.  A block takes one contiguous stretch of the points, each of
// its wavefronts a quarter of it.  While the 64 points of an iteration belong to one cloud (the
// usual layout: clouds stored one after another) the lanes keep running minima / maxima in
// registers, reduced over the wavefront when the cloud changes or the stretch ends.  Results
// meet in LDS for the first eight clouds of the stretch, and leave the block as one atomic per
// cloud and dimension: thousands of wavefronts sending their own to the same few addresses
// took 54 us on 763 k points in 8 clouds, the serial rate of an address.
constexpr int kAabbThreads = 256;
constexpr int kAabbLdsClouds = 8;

template <int D>
__global__ void __launch_bounds__(kAabbThreads) aabb_reduce_kernel(
    int64_t n, int64_t per_block, const float *__restrict__ pts, const int *__restrict__ bids,
    int batch, unsigned *mn, unsigned *mx) {
  __shared__ unsigned lmn[kAabbLdsClouds * D], lmx[kAabbLdsClouds * D];
  const unsigned none_lo = enc_float(FLT_MAX), none_hi = enc_float(-FLT_MAX);
  for (int t = threadIdx.x; t < kAabbLdsClouds * D; t += kAabbThreads) {
    lmn[t] = none_lo;
    lmx[t] = none_hi;
  }
  __syncthreads();
  const int64_t block_first = (int64_t)blockIdx.x * per_block;
  const int b_first = block_first < n ? bids[block_first] : 0;
  const int64_t per_wave = per_block / (kAabbThreads / kWave);
  const int64_t first = block_first + (threadIdx.x / kWave) * per_wave;
  const int64_t last = first + per_wave < n ? first + per_wave : n;
  auto flush = [&](int b, Bounds<D> &box) {
    const int e = b - b_first;
    if (e >= 0 && e < kAabbLdsClouds) box.flush(lmn + e * D, lmx + e * D);
    else box.flush(mn + (int64_t)b * D, mx + (int64_t)b * D);
  };
  Bounds<D> box;
  int cur = -1;                     // cloud of the running minima / maxima (wave-uniform)
  // Four times 64 points in flight: one after the other they are a chain of waits (eight: the same).
  constexpr int kAhead = 4;
  for (int64_t base = first; base < last; base += kAhead * kWave) {
    int b[kAhead];
    float p[kAhead][D];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {            // past the end: the last point again
      const int64_t at = base + u * kWave + lane_id(), i = at < last ? at : last - 1;
      b[u] = bids[i];
#pragma unroll
      for (int d = 0; d < D; ++d) p[u][d] = pts[i * D + d];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      add_points<D>(base + u * kWave + lane_id() < last, b[u], p[u], batch >= kWave ? 3 : kWave, box,
                    cur, flush, [&](int b, const float *p) {
#pragma unroll
                      for (int d = 0; d < D; ++d) {
                        atomicMin(&mn[(int64_t)b * D + d], enc_float(p[d]));
                        atomicMax(&mx[(int64_t)b * D + d], enc_float(p[d]));
                      }
                    });
  }
  if (cur >= 0) flush(cur, box);
  __syncthreads();
  for (int t = threadIdx.x; t < kAabbLdsClouds * D; t += kAabbThreads) {
    const int64_t o = (int64_t)b_first * D + t;
    if (lmn[t] != none_lo) atomicMin(&mn[o], lmn[t]);
    if (lmx[t] != none_hi) atomicMax(&mx[o], lmx[t]);
  }
}

// min - 1e-9f, max + 1e-9f, scaled minimum and cells of one (cloud, dimension), in the fp32
// expressions of the reference's Python glue.
struct CellExtent {
  float lo, hi, smin;
  int cells;
};
__device__ __forceinline__ CellExtent finalize_extent(unsigned mn, unsigned mx, float cell) {
  CellExtent e;
  e.lo = dec_float(mn) - 1e-9f;
  e.hi = dec_float(mx) + 1e-9f;
  const float size = e.hi - e.lo;
  e.cells = (int)ceilf(size / cell);
  e.smin = e.lo / cell;
  return e;
}

// One block: boxes decoded in place, grid shape, scaled minima, reciprocal cell size.
template <int D>
__global__ void __launch_bounds__(256) grid_finalize_kernel(int batch,
                                                            const float *__restrict__ cell,
                                                            float *aabb_min, float *aabb_max,
                                                            int *num_cells, float *smin,
                                                            float *inv_cell) {
  __shared__ int nc[D];
  if (threadIdx.x < D) nc[threadIdx.x] = 1;
  __syncthreads();
  for (int t = threadIdx.x; t < batch * D; t += blockDim.x) {
    const int d = t % D;
    const CellExtent e = finalize_extent(reinterpret_cast<unsigned *>(aabb_min)[t],
                                         reinterpret_cast<unsigned *>(aabb_max)[t], cell[d]);
    aabb_min[t] = e.lo;
    aabb_max[t] = e.hi;
    smin[t] = e.smin;
    atomicMax(&nc[d], e.cells);
  }
  __syncthreads();
  if (threadIdx.x < D) {
    num_cells[threadIdx.x] = nc[threadIdx.x];
    inv_cell[threadIdx.x] = 1.0f / cell[threadIdx.x];
  }
}

// Largest batch * D whose extents a block keeps in LDS.
constexpr int kGridLdsExtents = 512;

// What a grid is made of; arrays of outputs in the caller's hands.
struct GridArrays {
  float *aabb_min, *aabb_max;
  int *num_cells;
  float *smin, *inv_cell;
  int64_t *keys, *sorted_keys;
  int *sorted_idx;
  float *sorted_pts;
  int *sorted_bids;
};

// Grid shape and keys in one launch, from the encoded boxes mn, mx: every block derives the
// shape from the batch * D extents for itself (a few dozen values from L2), block 0 writes it
// out (and to shape_host, pinned host memory the caller waits for).  Beside the 64-bit keys the
// block stores their lower halves and the digit histogram of its tile for the sort.
template <int D>
__global__ void __launch_bounds__(kSortThreads) grid_keys_kernel(
    int64_t n, int batch, int nb, const float *__restrict__ pts, const int *__restrict__ bids,
    const float *__restrict__ cell, const unsigned *__restrict__ mn,
    const unsigned *__restrict__ mx, GridArrays g, unsigned *__restrict__ keys32,
    int *__restrict__ hist, int *shape_host) {
  __shared__ int nc[D];
  __shared__ float smin[kGridLdsExtents];
  __shared__ int bins[kSortRadix];
  bins[threadIdx.x] = 0;
  if (threadIdx.x < D) nc[threadIdx.x] = 1;
  __syncthreads();
  for (int t = threadIdx.x; t < batch * D; t += kSortThreads) {
    const CellExtent e = finalize_extent(mn[t], mx[t], cell[t % D]);
    smin[t] = e.smin;
    atomicMax(&nc[t % D], e.cells);
    if (blockIdx.x == 0) {
      g.aabb_min[t] = e.lo;
      g.aabb_max[t] = e.hi;
      g.smin[t] = e.smin;
    }
  }
  __syncthreads();
  GridShape<D> shape;
  float ic[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    shape.n[d] = nc[d];
    ic[d] = 1.0f / cell[d];
  }
  if (blockIdx.x == 0 && threadIdx.x < D) {
    g.num_cells[threadIdx.x] = nc[threadIdx.x];
    g.inv_cell[threadIdx.x] = ic[threadIdx.x];
    if (shape_host)
      __hip_atomic_store(&shape_host[threadIdx.x], nc[threadIdx.x], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k) {
    const int64_t i = base + k * kSortThreads + threadIdx.x;
    if (i < n) {
      const int b = bids[i];
      float p[D];
#pragma unroll
      for (int d = 0; d < D; ++d) p[d] = pts[i * D + d];
      int c[D];
      cell_of_point<D>(p, smin + b * D, ic, shape, c);
      const int64_t key = key_of_cell<D>(c, shape, b);
      g.keys[i] = key;
      keys32[i] = (unsigned)key;
      atomicAdd(&bins[(~(unsigned)key) & (kSortRadix - 1)], 1);
    }
  }
  __syncthreads();
  hist[(int64_t)threadIdx.x * nb + blockIdx.x] = bins[threadIdx.x];
}

// The whole grid of a small cloud (up to 16 384 points) in one launch of one block: boxes,
// shape, keys, sort (small_sort.h), gathers.  As separate launches the same steps take 57 us of
// kernels on 16 x 1024 points, plus the gaps between eight launches and a host round trip for
// the grid shape.  kOrderOnly: the points are centres of a grid that is there already
// (num_cells, smin, inv_cell given); their order by cell key, and coordinates and cloud ids in
// that order.
//
// kByCloud: the sort is bound by the instructions of one compute unit.  A batch whose clouds
// follow one another (ids in ascending order, as clouds are put together, or in descending order,
// as a grid leaves them for the next level) is sorted cloud by cloud, a block each: the cloud is
// the highest part of the key, so the points of cloud b go to the places before those of b - 1, by
// the cell part of their keys.  Every block looks at all points for the boxes and at all ids for
// the order; out of it, block 0 sorts everything.  16 384 points in 1 / 2 / 4 / 16 / 64 / 128
// clouds: 64 / 73 / 71 / 70 / 69 / 75 us with one block, 64 / 45 / 31 / 23 / 24 / 31 us by cloud
// (one cloud has one block either way), 6000 in 16: 35 and 21 us; ids out of order 82 and 87 us.
struct SmallGridLds {
  SmallSortLds sort;
  unsigned mn[kGridLdsExtents], mx[kGridLdsExtents];
  float smin[kGridLdsExtents];
  int nc[kMaxDims];
  int lo, hi, up, down;                  // points of the block's cloud, where its ids lead
};

template <int D, bool kOrderOnly, bool kByCloud>
__global__ void __launch_bounds__(kSmallThreads) grid_small_kernel(
    int n, int batch, const float *__restrict__ pts, const int *__restrict__ bids,
    const float *__restrict__ cell, GridArrays g) {
  extern __shared__ __align__(16) char lds_raw[];
  SmallGridLds &s = *reinterpret_cast<SmallGridLds *>(lds_raw);
  const int t = threadIdx.x, lane = lane_id();
  int first = small_first(n), last = small_last(n);
  const int cloud = kByCloud ? blockIdx.x : 0;
  if (kByCloud && t == 0) s.lo = s.hi = s.up = s.down = 0;
  auto find_cloud = [&](int i, int b, int before) {  // point i is of cloud b, the one before it
    if (before < b) s.up = 1;
    if (before > b) s.down = 1;
    if (b == cloud && before != b) s.lo = i;
    if (before == cloud && before != b) s.hi = i;
    if (b == cloud && i == n - 1) s.hi = n;
  };
  GridShape<D> shape;
  float ic[D];
  if (kOrderOnly) {
    if (kByCloud) {
      __syncthreads();
      constexpr int kAhead = 4;
      for (int base = first; base < last; base += kAhead * kWave) {
        int b[kAhead], before[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const int i = base + u * kWave + lane < last ? base + u * kWave + lane : last - 1;
          b[u] = bids[i];
          before[u] = bids[i > 0 ? i - 1 : 0];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
          if (__any(b[u] != before[u]) || base + (u + 1) * kWave >= n)
            if (base + u * kWave + lane < last)
              find_cloud(base + u * kWave + lane, b[u], before[u]);
      }
      __syncthreads();
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      shape.n[d] = g.num_cells[d];
      ic[d] = g.inv_cell[d];
    }
  } else {
    if (t < batch * D) {
      s.mn[t] = enc_float(FLT_MAX);
      s.mx[t] = enc_float(-FLT_MAX);
    }
    if (t < D) s.nc[t] = 1;
    __syncthreads();
    Bounds<D> box;
    int cur = -1;
    // kAhead times 64 points in flight: every block reads all points, and iteration by iteration
    // that is a chain of up to sixteen waits (16 clouds of 8659 points in all: 20 -> 14 us, 2 x 1024
    // 15 -> 12)
    constexpr int kAhead = 4;
    for (int base = first; base < last; base += kAhead * kWave) {
      int b[kAhead], before[kAhead];
      float p[kAhead][D];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {            // past the end: the last point again
        const int i = base + u * kWave + lane < last ? base + u * kWave + lane : last - 1;
        b[u] = bids[i];
        if (kByCloud) before[u] = bids[i > 0 ? i - 1 : 0];
#pragma unroll
        for (int d = 0; d < D; ++d) p[u][d] = pts[(int64_t)i * D + d];
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int i = base + u * kWave + lane;
        const bool live = i < last;
        // (nothing to see where the 64 points and the one before them are of one cloud)
        if (kByCloud && (__any(b[u] != before[u]) || base + (u + 1) * kWave >= n)) {
          if (live) find_cloud(i, b[u], before[u]);
        }
        add_points<D>(live, b[u], p[u], 1, box, cur,
                      [&](int b, Bounds<D> &box) { box.flush(s.mn + b * D, s.mx + b * D); },
                      [&](int b, const float *p) {
#pragma unroll
                        for (int d = 0; d < D; ++d) {
                          atomicMin(&s.mn[b * D + d], enc_float(p[d]));
                          atomicMax(&s.mx[b * D + d], enc_float(p[d]));
                        }
                      });
      }
    }
    if (cur >= 0) box.flush(s.mn + cur * D, s.mx + cur * D);
    __syncthreads();
    if (t < batch * D) {
      const CellExtent e = finalize_extent(s.mn[t], s.mx[t], cell[t % D]);
      if (cloud == 0) {
        g.aabb_min[t] = e.lo;
        g.aabb_max[t] = e.hi;
        g.smin[t] = e.smin;
      }
      s.smin[t] = e.smin;
      atomicMax(&s.nc[t % D], e.cells);
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < D; ++d) {
      shape.n[d] = s.nc[d];
      ic[d] = 1.0f / cell[d];
    }
    if (t < D && cloud == 0) {
      g.num_cells[t] = s.nc[t];
      g.inv_cell[t] = 1.0f / cell[t];
    }
  }
  // the block's points, and where the sorted ones go
  int begin = 0, count = n, dest = 0;
  if (kByCloud) {
    if (s.up == 0 || s.down == 0) {
      begin = s.lo;
      count = s.hi - s.lo;
      dest = s.down ? s.lo : n - s.hi;
      if (count == 0) return;
      first = begin + small_first(count);
      last = begin + small_last(count);
    } else if (cloud > 0) {
      return;
    }
  }
  uint64_t cells = 1;
#pragma unroll
  for (int d = 0; d < D; ++d) cells *= (uint64_t)shape.n[d];
  const int64_t below = kByCloud && count < n ? (int64_t)cells * cloud : 0;  // keys of the clouds before
  if (count == n) cells *= (uint64_t)(batch > 0 ? batch : 1);
  const int bits = cells > 1 ? 64 - __clzll((long long)(cells - 1)) : 1;
  for (int i = first + lane; i < last; i += kWave) {
    const int b = bids[i];
    float p[D], m[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      p[d] = pts[(int64_t)i * D + d];
      m[d] = kOrderOnly ? g.smin[(int64_t)b * D + d] : s.smin[b * D + d];
    }
    int c[D];
    cell_of_point<D>(p, m, ic, shape, c);
    g.keys[i] = key_of_cell<D>(c, shape, b);
  }
  __threadfence_block();
  __syncthreads();                       // the keys are in memory for the whole block
  int item[kSmallRounds];
  small_sort_any(count, bits, g.keys + begin, below, item, s.sort);
#pragma unroll
  for (int r = 0; r < kSmallRounds; ++r) {
    if (first + r * kWave + lane < last) {
      const int from = begin + item[r], i = dest + (first - begin) + r * kWave + lane;
      g.sorted_idx[i] = from;
      if (!kOrderOnly || g.sorted_keys) g.sorted_keys[i] = g.keys[from];
#pragma unroll
      for (int d = 0; d < D; ++d) g.sorted_pts[(int64_t)i * D + d] = pts[(int64_t)from * D + d];
      g.sorted_bids[i] = bids[from];
    }
  }
}

// inverse[order[i]] = i
__global__ void __launch_bounds__(256) invert_order_kernel(int64_t n, const int *__restrict__ order,
                                                           int *__restrict__ inverse) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    inverse[order[i]] = (int)i;
}

// Clouds up to which each gets a block: half the compute units, a block fills one.
constexpr int kMaxCloudBlocks = 128;

template <int D, bool kOrderOnly>
static int launch_small(hipStream_t s, int64_t n, int batch, const float *points,
                        const int *batch_ids, const float *cell, const GridArrays &g) {
  const bool by_cloud = batch > 1 && batch <= kMaxCloudBlocks;
  auto kernel = by_cloud ? grid_small_kernel<D, kOrderOnly, true>
                         : grid_small_kernel<D, kOrderOnly, false>;
  MCCNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)sizeof(SmallGridLds)));
  hipLaunchKernelGGL(kernel, dim3(by_cloud ? batch : 1), dim3(kSmallThreads),
                     sizeof(SmallGridLds), s, (int)n, batch, points, batch_ids, cell, g);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static int reduce_boxes(hipStream_t s, int64_t n, int num_dims, const float *points,
                        const int *batch_ids, int batch, unsigned *mn, unsigned *mx) {
  const int count = batch * num_dims;
  hipLaunchKernelGGL(aabb_init_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, s, count, mn, mx);
  MCCNN_LAUNCH_CHECK();
  if (n == 0) return MCCNN_OK;
  // Stretches of at least 1024 points, at most 256 or 512 blocks.  Every block ends in a few minima and
  // maxima of the same words of memory, one after the other, which were most of the time of 745
  // blocks; the words of many clouds are others, and long stretches are better read by more blocks.
  // us at 256 / 512 / 1024 blocks, 1, 8, 16 and 64 clouds: 763 k points 7.6 / 10.6 / 11.4,
  // 7.5 / 8.5 / 9.7, 7.3 / 7.0 / 8.1, 7.0 / 6.4 / 6.4; 3 M 14.8 / 13.6 / 17.9, 14.1 / 12.2 / 15.2,
  // 14.1 / 11.6 / 13.3, 14.0 / 10.4 / 10.3; 8 M 30 / 22 / 21 to 28; 300 k 6 to 7 all.  (64 points in
  // flight and up to 1024 blocks: 763 k 12.7, 10.7, 9.3, 6.8; 3 M 19.9, 17.2, 15.2, 11.9.  All of one
  // grid after another; 800 k points in 4 clouds between the kernels of a whole pass 9.3, 11.8 before.)
  const int64_t most = batch >= 16 || n >= (int64_t)1 << 21 ? 512 : 256;
  int64_t per_block = (n + most - 1) / most;
  per_block = (per_block < 1024 ? 1024 : per_block + 255) / 256 * 256;
  MCCNN_DIM_SWITCH(num_dims,
                   hipLaunchKernelGGL(aabb_reduce_kernel<D>, dim3(blocks_for(n, (int)per_block)),
                                      dim3(kAabbThreads), 0, s, n, per_block, points, batch_ids,
                                      batch, mn, mx));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

}  // namespace mccnn

using namespace mccnn;

extern "C" int mccnn_compute_keys(mccnn_stream_t stream, int64_t num_pts, int num_dims,
                                  const float *points, int64_t batch_ids_len,
                                  const int32_t *batch_ids, int64_t aabb_rows, int aabb_dims,
                                  const float *scaled_aabb_min, int num_cells_len,
                                  const int32_t *num_cells, int inv_cell_sizes_len,
                                  const float *inv_cell_sizes, int64_t *keys_out) {
  MCCNN_REQUIRE(valid_dims(num_dims), "ComputeKeys expects a valid number of dimensions (got %d)",
                num_dims);
  MCCNN_REQUIRE(num_pts >= 0 && aabb_rows >= 0, "ComputeKeys expects non-negative sizes");
  MCCNN_REQUIRE(batch_ids_len == num_pts,
                "ComputeKeys expects the same number of batch ids as number of points");
  MCCNN_REQUIRE(aabb_dims == num_dims,
                "ComputeKeys expects aabb with the same number of dimensions as the points");
  MCCNN_REQUIRE(num_cells_len == num_dims,
                "ComputeKeys expects number of cells with the same number of dimensions as the "
                "points");
  MCCNN_REQUIRE(inv_cell_sizes_len == num_dims,
                "ComputeKeys expects cell sizes with the same number of dimensions as the points");
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(points && batch_ids && scaled_aabb_min && num_cells && inv_cell_sizes && keys_out,
                "ComputeKeys received a null tensor");
  const unsigned grid = blocks_for(num_pts, 256);
  MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(compute_keys_kernel<D>, dim3(grid), dim3(256), 0,
                                                as_stream(stream), num_pts, points, batch_ids,
                                                scaled_aabb_min, num_cells, inv_cell_sizes,
                                                (int64_t *)keys_out));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_gather_points(mccnn_stream_t stream, int64_t num_pts, int num_dims,
                                   const float *points, const int32_t *batch_ids,
                                   const int32_t *indices, float *points_out,
                                   int32_t *batch_ids_out) {
  MCCNN_REQUIRE(valid_dims(num_dims), "gather_points expects a valid number of dimensions");
  MCCNN_REQUIRE(num_pts >= 0, "gather_points expects a non-negative size");
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(points && batch_ids && indices && points_out && batch_ids_out,
                "gather_points received a null tensor");
  const unsigned grid = blocks_for(num_pts, 256);
  MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(gather_points_kernel<D>, dim3(grid), dim3(256), 0,
                                                as_stream(stream), num_pts, points, batch_ids,
                                                indices, points_out, batch_ids_out));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_build_grid_ds(mccnn_stream_t stream, int64_t num_pts,
                                   const int64_t *sorted_keys, int num_cells_len,
                                   const int32_t *num_cells, int num_cells_host_len,
                                   const int32_t *num_cells_host, int batch_size,
                                   int32_t *ds_out) {
  MCCNN_REQUIRE(batch_size > 0, "BuildGridDs requires a positive batch size");
  MCCNN_REQUIRE(valid_dims(num_cells_len), "BuildGridDs expects a valid number of dimensions");
  MCCNN_REQUIRE(num_cells_host_len == num_cells_len,
                "BuildGridDs expects number of cells with the same dimensions in both parameters");
  MCCNN_REQUIRE(num_pts >= 0 && num_cells && num_cells_host && ds_out,
                "BuildGridDs received a null tensor");
  MCCNN_REQUIRE(num_cells_host[0] > 0 && num_cells_host[1] > 0,
                "BuildGridDs expects a positive number of cells");
  const int64_t cols = (int64_t)batch_size * num_cells_host[0] * num_cells_host[1];
  MCCNN_REQUIRE(cols * 2 < ((int64_t)1 << 31), "BuildGridDs table too large");
  int rc = fill_zero(as_stream(stream), ds_out, sizeof(int32_t) * 2 * (size_t)cols);
  if (rc != MCCNN_OK) return rc;
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(sorted_keys, "BuildGridDs received a null tensor");
  const unsigned grid = blocks_for(num_pts, 256);
  MCCNN_DIM_SWITCH(num_cells_len,
                   hipLaunchKernelGGL(build_grid_ds_kernel<D>, dim3(grid), dim3(256), 0,
                                      as_stream(stream), num_pts, (const int64_t *)sorted_keys,
                                      num_cells, (int2 *)ds_out));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_grid_setup(mccnn_stream_t stream, int64_t num_pts, int num_dims,
                                const float *points, const int32_t *batch_ids, int batch_size,
                                const float *cell_sizes, float *aabb_min_out, float *aabb_max_out,
                                int32_t *num_cells_out, float *scaled_aabb_min_out,
                                float *inv_cell_sizes_out) {
  MCCNN_REQUIRE(valid_dims(num_dims), "grid_setup expects a valid number of dimensions");
  MCCNN_REQUIRE(batch_size > 0, "grid_setup requires a positive batch size");
  MCCNN_REQUIRE(num_pts >= 0 && cell_sizes && aabb_min_out && aabb_max_out && num_cells_out &&
                    scaled_aabb_min_out && inv_cell_sizes_out,
                "grid_setup received a null tensor");
  MCCNN_REQUIRE(num_pts == 0 || (points && batch_ids), "grid_setup received a null tensor");
  hipStream_t s = as_stream(stream);
  int rc = reduce_boxes(s, num_pts, num_dims, points, batch_ids, batch_size,
                        (unsigned *)aabb_min_out, (unsigned *)aabb_max_out);
  if (rc != MCCNN_OK) return rc;
  MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(grid_finalize_kernel<D>, dim3(1), dim3(256), 0, s,
                                                batch_size, cell_sizes, aabb_min_out, aabb_max_out,
                                                num_cells_out, scaled_aabb_min_out,
                                                inv_cell_sizes_out));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static unsigned capped_grid(int64_t work) {
  if (work > (int64_t)1 << 26) work = (int64_t)1 << 26;
  return blocks_for(work, 256);
}

extern "C" int mccnn_original_neighbor_ids(mccnn_stream_t stream, int64_t num_neighbors,
                                           const int32_t *neighbors,
                                           const int32_t *sorted_indices,
                                           int32_t *original_neighbors_out) {
  MCCNN_REQUIRE(num_neighbors >= 0, "original_neighbor_ids expects a non-negative size");
  if (num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(neighbors && sorted_indices && original_neighbors_out,
                "original_neighbor_ids received a null tensor");
  hipLaunchKernelGGL(original_ids_kernel, dim3(capped_grid(num_neighbors)), dim3(256), 0,
                     as_stream(stream), num_neighbors, (const int2 *)neighbors, sorted_indices,
                     (int2 *)original_neighbors_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_swapped_pairs(mccnn_stream_t stream, int64_t num_neighbors,
                                   const int32_t *neighbors, const int32_t *pair_order,
                                   int32_t *swapped_out) {
  MCCNN_REQUIRE(num_neighbors >= 0, "swapped_pairs expects a non-negative size");
  if (num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(neighbors && pair_order && swapped_out, "swapped_pairs received a null tensor");
  hipLaunchKernelGGL(swapped_pairs_kernel, dim3(capped_grid(num_neighbors)), dim3(256), 0,
                     as_stream(stream), num_neighbors, (const int2 *)neighbors, pair_order,
                     (int2 *)swapped_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_gather_pdf_column(mccnn_stream_t stream, int64_t num_neighbors,
                                       const int32_t *neighbors, int column, const float *pdf,
                                       float *pdf_per_pair_out) {
  MCCNN_REQUIRE(num_neighbors >= 0, "gather_pdf expects a non-negative size");
  MCCNN_REQUIRE(column == 0 || column == 1, "gather_pdf expects column 0 or 1 (got %d)", column);
  if (num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(neighbors && pdf && pdf_per_pair_out, "gather_pdf received a null tensor");
  hipLaunchKernelGGL(gather_pdf_kernel, dim3(capped_grid(num_neighbors)), dim3(256), 0,
                     as_stream(stream), num_neighbors, (const int2 *)neighbors, column, pdf,
                     pdf_per_pair_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_gather_pdf_both(mccnn_stream_t stream, int64_t num_neighbors,
                                     const int32_t *neighbors, const int32_t *transposed,
                                     const float *pdf, float *pdf_per_pair_out,
                                     float *pdf_per_transposed_out) {
  MCCNN_REQUIRE(num_neighbors >= 0, "gather_pdf expects a non-negative size");
  if (num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(neighbors && transposed && pdf && pdf_per_pair_out && pdf_per_transposed_out,
                "gather_pdf received a null tensor");
  hipLaunchKernelGGL(gather_pdf_both_kernel, dim3(capped_grid(num_neighbors)), dim3(256), 0,
                     as_stream(stream), num_neighbors, (const int2 *)neighbors,
                     (const int2 *)transposed, pdf, pdf_per_pair_out, pdf_per_transposed_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_gather_pdf(mccnn_stream_t stream, int64_t num_neighbors,
                                const int32_t *neighbors, const float *pdf,
                                float *pdf_per_pair_out) {
  return mccnn_gather_pdf_column(stream, num_neighbors, neighbors, 0, pdf, pdf_per_pair_out);
}

extern "C" int mccnn_gather_rows(mccnn_stream_t stream, int64_t num_rows, int num_cols,
                                 const float *src, const int32_t *indices, float *out) {
  MCCNN_REQUIRE(num_rows >= 0, "gather_rows expects a non-negative size");
  MCCNN_REQUIRE(num_cols > 0 && num_cols % 4 == 0,
                "gather_rows expects a row length that is a multiple of 4 (got %d)", num_cols);
  if (num_rows == 0) return MCCNN_OK;
  MCCNN_REQUIRE(src && indices && out, "gather_rows received a null tensor");
  const int64_t total = num_rows * (num_cols / 4);
  hipLaunchKernelGGL(gather_rows_kernel, dim3(capped_grid(total)), dim3(256), 0,
                     as_stream(stream), total, num_cols / 4, (const float4 *)src, indices,
                     (float4 *)out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_gather_i32(mccnn_stream_t stream, int64_t count, const int32_t *src,
                                const int32_t *indices, int32_t *out) {
  MCCNN_REQUIRE(count >= 0, "gather_i32 expects a non-negative size");
  if (count == 0) return MCCNN_OK;
  MCCNN_REQUIRE(src && indices && out, "gather_i32 received a null tensor");
  hipLaunchKernelGGL(gather_i32_kernel, dim3(capped_grid(count)), dim3(256), 0,
                     as_stream(stream), count, src, indices, out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_invert_order(mccnn_stream_t stream, int64_t count, const int32_t *order,
                                  int32_t *inverse_out) {
  MCCNN_REQUIRE(count >= 0, "invert_order expects a non-negative size");
  if (count == 0) return MCCNN_OK;
  MCCNN_REQUIRE(order && inverse_out, "invert_order received a null tensor");
  hipLaunchKernelGGL(invert_order_kernel, dim3(capped_grid(count)), dim3(256), 0,
                     as_stream(stream), count, order, inverse_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

// The grid of pylib/pc/Grid.py:32-64 in one call.  Up to 16 384 points in clouds whose extents
// (batch * dims) fit a block's 512: one launch, no host
// round trip unless the caller asks for the shape.  Beyond that: boxes, shape and keys (three
// launches), the host copy of the shape -- it sizes the key width of the sort and, for the
// caller, the grid table --, three launches per digit of the sort, the last of which gathers
// the points.
extern "C" size_t mccnn_build_grid_workspace_bytes(int64_t num_pts) {
  if (num_pts < 0) num_pts = 0;
  return carve_sort_workspace(nullptr, num_pts).bytes + align256(sizeof(unsigned) * (size_t)num_pts) +
         2 * align256(sizeof(unsigned) * kGridLdsExtents);
}

extern "C" int64_t mccnn_build_grid_single_launch_max(void) { return kSmallMax; }

static bool extents_fit(int num_dims, int batch_size) {
  return batch_size > 0 && (int64_t)batch_size * num_dims <= kGridLdsExtents;
}

extern "C" int mccnn_build_grid_is_single_launch(int64_t num_pts, int num_dims, int batch_size) {
  return num_pts > 0 && num_pts <= kSmallMax && extents_fit(num_dims, batch_size);
}

static int key_bits_for(int batch, int num_dims, const int32_t *cells) {
  unsigned long long total = (unsigned long long)(batch > 0 ? batch : 1);
  for (int d = 0; d < num_dims; ++d) total *= (unsigned long long)cells[d];
  int bits = 1;
  while (bits < 64 && (1ull << bits) < total) ++bits;
  return bits;
}

static int build_grid(mccnn_stream_t stream, int64_t num_pts, int num_dims, const float *points,
                      const int32_t *batch_ids, int batch_size, const float *cell_sizes,
                      const GridArrays &g, void *workspace, size_t workspace_bytes,
                      bool shape_is_pinned, int32_t *num_cells_out_host, int *key_bits_out_host) {
  MCCNN_REQUIRE(valid_dims(num_dims), "build_grid expects a valid number of dimensions");
  MCCNN_REQUIRE(num_pts >= 0 && num_pts < ((int64_t)1 << 31), "build_grid expects 0 <= num_pts < 2^31");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_build_grid_workspace_bytes(num_pts),
                "build_grid workspace too small");
  const bool want_shape = num_cells_out_host != nullptr;
  MCCNN_REQUIRE(want_shape == (key_bits_out_host != nullptr),
                "build_grid expects both host outputs, the grid shape and the key width, or neither");
  const bool single_launch = mccnn_build_grid_is_single_launch(num_pts, num_dims, batch_size);
  MCCNN_REQUIRE(want_shape || single_launch,
                "build_grid needs host outputs for the grid shape and the key width");
  hipStream_t s = as_stream(stream);
  if (num_pts > 0 && extents_fit(num_dims, batch_size)) {
    MCCNN_REQUIRE(points && batch_ids && cell_sizes && g.aabb_min && g.aabb_max && g.num_cells &&
                      g.smin && g.inv_cell && g.keys && g.sorted_keys && g.sorted_idx &&
                      g.sorted_pts && g.sorted_bids && workspace,
                  "build_grid received a null tensor");
    if (single_launch) {
      int rc = MCCNN_OK;
      MCCNN_DIM_SWITCH(num_dims, rc = (launch_small<D, false>(s, num_pts, batch_size, points, batch_ids,
                                                              cell_sizes, g)));
      if (rc != MCCNN_OK || !want_shape) return rc;
      MCCNN_HIP_CHECK(hipMemcpyAsync(num_cells_out_host, g.num_cells, sizeof(int32_t) * num_dims,
                                     hipMemcpyDeviceToHost, s));
      MCCNN_HIP_CHECK(hipStreamSynchronize(s));
      *key_bits_out_host = key_bits_for(batch_size, num_dims, num_cells_out_host);
      return MCCNN_OK;
    }
    const SortWorkspace w = carve_sort_workspace(workspace, num_pts);
    char *p = (char *)workspace + w.bytes;
    unsigned *keys32 = (unsigned *)p;
    p += align256(sizeof(unsigned) * (size_t)num_pts);
    unsigned *mn = (unsigned *)p, *mx = (unsigned *)(p + align256(sizeof(unsigned) * kGridLdsExtents));
    int rc = reduce_boxes(s, num_pts, num_dims, points, batch_ids, batch_size, mn, mx);
    if (rc != MCCNN_OK) return rc;
    const int nb = (int)((num_pts + kSortTile - 1) / kSortTile);
    if (shape_is_pinned)
      for (int d = 0; d < num_dims; ++d) num_cells_out_host[d] = -1;
    MCCNN_DIM_SWITCH(num_dims,
                     hipLaunchKernelGGL(grid_keys_kernel<D>, dim3(nb), dim3(kSortThreads), 0, s,
                                        num_pts, batch_size, nb, points, batch_ids, cell_sizes, mn,
                                        mx, g, keys32, w.hist,
                                        shape_is_pinned ? num_cells_out_host : (int32_t *)nullptr));
    MCCNN_LAUNCH_CHECK();
    if (shape_is_pinned) {
      rc = wait_for_host_values(s, num_cells_out_host, num_dims);
      if (rc != MCCNN_OK) return rc;
    } else {
      MCCNN_HIP_CHECK(hipMemcpyAsync(num_cells_out_host, g.num_cells, sizeof(int32_t) * num_dims,
                                     hipMemcpyDeviceToHost, s));
      MCCNN_HIP_CHECK(hipStreamSynchronize(s));
    }
    const int bits = key_bits_for(batch_size, num_dims, num_cells_out_host);
    *key_bits_out_host = bits;
    if (bits <= 32) {
      const SortedPoints out = {points, batch_ids, g.sorted_pts, g.sorted_bids};
      return sort_grid_keys(s, num_dims, num_pts, bits, keys32, w, g.sorted_keys, g.sorted_idx,
                            out);
    }
  } else {
    int rc = mccnn_grid_setup(stream, num_pts, num_dims, points, batch_ids, batch_size, cell_sizes,
                              g.aabb_min, g.aabb_max, g.num_cells, g.smin, g.inv_cell);
    if (rc != MCCNN_OK) return rc;
    rc = mccnn_compute_keys(stream, num_pts, num_dims, points, num_pts, batch_ids, batch_size,
                            num_dims, g.smin, num_dims, g.num_cells, num_dims, g.inv_cell, g.keys);
    if (rc != MCCNN_OK) return rc;
    MCCNN_HIP_CHECK(hipMemcpyAsync(num_cells_out_host, g.num_cells, sizeof(int32_t) * num_dims,
                                   hipMemcpyDeviceToHost, s));
    MCCNN_HIP_CHECK(hipStreamSynchronize(s));
    *key_bits_out_host = key_bits_for(batch_size, num_dims, num_cells_out_host);
  }
  // keys wider than 32 bits, or more clouds than a block keeps the extents of
  int rc = mccnn_sort_keys_descending(stream, num_pts, *key_bits_out_host, g.keys, g.sorted_keys,
                                      g.sorted_idx, workspace, workspace_bytes);
  if (rc != MCCNN_OK) return rc;
  return mccnn_gather_points(stream, num_pts, num_dims, points, batch_ids, g.sorted_idx,
                             g.sorted_pts, g.sorted_bids);
}

extern "C" int mccnn_build_grid(mccnn_stream_t stream, int64_t num_pts, int num_dims,
                                const float *points, const int32_t *batch_ids, int batch_size,
                                const float *cell_sizes, float *aabb_min_out,
                                float *aabb_max_out, int32_t *num_cells_out,
                                float *scaled_aabb_min_out, float *inv_cell_sizes_out,
                                int64_t *keys_out, int64_t *sorted_keys_out,
                                int32_t *sorted_indices_out, float *sorted_points_out,
                                int32_t *sorted_batch_ids_out, void *workspace,
                                size_t workspace_bytes, int32_t *num_cells_out_host,
                                int *key_bits_out_host) {
  MCCNN_REQUIRE(num_cells_out_host && key_bits_out_host,
                "build_grid needs host outputs for the grid shape and the key width");
  const GridArrays g = {aabb_min_out, aabb_max_out, num_cells_out, scaled_aabb_min_out,
                        inv_cell_sizes_out, keys_out, sorted_keys_out, sorted_indices_out,
                        sorted_points_out, sorted_batch_ids_out};
  return build_grid(stream, num_pts, num_dims, points, batch_ids, batch_size, cell_sizes, g,
                    workspace, workspace_bytes, false, num_cells_out_host, key_bits_out_host);
}

extern "C" int mccnn_build_grid_pinned(mccnn_stream_t stream, int64_t num_pts, int num_dims,
                                       const float *points, const int32_t *batch_ids,
                                       int batch_size, const float *cell_sizes,
                                       float *aabb_min_out, float *aabb_max_out,
                                       int32_t *num_cells_out, float *scaled_aabb_min_out,
                                       float *inv_cell_sizes_out, int64_t *keys_out,
                                       int64_t *sorted_keys_out, int32_t *sorted_indices_out,
                                       float *sorted_points_out, int32_t *sorted_batch_ids_out,
                                       void *workspace, size_t workspace_bytes,
                                       int32_t *num_cells_out_pinned, int *key_bits_out_host) {
  const GridArrays g = {aabb_min_out, aabb_max_out, num_cells_out, scaled_aabb_min_out,
                        inv_cell_sizes_out, keys_out, sorted_keys_out, sorted_indices_out,
                        sorted_points_out, sorted_batch_ids_out};
  return build_grid(stream, num_pts, num_dims, points, batch_ids, batch_size, cell_sizes, g,
                    workspace, workspace_bytes, true, num_cells_out_pinned, key_bits_out_host);
}

// Centres in the order of their cells in a grid that is there already: order, coordinates and
// cloud ids.  Up to 16 384 centres one launch; beyond that keys, sort and gather, for which the
// key width of the grid is needed.
extern "C" int mccnn_order_centres(mccnn_stream_t stream, int64_t num_samples, int num_dims,
                                   const float *samples, const int32_t *sample_batch_ids,
                                   int batch_size, const int32_t *num_cells,
                                   const float *scaled_aabb_min, const float *inv_cell_sizes,
                                   int key_bits, void *workspace, size_t workspace_bytes,
                                   int32_t *order_out, float *points_out,
                                   int32_t *batch_ids_out) {
  return mccnn_order_centres_keys(stream, num_samples, num_dims, samples, sample_batch_ids,
                                  batch_size, num_cells, scaled_aabb_min, inv_cell_sizes, key_bits,
                                  workspace, workspace_bytes, order_out, points_out, batch_ids_out,
                                  nullptr);
}

extern "C" int mccnn_order_centres_keys(mccnn_stream_t stream, int64_t num_samples, int num_dims,
                                        const float *samples, const int32_t *sample_batch_ids,
                                        int batch_size, const int32_t *num_cells,
                                        const float *scaled_aabb_min,
                                        const float *inv_cell_sizes, int key_bits,
                                        void *workspace, size_t workspace_bytes,
                                        int32_t *order_out, float *points_out,
                                        int32_t *batch_ids_out, int64_t *sorted_keys_out) {
  MCCNN_REQUIRE(valid_dims(num_dims), "order_centres expects a valid number of dimensions");
  MCCNN_REQUIRE(num_samples >= 0 && num_samples < ((int64_t)1 << 31) && batch_size > 0,
                "order_centres expects 0 <= num_samples < 2^31 and a positive batch size");
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(samples && sample_batch_ids && num_cells && scaled_aabb_min && inv_cell_sizes &&
                    workspace && order_out && points_out && batch_ids_out,
                "order_centres received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_order_centres_workspace_bytes(num_samples),
                "order_centres workspace too small");
  hipStream_t s = as_stream(stream);
  if (num_samples <= kSmallMax) {
    const GridArrays g = {nullptr, nullptr, (int *)num_cells, (float *)scaled_aabb_min,
                          (float *)inv_cell_sizes, (int64_t *)workspace, sorted_keys_out,
                          order_out, points_out, batch_ids_out};
    int rc = MCCNN_OK;
    MCCNN_DIM_SWITCH(num_dims, rc = (launch_small<D, true>(s, num_samples, batch_size, samples,
                                                           sample_batch_ids, nullptr, g)));
    return rc;
  }
  char *p = (char *)workspace;
  int64_t *keys = (int64_t *)p, *sorted = (int64_t *)(p + align256(8 * (size_t)num_samples));
  if (sorted_keys_out) sorted = sorted_keys_out;
  void *ws = p + 2 * align256(8 * (size_t)num_samples);
  int rc = mccnn_compute_keys(stream, num_samples, num_dims, samples, num_samples,
                              sample_batch_ids, batch_size, num_dims, scaled_aabb_min, num_dims,
                              num_cells, num_dims, inv_cell_sizes, keys);
  if (rc != MCCNN_OK) return rc;
  rc = mccnn_sort_keys_descending(stream, num_samples, key_bits, keys, sorted, order_out, ws,
                                  carve_sort_workspace(nullptr, num_samples).bytes);
  if (rc != MCCNN_OK) return rc;
  return mccnn_gather_points(stream, num_samples, num_dims, samples, sample_batch_ids, order_out,
                             points_out, batch_ids_out);
}

extern "C" size_t mccnn_order_centres_workspace_bytes(int64_t num_samples) {
  if (num_samples < 0) num_samples = 0;
  return 2 * align256(8 * (size_t)num_samples) + carve_sort_workspace(nullptr, num_samples).bytes;
}
