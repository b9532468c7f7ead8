// Point-cloud sampling on the sorted grid
// (custom_ops/tfg_custom_ops/sampling/cc/ops/sampling_ops.cpp:131-194):
// mode 0 Poisson disk (count_sampling_pd_kernels.cu.cc:41-181), mode 1 cell
// average (sampling_avg_kernels.cu.cc:42-88).
//
// Occupied cells are found by flagging key changes and a prefix sum, so the
// cell list and both outputs keep the sorted order (the reference compacts with
// a global atomic counter and leaves the order to chance).  Poisson disk keeps
// the reference's 2^D cell-parity launches; inside a launch one wavefront owns a
// cell and decides its points in order (details at the kernel).  Cell averages are
// summed serially in sorted order so that the result is bit-reproducible (later
// hierarchy levels derive integer keys from these points).
#include "common.h"
#include "fill.h"
#include "search.h"

namespace mccnn {

// cell_scan[i] = 1 at the first point of each occupied cell (scanned in place
// afterwards into "cells up to and including i").
__global__ void __launch_bounds__(256) flag_cell_starts_kernel(int64_t n,
                                                               const int64_t *__restrict__ keys,
                                                               int *__restrict__ cell_scan) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    cell_scan[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1 : 0;
}

__global__ void __launch_bounds__(256) store_cell_starts_kernel(int64_t n,
                                                                const int64_t *__restrict__ keys,
                                                                const int *__restrict__ cell_scan,
                                                                int *__restrict__ first_idx) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    if (i == 0 || keys[i] != keys[i - 1]) first_idx[cell_scan[i] - 1] = (int)i;
}

// The three steps -- flags, their prefix sum and the list of cells -- of up to 16 384 points in one
// launch of one block, with the number of cells in *total: launches cost more than the work there (4
// or 16 rounds of 1024 keys, all in flight; three levels of 16 x 1024 points 28 us and the gaps of nine
// launches, 17 and those of three).  Beyond, one compute unit is too few.
constexpr int kStartThreads = 1024, kStartWaves = kStartThreads / kWave;
constexpr int64_t kStartMax = 16 * kStartThreads;

template <int kStartRounds>
__global__ void __launch_bounds__(kStartThreads) cell_starts_block_kernel(
    int n, const int64_t *__restrict__ keys, int *__restrict__ first_idx, int64_t *total) {
  constexpr int kParts = kStartRounds * kStartWaves;
  __shared__ int before[kParts];                 // cells that start in (round, wavefront), then before it
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  int64_t key[kStartRounds], prev[kStartRounds];
#pragma unroll
  for (int r = 0; r < kStartRounds; ++r) {       // (past the end: the last point again)
    const int i = r * kStartThreads + t < n ? r * kStartThreads + t : n - 1;
    key[r] = keys[i];
    prev[r] = keys[i > 0 ? i - 1 : 0];
  }
  uint64_t starts[kStartRounds];
#pragma unroll
  for (int r = 0; r < kStartRounds; ++r) {
    const int i = r * kStartThreads + t;
    starts[r] = __ballot(i < n && (i == 0 || key[r] != prev[r]));
    if (lane == 0) before[r * kStartWaves + wave] = __popcll(starts[r]);
  }
  __syncthreads();
  if (wave == 0) {
    constexpr int kEach = kParts / kWave;
    int count[kEach], sum = 0;
#pragma unroll
    for (int k = 0; k < kEach; ++k) sum += count[k] = before[kEach * lane + k];
    const int incl = wave_inclusive_scan(sum);
    int run = incl - sum;
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
      before[kEach * lane + k] = run;
      run += count[k];
    }
    if (lane == kWave - 1)
      __hip_atomic_store(total, (int64_t)incl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kStartRounds; ++r)
    if ((starts[r] >> lane) & 1)
      first_idx[before[r * kStartWaves + wave] + __popcll(starts[r] & ((1ull << lane) - 1ull))] =
          r * kStartThreads + t;
}

// Parity class of every occupied cell (bit d = parity of the cell index in dim d), and how many
// cells every class has.
constexpr int kMaxClasses = 1 << kMaxDims;

template <int D>
__global__ void __launch_bounds__(256) cell_class_kernel(
    const int64_t *__restrict__ num_cells_total /*device*/, const int64_t *__restrict__ keys,
    const int *__restrict__ num_cells, const int *__restrict__ first_idx,
    int *__restrict__ cell_class, int *__restrict__ class_counts) {
  __shared__ int counts[1 << D];
  const int64_t cells = *num_cells_total;
  if ((int64_t)blockIdx.x * blockDim.x >= cells) return;
  if (threadIdx.x < (1 << D)) counts[threadIdx.x] = 0;
  __syncthreads();
  const int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (u < cells) {
    // decode the cell index of the key (batch digit dropped)
    int64_t aux = keys[first_idx[u]];
    int cls = 0;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const int nd = num_cells[d];
      const int cd = (int)(aux % nd);
      aux /= nd;
      cls |= (cd & 1) << d;
    }
    cell_class[u] = cls;
    atomicAdd(&counts[cls], 1);
  }
  __syncthreads();
  if (threadIdx.x < (1 << D) && counts[threadIdx.x] > 0)
    atomicAdd(&class_counts[threadIdx.x], counts[threadIdx.x]);
}

// The cells of every class, one class after the other.  Their order inside a class does not
// matter: cells of one class are decided independently.  `cursors` starts at zero.
template <int D>
__global__ void __launch_bounds__(256) class_list_kernel(
    const int64_t *__restrict__ num_cells_total /*device*/, const int *__restrict__ cell_class,
    const int *__restrict__ class_counts, int *__restrict__ cursors, int *__restrict__ list) {
  __shared__ int counts[1 << D], base[1 << D];
  const int64_t cells = *num_cells_total;
  if ((int64_t)blockIdx.x * blockDim.x >= cells) return;
  if (threadIdx.x < (1 << D)) counts[threadIdx.x] = 0;
  __syncthreads();
  const int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int cls = 0, rank = 0;
  if (u < cells) {
    cls = cell_class[u];
    rank = atomicAdd(&counts[cls], 1);
  }
  __syncthreads();
  if (threadIdx.x < (1 << D)) {
    int start = 0;
    for (int c = 0; c < (int)threadIdx.x; ++c) start += class_counts[c];
    const int mine = counts[threadIdx.x];
    base[threadIdx.x] = start + (mine > 0 ? atomicAdd(&cursors[threadIdx.x], mine) : 0);
  }
  __syncthreads();
  if (u < cells) list[base[cls] + rank] = (int)u;
}

// One pass of the Poisson-disk selection, over the cells of parity class `call`: a wavefront takes
// a cell and decides its points in ascending sorted index, their neighbour lists spread over its
// lanes; a point is selected unless one of its neighbours already is.  Cells of one class are at
// least a cell apart, so only the wavefront's own selections can change under it during a pass.
// Points are taken four at a time: their lists and the selections these meet are requested
// together (the lists one batch ahead), and whether a point of the batch hides a later one is
// seen from the indices in registers.  A pass is a chain of loads; point by point, and with a
// wavefront for every cell there could be of any class, 16 passes over 4 x 200 k points took
// 528 us, 205 us now.
constexpr int kDiskBatch = 4, kDiskLists = 2;      // points decided together; 64 neighbours each
constexpr int kDiskBlocks = 2048;                  // wavefronts for every slot of the chip

__global__ void __launch_bounds__(256) poisson_pass_kernel(
    int64_t n, int call, const int64_t *__restrict__ num_cells_total /*device*/,
    const int *__restrict__ class_counts, const int *__restrict__ list,
    const int2 *__restrict__ nbrs, const int *__restrict__ ranges,
    const int *__restrict__ first_idx, int *used) {
  const int lane = lane_id();
  int offset = 0;
  for (int c = 0; c < call; ++c) offset += class_counts[c];
  const int mine = class_counts[call];
  const int64_t cells = *num_cells_total;
  const int waves = gridDim.x * (256 / kWave);
  auto selected = [&](int i) {
    return __hip_atomic_load(&used[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0;
  };
  // Loads that follow observe the wavefront's selections so far.  They are the only ones that can
  // change what it reads during a pass, so the accesses to `used` have workgroup scope: they go
  // through the compute unit's cache and its XCD's L2.  (With device scope every look at `used`
  // goes past both, to the memory-side cache.)
  auto settle = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  for (int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (256 / kWave) + threadIdx.x / kWave));
       w < mine; w += waves) {
    const int u = list[offset + w];
    const int first = first_idx[u];
    const int last = u + 1 < cells ? first_idx[u + 1] : (int)n;
    // ends of the lists of 64 points at a time: lane l holds that of point chunk + l
    for (int chunk = first; chunk < last; chunk += kWave) {
      const int points = last - chunk < kWave ? last - chunk : kWave;
      const int my_end = lane < points ? ranges[chunk + lane] : 0;
      const int before = chunk > 0 ? ranges[chunk - 1] : 0;
      auto list_begin = [&](int p) {
        return p > 0 ? __builtin_amdgcn_readlane(my_end, p - 1) : before;
      };
      auto list_end = [&](int p) { return __builtin_amdgcn_readlane(my_end, p); };
      struct Lists {
        int idx[kDiskBatch][kDiskLists];           // -1 past the end
      };
      auto fetch = [&](int p0) {
        Lists l;
#pragma unroll
        for (int k = 0; k < kDiskBatch; ++k) {
          const bool there = p0 + k < points;
          const int a = there ? list_begin(p0 + k) : 0, b = there ? list_end(p0 + k) : 0;
#pragma unroll
          for (int q = 0; q < kDiskLists; ++q) {
            const int m = a + q * kWave + lane;
            l.idx[k][q] = m < b ? nbrs[m].x : -1;
          }
        }
        return l;
      };
      Lists cur = fetch(0);
      for (int p0 = 0; p0 < points; p0 += kDiskBatch) {
        // (requested without branches, for lanes past a list's end at point 0: all are in flight
        // before the first is looked at)
        bool flag[kDiskBatch][kDiskLists], hit[kDiskBatch];
#pragma unroll
        for (int k = 0; k < kDiskBatch; ++k)
#pragma unroll
          for (int q = 0; q < kDiskLists; ++q)
            flag[k][q] = selected(cur.idx[k][q] < 0 ? 0 : cur.idx[k][q]);
        const Lists next = fetch(p0 + kDiskBatch);
#pragma unroll
        for (int k = 0; k < kDiskBatch; ++k) {
          hit[k] = false;
#pragma unroll
          for (int q = 0; q < kDiskLists; ++q) hit[k] |= flag[k][q] && cur.idx[k][q] >= 0;
        }
        bool pending = false;                      // selections that may not have reached memory
#pragma unroll
        for (int k = 0; k < kDiskBatch; ++k) {
          if (p0 + k >= points) break;
          bool taken = hit[k];
          const int more = list_begin(p0 + k) + kDiskLists * kWave, b = list_end(p0 + k);
          if (more < b) {                          // neighbours past the registers
            if (pending) settle();
            pending = false;
            for (int m = more + lane; m < b; m += kWave) taken |= selected(nbrs[m].x);
          }
          if (__any(taken)) continue;
          const int i = chunk + p0 + k;
          if (lane == 0)
            __hip_atomic_store(&used[i], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          // later points of the batch that list it
#pragma unroll
          for (int j = k + 1; j < kDiskBatch; ++j)
#pragma unroll
            for (int q = 0; q < kDiskLists; ++q) hit[j] |= cur.idx[j][q] == i;
          pending = true;
        }
        if (pending) settle();
        cur = next;
      }
    }
  }
}

// Where the points of the cells around every occupied cell lie: slices[u R + r], cell row r of cell
// u (rows as in the neighbour search).  A wavefront per row, 64 cells each, as in nbr_ranges_kernel.
constexpr int kRowWaves = 9;
template <int D>
__global__ void __launch_bounds__(kRowWaves * kWave) cell_rows_kernel(
    int64_t n, const int64_t *__restrict__ num_cells_total /*device*/,
    const int64_t *__restrict__ keys, const int2 *__restrict__ ds,
    const int *__restrict__ num_cells, const int *__restrict__ first_idx,
    int2 *__restrict__ slices) {
  constexpr int R = OffsetInfo<D>::count(), OD = OffsetInfo<D>::kDims;
  const int r = kRowWaves * blockIdx.y +
                __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int64_t u = (int64_t)blockIdx.x * kWave + lane_id();
  if (u >= *num_cells_total) return;
  const GridShape<D> g = load_shape<D>(num_cells);
  int cell[D];
  int64_t aux = keys[first_idx[u]];
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    cell[d] = (int)(aux % g.n[d]);
    aux /= g.n[d];
  }
  const int b = (int)aux;
  bool inside = true;
  int digits = r;
#pragma unroll
  for (int d = OD - 1; d >= 0; --d) {
    cell[d] += 1 - digits % 3;
    digits /= 3;
    inside = inside && cell[d] >= 0 && cell[d] < g.n[d];
  }
  KeyRange range = {make_int2(0, 0), 0, 1};
  if (inside) {
    range.span = make_int2(0, (int)n);
    if (ds) range.span = ds[((int64_t)b * g.n[0] + cell[0]) * g.n[1] + cell[1]];
    if (range.span.y <= range.span.x) range.span = make_int2(0, 0);
    else if (!(D == 2 && ds)) {
      range.maxk = range.mink = key_of_cell<D>(cell, g, b);
      if (D > 2) {                                // the cells before and behind in the last dim
        range.maxk += cell[D - 1] < g.n[D - 1] - 1 ? 1 : 0;
        range.mink -= cell[D - 1] > 0 ? 1 : 0;
      }
    }
  }
  int2 slice;
  find_slices<1>(&range, keys, &slice);
  slices[u * R + r] = slice;
}

// One pass of the Poisson-disk selection without a pair table: the same decisions, since a point's
// neighbours are the points of the cells around it within the radius, and only selected ones
// matter.  Those are few -- selected points are a radius apart, at most 90 of them fit into 3 x 3 x 3
// cells of a radius -- and are the same for all points of a cell but for the cell's own: a wavefront
// takes a cell, gathers the selected points around it into its registers, two a lane, and decides
// the cell's points in ascending sorted index without another load, each against all of
// them at once.  Where they do not fit (radii well below the cell size, more than three dimensions)
// the points are decided from memory.  Cells of one class are at least a cell apart, so only the
// wavefront's own selections change under it during a pass.  A pass is latency: four dependent
// loads and the decisions of a cell, one round of wavefronts for 64 k cells.
// 16 passes over 4 x 200 k points of 52 neighbours 203 -> 129 us, the cell rows 27, and the table they no
// longer need 480.
constexpr int kListed = 2 * kWave;

template <int D>
__global__ void __launch_bounds__(256) poisson_cells_kernel(
    int64_t n, int call, const int64_t *__restrict__ num_cells_total /*device*/,
    const int *__restrict__ class_counts, const int *__restrict__ list,
    const int2 *__restrict__ slices, const int *__restrict__ first_idx,
    const float *__restrict__ pts, const float *__restrict__ inv_radii, int *used) {
  constexpr int R = OffsetInfo<D>::count(), kSlices = 9;
  __shared__ int found[256 / kWave][kListed];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  int offset = 0;
  for (int c = 0; c < call; ++c) offset += class_counts[c];
  const int mine = class_counts[call];
  const int64_t cells = *num_cells_total;
  const int waves = gridDim.x * (256 / kWave);
  float ir[D];
#pragma unroll
  for (int d = 0; d < D; ++d) ir[d] = inv_radii[d];
  auto near = [&](const float *s, const float *q) {
    float diff[D];
#pragma unroll
    for (int d = 0; d < D; ++d) diff[d] = s[d] - q[d];
    return within_radius<D>(true, diff, ir);
  };
  // Loads that follow observe the wavefront's selections so far (accesses of workgroup scope).
  auto settle = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  for (int w = blockIdx.x * (256 / kWave) + wave; w < mine; w += waves) {
    const int u = list[offset + w];
    const int first = first_idx[u];
    const int last = u + 1 < cells ? first_idx[u + 1] : (int)n;
    int cnt = 0;                                  // selected points around the cell
    auto append = [&](bool selected, int j) {
      const unsigned long long mask = __ballot(selected);
      const int pos = cnt + __builtin_amdgcn_mbcnt_hi(
                                (unsigned)(mask >> 32),
                                __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
      if (selected && pos < kListed) found[wave][pos] = j;
      cnt += __popcll(mask);
    };
    wave_lds_sync();                              // the list of the cell before has been read
    for (int r0 = 0; r0 < R; r0 += kSlices) {
      const int2 row = lane < kSlices ? slices[(int64_t)u * R + r0 + lane] : make_int2(0, 0);
      int lo[kSlices], hi[kSlices], flag[kSlices];
#pragma unroll
      for (int i = 0; i < kSlices; ++i) {         // (requested without branches)
        lo[i] = __builtin_amdgcn_readlane(row.x, i);
        hi[i] = __builtin_amdgcn_readlane(row.y, i);
        flag[i] = used[lo[i] + lane < hi[i] ? lo[i] + lane : 0];
      }
#pragma unroll
      for (int i = 0; i < kSlices; ++i) {
        append(flag[i] != 0 && lo[i] + lane < hi[i], lo[i] + lane);
        for (int j = lo[i] + kWave; j < hi[i]; j += kWave)
          append(j + lane < hi[i] && used[j + lane < hi[i] ? j + lane : 0] != 0, j + lane);
      }
    }
    wave_lds_sync();
    bool listed = cnt <= kListed;                 // all of them are in the registers
    float qa[D], qb[D];                           // no point: nothing is near it
#pragma unroll
    for (int d = 0; d < D; ++d) qa[d] = qb[d] = __builtin_nanf("");
    if (listed) {
      if (lane < cnt) {
        const int64_t j = found[wave][lane];
#pragma unroll
        for (int d = 0; d < D; ++d) qa[d] = pts[j * D + d];
      }
      if (lane + kWave < cnt) {
        const int64_t j = found[wave][lane + kWave];
#pragma unroll
        for (int d = 0; d < D; ++d) qb[d] = pts[j * D + d];
      }
    }
    for (int chunk = first; chunk < last; chunk += kWave) {
      const int points = last - chunk < kWave ? last - chunk : kWave;
      float own[D];
#pragma unroll
      for (int d = 0; d < D; ++d)
        own[d] = pts[(int64_t)(lane < points ? chunk + lane : chunk) * D + d];
      for (int k = 0; k < points; ++k) {
        float s[D];
#pragma unroll
        for (int d = 0; d < D; ++d)
          s[d] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(own[d]), k));
        bool taken;
        if (listed) {
          taken = near(s, qa);
          if (cnt > kWave) taken |= near(s, qb);
        } else {
          taken = false;
          for (int r = 0; r < R; ++r) {
            const int2 row = slices[(int64_t)u * R + r];
            for (int j = row.x + lane; j < row.y; j += kWave) {
              if (!__hip_atomic_load(&used[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
                continue;
              float q[D];
#pragma unroll
              for (int d = 0; d < D; ++d) q[d] = pts[(int64_t)j * D + d];
              taken |= near(s, q);
            }
          }
        }
        if (__any(taken)) continue;
        if (lane == 0)
          __hip_atomic_store(&used[chunk + k], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
        for (int d = 0; d < D; ++d) {
          qa[d] = lane == cnt ? s[d] : qa[d];
          qb[d] = lane + kWave == cnt ? s[d] : qb[d];
        }
        ++cnt;
        listed = listed && cnt <= kListed;
        if (!listed) settle();
      }
    }
  }
}

template <int D>
__global__ void __launch_bounds__(256) store_selected_kernel(
    int64_t n, const float *__restrict__ pts, const int *__restrict__ bids,
    const int *__restrict__ used, const int *__restrict__ sel_scan, float *__restrict__ out_pts,
    int *__restrict__ out_bids, int *__restrict__ out_idx) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (used[i]) {
      const int64_t pos = sel_scan[i] - 1;
#pragma unroll
      for (int d = 0; d < D; ++d) out_pts[pos * D + d] = pts[i * D + d];
      out_bids[pos] = bids[i];
      out_idx[pos] = (int)i;
    }
  }
}

template <int D>
__global__ void __launch_bounds__(256) cell_average_kernel(
    int64_t n, int64_t cells, const float *__restrict__ pts, const int64_t *__restrict__ keys,
    const int *__restrict__ num_cells, const int *__restrict__ first_idx,
    float *__restrict__ out_pts, int *__restrict__ out_bids, int *__restrict__ out_idx) {
  int64_t total = 1;
#pragma unroll
  for (int d = 0; d < D; ++d) total *= num_cells[d];
  for (int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; u < cells;
       u += (int64_t)gridDim.x * blockDim.x) {
    int64_t i = first_idx[u];
    const int64_t key = keys[i];
    float acc[D];
#pragma unroll
    for (int d = 0; d < D; ++d) acc[d] = 0.0f;
    int cnt = 0;
    while (i < n && keys[i] == key) {
#pragma unroll
      for (int d = 0; d < D; ++d) acc[d] = acc[d] + pts[i * D + d];
      ++cnt;
      ++i;
    }
    const float fc = (float)cnt;
#pragma unroll
    for (int d = 0; d < D; ++d) out_pts[u * D + d] = acc[d] / fc;
    out_bids[u] = (int)(key / total);
    out_idx[u] = first_idx[u];
  }
}

struct SamplingWorkspace {
  int *cell_scan;    // [n]
  int *first_idx;    // [n]
  int *used;         // [n], and behind it the counts and cursors of the parity classes
  int *class_counts, *cursors;
  int *sel_scan;     // [n]
  int *scan_scratch;
  int64_t *num_cells_total;
  int64_t *num_selected;
  int2 *slices;      // [n, cell rows], of a selection without a pair table
  size_t bytes;
};

// `slices_per_cell`: 0 where the selection has a pair table.
static SamplingWorkspace carve_sampling_workspace(void *ws, int64_t n, int slices_per_cell = 0) {
  char *p = (char *)ws;
  SamplingWorkspace w;
  size_t off = 0;
  const size_t arr = align256(sizeof(int) * (size_t)n);
  w.cell_scan = (int *)(p + off); off += arr;
  w.first_idx = (int *)(p + off); off += arr;
  w.used = (int *)(p + off); off += arr;
  w.class_counts = (int *)(p + off); off += sizeof(int) * kMaxClasses;
  w.cursors = (int *)(p + off); off += sizeof(int) * kMaxClasses;
  w.sel_scan = (int *)(p + off); off += arr;
  w.scan_scratch = (int *)(p + off); off += align256(sizeof(int) * scan_scratch_ints(n));
  w.num_cells_total = (int64_t *)(p + off); off += 256;
  w.num_selected = (int64_t *)(p + off); off += 256;
  w.slices = (int2 *)(p + off); off += align256(sizeof(int2) * (size_t)n * slices_per_cell);
  w.bytes = off;
  return w;
}

__global__ void __launch_bounds__(256) copy_i32_kernel(int64_t n, const int *__restrict__ src,
                                                       int *__restrict__ dst) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

}  // namespace mccnn

using namespace mccnn;

extern "C" size_t mccnn_sampling_workspace_bytes(int64_t num_pts) {
  if (num_pts < 0) num_pts = 0;
  return carve_sampling_workspace(nullptr, num_pts).bytes;
}

extern "C" size_t mccnn_sampling_grid_workspace_bytes(int num_dims, int64_t num_pts) {
  if (!valid_dims(num_dims) || num_pts < 0) return 0;
  return carve_sampling_workspace(nullptr, num_pts, offsets_for(num_dims)).bytes;
}

// What a selection without a pair table has in its place.
struct DiskGrid {
  const float *inv_radii;
  const int2 *ds;          // column table, or null: the keys are searched
};

static int sampling_count(mccnn_stream_t stream, int mode, int64_t num_pts, int num_dims,
                                    const float *points, int64_t batch_ids_len,
                                    const int32_t *batch_ids, int64_t point_keys_len,
                                    const int64_t *point_keys, int num_cells_len,
                                    const int32_t *num_cells, int64_t num_neighbors,
                                    int neighbors_rank, int neighbors_cols,
                                    const int32_t *neighbors, int64_t ranges_len,
                                    const int32_t *ranges, void *workspace,
                                    size_t workspace_bytes, bool pinned, int64_t *num_sampled_out_host,
                                    const DiskGrid *disk = nullptr) {
  MCCNN_REQUIRE(mode >= 0 && mode < 2, "Sampling requires a valid sampling mode");
  MCCNN_REQUIRE(valid_dims(num_dims), "Sampling expects a valid number of dimensions");
  MCCNN_REQUIRE(batch_ids_len == num_pts,
                "Sampling expects the same number of batch ids as number of points");
  MCCNN_REQUIRE(point_keys_len == num_pts,
                "Sampling expects the same number of keys as number of points");
  MCCNN_REQUIRE(num_cells_len == num_dims,
                "Sampling expects a number of dimensions in num_cells equal to the number of "
                "dimensions in the input points");
  MCCNN_REQUIRE(neighbors_rank == 2 && neighbors_cols == 2,
                "Sampling expects a neighbor tensor with 2 dimensions and 2 indices per neighbor");
  MCCNN_REQUIRE(ranges_len == num_pts,
                "Sampling expects the same number of points in ranges as in the points tensor");
  MCCNN_REQUIRE(num_pts >= 0 && num_pts < ((int64_t)1 << 31) && num_neighbors >= 0,
                "Sampling expects sizes in [0, 2^31)");
  MCCNN_REQUIRE(num_sampled_out_host, "Sampling received a null output");
  *num_sampled_out_host = 0;
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(points && batch_ids && point_keys && num_cells && workspace &&
                    (disk ? disk->inv_radii != nullptr
                          : ranges && (neighbors || num_neighbors == 0)),
                "Sampling received a null tensor");
  const SamplingWorkspace w =
      carve_sampling_workspace(workspace, num_pts, disk ? offsets_for(num_dims) : 0);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "Sampling workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  hipStream_t s = as_stream(stream);
  const unsigned grid = blocks_for(num_pts, 256);
  // pinned: the last count goes straight to the host
  if (pinned) *num_sampled_out_host = -1;
  int64_t *cells = pinned && mode == 1 ? num_sampled_out_host : w.num_cells_total;
  int rc = MCCNN_OK;
  if (num_pts <= kStartMax) {
    auto kernel = num_pts <= 4 * kStartThreads ? cell_starts_block_kernel<4>
                                               : cell_starts_block_kernel<16>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kStartThreads), 0, s, (int)num_pts,
                       (const int64_t *)point_keys, w.first_idx, cells);
    MCCNN_LAUNCH_CHECK();
  } else {
    hipLaunchKernelGGL(flag_cell_starts_kernel, dim3(grid), dim3(256), 0, s, num_pts,
                       (const int64_t *)point_keys, w.cell_scan);
    MCCNN_LAUNCH_CHECK();
    rc = inclusive_scan_i32(s, num_pts, w.cell_scan, w.scan_scratch, cells);
    if (rc != MCCNN_OK) return rc;
    hipLaunchKernelGGL(store_cell_starts_kernel, dim3(grid), dim3(256), 0, s, num_pts,
                       (const int64_t *)point_keys, w.cell_scan, w.first_idx);
    MCCNN_LAUNCH_CHECK();
  }
  const int64_t *result = w.num_cells_total;
  if (mode == 0) {
    rc = fill_zero(s, w.used, (char *)(w.cursors + kMaxClasses) - (char *)w.used);
    if (rc != MCCNN_OK) return rc;
    // at most num_pts occupied cells; the kernels read the true count on device.  The
    // classes live in sel_scan, which is only filled after the passes, their cells in cell_scan,
    // which the cells' starts have been taken from.
    MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(cell_class_kernel<D>, dim3(grid), dim3(256), 0, s,
                                                  w.num_cells_total, (const int64_t *)point_keys,
                                                  num_cells, w.first_idx, w.sel_scan,
                                                  w.class_counts));
    MCCNN_LAUNCH_CHECK();
    MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(class_list_kernel<D>, dim3(grid), dim3(256), 0, s,
                                                  w.num_cells_total, w.sel_scan, w.class_counts,
                                                  w.cursors, w.cell_scan));
    MCCNN_LAUNCH_CHECK();
    if (disk) {
      MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(
          cell_rows_kernel<D>,
          dim3(blocks_for(num_pts, kWave), (unsigned)(OffsetInfo<D>::count() / kRowWaves)),
          dim3(kRowWaves * kWave), 0, s, num_pts, w.num_cells_total, (const int64_t *)point_keys,
          disk->ds, num_cells, w.first_idx, w.slices));
      MCCNN_LAUNCH_CHECK();
    }
    unsigned wgrid = blocks_for(num_pts, 256 / kWave);
    if (wgrid > (unsigned)kDiskBlocks) wgrid = kDiskBlocks;
    for (int call = 0; call < (1 << num_dims); ++call) {
      if (disk)
        MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(
            poisson_cells_kernel<D>, dim3(wgrid), dim3(256), 0, s, num_pts, call,
            w.num_cells_total, w.class_counts, w.cell_scan, w.slices, w.first_idx, points,
            disk->inv_radii, w.used))
      else
        hipLaunchKernelGGL(poisson_pass_kernel, dim3(wgrid), dim3(256), 0, s, num_pts, call,
                           w.num_cells_total, w.class_counts, w.cell_scan,
                           (const int2 *)neighbors, ranges, w.first_idx, w.used);
      MCCNN_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(copy_i32_kernel, dim3(grid), dim3(256), 0, s, num_pts, w.used, w.sel_scan);
    MCCNN_LAUNCH_CHECK();
    rc = inclusive_scan_i32(s, num_pts, w.sel_scan, w.scan_scratch,
                            pinned ? num_sampled_out_host : w.num_selected);
    if (rc != MCCNN_OK) return rc;
    result = w.num_selected;
  }
  if (pinned) return wait_for_host_values(s, num_sampled_out_host, 1);
  MCCNN_HIP_CHECK(hipMemcpyAsync(num_sampled_out_host, result, sizeof(int64_t),
                                 hipMemcpyDeviceToHost, s));
  MCCNN_HIP_CHECK(hipStreamSynchronize(s));
  return MCCNN_OK;
}

extern "C" int mccnn_sampling_count(
    mccnn_stream_t stream, int mode, int64_t num_pts, int num_dims, const float *points,
    int64_t batch_ids_len, const int32_t *batch_ids, int64_t point_keys_len,
    const int64_t *point_keys, int num_cells_len, const int32_t *num_cells, int64_t num_neighbors,
    int neighbors_rank, int neighbors_cols, const int32_t *neighbors, int64_t ranges_len,
    const int32_t *ranges, void *workspace, size_t workspace_bytes, int64_t *num_sampled_out_host) {
  return sampling_count(stream, mode, num_pts, num_dims, points, batch_ids_len, batch_ids,
                        point_keys_len, point_keys, num_cells_len, num_cells, num_neighbors,
                        neighbors_rank, neighbors_cols, neighbors, ranges_len, ranges, workspace,
                        workspace_bytes, false, num_sampled_out_host);
}

extern "C" int mccnn_sampling_count_pinned(
    mccnn_stream_t stream, int mode, int64_t num_pts, int num_dims, const float *points,
    int64_t batch_ids_len, const int32_t *batch_ids, int64_t point_keys_len,
    const int64_t *point_keys, int num_cells_len, const int32_t *num_cells, int64_t num_neighbors,
    int neighbors_rank, int neighbors_cols, const int32_t *neighbors, int64_t ranges_len,
    const int32_t *ranges, void *workspace, size_t workspace_bytes, int64_t *num_sampled_out_pinned) {
  return sampling_count(stream, mode, num_pts, num_dims, points, batch_ids_len, batch_ids,
                        point_keys_len, point_keys, num_cells_len, num_cells, num_neighbors,
                        neighbors_rank, neighbors_cols, neighbors, ranges_len, ranges, workspace,
                        workspace_bytes, true, num_sampled_out_pinned);
}

extern "C" int mccnn_sampling_grid_count_pinned(
    mccnn_stream_t stream, int64_t num_pts, int num_dims, const float *points,
    const int32_t *batch_ids, const int64_t *point_keys, const int32_t *grid_ds,
    const int32_t *num_cells, const float *inv_radii, void *workspace, size_t workspace_bytes,
    int64_t *num_sampled_out_pinned) {
  const DiskGrid disk = {inv_radii, (const int2 *)grid_ds};
  return sampling_count(stream, 0, num_pts, num_dims, points, num_pts, batch_ids, num_pts,
                        point_keys, num_dims, num_cells, 0, 2, 2, nullptr, num_pts, nullptr,
                        workspace, workspace_bytes, true, num_sampled_out_pinned, &disk);
}

extern "C" int mccnn_sampling_fill(mccnn_stream_t stream, int mode, int64_t num_pts, int num_dims,
                                   const float *points, const int32_t *batch_ids,
                                   const int64_t *point_keys, const int32_t *num_cells,
                                   void *workspace, size_t workspace_bytes, int64_t num_sampled,
                                   float *sample_pts_out, int32_t *sample_batch_ids_out,
                                   int32_t *sample_indices_out) {
  MCCNN_REQUIRE(mode >= 0 && mode < 2, "Sampling requires a valid sampling mode");
  MCCNN_REQUIRE(valid_dims(num_dims), "Sampling expects a valid number of dimensions");
  MCCNN_REQUIRE(num_pts >= 0 && num_sampled >= 0 && num_sampled <= num_pts,
                "Sampling expects 0 <= num_sampled <= num_pts");
  if (num_pts == 0 || num_sampled == 0) return MCCNN_OK;
  MCCNN_REQUIRE(points && batch_ids && point_keys && num_cells && workspace && sample_pts_out &&
                    sample_batch_ids_out && sample_indices_out,
                "Sampling received a null tensor");
  const SamplingWorkspace w = carve_sampling_workspace(workspace, num_pts);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "Sampling workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  hipStream_t s = as_stream(stream);
  if (mode == 0) {
    MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(store_selected_kernel<D>,
                                                  dim3(blocks_for(num_pts, 256)), dim3(256), 0, s,
                                                  num_pts, points, batch_ids, w.used, w.sel_scan,
                                                  sample_pts_out, sample_batch_ids_out,
                                                  sample_indices_out));
  } else {
    MCCNN_DIM_SWITCH(num_dims, hipLaunchKernelGGL(cell_average_kernel<D>,
                                                  dim3(blocks_for(num_sampled, 256)), dim3(256), 0,
                                                  s, num_pts, num_sampled, points,
                                                  (const int64_t *)point_keys, num_cells,
                                                  w.first_idx, sample_pts_out,
                                                  sample_batch_ids_out, sample_indices_out));
  }
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}
