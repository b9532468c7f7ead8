// Radius neighbour search on the sorted regular grid
// (custom_ops/tfg_custom_ops/find_neighbors/cc/ops/find_neighbors_ops.cpp:86-250).
//
// Three stages, all deterministic:
//   ranges  one lane per (centre, cell offset): the column of the 2-D table and
//           a binary search over the descending keys give the contiguous slice
//           of sorted points that lies in the offset cell row
//           (find_ranges_grid_ds_kernels.cu.cc:48-235);
//   count   8 lanes per centre stride over the slices and test
//           |(s - p) * inv_radii| < 1 (count_neighbors_kernels.cu.cc:83-86; as the
//           squared length against 1, which decides identically);
//   fill    the hits that the count pass has left as bits, one word per lane and window of
//           trips; the slot of a hit is the centre's start offset plus a ballot prefix inside
//           the 8-lane group, so the pairs of a centre come out in ascending sorted-point index
//           without atomics or a sort.
// Offsets are enumerated so that the slices of a centre ascend in index.
// (The bits cost the count pass nothing: instead of a running number of hits a lane shifts each
// outcome into a word, one add with carry either way, and counts the word's bits at its end.)
// Small inputs are bound by launches: there the count pass finds its slices itself (every
// lane of a group searches one or two), and a grid without a column table, which would need
// the grid's shape on the host first, is searched over all of its keys.
// Compiled with -ffp-contract=off (the distance test decides integer output).
#include "common.h"
#include "fill.h"
#include "search.h"

namespace mccnn {

// 8 lanes per centre: with the unreachable cells left out a slice holds one or two cells,
// and a wavefront steps through the union of what its centres need, so narrow groups
// waste fewer lanes (16 lanes: 7 % slower on the dense case, 10 % on clustered clouds;
// 32 lanes: 25 % slower).
constexpr int kGroup = 8;                  // lanes per centre
constexpr int kNbrThreads = 256;
constexpr int kCentresPerBlock = kNbrThreads / kGroup;
constexpr int kTrips = 32;                 // trips of eight candidates listed at a time
// Windows of 32 trips whose hits the count pass keeps for the fill pass (64 bytes per centre):
// 21.6 trips on average where a centre has 37 neighbours.  Candidates behind them -- crowded
// centres, and the slices after the first nine from four dimensions on -- are tested again.
constexpr int kMaskWindows = 2;

// What a search needs of the grid, per dimension in registers.
template <int D>
struct SearchGrid {
  GridShape<D> g;
  float ic[D], rho[D];                 // rho: one cell in units of the radius
  __device__ __forceinline__ SearchGrid(const int *__restrict__ num_cells,
                                        const float *__restrict__ inv_cell,
                                        const float *__restrict__ inv_radii)
      : g(load_shape<D>(num_cells)) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      ic[d] = inv_cell[d];
      rho[d] = inv_radii[d] / ic[d];
    }
  }
};

// Cell row r of the neighbourhood of point p (cloud b).  `ds` is the column table, or null: then
// the whole key array [0, np) is searched.
template <int D>
__device__ __forceinline__ KeyRange cell_row_keys(const SearchGrid<D> &sg, const float *p, int b,
                                                  int r, int64_t np, const int2 *__restrict__ ds,
                                                  const float *__restrict__ smin) {
  constexpr int OD = OffsetInfo<D>::kDims;
  const GridShape<D> &g = sg.g;
  float m[D];
#pragma unroll
  for (int d = 0; d < D; ++d) m[d] = smin[(int64_t)b * D + d];
  int cell[D];
  cell_of_point<D>(p, m, sg.ic, g, cell);
  // The centre in cell units, as the keys were computed, and what rounding can have
  // moved a point across a cell face: a point filed under cell x has a true
  // coordinate within `slack` of [x, x + 1) (outermost cells: unbounded outwards).
  float rel[D], slack[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const float prod = p[d] * sg.ic[d];
    rel[d] = prod - m[d];
    slack[d] = 9.6e-7f * (fabsf(prod) + fabsf(m[d]) + 1.0f);       // 8 float epsilons
  }
  // offset digits, most significant = dim 0, value 1 - digit (descending); g2 = lower
  // bound of the squared scaled distance to any point of the offset cell row, taken
  // over the offset dimensions
  bool inside = true;
  float g2 = 0.0f;
#pragma unroll
  for (int d = OD - 1; d >= 0; --d) {
    const int off = 1 - (r % 3);
    r /= 3;
    float gap = off < 0 ? rel[d] - (float)cell[d]
                        : (off > 0 ? (float)(cell[d] + 1) - rel[d] : 0.0f);
    gap = fmaxf(gap - slack[d], 0.0f) * sg.rho[d];
    g2 += gap * gap;
    cell[d] += off;
    inside = inside && cell[d] >= 0 && cell[d] < g.n[d];
  }
  // Cells that no pair of the exact test can come from are left out: every candidate
  // dropped here has a scaled distance of at least sqrt(1 + 1e-5) > 1, whatever the
  // rounding of the test itself (a few 1e-7), so the pairs found do not change.
  g2 *= 0.99999f;
  const KeyRange none = {make_int2(0, 0), 0, 1};
  if (!inside || !(g2 < 1.0f)) return none;
  int2 span = make_int2(0, (int)np);
  if (ds) span = ds[((int64_t)b * g.n[0] + cell[0]) * g.n[1] + cell[1]];
  if (span.y <= span.x) return none;
  if (D == 2 && ds) return KeyRange{span, 0, 1};
  const int64_t aux = key_of_cell<D>(cell, g, b);
  int64_t maxk = aux, mink = aux;
  if (D > 2) {
    const int w = cell[D - 1], nw = g.n[D - 1];
    // last dimension: the cells w - 1 .. w + 1 of the reference, cut to those the
    // sphere can reach given the offset in the other dimensions (out-of-range
    // coordinates belong to the outermost cells).  The approximate root and reciprocal are off by
    // a few 1e-7, what is left out keeps a distance of 1e-5.
    const float reach = __builtin_amdgcn_sqrtf(1.0f - g2) *
                            __builtin_amdgcn_rcpf(sg.rho[D - 1]) * 1.00001f + slack[D - 1];
    int wlo = (int)floorf(fmaxf(rel[D - 1] - reach, -1.0f));
    int whi = (int)floorf(fminf(rel[D - 1] + reach, (float)nw));
    wlo = wlo < 0 ? 0 : (wlo > nw - 1 ? nw - 1 : wlo);
    whi = whi < 0 ? 0 : (whi > nw - 1 ? nw - 1 : whi);
    wlo = wlo > w - 1 ? wlo : (w > 0 ? w - 1 : 0);
    whi = whi < w + 1 ? whi : (w < nw - 1 ? w + 1 : nw - 1);
    if (whi < wlo) return none;
    maxk = aux + (whi - w);
    mink = aux + (wlo - w);
  }
  return KeyRange{span, maxk, mink};
}

// One block per 64 centres and nine slices of each, a wavefront per slice: which cell row it is, and
// all that follows from it, is then the same for the lanes, and 64 neighbouring centres look
// for the slice in the same few columns.  Bound by instruction issue (one lane per centre and
// slice, numbered through: 413 vector instructions per wavefront, units busy for 80 % of the time;
// 763 k centres x 37 pairs 90 -> 82 us, 200 k x 52 in each of four clouds 145 -> 108).
// The slices lie by number, [R, ns]: stored and read as runs of centres.
constexpr int kRowWaves = 9;
template <int D>
__global__ void __launch_bounds__(kRowWaves * kWave) nbr_ranges_kernel(
    int64_t ns, const float *__restrict__ samples, const int *__restrict__ sbids, int64_t np,
    const int64_t *__restrict__ keys, const int2 *__restrict__ ds,
    const int *__restrict__ num_cells, const float *__restrict__ smin,
    const float *__restrict__ inv_cell, const float *__restrict__ inv_radii,
    int2 *__restrict__ ranges) {
  const int r = kRowWaves * blockIdx.y +
                __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int64_t c = (int64_t)blockIdx.x * kWave + lane_id();
  if (c >= ns) return;
  const SearchGrid<D> sg(num_cells, inv_cell, inv_radii);
  float p[D];
#pragma unroll
  for (int d = 0; d < D; ++d) p[d] = samples[c * D + d];
  const KeyRange range = cell_row_keys<D>(sg, p, sbids[c], r, np, ds, smin);
  int2 slice;
  find_slices<1>(&range, keys, &slice);
  ranges[r * ns + c] = slice;
}

// What a visit of a centre's candidates produces.
enum class Visit {
  kCount,      // counts[c] = number of hits (clamped to max_neighs when > 0)
  kFill,       // the pairs of centre c from its start offset on
  kDensity,    // density[c]: the kernel density of centre c over its hits (DensitySums)
};

// The kernel density of a centre, summed as compute_pdf_kernel (pdf.hip) sums it over the pair
// table: there G lanes take the pairs of a centre in turn, and G goes by the mean length of a
// list, which nobody knows before all centres are visited.  So the three sums are kept side by
// side and grid_density_select_kernel takes the one that the table would have given: the same
// bits whether a cloud's pairs are at hand or not (a difference in the last place moves a
// network's activations across kinks: one classifier pass in ten had gradients off by 2e-4).
// The eight lanes of a group hold one candidate each; a trip's hits go to the lane of their
// number in the list modulo eight.  Against one plain sum per lane: 17.3 -> 20.6 us for 16 384
// points of the three-level network, and 3.8 us of the selecting launch.
struct DensitySums {
  float four = 0.0f, eight = 0.0f, low = 0.0f, high = 0.0f;   // high: sixteenths 8..15
  // value of this lane's hit (0 without one), the group's hits as bits, hits of earlier trips
  __device__ __forceinline__ void add(float value, unsigned hits, int sub, int group, int found) {
    const int rank = __popc(hits & ((1u << sub) - 1u)), count = __popc(hits);
    const int slot = (hits >> sub) & 1u ? found + rank : found + count + (sub - rank);
    const float w = __int_as_float(
        __builtin_amdgcn_ds_permute(4 * (group + (slot & 7)), __float_as_int(value)));
    eight += w;
    if (((found + ((sub - found) & 7)) >> 3) & 1) high += w;
    else low += w;
    const int first = (found + ((sub - found) & 3)) & 7;
    four += __shfl(w, first, 8);
    four += __shfl(w, first ^ 4, 8);
  }
  __device__ __forceinline__ void finish() {
#pragma unroll
    for (int off = 2; off > 0; off >>= 1) four += __shfl_xor(four, off, kWave);
    low += high;
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) {
      eight += __shfl_xor(eight, off, kWave);
      low += __shfl_xor(low, off, kWave);
    }
  }
};

// One pair's part, with the contractions of pdf.hip (this file is built without any): those of
// the sum of squares, and those inside the exponential.
template <int D>
__device__ __forceinline__ float density_term(const float *diff, const float *scale) {
#pragma clang fp contract(fast)
  float e = 0.0f;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const float u = diff[d] * scale[d];
    e += u * u;
  }
  return expf(-0.5f * e);
}

struct VisitSearch {                  // for kSearch: the grid to find the slices in
  const int *sbids;
  int64_t np;
  const int64_t *keys;
  const int2 *ds;
  const int *num_cells;
  const float *smin, *inv_cell;
};

// kSearch: the lanes of a group find the centre's slices themselves (kCount also stores them
// for the fill pass); otherwise `ranges` holds them.
template <int D, Visit kVisit, bool kSearch>
__global__ void __launch_bounds__(kNbrThreads) nbr_visit_kernel(
    int64_t ns, const float *__restrict__ samples, const float *__restrict__ pts,
    int2 *ranges, unsigned *masks, const float *__restrict__ inv_radii, int max_neighs,
    VisitSearch search,
    int *__restrict__ counts, const int *__restrict__ ends, int2 *__restrict__ nbrs,
    int64_t *__restrict__ truncated, int64_t capacity, const float *__restrict__ inv_bandwidth,
    int mode, float *__restrict__ density /* kDensity: [3, ns], counts: hits per wavefront */) {
  constexpr int R = OffsetInfo<D>::count();
  constexpr int kAhead = 4;                        // trips in flight
  __shared__ __align__(16) int2 trips[kCentresPerBlock][kTrips + kAhead];
  const int sub = threadIdx.x & (kGroup - 1);
  const int lane = lane_id();
  float ir[D];
#pragma unroll
  for (int d = 0; d < D; ++d) ir[d] = inv_radii[d];
  const int64_t c = (int64_t)blockIdx.x * kCentresPerBlock + threadIdx.x / kGroup;
  if (c >= ns) return;
  float s[D];
#pragma unroll
  for (int d = 0; d < D; ++d) s[d] = samples[c * D + d];
  const int limit = max_neighs > 0 ? max_neighs : 0x7fffffff;
  int found = 0;                                   // hits so far (kCount: of this lane)
  int64_t start = 0;
  if (kVisit == Visit::kFill) start = c > 0 ? ends[c - 1] : 0;
  float scale[D], norm = 1.0f;                     // kDensity, as compute_pdf (pdf.hip)
  DensitySums sums;
  if (kVisit == Visit::kDensity) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const float bw = mode == 0 ? inv_bandwidth[d] : sqrtf((float)ns);
      scale[d] = bw * ir[d];
      norm *= bw * 0.39894228f;
    }
  }
  const bool upper = lane >= 32;                                // the group's bits in a ballot
  const int shift = lane & 24;
  const unsigned below = (1u << sub) - 1u;
  int2 *const list = nbrs + start;                              // kFill: the centre's pairs,
  const int64_t space = capacity - start;                       // and how many are stored
  const int most = (int)(space < limit ? (space > 0 ? space : 0) : limit);
  auto hits_of = [&](uint64_t ballot) {                         // of the group
    return ((upper ? (unsigned)(ballot >> 32) : (unsigned)ballot) >> shift) & 0xffu;
  };
  auto inside = [&](bool live, const float *q, float *diff) {
#pragma unroll
    for (int d = 0; d < D; ++d) diff[d] = s[d] - q[d];
    return within_radius<D>(live, diff, ir);
  };
  auto store_pair = [&](bool hit, int j) {                      // kGroup candidates of the centre
    const unsigned hits = hits_of(__ballot(hit));
    const int slot = found + __popc(hits & below);
    if (hit && slot < most) list[slot] = make_int2(j, (int)c);
    found += __popc(hits);
  };
  // The slices of the centre, nine at a time (their number is a power of three): lane `sub`
  // fetches or finds one, the first lane the ninth as well.  They are cut into trips of eight
  // candidates whose bounds go into LDS, and the group walks the list of trips, four in flight,
  // without a branch but the end of the list.  The count pass is bound by instruction issue (its vector
  // instructions, at four cycles each, fill the time), the fill pass for three quarters.  Slice by slice a trip took 45 instructions, a third
  // of them for the exec mask, and a wavefront took in each slice the trips of its fullest centre;
  // the list takes 24, and 14 in the fill pass, which neither loads nor tests the candidates.
  // 763 k centres x 37 pairs: count 150 -> 116 us, fill 216 -> 121; densities of 16 384 points
  // straight from the grid 19.4 -> 16.2.  (Two trips in flight: 125 and 118.)
  constexpr int kSlices = kGroup + 1;
  static_assert(R % kSlices == 0, "slices come in nines");
  int2 *const trip = trips[threadIdx.x / kGroup];
  for (int r0 = 0; r0 < R; r0 += kSlices) {
    int2 mine[2] = {make_int2(0, 0), make_int2(0, 0)};          // slices r0 + sub and r0 + kGroup
    if constexpr (kSearch) {
      const SearchGrid<D> sg(search.num_cells, search.inv_cell, inv_radii);
      const int b = search.sbids[c];
      KeyRange range[2] = {
          cell_row_keys<D>(sg, s, b, r0 + sub, search.np, search.ds, search.smin),
          cell_row_keys<D>(sg, s, b, r0 + kGroup, search.np, search.ds, search.smin)};
      if (sub != 0) range[1] = KeyRange{make_int2(0, 0), 0, 1};
      find_slices<2>(range, search.keys, mine);
      if (kVisit == Visit::kCount) {
        ranges[(r0 + sub) * ns + c] = mine[0];
        if (sub == 0) ranges[(r0 + kGroup) * ns + c] = mine[1];
      }
      mine[1] = make_int2(__shfl(mine[1].x, 0, kGroup), __shfl(mine[1].y, 0, kGroup));
    } else {
      mine[0] = ranges[(r0 + sub) * ns + c];
      mine[1] = ranges[(r0 + kGroup) * ns + c];
    }
    const int n0 = (mine[0].y - mine[0].x + kGroup - 1) / kGroup;
    const int n1 = (mine[1].y - mine[1].x + kGroup - 1) / kGroup;
    int upto = n0;                                              // trips of slices r0 .. r0 + sub
#pragma unroll
    for (int off = 1; off < kGroup; off *= 2) {
      const int o = __shfl_up(upto, off, kGroup);
      upto += sub >= off ? o : 0;
    }
    const int before1 = __shfl(upto, kGroup - 1, kGroup), total = before1 + n1;
    // (as many windows as the group has: the wavefront's other groups have lists of their own)
    for (int t0 = 0; t0 < total; t0 += kTrips) {                // a window of the trips
      group_lds_sync();                                         // the window before has been read
      const int first = upto - n0 - t0;
      for (int k = first < 0 ? -first : 0; k < n0 && first + k < kTrips; ++k)
        trip[first + k] = make_int2(mine[0].x + kGroup * k, mine[0].y);
      for (int k = sub; k < n1; k += kGroup)
        if (before1 + k - t0 >= 0 && before1 + k - t0 < kTrips)
          trip[before1 + k - t0] = make_int2(mine[1].x + kGroup * k, mine[1].y);
      const int n = total - t0 < kTrips ? total - t0 : kTrips;
      if (sub < kAhead) trip[n + sub] = make_int2(0, 0);        // (no candidates)
      group_lds_sync();
      const bool masked = r0 == 0 && t0 < kTrips * kMaskWindows;
      const int64_t mask_at = ((int64_t)(t0 / kTrips) * ns + c) * kGroup + sub;
      if (kVisit == Visit::kFill && masked) {
        unsigned word = masks[mask_at];
        for (int t = 0; t < n; t += kAhead) {
#pragma unroll
          for (int u = 0; u < kAhead; ++u) {
            store_pair((int)word < 0, trip[t + u].x + sub);
            word <<= 1;
          }
        }
        continue;
      }
      unsigned word = 0;                                        // kCount: this lane's hits
      for (int t = 0; t < n; t += kAhead) {
        int j[kAhead];
        bool live[kAhead];
        float q[kAhead][D];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const int2 span = trip[t + u];
          j[u] = span.x + sub;
          live[u] = j[u] < span.y;
          const int from = live[u] ? j[u] : span.x;             // some point: the trip's first
#pragma unroll
          for (int d = 0; d < D; ++d) q[u][d] = pts[(int64_t)from * D + d];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          float diff[D];
          const bool hit = inside(live[u], q[u], diff);
          if (kVisit == Visit::kCount) {
            word = word + word + (hit ? 1u : 0u);
          } else if (kVisit == Visit::kFill) {
            store_pair(hit, j[u]);
          } else {
            const unsigned hits = hits_of(__ballot(hit));
            if (hits != 0) {                   // the same for the lanes of a group
              sums.add(hit ? density_term<D>(diff, scale) : 0.0f, hits, sub, lane & ~(kGroup - 1),
                       found);
              found += __popc(hits);
            }
          }
        }
      }
      if (kVisit == Visit::kCount) {
        found += __popc(word);
        if (masked) masks[mask_at] = word << (kTrips - (n + kAhead - 1) / kAhead * kAhead);
      }
    }
  }
  if (kVisit == Visit::kCount) {
#pragma unroll
    for (int off = kGroup / 2; off > 0; off >>= 1) found += __shfl_xor(found, off, kWave);
    if (sub == 0) {
      counts[c] = found < limit ? found : limit;
      // some centre lost pairs to max_neighs (every writer stores the same value)
      if (truncated && found > limit) *truncated = 1;
    }
  }
  if (kVisit == Visit::kDensity) {
    sums.finish();
    if (sub == 0) {
      density[c] = sums.four * norm;
      density[ns + c] = sums.eight * norm;
      density[2 * ns + c] = sums.low * norm;
    }
    int pairs = 0;                      // of the wavefront's centres (those past the end have left)
    const int64_t first = c - lane / kGroup;
#pragma unroll
    for (int g = 0; g < kWave / kGroup; ++g)
      if (first + g < ns) pairs += __builtin_amdgcn_readlane(found, g * kGroup);
    if (lane == 0) counts[first / (kWave / kGroup)] = pairs;
  }
}

// The sums that compute_pdf would have taken for lists of this mean length (the rule of
// mccnn_compute_pdf).  Every block adds up all counts: 8 KB for 16 384 points, 400 KB from L2 for
// 800 000, and few blocks do.
constexpr int kSelectThreads = 1024, kSelectBlocks = 64;
__global__ void __launch_bounds__(kSelectThreads) grid_density_select_kernel(
    int64_t n, int64_t parts, const int *__restrict__ counts, const float *__restrict__ sums,
    float *__restrict__ pdf) {
  __shared__ int64_t part[kSelectThreads / kWave];
  int64_t pairs = 0;
  for (int64_t i = threadIdx.x; i < parts; i += blockDim.x) pairs += counts[i];
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) pairs += __shfl_xor(pairs, off, kWave);
  if (lane_id() == 0) part[threadIdx.x / kWave] = pairs;
  __syncthreads();
  pairs = 0;
  for (int w = 0; w < kSelectThreads / kWave; ++w) pairs += part[w];
  const int64_t mean = pairs / n;
  const float *from = sums + (mean <= 16 ? 0 : mean <= 96 ? n : 2 * n);
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < n;
       c += (int64_t)gridDim.x * blockDim.x)
    pdf[c] = from[c];
}

// Centres up to which the count pass finds its slices itself: 16 384 centres are 512 blocks,
// one launch of latency; beyond that the searches of a group's lanes (nine slices, eight
// lanes) cost more than a launch of one lane per slice (763 k centres: 88 us for the slices).
constexpr int64_t kSearchInVisit = 16384;

struct NbrWorkspace {
  int2 *ranges;
  unsigned *masks;       // [kMaskWindows, ns, kGroup]: what the count pass tells the fill pass
  int *scan_scratch;
  int64_t *total;
  size_t bytes;
};

static NbrWorkspace carve_nbr_workspace(void *ws, int d, int64_t ns) {
  char *p = (char *)ws;
  NbrWorkspace w;
  size_t off = 0;
  w.ranges = (int2 *)(p + off);
  off += align256(sizeof(int2) * (size_t)ns * offsets_for(d));
  w.masks = (unsigned *)(p + off);
  off += align256(sizeof(unsigned) * (size_t)ns * kGroup * kMaskWindows);
  w.scan_scratch = (int *)(p + off);
  off += align256(sizeof(int) * scan_scratch_ints(ns));
  w.total = (int64_t *)(p + off);
  off += 256;
  w.bytes = off;
  return w;
}

// Pair table regrouped for another order of the centres: slot q takes the
// segment of centre order[q].  counts pass, then (after the scan) a copy pass;
// the centre column is rewritten to the slot.
__global__ void __launch_bounds__(256) segment_counts_kernel(int64_t n, const int *__restrict__ ranges,
                                                             const int *__restrict__ order,
                                                             int *__restrict__ counts) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int i = order[q];
  counts[q] = ranges[i] - (i > 0 ? ranges[i - 1] : 0);
}

// `map` (optional) replaces the point index by map[index]; either output may be null, pdf_out
// takes the density of the pair's point.  A wavefront takes `slots` <= 16 consecutive slots, whose
// pairs are one contiguous stretch of the output, and walks that stretch 64 pairs at a time, four
// times 64 in flight; a lane finds its pair's slot by a binary search among the slots' ends.
// (With 16 lanes on one slot the four dependent loads of a slot -- its centre, the segment, the
// pair, the mapped index -- stood behind each other for every 37 pairs: 174 us per output of 28 M
// pairs, 121 us now.)
constexpr int kCopySlots = 16, kCopyAhead = 4;

__global__ void __launch_bounds__(256) segment_copy_kernel(
    int64_t n, int slots, const int *__restrict__ ranges, const int *__restrict__ order,
    const int2 *__restrict__ pairs, const int *__restrict__ ranges_out,
    const int *__restrict__ map, int2 *__restrict__ pairs_out, const float *__restrict__ pdf,
    float *__restrict__ pdf_out) {
  const int lane = lane_id();
  const int64_t q0 = ((int64_t)blockIdx.x * (256 / kWave) + threadIdx.x / kWave) * slots;
  if (q0 >= n) return;
  // lane i < slots: end of slot q0 + i in the output and how far before it its pairs are read
  int end = 0x7fffffff, shift = 0;
  const int64_t q = q0 + lane;
  if (lane < slots && q < n) {
    const int i = order[q];
    end = ranges_out[q];
    shift = (i > 0 ? ranges[i - 1] : 0) - (q > 0 ? ranges_out[q - 1] : 0);
  }
  const int first = q0 > 0 ? ranges_out[q0 - 1] : 0;
  const int last = ranges_out[(q0 + slots < n ? q0 + slots : n) - 1];
  for (int64_t m0 = first; m0 < last; m0 += kWave * kCopyAhead) {
    int slot[kCopyAhead], j[kCopyAhead];
#pragma unroll
    for (int u = 0; u < kCopyAhead; ++u) {
      const int64_t m = m0 + u * kWave + lane;
      slot[u] = 0;                                  // ends up to m: 0 .. 15 of the first 15
#pragma unroll
      for (int step = kCopySlots / 2; step > 0; step >>= 1)
        if (__shfl(end, slot[u] + step - 1, kWave) <= m) slot[u] += step;
      const int from = __shfl(shift, slot[u], kWave);
      j[u] = m < last ? pairs[m + from].x : 0;
    }
    if (pairs_out) {
#pragma unroll
      for (int u = 0; u < kCopyAhead; ++u) {
        const int64_t m = m0 + u * kWave + lane;
        if (m < last) pairs_out[m] = make_int2(map ? map[j[u]] : j[u], (int)q0 + slot[u]);
      }
    }
    if (pdf_out) {
#pragma unroll
      for (int u = 0; u < kCopyAhead; ++u) {
        const int64_t m = m0 + u * kWave + lane;
        if (m < last) pdf_out[m] = pdf[j[u]];
      }
    }
  }
}

}  // namespace mccnn

using namespace mccnn;

extern "C" size_t mccnn_find_neighbors_workspace_bytes(int num_dims, int64_t num_samples) {
  if (!valid_dims(num_dims) || num_samples < 0) return 0;
  return carve_nbr_workspace(nullptr, num_dims, num_samples).bytes;
}

static int launch_ranges(hipStream_t s, int num_dims, int64_t ns, const float *samples,
                         const float *inv_radii, const VisitSearch &g, int2 *slices) {
  const dim3 grid(blocks_for(ns, kWave), (unsigned)(offsets_for(num_dims) / kRowWaves));
  MCCNN_DIM_SWITCH(num_dims,
                   hipLaunchKernelGGL(nbr_ranges_kernel<D>, grid, dim3(kRowWaves * kWave), 0, s, ns,
                                      samples, g.sbids, g.np, g.keys, g.ds, g.num_cells, g.smin,
                                      g.inv_cell, inv_radii, slices));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static int launch_count(hipStream_t s, int num_dims, int64_t ns, const float *samples,
                        const float *points, const NbrWorkspace &w, const float *inv_radii,
                        int max_neighs, const VisitSearch *search, int *counts,
                        int64_t *truncated) {
  const dim3 grid(blocks_for(ns, kCentresPerBlock)), block(kNbrThreads);
  if (search)
    MCCNN_DIM_SWITCH(num_dims,
                     hipLaunchKernelGGL((nbr_visit_kernel<D, Visit::kCount, true>), grid, block, 0,
                                        s, ns, samples, points, w.ranges, w.masks, inv_radii,
                                        max_neighs, *search, counts, (const int *)nullptr, (int2 *)nullptr,
                                        truncated, (int64_t)0, (const float *)nullptr, 0,
                                        (float *)nullptr))
  else
    MCCNN_DIM_SWITCH(num_dims,
                     hipLaunchKernelGGL((nbr_visit_kernel<D, Visit::kCount, false>), grid, block,
                                        0, s, ns, samples, points, w.ranges, w.masks, inv_radii,
                                        max_neighs, VisitSearch{}, counts, (const int *)nullptr,
                                        (int2 *)nullptr, truncated, (int64_t)0,
                                        (const float *)nullptr, 0, (float *)nullptr))
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static int launch_fill(hipStream_t s, int num_dims, int64_t ns, const float *samples,
                       const float *points, const NbrWorkspace &w, const float *inv_radii,
                       int max_neighs, const int *ends, int32_t *neighbors, int64_t capacity) {
  MCCNN_DIM_SWITCH(num_dims,
                   hipLaunchKernelGGL((nbr_visit_kernel<D, Visit::kFill, false>),
                                      dim3(blocks_for(ns, kCentresPerBlock)), dim3(kNbrThreads), 0,
                                      s, ns, samples, points, w.ranges, w.masks, inv_radii,
                                      max_neighs, VisitSearch{}, (int *)nullptr, ends, (int2 *)neighbors,
                                      (int64_t *)nullptr, capacity, (const float *)nullptr, 0,
                                      (float *)nullptr));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

// `facts_out_host` (optional, two values): [0] 1 if some centre lost pairs to max_neighs,
// [1] 1 if the centres are the searched points themselves (same address, same count).
static int find_neighbors_count_impl(
    mccnn_stream_t stream, int64_t num_samples, int num_dims, const float *samples,
    int64_t sample_batch_ids_len, const int32_t *sample_batch_ids, int64_t num_pts, int pts_dims,
    const float *points, int64_t point_keys_len, const int64_t *point_keys, int ds_rank,
    int ds_batch, int ds_nx, int ds_ny, int ds_last, const int32_t *grid_ds, int num_cells_len,
    const int32_t *num_cells, int aabb_dims, const float *scaled_aabb_min, int inv_cell_sizes_len,
    const float *inv_cell_sizes, int inv_radii_len, const float *inv_radii, int max_neighs,
    void *workspace, size_t workspace_bytes, int32_t *ranges_out,
    int64_t *num_neighbors_out_host, int64_t *facts_out_host, bool to_host = true) {
  int64_t unused_total = 0;
  if (!to_host) num_neighbors_out_host = &unused_total;   // the total stays in the workspace
  MCCNN_REQUIRE(valid_dims(num_dims), "FindNeighbors expects a valid number of dimensions");
  MCCNN_REQUIRE(num_cells_len == num_dims,
                "FindNeighbors expects a number of dimensions in num_cells equal to the number of "
                "dimensions in the input points");
  MCCNN_REQUIRE(pts_dims == num_dims,
                "FindNeighbors expects a number of dimensions in points equal to the number of "
                "dimensions in the samples");
  MCCNN_REQUIRE(aabb_dims == num_dims,
                "FindNeighbors expects a number of dimensions in scaled_aabb_min equal to the "
                "number of dimensions in the input points");
  MCCNN_REQUIRE(inv_cell_sizes_len == num_dims,
                "FindNeighbors expects a number of dimensions in inv_cell_sizes equal to the "
                "number of dimensions in the input points");
  MCCNN_REQUIRE(inv_radii_len == num_dims,
                "FindNeighbors expects a number of dimensions in inv_radii equal to the number of "
                "dimensions in the input points");
  MCCNN_REQUIRE(sample_batch_ids_len == num_samples,
                "FindNeighbors expects the same number of batch ids as samples");
  MCCNN_REQUIRE(point_keys_len == num_pts,
                "FindNeighbors expects the same number of keys as points");
  MCCNN_REQUIRE(ds_rank == 4 && ds_last == 2,
                "FindNeighbors expects a grid acceleration data structure with the right format "
                "(B, X, Y, 2)");
  MCCNN_REQUIRE(ds_batch > 0 && ds_nx > 0 && ds_ny > 0,
                "FindNeighbors expects a non-empty grid acceleration data structure");
  MCCNN_REQUIRE(num_samples >= 0 && num_pts >= 0 && num_samples < ((int64_t)1 << 31) &&
                    num_pts < ((int64_t)1 << 31),
                "FindNeighbors expects sizes in [0, 2^31)");
  MCCNN_REQUIRE(num_neighbors_out_host, "FindNeighbors received a null output");
  *num_neighbors_out_host = 0;
  if (facts_out_host) {
    facts_out_host[0] = 0;
    facts_out_host[1] = samples == points && num_samples == num_pts ? 1 : 0;
  }
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(samples && sample_batch_ids && grid_ds && num_cells && scaled_aabb_min &&
                    inv_cell_sizes && inv_radii && ranges_out && workspace,
                "FindNeighbors received a null tensor");
  MCCNN_REQUIRE(num_pts == 0 || (points && point_keys), "FindNeighbors received a null tensor");
  const NbrWorkspace w = carve_nbr_workspace(workspace, num_dims, num_samples);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "FindNeighbors workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  hipStream_t s = as_stream(stream);
  const VisitSearch search = {sample_batch_ids, num_pts, (const int64_t *)point_keys,
                              (const int2 *)grid_ds, num_cells, scaled_aabb_min, inv_cell_sizes};
  int rc = launch_ranges(s, num_dims, num_samples, samples, inv_radii, search, w.ranges);
  if (rc != MCCNN_OK) return rc;
  // truncation can only happen with max_neighs > 0: only then is the flag cleared and read
  int64_t *truncated = facts_out_host && max_neighs > 0 ? w.total + 1 : nullptr;
  if (truncated) {
    int rc0 = fill_zero(s, truncated, sizeof(int64_t));
    if (rc0 != MCCNN_OK) return rc0;
  }
  rc = launch_count(s, num_dims, num_samples, samples, points, w, inv_radii, max_neighs, nullptr,
                    ranges_out, truncated);
  if (rc != MCCNN_OK) return rc;
  rc = inclusive_scan_i32(s, num_samples, ranges_out, w.scan_scratch, w.total);
  if (rc != MCCNN_OK) return rc;
  if (!to_host) return MCCNN_OK;
  MCCNN_HIP_CHECK(hipMemcpyAsync(num_neighbors_out_host, w.total, sizeof(int64_t),
                                 hipMemcpyDeviceToHost, s));
  if (truncated)
    MCCNN_HIP_CHECK(hipMemcpyAsync(facts_out_host, truncated, sizeof(int64_t),
                                   hipMemcpyDeviceToHost, s));
  MCCNN_HIP_CHECK(hipStreamSynchronize(s));
  // the scan saturates partial sums at 2^31 - 1, so a total from there on is a lower bound
  MCCNN_REQUIRE(*num_neighbors_out_host < (((int64_t)1 << 31) - 1),
                "FindNeighbors found at least %lld pairs; the int32 offsets of the op contract "
                "hold fewer than 2^31 - 1",
                (long long)*num_neighbors_out_host);
  return MCCNN_OK;
}

extern "C" int mccnn_find_neighbors_count(
    mccnn_stream_t stream, int64_t num_samples, int num_dims, const float *samples,
    int64_t sample_batch_ids_len, const int32_t *sample_batch_ids, int64_t num_pts, int pts_dims,
    const float *points, int64_t point_keys_len, const int64_t *point_keys, int ds_rank,
    int ds_batch, int ds_nx, int ds_ny, int ds_last, const int32_t *grid_ds, int num_cells_len,
    const int32_t *num_cells, int aabb_dims, const float *scaled_aabb_min, int inv_cell_sizes_len,
    const float *inv_cell_sizes, int inv_radii_len, const float *inv_radii, int max_neighs,
    void *workspace, size_t workspace_bytes, int32_t *ranges_out,
    int64_t *num_neighbors_out_host) {
  return find_neighbors_count_impl(
      stream, num_samples, num_dims, samples, sample_batch_ids_len, sample_batch_ids, num_pts,
      pts_dims, points, point_keys_len, point_keys, ds_rank, ds_batch, ds_nx, ds_ny, ds_last,
      grid_ds, num_cells_len, num_cells, aabb_dims, scaled_aabb_min, inv_cell_sizes_len,
      inv_cell_sizes, inv_radii_len, inv_radii, max_neighs, workspace, workspace_bytes, ranges_out,
      num_neighbors_out_host, nullptr);
}

extern "C" int mccnn_find_neighbors_count_facts(
    mccnn_stream_t stream, int64_t num_samples, int num_dims, const float *samples,
    int64_t sample_batch_ids_len, const int32_t *sample_batch_ids, int64_t num_pts, int pts_dims,
    const float *points, int64_t point_keys_len, const int64_t *point_keys, int ds_rank,
    int ds_batch, int ds_nx, int ds_ny, int ds_last, const int32_t *grid_ds, int num_cells_len,
    const int32_t *num_cells, int aabb_dims, const float *scaled_aabb_min, int inv_cell_sizes_len,
    const float *inv_cell_sizes, int inv_radii_len, const float *inv_radii, int max_neighs,
    void *workspace, size_t workspace_bytes, int32_t *ranges_out,
    int64_t *num_neighbors_out_host, int64_t *facts_out_host) {
  MCCNN_REQUIRE(facts_out_host, "FindNeighbors received a null output");
  return find_neighbors_count_impl(
      stream, num_samples, num_dims, samples, sample_batch_ids_len, sample_batch_ids, num_pts,
      pts_dims, points, point_keys_len, point_keys, ds_rank, ds_batch, ds_nx, ds_ny, ds_last,
      grid_ds, num_cells_len, num_cells, aabb_dims, scaled_aabb_min, inv_cell_sizes_len,
      inv_cell_sizes, inv_radii_len, inv_radii, max_neighs, workspace, workspace_bytes, ranges_out,
      num_neighbors_out_host, facts_out_host);
}

extern "C" int mccnn_find_neighbors_fill(
    mccnn_stream_t stream, int64_t num_samples, int num_dims, const float *samples,
    const int32_t *sample_batch_ids, int64_t num_pts, const float *points,
    const int64_t *point_keys, const int32_t *grid_ds, const int32_t *num_cells,
    const float *scaled_aabb_min, const float *inv_cell_sizes, const float *inv_radii,
    int max_neighs, void *workspace, size_t workspace_bytes, const int32_t *ranges,
    int64_t num_neighbors, int32_t *neighbors_out) {
  (void)sample_batch_ids; (void)point_keys; (void)grid_ds; (void)num_cells;
  (void)scaled_aabb_min; (void)inv_cell_sizes; (void)num_pts;
  MCCNN_REQUIRE(valid_dims(num_dims), "FindNeighbors expects a valid number of dimensions");
  MCCNN_REQUIRE(num_samples >= 0 && num_neighbors >= 0, "FindNeighbors expects non-negative sizes");
  if (num_samples == 0 || num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(samples && points && inv_radii && ranges && neighbors_out && workspace,
                "FindNeighbors received a null tensor");
  const NbrWorkspace w = carve_nbr_workspace(workspace, num_dims, num_samples);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "FindNeighbors workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  return launch_fill(as_stream(stream), num_dims, num_samples, samples, points, w, inv_radii,
                     max_neighs, ranges, neighbors_out, (int64_t)1 << 62);
}

// count_out[0] = pairs found, count_out[1] = 1 if they do not fit the capacity
__global__ void publish_neighbor_count_kernel(const int64_t *__restrict__ total, int64_t capacity,
                                              int64_t *__restrict__ count_out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    count_out[0] = *total;
    count_out[1] = *total > capacity ? 1 : 0;
  }
}

extern "C" int mccnn_find_neighbors_bounded(
    mccnn_stream_t stream, int64_t num_samples, int num_dims, const float *samples,
    const int32_t *sample_batch_ids, int64_t num_pts, const float *points,
    const int64_t *point_keys, int ds_batch, int ds_nx, int ds_ny, const int32_t *grid_ds,
    const int32_t *num_cells, const float *scaled_aabb_min, const float *inv_cell_sizes,
    const float *inv_radii, int max_neighs, void *workspace, size_t workspace_bytes,
    int64_t capacity, int32_t *ranges_out, int32_t *neighbors_out, int64_t *count_out_device) {
  MCCNN_REQUIRE(capacity >= 0 && capacity < ((int64_t)1 << 31),
                "find_neighbors_bounded expects a capacity in [0, 2^31)");
  MCCNN_REQUIRE(count_out_device && (capacity == 0 || neighbors_out),
                "find_neighbors_bounded received a null output");
  int rc = find_neighbors_count_impl(
      stream, num_samples, num_dims, samples, num_samples, sample_batch_ids, num_pts, num_dims,
      points, num_pts, point_keys, 4, ds_batch, ds_nx, ds_ny, 2, grid_ds, num_dims, num_cells,
      num_dims, scaled_aabb_min, num_dims, inv_cell_sizes, num_dims, inv_radii, max_neighs,
      workspace, workspace_bytes, ranges_out, nullptr, nullptr, false);
  if (rc != MCCNN_OK) return rc;
  hipStream_t s = as_stream(stream);
  if (num_samples == 0) return fill_zero(s, count_out_device, 2 * sizeof(int64_t));
  const NbrWorkspace w = carve_nbr_workspace(workspace, num_dims, num_samples);
  hipLaunchKernelGGL(publish_neighbor_count_kernel, dim3(1), dim3(64), 0, s, w.total, capacity,
                     count_out_device);
  MCCNN_LAUNCH_CHECK();
  if (capacity == 0) return MCCNN_OK;
  return launch_fill(s, num_dims, num_samples, samples, points, w, inv_radii, max_neighs,
                     ranges_out, neighbors_out, capacity);
}

// Both halves of a count by a caller that has the grid in hand: slices, counts, end offsets and
// their total in `total` (device or pinned memory), with kScanFlag where *truncated has been set.
static int search_counts(hipStream_t s, int64_t num_samples, int num_dims, const float *samples,
                         const int32_t *sample_batch_ids, int64_t num_pts, const float *points,
                         const int64_t *point_keys, const int32_t *grid_ds,
                         const int32_t *num_cells, const float *scaled_aabb_min,
                         const float *inv_cell_sizes, const float *inv_radii, int max_neighs,
                         const NbrWorkspace &w, int32_t *ranges_out, int64_t *total,
                         int64_t *truncated) {
  const bool in_visit = num_samples <= kSearchInVisit;
  const VisitSearch search = {sample_batch_ids, num_pts, (const int64_t *)point_keys,
                              (const int2 *)grid_ds, num_cells, scaled_aabb_min, inv_cell_sizes};
  int rc = MCCNN_OK;
  if (!in_visit)
    rc = launch_ranges(s, num_dims, num_samples, samples, inv_radii, search, w.ranges);
  if (rc != MCCNN_OK) return rc;
  rc = launch_count(s, num_dims, num_samples, samples, points, w, inv_radii, max_neighs,
                    in_visit ? &search : nullptr, ranges_out, truncated);
  if (rc != MCCNN_OK) return rc;
  return inclusive_scan_i32(s, num_samples, ranges_out, w.scan_scratch, total, truncated);
}

// The count half of a search by a caller that has the grid in hand (no argument checks beyond
// sizes and null pointers), with or without the grid's column table, and with the outcome in
// pinned host memory.
extern "C" int mccnn_search_count(mccnn_stream_t stream, int64_t num_samples, int num_dims,
                                  const float *samples, const int32_t *sample_batch_ids,
                                  int64_t num_pts, const float *points, const int64_t *point_keys,
                                  const int32_t *grid_ds, const int32_t *num_cells,
                                  const float *scaled_aabb_min, const float *inv_cell_sizes,
                                  const float *inv_radii, int max_neighs, void *workspace,
                                  size_t workspace_bytes, int32_t *ranges_out,
                                  int64_t *result_pinned) {
  MCCNN_REQUIRE(valid_dims(num_dims), "search_count expects a valid number of dimensions");
  MCCNN_REQUIRE(num_samples >= 0 && num_pts >= 0 && num_samples < ((int64_t)1 << 31) &&
                    num_pts < ((int64_t)1 << 31),
                "search_count expects sizes in [0, 2^31)");
  MCCNN_REQUIRE(result_pinned, "search_count received a null output");
  result_pinned[0] = result_pinned[1] = 0;
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(samples && sample_batch_ids && num_cells && scaled_aabb_min && inv_cell_sizes &&
                    inv_radii && ranges_out && workspace && (num_pts == 0 || (points && point_keys)),
                "search_count received a null tensor");
  const NbrWorkspace w = carve_nbr_workspace(workspace, num_dims, num_samples);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "search_count workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  hipStream_t s = as_stream(stream);
  result_pinned[0] = -1;
  int rc = search_counts(s, num_samples, num_dims, samples, sample_batch_ids, num_pts, points,
                         point_keys, grid_ds, num_cells, scaled_aabb_min, inv_cell_sizes, inv_radii,
                         max_neighs, w, ranges_out, result_pinned,
                         max_neighs > 0 ? result_pinned + 1 : nullptr);
  if (rc != MCCNN_OK) return rc;
  rc = wait_for_host_values(s, result_pinned, 1);
  if (rc != MCCNN_OK) return rc;
  // (the total's word holds the flag: the flag's own is not known to have arrived)
  const int64_t total = result_pinned[0];
  result_pinned[0] = total & ~kScanFlag;
  result_pinned[1] = total & kScanFlag ? 1 : 0;
  MCCNN_REQUIRE(result_pinned[0] < (((int64_t)1 << 31) - 1),
                "FindNeighbors found at least %lld pairs; the int32 offsets of the op contract "
                "hold fewer than 2^31 - 1",
                (long long)result_pinned[0]);
  return MCCNN_OK;
}

extern "C" int mccnn_search_known(mccnn_stream_t stream, int64_t num_samples, int num_dims,
                                  const float *samples, const int32_t *sample_batch_ids,
                                  int64_t num_pts, const float *points, const int64_t *point_keys,
                                  const int32_t *grid_ds, const int32_t *num_cells,
                                  const float *scaled_aabb_min, const float *inv_cell_sizes,
                                  const float *inv_radii, void *workspace, size_t workspace_bytes,
                                  int64_t num_neighbors, int32_t *ranges_out,
                                  int32_t *neighbors_out) {
  MCCNN_REQUIRE(valid_dims(num_dims), "search_known expects a valid number of dimensions");
  MCCNN_REQUIRE(num_samples >= 0 && num_pts >= 0 && num_samples < ((int64_t)1 << 31) &&
                    num_pts < ((int64_t)1 << 31) && num_neighbors >= 0 &&
                    num_neighbors < ((int64_t)1 << 31),
                "search_known expects sizes in [0, 2^31)");
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(samples && sample_batch_ids && num_cells && scaled_aabb_min && inv_cell_sizes &&
                    inv_radii && ranges_out && workspace && (num_pts == 0 || (points && point_keys)) &&
                    (num_neighbors == 0 || neighbors_out),
                "search_known received a null tensor");
  const NbrWorkspace w = carve_nbr_workspace(workspace, num_dims, num_samples);
  MCCNN_REQUIRE(workspace_bytes >= w.bytes, "search_known workspace too small (%zu < %zu)",
                workspace_bytes, w.bytes);
  hipStream_t s = as_stream(stream);
  int rc = search_counts(s, num_samples, num_dims, samples, sample_batch_ids, num_pts, points,
                         point_keys, grid_ds, num_cells, scaled_aabb_min, inv_cell_sizes, inv_radii,
                         0, w, ranges_out, w.total, nullptr);
  if (rc != MCCNN_OK || num_neighbors == 0) return rc;
  return launch_fill(s, num_dims, num_samples, samples, points, w, inv_radii, 0, ranges_out,
                     neighbors_out, num_neighbors);
}

struct DensityWorkspace {
  int2 *slices;
  float *sums;          // [3, n]
  int *counts;          // pairs per wavefront of the visit
  int64_t parts;
  size_t bytes;
};

static DensityWorkspace carve_density_workspace(void *ws, int d, int64_t n) {
  char *p = (char *)ws;
  DensityWorkspace w;
  size_t off = 0;
  w.slices = (int2 *)(p + off);
  off += n <= kSearchInVisit ? 256 : align256(sizeof(int2) * (size_t)n * offsets_for(d));
  w.sums = (float *)(p + off);
  off += align256(3 * sizeof(float) * (size_t)n);
  w.parts = (n + kWave / kGroup - 1) / (kWave / kGroup);
  w.counts = (int *)(p + off);
  off += align256(sizeof(int) * (size_t)w.parts);
  w.bytes = off;
  return w;
}

extern "C" size_t mccnn_grid_density_workspace_bytes(int num_dims, int64_t num_pts) {
  if (!valid_dims(num_dims) || num_pts < 0) return 0;
  return carve_density_workspace(nullptr, num_dims, num_pts).bytes;
}

// Kernel density of the grid's own points straight from the grid: what compute_pdf gives on the
// pair table of the points among themselves, bit for bit, without the table (its count, the host
// round trip for its size, the 8 bytes per pair written and read).
extern "C" int mccnn_grid_density(mccnn_stream_t stream, int64_t num_pts, int num_dims,
                                  const float *points, const int32_t *batch_ids,
                                  const int64_t *point_keys, const int32_t *grid_ds,
                                  const int32_t *num_cells, const float *scaled_aabb_min,
                                  const float *inv_cell_sizes, const float *inv_radii,
                                  const float *inv_bandwidth, int mode, void *workspace,
                                  size_t workspace_bytes, float *pdf_out) {
  MCCNN_REQUIRE(valid_dims(num_dims), "grid_density expects a valid number of dimensions");
  MCCNN_REQUIRE(mode == 0 || mode == 1, "grid_density expects mode 0 or 1");
  MCCNN_REQUIRE(num_pts >= 0 && num_pts < ((int64_t)1 << 31), "grid_density expects a size in [0, 2^31)");
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(points && batch_ids && point_keys && num_cells && scaled_aabb_min &&
                    inv_cell_sizes && inv_radii && inv_bandwidth && workspace && pdf_out,
                "grid_density received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_grid_density_workspace_bytes(num_dims, num_pts),
                "grid_density workspace too small");
  hipStream_t s = as_stream(stream);
  const DensityWorkspace w = carve_density_workspace(workspace, num_dims, num_pts);
  const VisitSearch search = {batch_ids, num_pts, (const int64_t *)point_keys,
                              (const int2 *)grid_ds, num_cells, scaled_aabb_min, inv_cell_sizes};
  const dim3 grid(blocks_for(num_pts, kCentresPerBlock)), block(kNbrThreads);
#define MCCNN_DENSITY_VISIT(kSearch_, search_)                                                  \
  MCCNN_DIM_SWITCH(num_dims,                                                                    \
                   hipLaunchKernelGGL((nbr_visit_kernel<D, Visit::kDensity, kSearch_>), grid,   \
                                      block, 0, s, num_pts, points, points, w.slices,            \
                                      (unsigned *)nullptr, inv_radii,                            \
                                      0, search_, w.counts, (const int *)nullptr,               \
                                      (int2 *)nullptr, (int64_t *)nullptr, (int64_t)0,          \
                                      inv_bandwidth, mode, w.sums))
  if (num_pts <= kSearchInVisit) {
    MCCNN_DENSITY_VISIT(true, search);
  } else {
    const int rc = launch_ranges(s, num_dims, num_pts, points, inv_radii, search, w.slices);
    if (rc != MCCNN_OK) return rc;
    MCCNN_DENSITY_VISIT(false, VisitSearch{});
  }
#undef MCCNN_DENSITY_VISIT
  MCCNN_LAUNCH_CHECK();
  const int64_t blocks = (num_pts + kSelectThreads - 1) / kSelectThreads;
  hipLaunchKernelGGL(grid_density_select_kernel,
                     dim3((unsigned)(blocks < kSelectBlocks ? blocks : kSelectBlocks)),
                     dim3(kSelectThreads), 0, s, num_pts, w.parts, w.counts, w.sums, pdf_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" size_t mccnn_reorder_neighbors_workspace_bytes(int64_t num_samples) {
  if (num_samples < 0) return 0;
  return align256(sizeof(int) * scan_scratch_ints(num_samples)) + align256(sizeof(int64_t));
}

extern "C" int mccnn_reorder_neighbors(mccnn_stream_t stream, int64_t num_samples,
                                       const int32_t *ranges, int64_t num_neighbors,
                                       const int32_t *neighbors, const int32_t *centre_order,
                                       void *workspace, size_t workspace_bytes,
                                       int32_t *ranges_out, int32_t *neighbors_out) {
  MCCNN_REQUIRE(num_samples >= 0 && num_neighbors >= 0 && num_neighbors < ((int64_t)1 << 31),
                "reorder_neighbors expects sizes in [0, 2^31)");
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && centre_order && ranges_out && workspace &&
                    (num_neighbors == 0 || (neighbors && neighbors_out)),
                "reorder_neighbors received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_reorder_neighbors_workspace_bytes(num_samples),
                "reorder_neighbors workspace too small");
  int rc = mccnn_reorder_ranges(stream, num_samples, ranges, centre_order, workspace,
                                workspace_bytes, ranges_out);
  if (rc != MCCNN_OK) return rc;
  return mccnn_reorder_pairs(stream, num_samples, ranges, num_neighbors, neighbors, centre_order,
                             ranges_out, nullptr, neighbors_out, nullptr, nullptr);
}

// The two halves by themselves: the end offsets of the regrouped table, and any of its columns
// -- the pairs, the pairs with original point ids, the per-pair densities -- without the
// regrouped table in memory first.
extern "C" int mccnn_reorder_ranges(mccnn_stream_t stream, int64_t num_samples,
                                    const int32_t *ranges, const int32_t *centre_order,
                                    void *workspace, size_t workspace_bytes,
                                    int32_t *ranges_out) {
  MCCNN_REQUIRE(num_samples >= 0, "reorder_ranges expects a non-negative size");
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && centre_order && ranges_out && workspace,
                "reorder_ranges received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_reorder_neighbors_workspace_bytes(num_samples),
                "reorder_ranges workspace too small");
  hipStream_t s = as_stream(stream);
  int *scratch = (int *)workspace;
  int64_t *total = (int64_t *)((char *)workspace +
                               align256(sizeof(int) * scan_scratch_ints(num_samples)));
  hipLaunchKernelGGL(segment_counts_kernel, dim3(blocks_for(num_samples, 256)), dim3(256), 0, s,
                     num_samples, ranges, centre_order, ranges_out);
  MCCNN_LAUNCH_CHECK();
  return inclusive_scan_i32(s, num_samples, ranges_out, scratch, total);
}

extern "C" int mccnn_reorder_pairs(mccnn_stream_t stream, int64_t num_samples,
                                   const int32_t *ranges, int64_t num_neighbors,
                                   const int32_t *neighbors, const int32_t *centre_order,
                                   const int32_t *ranges_out, const int32_t *point_map,
                                   int32_t *neighbors_out, const float *pdf,
                                   float *pdf_per_pair_out) {
  MCCNN_REQUIRE(num_samples >= 0 && num_neighbors >= 0 && num_neighbors < ((int64_t)1 << 31),
                "reorder_pairs expects sizes in [0, 2^31)");
  if (num_samples == 0 || num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && neighbors && centre_order && ranges_out &&
                    (neighbors_out || pdf_per_pair_out) && (!pdf_per_pair_out || pdf),
                "reorder_pairs received a null tensor");
  // few slots: a wavefront each for four of them, or the chip is not filled
  const int slots = num_samples >= 131072 ? kCopySlots : 4;
  hipLaunchKernelGGL(segment_copy_kernel, dim3(blocks_for(num_samples, slots * (256 / kWave))),
                     dim3(256), 0, as_stream(stream), num_samples, slots, ranges, centre_order,
                     (const int2 *)neighbors, ranges_out, point_map, (int2 *)neighbors_out, pdf,
                     pdf_per_pair_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}
