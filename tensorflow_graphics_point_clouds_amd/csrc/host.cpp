// Host path of the layers and of the point-cloud structures: the sequences of C-ABI calls
// that make up a grid, a neighbour search or a layer pass, issued from C++ on tensors.
//
// A pass over a few thousand points is bound by what happens between the kernels: with every
// C-ABI call made through ctypes (6 to 8 us each with its argument objects) and every
// intermediate tensor, pad and permutation made in Python, a forward call on 2 x 1024 points
// took 375 us for 109 us of kernels.  The functions here allocate with the caching allocator,
// run on the current stream of the current device, release the interpreter lock, and keep no
// state between calls but a pool of pinned 256-byte blocks (as many as threads were ever
// waiting for a device count at the same time).
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <mutex>
#include <utility>
#include <vector>

#include "../../include/mccnn_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------ errors, pointers ----

struct InvalidArgument : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check(int rc) {
  if (rc == MCCNN_OK) return;
  const std::string msg = mccnn_last_error();
  if (rc == MCCNN_INVALID_ARGUMENT) throw InvalidArgument(msg);
  throw std::runtime_error("HIP error in libmccnn_hip: " + msg);
}

void hip_check(hipError_t e) {
  if (e != hipSuccess) throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e));
}

void *raw(const Tensor &t, at::ScalarType type) {
  if (!t.defined()) return nullptr;
  TORCH_CHECK_TYPE(t.is_cuda(), "expected a GPU tensor, got one on ", t.device());
  TORCH_CHECK_TYPE(t.scalar_type() == type, "expected dtype ", type, ", got ", t.scalar_type());
  TORCH_CHECK_TYPE(t.is_contiguous(), "expected a contiguous tensor");
  return t.data_ptr();
}
float *f32(const Tensor &t) { return static_cast<float *>(raw(t, at::kFloat)); }
int32_t *i32(const Tensor &t) { return static_cast<int32_t *>(raw(t, at::kInt)); }
int64_t *i64(const Tensor &t) { return static_cast<int64_t *>(raw(t, at::kLong)); }
Tensor opt(const OptTensor &t) { return t.has_value() ? *t : Tensor(); }

hipStream_t current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

Tensor empty_f32(at::IntArrayRef sizes, const Tensor &like) {
  return at::empty(sizes, like.options().dtype(at::kFloat).requires_grad(false));
}
Tensor empty_i32(at::IntArrayRef sizes, const Tensor &like) {
  return at::empty(sizes, like.options().dtype(at::kInt).requires_grad(false));
}
Tensor empty_i64(at::IntArrayRef sizes, const Tensor &like) {
  return at::empty(sizes, like.options().dtype(at::kLong).requires_grad(false));
}
Tensor workspace(size_t bytes, const Tensor &like) {
  return at::empty({(int64_t)(bytes ? bytes : 1)},
                   like.options().dtype(at::kByte).requires_grad(false));
}

int64_t dim(const Tensor &t, int64_t axis) { return t.dim() > axis ? t.size(axis) : -1; }

int compute_units() {
  static thread_local int device = -1, cus = 0;
  int d = 0;
  hip_check(hipGetDevice(&d));
  if (d != device) {
    hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, d));
    device = d;
  }
  return cus;
}

// A block of pinned host memory for the counts a call waits for, taken from a pool.
class PinnedBlock {
 public:
  PinnedBlock() {
    {
      std::lock_guard<std::mutex> lock(mutex());
      if (!pool().empty()) {
        p_ = pool().back();
        pool().pop_back();
      }
    }
    // (coherent: the host reads what a kernel has stored while the kernel still runs)
    if (!p_) hip_check(hipHostMalloc(&p_, 256, hipHostMallocCoherent));
  }
  ~PinnedBlock() {
    std::lock_guard<std::mutex> lock(mutex());
    pool().push_back(p_);
  }
  PinnedBlock(const PinnedBlock &) = delete;
  int64_t *words() { return static_cast<int64_t *>(p_); }
  int32_t *ints() { return static_cast<int32_t *>(p_); }

 private:
  static std::mutex &mutex() { static std::mutex *m = new std::mutex; return *m; }
  static std::vector<void *> &pool() { static auto *v = new std::vector<void *>; return *v; }
  void *p_ = nullptr;
};

// ------------------------------------------------------------------------- timing ----
// The counterpart of the regions of _lib.py for the calls made here: a pair of events
// around every call while timing is on.

struct TimedCall {
  const char *name;
  hipEvent_t start, end;
};
std::mutex g_timing_mutex;
std::atomic<bool> g_timing{false};
std::vector<TimedCall> g_timed;

class Region {
 public:
  Region(const char *name, hipStream_t s) : on_(g_timing.load(std::memory_order_relaxed)), s_(s) {
    if (!on_) return;
    c_.name = name;
    hip_check(hipEventCreate(&c_.start));
    hip_check(hipEventCreate(&c_.end));
    hip_check(hipEventRecord(c_.start, s_));
  }
  ~Region() {
    if (!on_) return;
    (void)hipEventRecord(c_.end, s_);
    std::lock_guard<std::mutex> lock(g_timing_mutex);
    g_timed.push_back(c_);
  }

 private:
  bool on_;
  hipStream_t s_;
  TimedCall c_{};
};

void start_timing() {
  std::lock_guard<std::mutex> lock(g_timing_mutex);
  g_timed.clear();
  g_timing = true;
}

std::vector<std::pair<std::string, double>> collect_timing() {
  g_timing = false;
  hip_check(hipDeviceSynchronize());
  std::vector<std::pair<std::string, double>> out;
  std::lock_guard<std::mutex> lock(g_timing_mutex);
  for (auto &c : g_timed) {
    float ms = 0.0f;
    hip_check(hipEventElapsedTime(&ms, c.start, c.end));
    out.emplace_back(c.name, ms);
    (void)hipEventDestroy(c.start);
    (void)hipEventDestroy(c.end);
  }
  g_timed.clear();
  return out;
}

// --------------------------------------------------------------------------- grid ----

Tensor compute_keys(const Tensor &points, const Tensor &bids, const Tensor &smin,
                    const Tensor &num_cells, const Tensor &inv_cell) {
  Tensor keys = empty_i64({points.size(0)}, points);
  hipStream_t s = current_stream();
  Region r("compute_keys", s);
  check(mccnn_compute_keys(s, points.size(0), (int)dim(points, 1), f32(points), bids.size(0),
                           i32(bids), smin.size(0), (int)dim(smin, 1), f32(smin),
                           (int)num_cells.size(0), i32(num_cells), (int)inv_cell.size(0),
                           f32(inv_cell), i64(keys)));
  return keys;
}

struct GridTensors {
  Tensor aabb_min, aabb_max, num_cells, smin, inv_cell, keys, sorted_keys, sorted_indices,
      sorted_points, sorted_bids;
  std::vector<int64_t> cells_host;   // empty: the shape has not been waited for
  int64_t key_bits = 0;
};

// The grid of a point cloud (pylib/pc/Grid.py:32-84).
GridTensors build_grid(const Tensor &points, const Tensor &bids, int64_t batch,
                       const Tensor &cell_sizes) {
  const int64_t n = points.size(0), d = points.size(1);
  if (cell_sizes.numel() < d)
    throw InvalidArgument("BuildGrid expects a cell size for each of the points' dimensions");
  if (bids.size(0) != n)
    throw InvalidArgument("BuildGrid expects the same number of batch ids as number of points");
  GridTensors g;
  g.aabb_min = empty_f32({batch, d}, points);
  g.aabb_max = empty_f32({batch, d}, points);
  g.num_cells = empty_i32({d}, points);
  g.smin = empty_f32({batch, d}, points);
  g.inv_cell = empty_f32({d}, points);
  g.keys = empty_i64({n}, points);
  g.sorted_keys = empty_i64({n}, points);
  g.sorted_indices = empty_i32({n}, points);
  g.sorted_points = empty_f32({n, d}, points);
  g.sorted_bids = empty_i32({n}, points);
  Tensor ws = workspace(mccnn_build_grid_workspace_bytes(n), points);
  hipStream_t s = current_stream();
  Region r("build_grid", s);
  auto call = [&](int32_t *cells, int *bits) {
    check(mccnn_build_grid_pinned(s, n, (int)d, f32(points), i32(bids), (int)batch,
                                  f32(cell_sizes), f32(g.aabb_min), f32(g.aabb_max),
                                  i32(g.num_cells), f32(g.smin), f32(g.inv_cell), i64(g.keys),
                                  i64(g.sorted_keys), i32(g.sorted_indices), f32(g.sorted_points),
                                  i32(g.sorted_bids), ws.data_ptr(), ws.numel(), cells, bits));
  };
  if (mccnn_build_grid_is_single_launch(n, (int)d, (int)batch)) {
    call(nullptr, nullptr);
    return g;
  }
  PinnedBlock host;
  int bits = 1;
  call(host.ints(), &bits);
  for (int64_t i = 0; i < d; ++i) g.cells_host.push_back(host.ints()[i]);
  g.key_bits = bits;
  return g;
}

void check_search(const Tensor &samples, const Tensor &sbids, const Tensor &num_cells,
                  const Tensor &smin, const Tensor &inv_cell);

// Centres in the order of their cells in a grid -> (order, coordinates, cloud ids, cell keys or
// nothing unless `want_keys`).
std::tuple<Tensor, Tensor, Tensor, OptTensor> order_centres(
    const Tensor &samples, const Tensor &bids, int64_t batch, const Tensor &num_cells,
    const Tensor &smin, const Tensor &inv_cell, int64_t key_bits, bool want_keys) {
  check_search(samples, bids, num_cells, smin, inv_cell);
  const int64_t n = samples.size(0), d = samples.size(1);
  Tensor order = empty_i32({n}, samples), pts = empty_f32({n, d}, samples),
         out_bids = empty_i32({n}, samples);
  OptTensor keys;
  if (want_keys) keys = empty_i64({n}, samples);
  Tensor ws = workspace(mccnn_order_centres_workspace_bytes(n), samples);
  hipStream_t s = current_stream();
  Region r("order_centres", s);
  check(mccnn_order_centres_keys(s, n, (int)d, f32(samples), i32(bids), (int)batch,
                                 i32(num_cells), f32(smin), f32(inv_cell), (int)key_bits,
                                 ws.data_ptr(), ws.numel(), i32(order), f32(pts), i32(out_bids),
                                 keys ? i64(*keys) : nullptr));
  return {order, pts, out_bids, keys};
}

Tensor invert_order(const Tensor &order) {
  Tensor out = empty_i32({order.size(0)}, order);
  hipStream_t s = current_stream();
  Region r("invert_order", s);
  check(mccnn_invert_order(s, order.size(0), i32(order), i32(out)));
  return out;
}

Tensor build_grid_ds(const Tensor &sorted_keys, const Tensor &num_cells,
                     const std::vector<int32_t> &host, int64_t batch) {
  if (batch <= 0) throw InvalidArgument("BuildGridDs requires a positive batch size");
  if (host.size() < 2) throw InvalidArgument("BuildGridDs expects a valid number of dimensions");
  hipStream_t s = current_stream();
  Tensor ds = empty_i32({batch, std::max(host[0], 0), std::max(host[1], 0), 2}, sorted_keys);
  Region r("build_grid_ds", s);
  check(mccnn_build_grid_ds(s, sorted_keys.size(0), i64(sorted_keys), (int)num_cells.size(0),
                            i32(num_cells), (int)host.size(), host.data(), (int)batch, i32(ds)));
  return ds;
}

// ---------------------------------------------------------------------- neighbours ----

// -> (ranges, neighbors, whether the table is an untruncated self-neighbourhood)
std::tuple<Tensor, Tensor, bool> find_neighbors(const Tensor &samples, const Tensor &sbids,
                                                const Tensor &points, const Tensor &keys,
                                                const Tensor &ds, const Tensor &num_cells,
                                                const Tensor &smin, const Tensor &inv_cell,
                                                const Tensor &inv_radii, int64_t max_neighs) {
  const int64_t ns = samples.size(0);
  const int nd = (int)dim(samples, 1);
  Tensor ws = workspace(mccnn_find_neighbors_workspace_bytes(nd, ns), samples);
  Tensor ranges = empty_i32({ns}, samples);
  hipStream_t s = current_stream();
  PinnedBlock host;
  int64_t *total = host.words();
  total[0] = total[1] = total[2] = 0;
  {
    Region r("find_neighbors_count", s);
    check(mccnn_find_neighbors_count_facts(
        s, ns, nd, f32(samples), sbids.size(0), i32(sbids), points.size(0), (int)dim(points, 1),
        f32(points), keys.size(0), i64(keys), (int)ds.dim(), (int)dim(ds, 0), (int)dim(ds, 1),
        (int)dim(ds, 2), (int)dim(ds, 3), i32(ds), (int)num_cells.size(0), i32(num_cells),
        (int)dim(smin, 1), f32(smin), (int)inv_cell.size(0), f32(inv_cell),
        (int)inv_radii.size(0), f32(inv_radii), (int)max_neighs, ws.data_ptr(), ws.numel(),
        i32(ranges), total, total + 1));
  }
  const int64_t m = total[0];
  const bool symmetric = total[1] == 0 && total[2] == 1;
  Tensor neighbors = empty_i32({m, 2}, samples);
  Region r("find_neighbors_fill", s);
  check(mccnn_find_neighbors_fill(s, ns, nd, f32(samples), i32(sbids), points.size(0), f32(points),
                                  i64(keys), i32(ds), i32(num_cells), f32(smin), f32(inv_cell),
                                  f32(inv_radii), (int)max_neighs, ws.data_ptr(), ws.numel(),
                                  i32(ranges), m, i32(neighbors)));
  return {ranges, neighbors, symmetric};
}

// What find_neighbors asks of its arguments, for the entries below that skip its checks: a sample
// cloud, radii or a grid of another number of dimensions would be read out of range.
void check_search(const Tensor &samples, const Tensor &sbids, const Tensor &num_cells,
                  const Tensor &smin, const Tensor &inv_cell) {
  const int64_t d = dim(samples, 1);
  auto require = [](bool ok, const char *what) {
    if (!ok) throw InvalidArgument(std::string("FindNeighbors expects ") + what);
  };
  require(num_cells.numel() == d,
          "a number of dimensions in num_cells equal to the number of dimensions in the samples");
  require(dim(smin, 1) == d,
          "a number of dimensions in scaled_aabb_min equal to the number of dimensions in the "
          "samples");
  require(inv_cell.numel() == d,
          "a number of dimensions in inv_cell_sizes equal to the number of dimensions in the "
          "samples");
  require(sbids.size(0) == samples.size(0), "the same number of batch ids as samples");
}

void check_search(const Tensor &samples, const Tensor &sbids, const Tensor &points,
                  const Tensor &keys, const Tensor &num_cells, const Tensor &smin,
                  const Tensor &inv_cell, const Tensor &inv_radii) {
  check_search(samples, sbids, num_cells, smin, inv_cell);
  if (dim(points, 1) != dim(samples, 1))
    throw InvalidArgument("FindNeighbors expects a number of dimensions in points equal to the "
                          "number of dimensions in the samples");
  if (inv_radii.numel() != dim(samples, 1))
    throw InvalidArgument("FindNeighbors expects a number of dimensions in inv_radii equal to the "
                          "number of dimensions in the input points");
  if (keys.size(0) != points.size(0))
    throw InvalidArgument("FindNeighbors expects the same number of keys as points");
}

// The same for the structures of pc.py, which hold the grid: its column table is optional (for
// a small cloud it would need the grid's shape on the host first).
// -> (ranges, neighbors, whether a neighbourhood was cut at max_neighs)
std::tuple<Tensor, Tensor, bool> search(const Tensor &samples, const Tensor &sbids,
                                        const Tensor &points, const Tensor &keys,
                                        const OptTensor &ds, const Tensor &num_cells,
                                        const Tensor &smin, const Tensor &inv_cell,
                                        const Tensor &inv_radii, int64_t max_neighs) {
  check_search(samples, sbids, points, keys, num_cells, smin, inv_cell, inv_radii);
  const int64_t ns = samples.size(0);
  const int nd = (int)dim(samples, 1);
  Tensor ws = workspace(mccnn_find_neighbors_workspace_bytes(nd, ns), samples);
  Tensor ranges = empty_i32({ns}, samples);
  hipStream_t s = current_stream();
  PinnedBlock host;
  {
    Region r("find_neighbors_count", s);
    check(mccnn_search_count(s, ns, nd, f32(samples), i32(sbids), points.size(0), f32(points),
                             i64(keys), i32(opt(ds)), i32(num_cells), f32(smin), f32(inv_cell),
                             f32(inv_radii), (int)max_neighs, ws.data_ptr(), ws.numel(),
                             i32(ranges), host.words()));
  }
  const int64_t m = host.words()[0];
  const bool cut = host.words()[1] != 0;
  Tensor neighbors = empty_i32({m, 2}, samples);
  Region r("find_neighbors_fill", s);
  check(mccnn_find_neighbors_fill(s, ns, nd, f32(samples), i32(sbids), points.size(0), f32(points),
                                  i64(keys), nullptr, i32(num_cells), f32(smin), f32(inv_cell),
                                  f32(inv_radii), (int)max_neighs, ws.data_ptr(), ws.numel(),
                                  i32(ranges), m, i32(neighbors)));
  return {ranges, neighbors, cut};
}

// The same where the number of pairs is known: no host round trip -> (ranges, neighbors).
std::tuple<Tensor, Tensor> search_known(const Tensor &samples, const Tensor &sbids,
                                        const Tensor &points, const Tensor &keys,
                                        const Tensor &num_cells, const Tensor &smin,
                                        const Tensor &inv_cell, const Tensor &inv_radii,
                                        int64_t pairs) {
  check_search(samples, sbids, points, keys, num_cells, smin, inv_cell, inv_radii);
  const int64_t ns = samples.size(0);
  const int nd = (int)dim(samples, 1);
  Tensor ws = workspace(mccnn_find_neighbors_workspace_bytes(nd, ns), samples);
  Tensor ranges = empty_i32({ns}, samples), neighbors = empty_i32({pairs, 2}, samples);
  hipStream_t s = current_stream();
  Region r("transpose_neighbors", s);
  check(mccnn_search_known(s, ns, nd, f32(samples), i32(sbids), points.size(0), f32(points),
                           i64(keys), nullptr, i32(num_cells), f32(smin), f32(inv_cell),
                           f32(inv_radii), ws.data_ptr(), ws.numel(), pairs, i32(ranges),
                           i32(neighbors)));
  return {ranges, neighbors};
}

Tensor grid_density(const Tensor &points, const Tensor &bids, const Tensor &keys,
                    const OptTensor &ds, const Tensor &num_cells, const Tensor &smin,
                    const Tensor &inv_cell, const Tensor &inv_radii, const Tensor &inv_bandwidth,
                    int64_t mode) {
  check_search(points, bids, points, keys, num_cells, smin, inv_cell, inv_radii);
  const int64_t n = points.size(0);
  const int nd = (int)dim(points, 1);
  if (inv_bandwidth.numel() != nd)
    throw InvalidArgument("ComputePDF expects a number of dimensions in inv_bandwidth equal to the "
                          "number of dimensions in the input points");
  Tensor ws = workspace(mccnn_grid_density_workspace_bytes(nd, n), points);
  Tensor pdf = empty_f32({n}, points);
  hipStream_t s = current_stream();
  Region r("compute_pdf", s);
  check(mccnn_grid_density(s, n, nd, f32(points), i32(bids), i64(keys), i32(opt(ds)),
                           i32(num_cells), f32(smin), f32(inv_cell), f32(inv_radii),
                           f32(inv_bandwidth), (int)mode, ws.data_ptr(), ws.numel(), f32(pdf)));
  return pdf;
}

// Columns of the pair table regrouped for centres in the order `order`: the end offsets, the
// pairs (point indices through `map` if given), the density of every pair's point.
Tensor reorder_ranges(const Tensor &ranges, const Tensor &order) {
  const int64_t n = ranges.size(0);
  Tensor ws = workspace(mccnn_reorder_neighbors_workspace_bytes(n), ranges);
  Tensor out = empty_i32({n}, ranges);
  hipStream_t s = current_stream();
  Region r("reorder_neighbors", s);
  check(mccnn_reorder_ranges(s, n, i32(ranges), i32(order), ws.data_ptr(), ws.numel(), i32(out)));
  return out;
}

Tensor reorder_pairs(const Tensor &ranges, const Tensor &neighbors, const Tensor &order,
                     const Tensor &ranges_out, const OptTensor &map) {
  Tensor out = empty_i32(neighbors.sizes(), neighbors);
  hipStream_t s = current_stream();
  Region r("reorder_neighbors", s);
  check(mccnn_reorder_pairs(s, ranges.size(0), i32(ranges), neighbors.size(0), i32(neighbors),
                            i32(order), i32(ranges_out), i32(opt(map)), i32(out), nullptr,
                            nullptr));
  return out;
}

Tensor reorder_pdf(const Tensor &ranges, const Tensor &neighbors, const Tensor &order,
                   const Tensor &ranges_out, const Tensor &pdf) {
  Tensor out = empty_f32({neighbors.size(0)}, neighbors);
  hipStream_t s = current_stream();
  Region r("gather_pdf", s);
  check(mccnn_reorder_pairs(s, ranges.size(0), i32(ranges), neighbors.size(0), i32(neighbors),
                            i32(order), i32(ranges_out), nullptr, nullptr, f32(pdf), f32(out)));
  return out;
}

Tensor original_neighbor_ids(const Tensor &neighbors, const Tensor &sorted_indices) {
  Tensor out = empty_i32(neighbors.sizes(), neighbors);
  hipStream_t s = current_stream();
  Region r("original_neighbor_ids", s);
  check(mccnn_original_neighbor_ids(s, neighbors.size(0), i32(neighbors), i32(sorted_indices),
                                    i32(out)));
  return out;
}

// -> (point_ranges, pair_order)
std::pair<Tensor, Tensor> transpose_neighbors(const Tensor &neighbors, int64_t num_pts) {
  const int64_t m = neighbors.size(0);
  Tensor ws = workspace(mccnn_transpose_neighbors_workspace_bytes(m, num_pts), neighbors);
  Tensor ranges = empty_i32({num_pts}, neighbors), order = empty_i32({m}, neighbors);
  hipStream_t s = current_stream();
  Region r("transpose_neighbors", s);
  check(mccnn_transpose_neighbors(s, m, i32(neighbors), num_pts, ws.data_ptr(), ws.numel(),
                                  i32(ranges), i32(order)));
  return {ranges, order};
}

Tensor swapped_pairs(const Tensor &neighbors, const Tensor &order) {
  Tensor out = empty_i32(neighbors.sizes(), neighbors);
  hipStream_t s = current_stream();
  Region r("swapped_pairs", s);
  check(mccnn_swapped_pairs(s, neighbors.size(0), i32(neighbors), i32(order), i32(out)));
  return out;
}

// Column 0 of a pair table and column 1 of its transpose -> (densities, densities).
std::pair<Tensor, Tensor> gather_pdf_both(const Tensor &neighbors, const Tensor &transposed,
                                          const Tensor &pdf) {
  const int64_t m = neighbors.size(0);
  if (transposed.size(0) != m) throw InvalidArgument("gather_pdf expects tables of equal length");
  Tensor out = empty_f32({m}, pdf), out_t = empty_f32({m}, pdf);
  hipStream_t s = current_stream();
  Region r("gather_pdf", s);
  check(mccnn_gather_pdf_both(s, m, i32(neighbors), i32(transposed), f32(pdf), f32(out), f32(out_t)));
  return {out, out_t};
}

Tensor gather_pdf(const Tensor &neighbors, int64_t column, const Tensor &pdf) {
  Tensor out = empty_f32({neighbors.size(0)}, neighbors);
  hipStream_t s = current_stream();
  Region r("gather_pdf", s);
  check(mccnn_gather_pdf_column(s, neighbors.size(0), i32(neighbors), (int)column, f32(pdf),
                                f32(out)));
  return out;
}

Tensor gather_i32(const Tensor &src, const Tensor &indices) {
  Tensor out = empty_i32({indices.size(0)}, indices);
  hipStream_t s = current_stream();
  Region r("gather_i32", s);
  check(mccnn_gather_i32(s, indices.size(0), i32(src), i32(indices), i32(out)));
  return out;
}

Tensor compute_pdf(const Tensor &points, const Tensor &neighbors, const Tensor &ranges,
                   const Tensor &inv_bandwidth, const Tensor &inv_radii, int64_t mode) {
  Tensor pdf = empty_f32({ranges.size(0)}, points);
  hipStream_t s = current_stream();
  Region r("compute_pdf", s);
  check(mccnn_compute_pdf(s, points.size(0), (int)dim(points, 1), f32(points), neighbors.size(0),
                          (int)neighbors.dim(), (int)dim(neighbors, 1), i32(neighbors),
                          ranges.size(0), i32(ranges), (int)inv_bandwidth.size(0),
                          f32(inv_bandwidth), (int)inv_radii.size(0), f32(inv_radii), (int)mode,
                          f32(pdf)));
  return pdf;
}

// The second half: -> (points, batch ids, indices).
std::tuple<Tensor, Tensor, Tensor> selected_points(int64_t mode, const Tensor &points,
                                                   const Tensor &bids, const Tensor &keys,
                                                   const Tensor &num_cells, const Tensor &ws,
                                                   int64_t k) {
  const int nd = (int)dim(points, 1);
  Tensor pts = empty_f32({k, nd}, points), out_bids = empty_i32({k}, points),
         idx = empty_i32({k}, points);
  hipStream_t s = current_stream();
  Region r("sampling_fill", s);
  check(mccnn_sampling_fill(s, (int)mode, points.size(0), nd, f32(points), i32(bids), i64(keys),
                            i32(num_cells), ws.data_ptr(), ws.numel(), k, f32(pts), i32(out_bids),
                            i32(idx)));
  return {pts, out_bids, idx};
}

// -> (points, batch ids, indices)
std::tuple<Tensor, Tensor, Tensor> sampling(const Tensor &points, const Tensor &bids,
                                            const Tensor &keys, const Tensor &num_cells,
                                            const Tensor &neighbors, const Tensor &ranges,
                                            int64_t mode) {
  const int64_t n = points.size(0);
  const int nd = (int)dim(points, 1);
  Tensor ws = workspace(mccnn_sampling_workspace_bytes(n), points);
  hipStream_t s = current_stream();
  PinnedBlock host;
  host.words()[0] = 0;
  {
    Region r("sampling_count", s);
    check(mccnn_sampling_count_pinned(s, (int)mode, n, nd, f32(points), bids.size(0), i32(bids),
                               keys.size(0), i64(keys), (int)num_cells.size(0), i32(num_cells),
                               neighbors.size(0), (int)neighbors.dim(), (int)dim(neighbors, 1),
                               i32(neighbors), ranges.size(0), i32(ranges), ws.data_ptr(),
                               ws.numel(), host.words()));
  }
  return selected_points(mode, points, bids, keys, num_cells, ws, host.words()[0]);
}

// Poisson-disk sampling of a grid's sorted points without their pair table.
std::tuple<Tensor, Tensor, Tensor> sampling_grid(const Tensor &points, const Tensor &bids,
                                                 const Tensor &keys, const OptTensor &ds,
                                                 const Tensor &num_cells,
                                                 const Tensor &inv_radii) {
  const int64_t n = points.size(0);
  const int nd = (int)dim(points, 1);
  if (bids.size(0) != n || keys.size(0) != n || num_cells.numel() != nd || inv_radii.numel() != nd)
    throw InvalidArgument("Sampling expects batch ids and keys per point, numbers of cells and radii "
                          "per dimension");
  Tensor ws = workspace(mccnn_sampling_grid_workspace_bytes(nd, n), points);
  hipStream_t s = current_stream();
  PinnedBlock host;
  host.words()[0] = 0;
  {
    Region r("sampling_count", s);
    check(mccnn_sampling_grid_count_pinned(s, n, nd, f32(points), i32(bids), i64(keys),
                                           i32(opt(ds)), i32(num_cells), f32(inv_radii),
                                           ws.data_ptr(), ws.numel(), host.words()));
  }
  return selected_points(0, points, bids, keys, num_cells, ws, host.words()[0]);
}

// ------------------------------------------------------------------ dense products ----

Tensor gather_rows(const Tensor &src, const Tensor &rows, int64_t first_col, int64_t cols,
                   int64_t out_cols) {
  const int64_t n = rows.defined() ? rows.size(0) : src.size(0);
  Tensor out = empty_f32({n, out_cols}, src);
  hipStream_t s = current_stream();
  Region r("gather_rows", s);
  check(mccnn_gather_rows_padded(s, n, i32(rows), f32(src), src.size(1), (int)first_col, (int)cols,
                                 (int)out_cols, f32(out)));
  return out;
}

int64_t product_tiles(int64_t n, int64_t f) {   // 128 x 128 tiles, 256 x 64 for odd multiples of 64
  return f % 128 == 0 ? (n + 127) / 128 * (f / 128) : (n + 255) / 256 * (f / 64);
}

enum class Product { kTiled, kRegisters, kLibrary };

// Which kernel multiplies [n, r] by [r, f].  Weights beyond the registers of a block of
// wavefronts (r f > 65536) take the tiled product, whose weights are handed over transposed,
// once its tiles give every compute unit one; smaller inputs take the register-resident
// product in blocks of w.  On the bf16 pipe the tiled kernel is also the faster one for
// smaller weights once there are one and a half tiles per compute unit ([763 063, 1024] x
// [1024, 64]: 0.82 against 0.93 ms inside the layer step; [30 000, 1024] x [1024, 64]: 0.087
// against 0.049 ms).
Product product_kind(int64_t n, int64_t r, int64_t f) {
  const int64_t tiles = f % 64 == 0 ? product_tiles(n, f) : 0, units = compute_units();
  if (mccnn_final_product_wt_supported((int)r, (int)f) &&
      ((r * f > 65536 && tiles >= units) ||
       (mccnn_split_products_enabled() && 2 * tiles >= 3 * units)))
    return Product::kTiled;
  return mccnn_final_product_supported((int)r, (int)f) ? Product::kRegisters : Product::kLibrary;
}

// x w for x [n, r]; `w` [r, f] and `wt` [f, r]: the one `kind` needs.  Rows of the result go
// to out_rows if given; columns from `cols` on (if given) are padding and may be left unwritten.
Tensor run_product(Product kind, const Tensor &x, const Tensor &w, const Tensor &wt,
                   const Tensor &out_rows, int64_t cols = 0) {
  const int64_t n = x.size(0), r = x.size(1);
  hipStream_t s = current_stream();
  if (kind == Product::kLibrary) {
    Region t("gemm_final", s);
    Tensor out = at::matmul(x, w);
    return out_rows.defined() ? at::empty_like(out).index_copy_(0, out_rows.to(at::kLong), out)
                              : out;
  }
  const int64_t f = kind == Product::kTiled ? wt.size(0) : w.size(1);
  Tensor out = empty_f32({n, f}, x);
  Region t("final_product", s);
  if (kind == Product::kTiled)
    check(mccnn_final_product_wt(s, n, (int)r, f32(x), (int)f, f32(wt), i32(out_rows), f32(out)));
  else
    check(mccnn_final_product_padded(s, n, (int)r, f32(x), (int)f, (int)(cols > 0 ? cols : f),
                                     f32(w), i32(out_rows), f32(out)));
  return out;
}

Tensor final_product(const Tensor &x, const Tensor &w) {
  const Product kind = product_kind(x.size(0), w.size(0), w.size(1));
  if (kind == Product::kTiled) return run_product(kind, x, Tensor(), w.t().contiguous(), Tensor());
  return run_product(kind, x, w.contiguous(), Tensor(), Tensor());
}

Tensor weight_grad_product(const Tensor &x, const Tensor &y) {
  const int64_t c = x.size(1), r = y.size(1);
  hipStream_t s = current_stream();
  if (!mccnn_weight_grad_product_supported((int)c, (int)r)) {
    Region t("gemm_dfinal", s);
    return at::matmul(x.t(), y);
  }
  Tensor ws = workspace(mccnn_weight_grad_product_workspace_bytes((int)c, (int)r), x);
  Tensor out = empty_f32({c, r}, x);
  Region t("weight_grad_product", s);
  check(mccnn_weight_grad_product(s, x.size(0), (int)c, f32(x), (int)r, f32(y), ws.data_ptr(),
                                  ws.numel(), f32(out)));
  return out;
}

Tensor projection_grad_product(const Tensor &x, const Tensor &w) {
  const int64_t f = x.size(1), r = w.size(0);
  hipStream_t s = current_stream();
  if (!mccnn_projection_grad_product_supported((int)f, (int)r)) {
    Region t("gemm_dproj", s);
    return at::matmul(x, w.t());
  }
  Tensor out = empty_f32({x.size(0), r}, x);
  Region t("projection_grad_product", s);
  check(mccnn_projection_grad_product(s, x.size(0), (int)f, f32(x), (int)r, f32(w), f32(out)));
  return out;
}

// dout W^T for dout [n, f] and W [r, f] of a layer.  Column counts without a kernel take that of
// the next multiple of 64 with zero columns in both operands where there is one: nearer to the
// exact sums than the library's product (48 columns: 9.5e-8 against 1.25e-7 of the result; 96:
// 1.4e-7 / 1.8e-7) and faster with the padding (400 000 x 48 x 1024: 309 against 590 us, x 96:
// 569 / 823 us, plus 30 to 60 us for the padded rows).
Tensor layer_projection_grad(const Tensor &dout, const Tensor &w) {
  const int64_t f = dout.size(1), wide = (f + 63) / 64 * 64;
  if (mccnn_projection_grad_product_supported((int)f, (int)w.size(0)) ||
      !mccnn_projection_grad_product_supported((int)wide, (int)w.size(0)))
    return projection_grad_product(dout, w);
  return projection_grad_product(gather_rows(dout, Tensor(), 0, f, wide),
                                 gather_rows(w, Tensor(), 0, f, wide));
}

// --------------------------------------------------------------------- convolutions ----

// The neighbourhood of a layer pass in grid order (`_SortedView` of pc.py), and how its pairs
// are weighted.  The transposed half is only there when a gradient will be asked for.
struct Geometry : torch::CustomClassHolder {
  Tensor points_in, points_out, table, ranges, table_t, ranges_t, point_rows, centre_rows;
  Tensor pdf, pdf_t, inv_radii, neg_inv_radii;
};

// Sizes of a layer: of its weights, and as the kernels run it.  A layer of several kernel
// MLPs runs as mlps / per independent convolutions of per * hidden_pad basis columns: kernel
// MLPs share no final weights (MCConv.py:180-194), so the dense products then cost that many
// times less than on the block-diagonal matrix.
struct Plan {
  int64_t dims, c, h, g, mlps;
  int64_t c_pad, h_pad, g_pad, per;
  int64_t act;
  int64_t k() const { return per * h_pad; }
  int64_t f() const { return per * g_pad; }
  // output columns without the padding that only follows them, in sixteens
  int64_t cols() const { return per == 1 ? (g + 15) / 16 * 16 : f(); }
  bool padded() const { return c_pad != c || h_pad != h || g_pad != g || per != 1; }
};

// What the kernels read of one sub-layer's weights.  Between the passes what the backward reads of
// it rides among the saved tensors, so that autograd frees it afterwards.
struct Packed {
  Tensor w, wt, w2, w2t, kw, kb;
  Product forward = Product::kRegisters;
  static constexpr size_t kTensors = 5;
  void save(variable_list &to) const { to.insert(to.end(), {w, w2, w2t, kw, kb}); }
  static Packed saved(const variable_list &from, size_t first) {
    return {from[first],     Tensor(),        from[first + 1],
            from[first + 2], from[first + 3], from[first + 4]};
  }
};

Packed pack(const Plan &p, int64_t first, const Tensor &final_weights,
            const Tensor &kw, const Tensor &kb, int64_t n_out, int64_t n_in, bool need_w,
            bool need_transposed) {
  Packed out;
  const int64_t k = p.k(), f = p.f(), r = p.c_pad * k;
  out.forward = product_kind(n_out, r, f);
  const Product transposed = product_kind(n_in, f * k, p.c_pad);
  const bool plain = !p.padded();
  if (need_w || out.forward != Product::kTiled)
    out.w = plain && p.mlps == 1 ? final_weights.view({r, f}) : empty_f32({r, f}, final_weights);
  if (out.forward == Product::kTiled) out.wt = empty_f32({f, r}, final_weights);
  if (need_transposed) {
    if (transposed == Product::kTiled) out.w2t = empty_f32({p.c_pad, f * k}, final_weights);
    else out.w2 = empty_f32({f * k, p.c_pad}, final_weights);
  }
  const bool kernel = kw.defined();
  if (kernel) {
    if (plain && p.mlps == 1) {
      out.kw = kw;
      out.kb = kb;
    } else {
      out.kw = empty_f32({p.per, p.dims, p.h_pad}, kw);
      out.kb = empty_f32({k}, kb);
    }
  }
  const bool pack_w = out.w.defined() && !(plain && p.mlps == 1);
  const bool pack_kernel = kernel && !(plain && p.mlps == 1);
  if (pack_w || out.wt.defined() || out.w2.defined() || out.w2t.defined() || pack_kernel) {
    hipStream_t s = current_stream();
    Region t("pack_layer_weights", s);
    check(mccnn_pack_layer_weights(
        s, (int)p.dims, (int)p.c, (int)p.h, (int)p.g, (int)first, (int)p.per, (int)p.c_pad,
        (int)p.h_pad, (int)p.g_pad, f32(final_weights), f32(kw), f32(kb),
        pack_w ? f32(out.w) : nullptr, f32(out.wt), f32(out.w2), f32(out.w2t),
        pack_kernel ? f32(out.kw) : nullptr, pack_kernel ? f32(out.kb) : nullptr));
  }
  return out;
}

// Layers of few input and more output channels take their gradients the other way round
// (feature_grads.hip): from G = dout W^T, which the kernel MLPs' gradients need anyway, instead of
// the transposed projection Q [N, F, K] of dout,
//     dfeat[j, c]  = sum_{i in T(j)} sum_k basis[ij, k] G[i, c, k],
//     dW[c, k, f]  = sum_i proj[i, c, k] dout[i, f],
// with the projection computed again.  What is written and read per centre then grows with C, not with
// F; what is gathered per pair grows with 16 C for the 4, 8 or 16 channels that are gathered, not with F.
// `wide`: the columns that dout and W are padded to for the products, 0 where this does not apply.
// From five columns per gathered channel on it is the faster one whatever the lists (two passes of
// 500 k points, other way / this way: KPConv 16 -> 96 1.47 with lists of 10, 0.95 with 55, 4 -> 32 1.14
// and 0.93, 7 -> 48 1.35 and 1.16; MCConv 16 -> 80 1.44 and 1.02, 4 -> 32 1.22 and 1.01); from three
// on with short lists only (MCConv 16 -> 48 and 64 1.15 and 1.22 with lists of 10, 0.86 with 37,
// KPConv 1.06 and 1.10, 0.79 and 0.78; 8 -> 32 1.08 and 0.98 with 10, with 25 0.98 and 0.89); with two never
// (16 -> 32 of 10: 0.89 and 0.78, of 37: 0.62 and 0.53).
int64_t narrow_columns(const Plan &p, int64_t n_out, int64_t pairs) {
  const int64_t f = p.f(), r = p.c_pad * p.k(), live = p.c <= 4 ? 4 : p.c <= 8 ? 8 : 16;
  const bool pays = f >= 5 * live || (f >= 3 * live && pairs <= 16 * n_out);
  if (p.k() != 16 || p.c_pad != 16 || f < 2 * p.c_pad || !pays ||
      (p.per != 1 && p.g_pad != p.g) || n_out * r >= (int64_t)1 << 30)
    return 0;
  const int64_t wide = f == 32 ? 32 : (f + 63) / 64 * 64;
  if (wide != f && p.per != 1) return 0;
  return mccnn_weight_grad_product_supported((int)wide, (int)r) &&
                 mccnn_projection_grad_product_supported((int)wide, (int)r)
             ? wide : 0;
}

// The product of the feature gradient, q w2.
Tensor transposed_product(const Tensor &q, const Packed &w, const Tensor &out_rows) {
  if (w.w2t.defined()) return run_product(Product::kTiled, q, Tensor(), w.w2t, out_rows);
  const bool covered = mccnn_final_product_supported((int)q.size(1), (int)w.w2.size(1));
  return run_product(covered ? Product::kRegisters : Product::kLibrary, q, w.w2, Tensor(),
                     out_rows);
}

Tensor mc_project(const Plan &p, const Packed &w, const Tensor &feats, const Tensor &pin,
                  const Tensor &pout, const Tensor &table, const Tensor &ranges,
                  const Tensor &inv_radii, const Tensor &pdf, const Tensor &out_rows) {
  const int64_t k = p.k(), c = feats.size(1);
  Tensor out = empty_f32({ranges.size(0), c * k}, feats);
  hipStream_t s = current_stream();
  Region t("mc_conv_project", s);
  check(mccnn_mc_conv_project(s, (int)p.dims, feats.size(0), f32(pin), (int)c, f32(feats),
                              ranges.size(0), f32(pout), table.size(0), i32(table), i32(ranges),
                              f32(inv_radii), (int)k, (int)p.per, (int)p.act, f32(w.kw),
                              f32(w.kb), f32(pdf), i32(out_rows), f32(out)));
  return out;
}

// Columns [first, first + cols) of the caller's rows cut out of a padded sub-layer result and
// joined: [n, mlps * g] from the sub-layers' [n, per * g_pad].
Tensor join_outputs(const Plan &p, std::vector<Tensor> &outs) {
  if (p.g_pad != p.g)
    for (auto &o : outs)
      o = o.view({o.size(0), p.per, p.g_pad}).slice(2, 0, p.g).reshape({o.size(0), p.per * p.g});
  return outs.size() == 1 ? outs[0] : at::cat(outs, 1);
}

// The rows of the upstream gradient that belong to sub-layer `first`, in the view's centre
// order and padded to its columns.
Tensor gather_upstream(const Plan &p, const Tensor &dout, const Tensor &rows, int64_t first) {
  if (p.g_pad == p.g) return gather_rows(dout, rows, first * p.g, p.per * p.g, p.per * p.g);
  if (p.per == 1) return gather_rows(dout, rows, first * p.g, p.g, p.g_pad);
  Tensor cols = dout.slice(1, first * p.g, (first + p.per) * p.g)
                    .reshape({dout.size(0), p.per, p.g});
  cols = at::constant_pad_nd(cols, {0, p.g_pad - p.g}, 0).view({dout.size(0), p.f()});
  return rows.defined() ? gather_rows(cols, rows, 0, p.f(), p.f()) : cols;
}

// The same with the columns padded to `wide` (one sub-layer of one kernel MLP, or wide as it is).
Tensor gather_upstream(const Plan &p, const Tensor &dout, const Tensor &rows, int64_t first,
                       int64_t wide) {
  return wide > p.f() || p.g_pad != p.g ? gather_rows(dout, rows, first * p.g, p.g, wide)
                                        : gather_upstream(p, dout, rows, first);
}

// W [r, f] with its columns padded to `wide`.
Tensor widen(const Tensor &w, int64_t wide) {
  return w.size(1) == wide ? w : gather_rows(w, Tensor(), 0, w.size(1), wide);
}

Tensor cut_columns(const Tensor &x, int64_t cols) {
  return x.size(1) == cols ? x : x.slice(1, 0, cols).contiguous();
}

// Whether the layer's two sub-layers run side by side, one launch of everything for both: inputs
// whose products keep the register-resident kernel, where a pass is chains of loads and launches.
// Per output element the sums are those of the sub-layers on their own.
// Layer of 6 -> 32 channels, 4 x 8 hidden units, 61 k points of 28 pairs: 592 -> 490 us for the pass, 53 -> 39
// launches.  Over 4 k to 200 k points, 6 to 128 inputs and 32 to 128 outputs the two apart take 1.0 (from
// 61 k points and 64 channels on, where the kernels' own time is all) to 1.7 times as long.
bool paired(const Plan &p, int64_t n_out, int64_t n_in, int64_t pairs, bool grads) {
  const int64_t f = p.f(), r = p.c_pad * p.k();
  if (p.mlps != 2 * p.per || p.k() != 16 || p.g_pad != p.g || p.cols() != f ||
      n_in * 2 * std::max(p.c_pad, f) >= (int64_t)1 << 30 || n_out * 2 * f >= (int64_t)1 << 30 ||
      product_kind(n_out, r, f) != Product::kRegisters)
    return false;
  return !grads || (narrow_columns(p, n_out, pairs) == 0 &&
                    product_kind(n_in, f * 16, p.c_pad) == Product::kRegisters &&
                    product_kind(n_in, 2 * f * 16, p.c_pad) == Product::kRegisters &&
                    mccnn_projection_grad_product_supported((int)(2 * f), (int)(2 * r)) &&
                    mccnn_weight_grad_product_supported((int)p.c_pad, (int)(2 * f * 16)));
}

// Both sub-layers' weights: w [2, r, f] where the forward product reads them, all [2 r, 2 f] as w
// of the saved ones, w2 [2 f k, c].
Packed pack_pair(const Plan &p, const Tensor &final_weights, const Tensor &kw, const Tensor &kb,
                 bool grads, Tensor *forward) {
  Packed out;
  const int64_t k = p.k(), f = p.f(), r = p.c_pad * k;
  *forward = empty_f32({2, r, f}, final_weights);
  if (grads) {
    out.w = empty_f32({2 * r, 2 * f}, final_weights);
    out.w2 = empty_f32({2 * f * k, p.c_pad}, final_weights);
  }
  out.kw = empty_f32({p.mlps, p.dims, p.h_pad}, kw);
  out.kb = empty_f32({2 * k}, kb);
  hipStream_t s = current_stream();
  Region t("pack_layer_weights", s);
  check(mccnn_pack_layer_weights_pair(s, (int)p.dims, (int)p.c, (int)p.h, (int)p.g, (int)p.per,
                                      (int)p.c_pad, (int)p.h_pad, (int)p.g_pad,
                                      f32(final_weights), f32(kw), f32(kb), f32(*forward),
                                      f32(out.w2), f32(out.kw), f32(out.kb), f32(out.w)));
  return out;
}

// Projections of both sub-layers, [n, 2, channels, 16]; `own`: feats hold channels of each.
Tensor mc_project_pair(const Plan &p, const Packed &w, const Tensor &feats, bool own,
                       const Tensor &pin, const Tensor &pout, const Tensor &table,
                       const Tensor &ranges, const Tensor &inv_radii, const Tensor &pdf,
                       const Tensor &out_rows) {
  const int64_t c = own ? feats.size(1) / 2 : feats.size(1);
  Tensor out = empty_f32({ranges.size(0), 2 * c * p.k()}, feats);
  hipStream_t s = current_stream();
  Region t("mc_conv_project", s);
  check(mccnn_mc_conv_project_pair(s, (int)p.dims, feats.size(0), f32(pin), (int)c, own ? 1 : 0,
                                   f32(feats), ranges.size(0), f32(pout), table.size(0),
                                   i32(table), i32(ranges), f32(inv_radii), (int)p.mlps,
                                   (int)p.act, f32(w.kw), f32(w.kb), f32(pdf), i32(out_rows),
                                   f32(out)));
  return out;
}

// The whole Monte-Carlo convolution (MCConv.py:137-194) on the grid-ordered view.  Forward:
// fused basis + projection, product with the final weights.  The projection writes its rows (of
// C K floats) to the centres' original positions, which costs it nothing; the product's rows of
// F floats do not scatter for free (16 455 rows x 2048 x 128: 108 us in order, 116 us to
// scattered rows).  Backward: the feature gradient is the same convolution
// run from the centres back to the points over the transposed pair table (no scatter),
//     Q[j, f, k]  = sum_{i in T(j)} basis[ij, k] dout[i, f]
//     dfeat[j, c] = sum_{f,k} Q[j, f, k] W[c, k, f]
//     dW[c, k, f] = sum_j feat[j, c] Q[j, f, k]
// and the kernel-MLP gradients come from dproj = dout W^T.  Rows of Q go to the points' original
// positions too, where the features there have the kernels' channel count.
struct McConv : torch::autograd::Function<McConv> {
  static Tensor forward(AutogradContext *ctx, const Tensor &features, const Tensor &kw,
                        const Tensor &kb, const Tensor &final_weights,
                        const c10::intrusive_ptr<Geometry> &geo, const Plan &p, bool grads) {
    const Tensor feats = gather_rows(features, geo->point_rows, 0, p.c, p.c_pad);
    const int64_t n_out = geo->ranges.size(0);
    std::vector<Tensor> outs;
    const int64_t pairs = geo->table.size(0);
    const bool narrow = grads && narrow_columns(p, n_out, pairs) > 0;
    variable_list saved = {feats, kw, kb, final_weights,
                           p.c == p.c_pad && !narrow ? features : Tensor()};
    const bool pair = paired(p, n_out, feats.size(0), pairs, grads);
    if (pair) {
      Tensor forward;
      const Packed w = pack_pair(p, final_weights, kw, kb, grads, &forward);
      const Tensor proj = mc_project_pair(p, w, feats, false, geo->points_in, geo->points_out,
                                          geo->table, geo->ranges, geo->inv_radii, geo->pdf,
                                          geo->centre_rows);
      Tensor out = empty_f32({n_out, 2 * p.f()}, feats);
      hipStream_t s = current_stream();
      Region t("final_product", s);
      check(mccnn_final_product_pair(s, n_out, (int)(proj.size(1) / 2), f32(proj), (int)p.f(),
                                     f32(forward), f32(out)));
      outs.push_back(out);
      if (grads) w.save(saved);
    }
    for (int64_t first = 0; first < p.mlps && !pair; first += p.per) {
      const Packed w = pack(p, first, final_weights, kw, kb, n_out, feats.size(0), grads,
                            grads && !narrow);
      const Tensor proj = mc_project(p, w, feats, geo->points_in, geo->points_out, geo->table,
                                     geo->ranges, geo->inv_radii, geo->pdf, geo->centre_rows);
      outs.push_back(run_product(w.forward, proj, w.w, w.wt, Tensor(), p.cols()));
      if (grads) w.save(saved);
    }
    if (grads) {
      ctx->save_for_backward(std::move(saved));
      ctx->saved_data["geo"] = c10::IValue::make_capsule(geo);
      ctx->saved_data["plan"] = std::vector<int64_t>{p.dims, p.c, p.h, p.g, p.mlps, p.c_pad,
                                                     p.h_pad, p.g_pad, p.per, p.act};
    }
    return join_outputs(p, outs);
  }

  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &feats = saved[0], &kw = saved[1], &kb = saved[2], &fw = saved[3],
                 &features = saved[4];
    const auto v = ctx->saved_data["plan"].toIntVector();
    const Plan p{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9]};
    const auto geo = c10::static_intrusive_pointer_cast<Geometry>(
        ctx->saved_data["geo"].toCapsule());
    const Tensor dout = grad_out[0].contiguous();
    const int64_t n_out = geo->ranges.size(0), k = p.k();
    const bool want_feat = ctx->needs_input_grad(0), want_kernel = ctx->needs_input_grad(1) ||
                                                                   ctx->needs_input_grad(2);
    const bool want_final = ctx->needs_input_grad(3);
    Tensor dfeat, dkw, dkb, dfinal;
    if (want_kernel) {
      dkw = at::empty_like(kw);
      dkb = at::empty_like(kb);
    }
    if (want_final) dfinal = at::empty_like(fw);
    const int64_t wide = narrow_columns(p, n_out, geo->table.size(0));
    if (wide > 0 && want_feat) dfeat = empty_f32({geo->ranges_t.size(0), p.c}, feats);
    hipStream_t s = current_stream();
    const bool pair = saved.size() == 5 + Packed::kTensors && p.mlps == 2 * p.per;
    if (pair) {
      const Packed w = Packed::saved(saved, 5);
      const int64_t f2 = 2 * p.f();
      const Tensor up = geo->centre_rows.defined() ? gather_rows(dout, geo->centre_rows, 0, f2, f2)
                                                   : dout;
      Tensor dkw_pad, dkb_pad, ddense;
      if (want_kernel) {
        const Tensor dproj = projection_grad_product(up, w.w);
        Tensor ws = workspace(mccnn_mc_conv_project_grads_workspace_bytes((int)p.dims, (int)(2 * k),
                                                                          n_out), feats);
        dkw_pad = empty_f32({p.mlps, p.dims, p.h_pad}, feats);
        dkb_pad = empty_f32({2 * k}, feats);
        Region t("mc_conv_project_grads", s);
        check(mccnn_mc_conv_project_grads(
            s, (int)p.dims, feats.size(0), f32(geo->points_in), (int)p.c_pad, f32(feats), n_out,
            f32(geo->points_out), geo->table.size(0), i32(geo->table), i32(geo->ranges),
            f32(geo->inv_radii), (int)(2 * k), (int)p.mlps, (int)p.act, f32(w.kw), f32(w.kb),
            f32(geo->pdf), f32(dproj), ws.data_ptr(), ws.numel(), nullptr, nullptr, nullptr,
            nullptr, f32(dkw_pad), f32(dkb_pad)));
      }
      if (want_feat || want_final) {
        const bool in_place = features.defined();
        const Tensor q = mc_project_pair(p, w, up, true, geo->points_out, geo->points_in,
                                         geo->table_t, geo->ranges_t, geo->neg_inv_radii,
                                         geo->pdf_t, in_place ? geo->point_rows : Tensor());
        if (want_feat) dfeat = transposed_product(q, w, in_place ? Tensor() : geo->point_rows);
        if (want_final) ddense = weight_grad_product(in_place ? features : feats, q);
      }
      if (want_final || want_kernel) {
        Region t("unpack_layer_grads", s);
        check(mccnn_unpack_layer_grads_pair(
            s, (int)p.dims, (int)p.c, (int)p.h, (int)p.g, (int)p.per, (int)p.c_pad, (int)p.h_pad,
            (int)p.g_pad, f32(ddense), f32(dkw_pad), f32(dkb_pad), f32(dfinal), f32(dkw),
            f32(dkb)));
      }
    }
    for (int64_t first = 0, i = 0; first < p.mlps && !pair; first += p.per, ++i) {
      const Packed w = Packed::saved(saved, 5 + i * Packed::kTensors);
      const Tensor up =
          geo->centre_rows.defined() || p.g_pad != p.g || p.per != p.mlps || wide > p.f()
              ? (wide > 0 ? gather_upstream(p, dout, geo->centre_rows, first, wide)
                          : gather_upstream(p, dout, geo->centre_rows, first)) : dout;
      const bool direct = !p.padded() && p.mlps == 1;      // gradients land in the caller's shapes
      Tensor dkw_pad, dkb_pad, ddense, dproj;
      if (want_kernel || (wide > 0 && want_feat))
        dproj = wide > 0 ? projection_grad_product(up, widen(w.w, wide))
                         : layer_projection_grad(up, w.w);
      if (want_kernel) {
        Tensor ws = workspace(mccnn_mc_conv_project_grads_workspace_bytes((int)p.dims, (int)k,
                                                                          n_out), feats);
        dkw_pad = direct ? dkw : empty_f32({p.per, p.dims, p.h_pad}, feats);
        dkb_pad = direct ? dkb : empty_f32({k}, feats);
        Region t("mc_conv_project_grads", s);
        check(mccnn_mc_conv_project_grads(
            s, (int)p.dims, feats.size(0), f32(geo->points_in), (int)p.c_pad, f32(feats), n_out,
            f32(geo->points_out), geo->table.size(0), i32(geo->table), i32(geo->ranges),
            f32(geo->inv_radii), (int)k, (int)p.per, (int)p.act, f32(w.kw), f32(w.kb),
            f32(geo->pdf), f32(dproj), ws.data_ptr(), ws.numel(), nullptr, nullptr, nullptr,
            nullptr, f32(dkw_pad), f32(dkb_pad)));
      }
      if (wide > 0) {
        if (want_feat) {
          Region t("mc_conv_gather_grads", s);
          check(mccnn_mc_conv_gather_grads(
              s, (int)p.dims, n_out, f32(geo->points_out), (int)p.c, (int)p.c_pad, f32(dproj),
              geo->ranges_t.size(0), f32(geo->points_in), geo->table_t.size(0),
              i32(geo->table_t), i32(geo->ranges_t), f32(geo->neg_inv_radii), (int)p.per,
              (int)p.act, f32(w.kw), f32(w.kb), f32(geo->pdf_t), i32(geo->point_rows),
              first > 0, f32(dfeat)));
        }
        dproj = Tensor();
        if (want_final)
          ddense = weight_grad_product(up, mc_project(p, w, feats, geo->points_in, geo->points_out,
                                                      geo->table, geo->ranges, geo->inv_radii,
                                                      geo->pdf, Tensor()));
      } else if (want_feat || want_final) {
        dproj = Tensor();
        const bool in_place = features.defined();
        const Tensor q = mc_project(p, w, up, geo->points_out, geo->points_in, geo->table_t,
                                    geo->ranges_t, geo->neg_inv_radii, geo->pdf_t,
                                    in_place ? geo->point_rows : Tensor());
        if (want_feat) {
          Tensor d = transposed_product(q, w, in_place ? Tensor() : geo->point_rows);
          if (dfeat.defined()) dfeat.add_(d);
          else dfeat = d;
        }
        if (want_final) ddense = weight_grad_product(in_place ? features : feats, q);
      }
      if (want_final || (want_kernel && !direct)) {
        const bool kernel = want_kernel && !direct;
        Region t("unpack_layer_grads", s);
        check((wide > 0 ? mccnn_unpack_layer_grads_wt : mccnn_unpack_layer_grads)(
            s, (int)p.dims, (int)p.c, (int)p.h, (int)p.g, (int)first, (int)p.per, (int)p.c_pad,
            (int)p.h_pad, (int)p.g_pad, f32(ddense), kernel ? f32(dkw_pad) : nullptr,
            kernel ? f32(dkb_pad) : nullptr, f32(dfinal), kernel ? f32(dkw) : nullptr,
            kernel ? f32(dkb) : nullptr));
      }
    }
    if (dfeat.defined()) dfeat = cut_columns(dfeat, p.c);
    return {dfeat, dkw, dkb, dfinal, Tensor(), Tensor(), Tensor()};
  }
};

// Rigid kernel-point convolution (KPConv.py:165-232) on the same view: the basis are the
// correlations with the kernel points, which need no gradient.
struct KpShape {
  int64_t num_kp, kind;
  double sigma;
};

Tensor kp_project(const KpShape &kp, const Tensor &kernel_points, int64_t k, const Tensor &feats,
                  const Tensor &pin, const Tensor &pout, const Tensor &table, const Tensor &ranges,
                  const Tensor &inv_radii, const Tensor &out_rows) {
  const int64_t c = feats.size(1);
  Tensor out = empty_f32({ranges.size(0), c * k}, feats);
  hipStream_t s = current_stream();
  Region t("kp_conv_project", s);
  check(mccnn_kp_conv_project(s, (int)kernel_points.size(1), feats.size(0), f32(pin), (int)c,
                              f32(feats), ranges.size(0), f32(pout), table.size(0), i32(table),
                              i32(ranges), f32(inv_radii), (int)kp.num_kp, f32(kernel_points),
                              (int)kp.kind, (float)kp.sigma, i32(out_rows), f32(out)));
  return out;
}

struct KpConv : torch::autograd::Function<KpConv> {
  static Tensor forward(AutogradContext *ctx, const Tensor &features, const Tensor &weights,
                        const Tensor &kernel_points, const c10::intrusive_ptr<Geometry> &geo,
                        const Plan &p, const KpShape &kp, bool grads) {
    const Tensor feats = gather_rows(features, geo->point_rows, 0, p.c, p.c_pad);
    const bool narrow = grads && narrow_columns(p, geo->ranges.size(0), geo->table.size(0)) > 0;
    const Packed w = pack(p, 0, weights, Tensor(), Tensor(), geo->ranges.size(0), feats.size(0),
                          narrow, grads && !narrow);
    const Tensor proj = kp_project(kp, kernel_points, p.k(), feats, geo->points_in,
                                   geo->points_out, geo->table, geo->ranges, geo->inv_radii,
                                   geo->centre_rows);
    Tensor out = run_product(w.forward, proj, w.w, w.wt, Tensor(), p.cols());
    if (grads) {
      // what the rows of Q are multiplied with (the features where they are, or padded ones), or
      // what is projected again
      variable_list saved = {p.c == p.c_pad && !narrow ? features : feats, weights, kernel_points};
      w.save(saved);
      ctx->save_for_backward(std::move(saved));
      ctx->saved_data["geo"] = c10::IValue::make_capsule(geo);
      ctx->saved_data["plan"] = std::vector<int64_t>{p.dims, p.c, p.h, p.g, p.mlps, p.c_pad,
                                                     p.h_pad, p.g_pad, p.per, p.act, kp.num_kp,
                                                     kp.kind};
      ctx->saved_data["sigma"] = kp.sigma;
    }
    return cut_columns(out, p.g);
  }

  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &weights = saved[1], &kernel_points = saved[2];
    const auto v = ctx->saved_data["plan"].toIntVector();
    const Plan p{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9]};
    const KpShape kp{v[10], v[11], ctx->saved_data["sigma"].toDouble()};
    const auto geo = c10::static_intrusive_pointer_cast<Geometry>(
        ctx->saved_data["geo"].toCapsule());
    const Packed w = Packed::saved(saved, 3);
    const Tensor dout = grad_out[0].contiguous();
    const int64_t n_out = geo->ranges.size(0);
    const int64_t wide = narrow_columns(p, n_out, geo->table.size(0));
    const Tensor up = geo->centre_rows.defined() || p.g_pad != p.g || wide > p.f()
                          ? (wide > 0 ? gather_upstream(p, dout, geo->centre_rows, 0, wide)
                                      : gather_upstream(p, dout, geo->centre_rows, 0)) : dout;
    Tensor dfeat, dweights;
    hipStream_t s = current_stream();
    if (wide > 0) {
      if (ctx->needs_input_grad(0)) {
        const Tensor dproj = projection_grad_product(up, widen(w.w, wide));
        dfeat = empty_f32({geo->ranges_t.size(0), p.c}, x);
        Region t("kp_conv_gather_grads", s);
        check(mccnn_kp_conv_gather_grads(
            s, (int)p.dims, n_out, f32(geo->points_out), (int)p.c, (int)p.c_pad, f32(dproj),
            geo->ranges_t.size(0), f32(geo->points_in), geo->table_t.size(0), i32(geo->table_t),
            i32(geo->ranges_t), f32(geo->neg_inv_radii), (int)kp.num_kp, f32(kernel_points),
            (int)kp.kind, (float)kp.sigma, i32(geo->point_rows), f32(dfeat)));
      }
      if (ctx->needs_input_grad(1)) {
        const Tensor ddense = weight_grad_product(
            up, kp_project(kp, kernel_points, p.k(), x, geo->points_in, geo->points_out,
                           geo->table, geo->ranges, geo->inv_radii, Tensor()));
        dweights = at::empty_like(weights);
        Region t("unpack_layer_grads", s);
        check(mccnn_unpack_layer_grads_wt(s, (int)p.dims, (int)p.c, (int)p.h, (int)p.g, 0, 1,
                                          (int)p.c_pad, (int)p.h_pad, (int)p.g_pad, f32(ddense),
                                          nullptr, nullptr, f32(dweights), nullptr, nullptr));
      }
    } else if (ctx->needs_input_grad(0) || ctx->needs_input_grad(1)) {
      const bool in_place = p.c == p.c_pad;
      const Tensor q = kp_project(kp, kernel_points, p.k(), up, geo->points_out, geo->points_in,
                                  geo->table_t, geo->ranges_t, geo->neg_inv_radii,
                                  in_place ? geo->point_rows : Tensor());
      if (ctx->needs_input_grad(0))
        dfeat = cut_columns(transposed_product(q, w, in_place ? Tensor() : geo->point_rows), p.c);
      if (ctx->needs_input_grad(1)) {
        const Tensor ddense = weight_grad_product(x, q);
        dweights = at::empty_like(weights);
        Region t("unpack_layer_grads", s);
        check(mccnn_unpack_layer_grads(s, (int)p.dims, (int)p.c, (int)p.h, (int)p.g, 0, 1,
                                       (int)p.c_pad, (int)p.h_pad, (int)p.g_pad, f32(ddense),
                                       nullptr, nullptr, f32(dweights), nullptr, nullptr));
      }
    }
    return {dfeat, dweights, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

c10::intrusive_ptr<Geometry> make_geometry(
    const Tensor &points_in, const Tensor &points_out, const Tensor &table, const Tensor &ranges,
    const OptTensor &table_t, const OptTensor &ranges_t, const Tensor &point_rows,
    const OptTensor &centre_rows, const OptTensor &pdf, const OptTensor &pdf_t,
    const Tensor &inv_radii, const OptTensor &neg_inv_radii) {
  auto g = c10::make_intrusive<Geometry>();
  g->points_in = points_in;
  g->points_out = points_out;
  g->table = table;
  g->ranges = ranges;
  g->table_t = opt(table_t);
  g->ranges_t = opt(ranges_t);
  g->point_rows = point_rows;
  g->centre_rows = opt(centre_rows);
  g->pdf = opt(pdf);
  g->pdf_t = opt(pdf_t);
  g->inv_radii = inv_radii;
  g->neg_inv_radii = opt(neg_inv_radii);
  return g;
}

Plan plan_of(const std::vector<int64_t> &v) {
  return {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9]};
}

// What the kernels take for granted about the operands of a layer.
void check_layer(const char *op, const Plan &p, const Tensor &features, const Tensor &points_in,
                 const Tensor &points_out, const Tensor &point_rows, const Tensor &final_weights,
                 int64_t weights_in) {
  auto require = [&](bool ok, const std::string &what) {
    if (!ok) throw InvalidArgument(std::string(op) + " expects " + what);
  };
  require(features.dim() == 2 && features.size(1) == p.c,
          std::to_string(p.c) + " input features (got " + std::to_string(dim(features, 1)) + ")");
  require(features.size(0) >= point_rows.size(0), "a row of features per point");
  require(dim(points_in, 1) == p.dims && dim(points_out, 1) == p.dims,
          "points of " + std::to_string(p.dims) + " dimensions");
  require(final_weights.numel() == weights_in * p.g, "weights of the layer's sizes");
}

Tensor mc_conv(const Tensor &features, const Tensor &kw, const Tensor &kb, const Tensor &fw,
               const std::vector<int64_t> &plan, bool grads, const Tensor &points_in,
               const Tensor &points_out, const Tensor &table, const Tensor &ranges,
               const OptTensor &table_t, const OptTensor &ranges_t, const Tensor &point_rows,
               const OptTensor &centre_rows, const Tensor &pdf, const OptTensor &pdf_t,
               const Tensor &inv_radii, const OptTensor &neg_inv_radii) {
  const Plan p = plan_of(plan);
  check_layer("MCConv", p, features, points_in, points_out, point_rows, fw, p.mlps * p.c * p.h);
  if (kw.numel() != p.mlps * p.dims * p.h || kb.numel() != p.mlps * p.h)
    throw InvalidArgument("MCConv expects kernel weights of the layer's sizes");
  return McConv::apply(features.contiguous(), kw.contiguous(), kb.contiguous(), fw.contiguous(),
                       make_geometry(points_in, points_out, table, ranges, table_t, ranges_t,
                                     point_rows, centre_rows, pdf, pdf_t, inv_radii,
                                     neg_inv_radii),
                       p, grads);
}

Tensor kp_conv(const Tensor &features, const Tensor &weights, const Tensor &kernel_points,
               const std::vector<int64_t> &plan, int64_t kind, double sigma, bool grads,
               const Tensor &points_in, const Tensor &points_out, const Tensor &table,
               const Tensor &ranges, const OptTensor &table_t, const OptTensor &ranges_t,
               const Tensor &point_rows, const OptTensor &centre_rows, const Tensor &inv_radii,
               const OptTensor &neg_inv_radii) {
  const Plan p = plan_of(plan);
  check_layer("KPConv", p, features, points_in, points_out, point_rows, weights, p.c * p.h);
  if (dim(kernel_points, 0) != p.h || dim(kernel_points, 1) != p.dims)
    throw InvalidArgument("KPConv expects kernel points of the layer's sizes");
  return KpConv::apply(features.contiguous(), weights.contiguous(), kernel_points,
                       make_geometry(points_in, points_out, table, ranges, table_t, ranges_t,
                                     point_rows, centre_rows, OptTensor(), OptTensor(), inv_radii,
                                     neg_inv_radii),
                       p, KpShape{kernel_points.size(0), kind, sigma}, grads);
}

// -------------------------------------------------------------------------- pooling ----

struct LocalPool : torch::autograd::Function<LocalPool> {
  static Tensor forward(AutogradContext *ctx, const Tensor &features, const Tensor &neighbors,
                        const Tensor &ranges, int64_t kind) {
    Tensor out = empty_f32({ranges.size(0), features.size(1)}, features);
    hipStream_t s = current_stream();
    {
      Region t("local_pool", s);
      check(mccnn_local_pool(s, (int)kind, features.size(0), (int)features.size(1), f32(features),
                             neighbors.size(0), i32(neighbors), ranges.size(0), i32(ranges),
                             f32(out)));
    }
    ctx->save_for_backward({features, neighbors, ranges, out});
    ctx->saved_data["kind"] = kind;
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &features = saved[0], &neighbors = saved[1], &ranges = saved[2], &out = saved[3];
    Tensor dfeat = at::empty_like(features);
    const Tensor grad = grad_out[0].contiguous();
    hipStream_t s = current_stream();
    Region t("local_pool_grads", s);
    check(mccnn_local_pool_grads(s, (int)ctx->saved_data["kind"].toInt(), features.size(0),
                                 (int)features.size(1), f32(features), neighbors.size(0),
                                 i32(neighbors), ranges.size(0), i32(ranges), f32(out), f32(grad),
                                 f32(dfeat)));
    return {dfeat, Tensor(), Tensor(), Tensor()};
  }
};

struct GlobalPool : torch::autograd::Function<GlobalPool> {
  static Tensor forward(AutogradContext *ctx, const Tensor &features, const Tensor &bids,
                        int64_t batch, int64_t kind) {
    Tensor out = empty_f32({batch, features.size(1)}, features);
    Tensor counts = empty_i32({batch}, features);
    hipStream_t s = current_stream();
    {
      Region t("global_pool", s);
      check(mccnn_global_pool(s, (int)kind, features.size(0), (int)features.size(1), f32(features),
                              i32(bids), (int)batch, f32(out), i32(counts)));
    }
    ctx->save_for_backward({features, bids, out, counts});
    ctx->saved_data["kind"] = kind;
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &features = saved[0], &bids = saved[1], &out = saved[2], &counts = saved[3];
    const int64_t kind = ctx->saved_data["kind"].toInt();
    Tensor dfeat = at::empty_like(features), tie;
    if (kind == 0) tie = at::empty_like(out);
    const Tensor grad = grad_out[0].contiguous();
    hipStream_t s = current_stream();
    Region t("global_pool_grads", s);
    check(mccnn_global_pool_grads(s, (int)kind, features.size(0), (int)features.size(1),
                                  f32(features), i32(bids), (int)out.size(0), f32(out),
                                  i32(counts), f32(grad), f32(tie), f32(dfeat)));
    return {dfeat, Tensor(), Tensor(), Tensor()};
  }
};

Tensor local_pool(const Tensor &features, const Tensor &neighbors, const Tensor &ranges,
                  int64_t kind) {
  return LocalPool::apply(features.contiguous(), neighbors, ranges, kind);
}
Tensor global_pool(const Tensor &features, const Tensor &bids, int64_t batch, int64_t kind) {
  return GlobalPool::apply(features.contiguous(), bids, batch, kind);
}

// ------------------------------------------------------------------------ basis_proj ----

Tensor basis_proj_raw(const Tensor &basis, const Tensor &features, const Tensor &neighbors,
                      const Tensor &ranges, const Tensor &order) {
  Tensor out = empty_f32({ranges.size(0), std::max<int64_t>(dim(features, 1), 0),
                          std::max<int64_t>(dim(basis, 1), 0)}, features);
  hipStream_t s = current_stream();
  Region t("basis_proj_ordered", s);
  check(mccnn_basis_proj_ordered(s, basis.size(0), (int)dim(basis, 1), f32(basis),
                                 features.size(0), (int)dim(features, 1), f32(features),
                                 neighbors.size(0), (int)neighbors.dim(), (int)dim(neighbors, 1),
                                 i32(neighbors), ranges.size(0), i32(ranges), i32(order),
                                 f32(out)));
  return out;
}

Tensor basis_proj_raw_opt(const Tensor &basis, const Tensor &features, const Tensor &neighbors,
                          const Tensor &ranges, const OptTensor &order) {
  return basis_proj_raw(basis, features, neighbors, ranges, opt(order));
}

Tensor neighbourhood_order(const Tensor &neighbors, const Tensor &ranges) {
  const int64_t n = ranges.size(0);
  Tensor order = empty_i32({n}, ranges);
  Tensor ws = workspace(mccnn_neighbourhood_order_workspace_bytes(n), ranges);
  hipStream_t s = current_stream();
  Region t("neighbourhood_order", s);
  check(mccnn_neighbourhood_order(s, n, neighbors.size(0), i32(neighbors), i32(ranges),
                                  ws.data_ptr(), ws.numel(), i32(order)));
  return order;
}

std::pair<Tensor, Tensor> basis_proj_grads_grouped(const Tensor &basis, const Tensor &features,
                                                   const Tensor &neighbors, const Tensor &ranges,
                                                   const Tensor &g, const Tensor &order) {
  Tensor dbasis = at::empty_like(basis), dfeat = at::empty_like(features);
  hipStream_t s = current_stream();
  Tensor ws = workspace(mccnn_basis_proj_grads_grouped_workspace_bytes(ranges.size(0),
                                                                       neighbors.size(0)), ranges);
  Region t("basis_proj_grads_grouped", s);
  check(mccnn_basis_proj_grads_grouped(s, features.size(0), (int)basis.size(1), f32(basis),
                                       (int)features.size(1), f32(features), neighbors.size(0),
                                       i32(neighbors), ranges.size(0), i32(ranges), i32(order),
                                       f32(g), ws.data_ptr(), ws.numel(), f32(dbasis),
                                       f32(dfeat)));
  return {dbasis, dfeat};
}

bool aligned16(const Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// whether the grouped kernels take over (anything they cannot check is left to the others' errors)
bool group_gradients(const Tensor &basis, const Tensor &features, const Tensor &neighbors,
                     const Tensor &ranges, const Tensor &g) {
  if (basis.dim() != 2 || features.dim() != 2 || neighbors.dim() != 2 || neighbors.size(1) != 2 ||
      basis.size(0) != neighbors.size(0) || g.dim() != 3 || g.size(0) != ranges.size(0) ||
      g.size(1) != features.size(1) || g.size(2) != basis.size(1))
    return false;
  return mccnn_basis_proj_grads_grouped_pays((int)features.size(1), (int)basis.size(1),
                                             ranges.size(0), neighbors.size(0)) &&
         aligned16(basis) && aligned16(features) && aligned16(g);
}

// -> (dbasis, dfeatures); with the transposed lists the feature gradient is summed per point
// from per-pair rows, in a fixed order
std::pair<Tensor, Tensor> basis_proj_grads(const Tensor &basis, const Tensor &features,
                                           const Tensor &neighbors, const Tensor &ranges,
                                           const Tensor &g, const OptTensor &order,
                                           const OptTensor &point_ranges,
                                           const OptTensor &pair_order) {
  if (!point_ranges.has_value() && group_gradients(basis, features, neighbors, ranges, g))
    return basis_proj_grads_grouped(basis, features, neighbors, ranges, g,
                                    neighbourhood_order(neighbors, ranges));
  Tensor dbasis = at::empty_like(basis), dfeat = at::empty_like(features);
  hipStream_t s = current_stream();
  if (point_ranges.has_value()) {
    Tensor rows = empty_f32({neighbors.size(0), features.size(1)}, features);
    Region t("basis_proj_grads_gathered", s);
    check(mccnn_basis_proj_grads_gathered(
        s, basis.size(0), (int)dim(basis, 1), f32(basis), features.size(0), (int)dim(features, 1),
        f32(features), neighbors.size(0), (int)neighbors.dim(), (int)dim(neighbors, 1),
        i32(neighbors), ranges.size(0), i32(ranges), (int)g.dim(), dim(g, 0), dim(g, 1), dim(g, 2),
        f32(g), i32(*point_ranges), i32(opt(pair_order)), f32(rows), f32(dbasis), f32(dfeat)));
  } else {
    Region t("basis_proj_grads_ordered", s);
    check(mccnn_basis_proj_grads_ordered(
        s, basis.size(0), (int)dim(basis, 1), f32(basis), features.size(0), (int)dim(features, 1),
        f32(features), neighbors.size(0), (int)neighbors.dim(), (int)dim(neighbors, 1),
        i32(neighbors), ranges.size(0), i32(ranges), i32(opt(order)), (int)g.dim(), dim(g, 0),
        dim(g, 1), dim(g, 2), f32(g), f32(dbasis), f32(dfeat)));
  }
  return {dbasis, dfeat};
}

struct BasisProj : torch::autograd::Function<BasisProj> {
  static Tensor forward(AutogradContext *ctx, const Tensor &basis, const Tensor &features,
                        const Tensor &neighbors, const Tensor &ranges, const OptTensor &order,
                        const OptTensor &point_ranges, const OptTensor &pair_order) {
    ctx->save_for_backward({basis, features, neighbors, ranges, opt(order), opt(point_ranges),
                            opt(pair_order)});
    return basis_proj_raw(basis, features, neighbors, ranges, opt(order));
  }
  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto s = ctx->get_saved_variables();
    auto given = [](const Tensor &t) { return t.defined() ? OptTensor(t) : OptTensor(); };
    const auto grads = basis_proj_grads(s[0], s[1], s[2], s[3], grad_out[0].contiguous(),
                                        given(s[4]), given(s[5]), given(s[6]));
    return {grads.first, grads.second, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor basis_proj_apply(const Tensor &basis, const Tensor &features, const Tensor &neighbors,
                        const Tensor &ranges, const OptTensor &order,
                        const OptTensor &point_ranges, const OptTensor &pair_order) {
  return BasisProj::apply(basis, features, neighbors, ranges, order, point_ranges, pair_order);
}

// ----------------------------------------------------- layers between the convolutions ----

bool recording_gradients() { return at::GradMode::is_enabled(); }

// Batch normalisation over the points + leaky activation.
struct NormAct : torch::autograd::Function<NormAct> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &weight,
                        const Tensor &bias, const Tensor &running_mean, const Tensor &running_var,
                        const OptTensor &batches, bool training, double momentum, double eps,
                        double slope) {
    auto norm = at::native_batch_norm(x, weight, bias, running_mean, running_var, training,
                                      momentum, eps);
    if (training && batches.has_value()) Tensor(*batches).add_(1);
    Tensor out = std::get<0>(norm);
    if (slope == 0.0) out.relu_();
    else if (slope != 1.0) at::leaky_relu_(out, slope);
    Tensor mean = std::get<1>(norm), inv = std::get<2>(norm);
    if (!training) {
      mean = running_mean.clone();
      inv = (running_var + eps).rsqrt();
    }
    ctx->save_for_backward({x, weight, bias, mean, inv, slope == 1.0 ? x : out});
    ctx->saved_data["training"] = training;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["slope"] = slope;
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto v = ctx->get_saved_variables();
    const Tensor &x = v[0], &weight = v[1], &bias = v[2], &out = v[5];
    const bool training = ctx->saved_data["training"].toBool();
    const double slope = ctx->saved_data["slope"].toDouble();
    variable_list grads(10);
    if (recording_gradients()) {          // gradients of gradients: through torch's operations
      Tensor mean = v[3], inv = v[4];
      if (training) {
        mean = x.mean(0);
        inv = (x.var(0, false) + ctx->saved_data["eps"].toDouble()).rsqrt();
      }
      const Tensor z = (x - mean) * inv * weight + bias;
      const Tensor y = slope == 1.0   ? z
                       : slope == 0.0 ? at::where(out <= 0, at::zeros_like(z), z)
                                      : at::where(out > 0, z, z * slope);
      variable_list wanted;
      std::vector<size_t> slots;
      for (size_t i = 0; i < 3; ++i)
        if (v[i].requires_grad()) {
          wanted.push_back(v[i]);
          slots.push_back(i);
        }
      const auto g = torch::autograd::grad({y}, wanted, {grad_out[0]}, true, true);
      for (size_t i = 0; i < slots.size(); ++i) grads[slots[i]] = g[i];
      return grads;
    }
    const Tensor g = grad_out[0].contiguous();
    if (ctx->needs_input_grad(0)) grads[0] = at::empty_like(x);
    grads[1] = at::empty_like(weight);
    grads[2] = at::empty_like(bias);
    Tensor ws = workspace(mccnn_norm_act_grads_workspace_bytes((int)x.size(1)), x);
    hipStream_t s = current_stream();
    Region t("norm_act_grads", s);
    check(mccnn_norm_act_grads(s, x.size(0), (int)x.size(1), f32(x), f32(out), f32(g), f32(v[3]),
                               f32(v[4]), f32(weight), training, (float)slope, ws.data_ptr(),
                               ws.numel(), f32(grads[0]), f32(grads[1]), f32(grads[2])));
    return grads;
  }
};

Tensor norm_act(const Tensor &x, const Tensor &weight, const Tensor &bias,
                const Tensor &running_mean, const Tensor &running_var, const OptTensor &batches,
                bool training, double momentum, double eps, double slope) {
  // the gradients take the side of 0 from the result
  if (!(slope >= 0.0)) throw InvalidArgument("norm_act expects a slope of at least 0");
  return NormAct::apply(x, weight, bias, running_mean, running_var, batches, training, momentum,
                        eps, slope);
}

// Per-point linear map with weights [R, F] and an optional bias of F elements.
struct Linear : torch::autograd::Function<Linear> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w,
                        const OptTensor &bias) {
    ctx->save_for_backward({x, w});
    if (bias.has_value()) ctx->saved_data["bias"] = bias->sizes().vec();
    Tensor out = x.mm(w);
    if (bias.has_value()) out.add_(*bias);
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grad_out) {
    const auto v = ctx->get_saved_variables();
    const Tensor &x = v[0], &w = v[1];
    const bool has_bias = ctx->saved_data.count("bias") > 0;
    variable_list grads(3);
    if (recording_gradients()) {          // gradients of gradients: through torch's operations
      grads[0] = grad_out[0].mm(w.t());
      grads[1] = x.t().mm(grad_out[0]);
      if (has_bias)
        grads[2] = grad_out[0].sum(0).view(ctx->saved_data["bias"].toIntVector());
      return grads;
    }
    const Tensor g = grad_out[0].contiguous();
    const int64_t n = x.size(0), r = w.size(0), f = w.size(1);
    hipStream_t s = current_stream();
    if (ctx->needs_input_grad(0)) {
      grads[0] = at::empty_like(x);
      Region t("linear_input_grads", s);
      check(mccnn_linear_input_grads(s, n, (int)r, f32(w), (int)f, f32(g), f32(grads[0])));
    }
    if (ctx->needs_input_grad(1) || (has_bias && ctx->needs_input_grad(2))) {
      grads[1] = at::empty_like(w);
      if (has_bias) grads[2] = empty_f32(ctx->saved_data["bias"].toIntVector(), w);
      if (n == 0) {
        grads[1].zero_();
        if (has_bias) grads[2].zero_();
        return grads;
      }
      Tensor ws = workspace(mccnn_linear_weight_grads_workspace_bytes(n, (int)r, (int)f), x);
      Region t("linear_weight_grads", s);
      check(mccnn_linear_weight_grads(s, n, (int)r, f32(x), (int)f, f32(g), ws.data_ptr(),
                                      ws.numel(), f32(grads[1]), f32(grads[2])));
    }
    return grads;
  }
};

Tensor linear(const Tensor &x, const Tensor &w, const OptTensor &bias) {
  return Linear::apply(x, w, bias);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  static py::object invalid_argument;
  m.def("set_error_class", [](py::object cls) { invalid_argument = std::move(cls); });
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const InvalidArgument &e) {
      PyErr_SetString(invalid_argument ? invalid_argument.ptr() : PyExc_ValueError, e.what());
    }
  });
  py::class_<GridTensors>(m, "GridTensors")
      .def_readonly("aabb_min", &GridTensors::aabb_min)
      .def_readonly("aabb_max", &GridTensors::aabb_max)
      .def_readonly("num_cells", &GridTensors::num_cells)
      .def_readonly("scaled_aabb_min", &GridTensors::smin)
      .def_readonly("inv_cell_sizes", &GridTensors::inv_cell)
      .def_readonly("keys", &GridTensors::keys)
      .def_readonly("sorted_keys", &GridTensors::sorted_keys)
      .def_readonly("sorted_indices", &GridTensors::sorted_indices)
      .def_readonly("sorted_points", &GridTensors::sorted_points)
      .def_readonly("sorted_batch_ids", &GridTensors::sorted_bids)
      .def_readonly("cells_host", &GridTensors::cells_host)
      .def_readonly("key_bits", &GridTensors::key_bits);
  using release = py::call_guard<py::gil_scoped_release>;
  m.def("start_timing", &start_timing);
  m.def("collect_timing", &collect_timing);
  m.def("compute_keys", &compute_keys, release());
  m.def("order_centres", &order_centres, py::arg("samples"), py::arg("batch_ids"),
        py::arg("batch_size"), py::arg("num_cells"), py::arg("scaled_aabb_min"),
        py::arg("inv_cell_sizes"), py::arg("key_bits"), py::arg("want_keys") = false, release());
  m.def("search_known", &search_known, release());
  m.def("invert_order", &invert_order, release());
  m.def("build_grid", &build_grid, release());
  m.def("build_grid_ds", &build_grid_ds, release());
  m.def("find_neighbors", &find_neighbors, release());
  m.def("search", &search, release());
  m.def("grid_density", &grid_density, release());
  m.def("reorder_ranges", &reorder_ranges, release());
  m.def("reorder_pairs", &reorder_pairs, release());
  m.def("reorder_pdf", &reorder_pdf, release());
  m.def("original_neighbor_ids", &original_neighbor_ids, release());
  m.def("transpose_neighbors", &transpose_neighbors, release());
  m.def("swapped_pairs", &swapped_pairs, release());
  m.def("gather_pdf", &gather_pdf, release());
  m.def("gather_pdf_both", &gather_pdf_both, release());
  m.def("gather_i32", &gather_i32, release());
  m.def("compute_pdf", &compute_pdf, release());
  m.def("sampling", &sampling, release());
  m.def("sampling_grid", &sampling_grid, release());
  m.def("final_product", &final_product, release());
  m.def("weight_grad_product", &weight_grad_product, release());
  m.def("projection_grad_product", &projection_grad_product, release());
  m.def("mc_conv", &mc_conv, release());
  m.def("kp_conv", &kp_conv, release());
  m.def("local_pool", &local_pool, release());
  m.def("global_pool", &global_pool, release());
  m.def("basis_proj", &basis_proj_raw_opt, release());
  m.def("norm_act", &norm_act, release());
  m.def("linear", &linear, release());
  m.def("basis_proj_apply", &basis_proj_apply, release());
  m.def("basis_proj_grads", &basis_proj_grads, release());
  m.def("basis_proj_grads_grouped", &basis_proj_grads_grouped, release());
  m.def("neighbourhood_order", &neighbourhood_order, release());
}
