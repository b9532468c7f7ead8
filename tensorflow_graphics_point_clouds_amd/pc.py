"""Thin counterparts of the reference's callers of the op path, on torch GPU
tensors: `PointCloud` (segmented and padded forms), `Grid`, `Neighborhood`, `sample`
and `PointHierarchy` (pylib/pc/PointCloud.py, Grid.py, Neighborhood.py,
sampling.py, PointHierarchy.py).  They only arrange arguments: bounding boxes,
grid shape, sort and gathers are kernels of libmccnn_hip.so as well.
"""
import enum
import math

import numpy as np

import torch

from . import _lib, tfg_custom_ops
_F32, _I32 = torch.float32, torch.int32


class KDEMode(enum.Enum):
    """pylib/pc/Neighborhood.py: constant bandwidth, bandwidth from the number of
    points, or no density estimate."""
    constant = 0
    num_points = 1
    no_pdf = 2


_vector_cache = {}       # (bytes of the host values, dims, device) -> shared device vector
_scalar_cache = {}       # (float, dims, device) -> one of the vectors above
_shared = {}             # id of a shared vector -> (the vector itself, its host values)
_derived_cache = {}      # (operation, id of a shared vector) -> shared result


def _share(t, values):
    """Registers a small read-only device vector under its own identity.  The entry keeps
    the tensor alive, so the id (and the memory behind it) cannot be handed to another
    tensor while the entry exists."""
    _shared[id(t)] = (t, values)
    return t


def _as_vector(value, dims, device):
    """`value` (a number, a sequence or a tensor) as a float32 [dims] tensor on
    `device`.  Host numbers are uploaded once per (value, dims, device) and the
    tensor is shared read-only afterwards: radii and cell sizes repeat in every
    layer of a network."""
    if isinstance(value, torch.Tensor):
        if id(value) in _shared and value.shape[0] == dims and value.device == device:
            return value                       # one of these vectors already
        t = value.to(dtype=_F32).reshape(-1)
        if t.numel() == 1:
            t = t.repeat(dims)
        return t.to(device).contiguous()
    if type(value) is float:                   # the usual argument, without a trip through numpy
        t = _scalar_cache.get((value, dims, device))
        if t is not None:
            return t
    host = np.asarray(value, dtype=np.float32).reshape(-1)
    key = (host.tobytes(), int(dims), str(device))
    t = _vector_cache.get(key)
    if t is None:
        t = torch.as_tensor(host)
        if t.numel() == 1:
            t = t.repeat(dims)
        t = t.to(device).contiguous()
        if len(_vector_cache) < 4096:
            _vector_cache[key] = _share(t, tuple(float(v) for v in t.tolist()))
    if type(value) is float and len(_scalar_cache) < 4096 and id(t) in _shared:
        _scalar_cache[(value, dims, device)] = t
    return t


def _derived(op, fn, t):
    """fn(t) for a small device vector; the vectors `_as_vector` keeps (shared,
    read-only) and what was derived from them get the result once instead of one
    kernel launch per use.  Shared vectors are recognised by object identity, never by
    address: a caller's own tensor always takes fn(t)."""
    entry = _shared.get(id(t))
    if entry is None or entry[0] is not t:
        return fn(t)
    r = _derived_cache.get((op, id(t)))
    if r is None:
        r = _derived_cache[(op, id(t))] = _share(fn(t), None)
    return r


def _reciprocal(t):
    return _derived("reciprocal", torch.reciprocal, t)


def _negative(t):
    return _derived("negative", torch.neg, t)


def _host_values(t):
    """The entries of a small device vector as a tuple of floats; no device round
    trip for the vectors `_as_vector` keeps."""
    entry = _shared.get(id(t))
    if entry is not None and entry[0] is t and entry[1] is not None and \
            len(entry[1]) == t.numel():
        return entry[1]
    return tuple(float(v) for v in t.tolist())


class AABB:
    """Axis-aligned bounding box per cloud (pylib/pc/PointCloud.py:23-66)."""

    def __init__(self, point_cloud):
        pts, ids = point_cloud._points.detach(), point_cloud._batch_ids.long()
        b, d = point_cloud._batch_size, pts.shape[1]
        index = ids[:, None].expand(-1, d)
        self._batch_shape = point_cloud._batch_shape
        self._aabb_min = torch.zeros((b, d), dtype=_F32, device=pts.device).scatter_reduce(
            0, index, pts, "amin", include_self=False) - 1e-9
        self._aabb_max = torch.zeros((b, d), dtype=_F32, device=pts.device).scatter_reduce(
            0, index, pts, "amax", include_self=False) + 1e-9

    def get_diameter(self, ord="euclidean"):
        """Norm of the box extent per cloud, [A1, ..., An] (or [B])."""
        extent = self._aabb_max - self._aabb_min
        diam = torch.linalg.vector_norm(extent, ord=2 if ord == "euclidean" else ord, dim=-1)
        return diam if self._batch_shape is None else diam.reshape(self._batch_shape)


class PointCloud:
    """Points with a cloud id per point (pylib/pc/PointCloud.py:68-290).

    points     [N, D] with `batch_ids` [N] or `sizes` (sum = N), or padded
               [A1, ..., An, V, D] with optional `sizes` [A1, ..., An] (the first
               sizes[a] rows of each cloud are real, the rest padding)
    batch_size number of clouds (default: from batch_ids / sizes / batch shape)

    Internally always the segmented form `_points` [N, D], `_batch_ids` [N]."""

    def __init__(self, points, batch_ids=None, batch_size=None, sizes=None):
        points = torch.as_tensor(points, dtype=_F32)
        dev = points.device
        self._sizes = None if sizes is None else torch.as_tensor(sizes, dtype=_I32, device=dev)
        self._batch_shape = None
        if points.dim() < 2:
            raise ValueError("expected points [N, D] or [A1, ..., An, V, D]")
        if points.dim() > 2:                                  # PointCloud.py:122-138
            self._batch_shape = tuple(points.shape[:-2])
            clouds, v = int(math.prod(self._batch_shape)), points.shape[-2]
            if self._sizes is None and points.shape[-1] > 0:     # no padding: every row is a point
                self._sizes = torch.full(self._batch_shape, v, dtype=_I32, device=dev)
                # a copy, as with sizes: the caller may refill a padded buffer
                self._points = points.reshape(clouds * v, -1).clone(
                    memory_format=torch.contiguous_format)
                self._batch_ids = torch.arange(clouds, dtype=_I32, device=dev)[:, None] \
                    .expand(clouds, v).reshape(-1).contiguous()    # (one cloud: still a view)
                self._batch_size = int(clouds if batch_size is None else batch_size)
                self._dimension = self._points.shape[1]
                return
            if self._sizes is None:
                self._sizes = torch.full(self._batch_shape, v, dtype=_I32, device=dev)
            if tuple(self._sizes.shape) != self._batch_shape:
                raise ValueError("sizes must have the batch shape %s" % (self._batch_shape,))
            flat_sizes = self._sizes.reshape(-1).long()
            if bool((flat_sizes > v).any()) or bool((flat_sizes < 0).any()):
                raise ValueError("sizes must lie in [0, V]")
            if batch_size is None:
                batch_size = clouds
            keep = (torch.arange(v, device=dev)[None, :] < flat_sizes[:, None]).reshape(-1)
            self._points = points.reshape(clouds * v, -1)[keep].contiguous()
            self._batch_ids = torch.repeat_interleave(
                torch.arange(clouds, dtype=_I32, device=dev), flat_sizes)
        else:                                                 # PointCloud.py:140-149
            self._points = points.contiguous()
            if batch_ids is None:
                if self._sizes is None:
                    raise ValueError("points [N, D] need batch_ids or sizes")
                flat_sizes = self._sizes.reshape(-1).long()
                if batch_size is None:
                    batch_size = flat_sizes.numel()
                batch_ids = torch.repeat_interleave(
                    torch.arange(flat_sizes.numel(), dtype=_I32, device=dev), flat_sizes)
            self._batch_ids = torch.as_tensor(batch_ids, dtype=_I32, device=dev).contiguous()
            if self._batch_ids.shape[0] != self._points.shape[0]:
                raise ValueError("expected one batch id (or sizes summing to one) per point")
            if batch_size is None:
                batch_size = int(self._batch_ids.max().item()) + 1 if self._points.shape[0] else 0
        self._batch_size = int(batch_size)
        self._dimension = self._points.shape[1]

    def get_AABB(self):
        """The bounding boxes, computed on the first call (PointCloud.py:235-247)."""
        if getattr(self, "_aabb", None) is None:
            self._aabb = AABB(self)
        return self._aabb

    def get_sizes(self):
        """Points per cloud, in the batch shape if one is set (PointCloud.py:184-204)."""
        if self._sizes is None:
            self._sizes = torch.bincount(self._batch_ids.long(),
                                         minlength=self._batch_size).to(_I32)
            if self._batch_shape is not None:
                self._sizes = self._sizes.reshape(self._batch_shape)
        return self._sizes

    def set_batch_shape(self, batch_shape):
        """PointCloud.py:262-290."""
        if batch_shape is None:
            self._batch_shape = None
            return
        batch_shape = tuple(int(b) for b in batch_shape)
        if int(math.prod(batch_shape)) != self._batch_size:
            raise ValueError("Incompatible batch size. Must be %d but is %d" %
                             (self._batch_size, int(math.prod(batch_shape))))
        self._batch_shape = batch_shape
        if self._sizes is not None:
            self._sizes = self._sizes.reshape(batch_shape)

    def get_unflatten(self, max_num_points=None):
        """data [N, ...] -> zero-padded [A1, ..., An, V, ...] (PointCloud.py:206-235):
        the rows of each cloud in their stored order."""
        sizes = self.get_sizes().reshape(-1).long()
        v = int(sizes.max().item()) if sizes.numel() else 0
        if max_num_points is not None:
            if max_num_points < v:
                raise ValueError("max_num_points must be at least the largest cloud")
            v = int(max_num_points)
        order = torch.argsort(self._batch_ids.long(), stable=True)
        starts = torch.cumsum(sizes, 0) - sizes
        sorted_ids = self._batch_ids.long()[order]
        slot = sorted_ids * v + (torch.arange(order.numel(), device=order.device) -
                                 starts[sorted_ids])
        shape = self._batch_shape if self._batch_shape is not None else (self._batch_size,)

        def unflatten(data):
            out = torch.zeros((self._batch_size * v,) + tuple(data.shape[1:]), dtype=data.dtype,
                              device=data.device)
            out[slot] = data[order]
            return out.reshape(tuple(shape) + (v,) + tuple(data.shape[1:]))

        return unflatten

    def flatten_features(self, features):
        """Features [N, C] (returned unchanged) or padded [A1, ..., An, V, C] ->
        [N, C] in the order of the stored points (pylib/pc/utils.py:75-94)."""
        if not isinstance(features, torch.Tensor) or features.dtype != _F32 or \
                features.device != self._points.device:
            features = torch.as_tensor(features, dtype=_F32, device=self._points.device)
        if features.dim() == 2:
            if features.shape[0] != self._points.shape[0]:
                raise ValueError("expected one feature row per point")
            return features
        sizes = self.get_sizes().reshape(-1).long()
        v, c = features.shape[-2], features.shape[-1]
        keep = (torch.arange(v, device=features.device)[None, :] < sizes[:, None]).reshape(-1)
        by_cloud = features.reshape(-1, c)[keep]          # rows grouped by cloud
        order = torch.argsort(self._batch_ids.long(), stable=True)
        out = torch.empty_like(by_cloud)
        out[order] = by_cloud
        return out

    def format_output(self, features, return_sorted=False, return_padded=False):
        """Layer output [N, C] as is, sorted by cloud id, or zero-padded to
        [A1, ..., An, V, C] (pylib/pc/layers/utils.py:22-49)."""
        if return_padded:
            return self.get_unflatten()(features)
        if return_sorted:
            return features[torch.argsort(self._batch_ids.long(), stable=True)]
        return features

    def get_points(self, id=None, max_num_points=None):
        """The points of cloud `id` (an int or an index into the batch shape), or all
        of them padded to [A1, ..., An, V, D] (PointCloud.py:151-182)."""
        if id is None:
            return self.get_unflatten(max_num_points)(self._points)
        if not isinstance(id, int):
            shape = self._batch_shape if self._batch_shape is not None else (self._batch_size,)
            id = int(torch.arange(self._batch_size).reshape(shape)[tuple(id)].item())
        if id >= self._batch_size or id < -self._batch_size:
            raise IndexError("batch index out of range")
        return self._points[self._batch_ids == id % self._batch_size]


class Grid:
    """Regular grid over a point cloud (pylib/pc/Grid.py:32-84): grid shape from
    the per-cloud bounding boxes, cell keys, stable descending sort, gathers."""

    def __init__(self, point_cloud, cell_sizes, aabb=None):
        # `aabb` is accepted for the reference's signature; like the reference
        # (Grid.py:42-44) the grid always takes the cloud's own bounding boxes
        pc = point_cloud
        self._point_cloud = pc
        self._batch_size = pc._batch_size
        self._cell_sizes = _as_vector(cell_sizes, pc._dimension, pc._points.device)
        g = _lib.host().build_grid(pc._points.detach(), pc._batch_ids, pc._batch_size,
                                   self._cell_sizes)
        self._aabb_min, self._aabb_max = g.aabb_min, g.aabb_max
        self._num_cells = g.num_cells
        self._scaled_aabb_min, self._inv_cell_sizes = g.scaled_aabb_min, g.inv_cell_sizes
        self._cur_keys, self._sorted_keys = g.keys, g.sorted_keys
        self._sorted_indices = g.sorted_indices
        self._sorted_points, self._sorted_batch_ids = g.sorted_points, g.sorted_batch_ids
        # host copy of the grid shape: sizes the key width and the column table.  A small
        # cloud's grid does not wait for it (None until somebody asks)
        self._shape = (g.cells_host, g.key_bits) if g.cells_host else None
        self._fast_DS = None
        self._sorted_positions = None
        self._self_neighborhoods = {}

    def _host_shape(self):
        if self._shape is None:
            cells = [int(v) for v in self._num_cells.tolist()]
            total = self._batch_size
            for v in cells:
                total *= v
            self._shape = (cells, max(1, (total - 1).bit_length()))
        return self._shape

    @property
    def _num_cells_host(self):
        return self._host_shape()[0]

    @property
    def _key_bits(self):
        return self._host_shape()[1]

    def sorted_positions(self):
        """Inverse of the sort: position of every original point in the sorted order."""
        if self._sorted_positions is None:
            self._sorted_positions = _lib.host().invert_order(self._sorted_indices)
        return self._sorted_positions

    def self_neighborhood(self, radii, max_neighbors=0):
        """The neighbourhood of the grid's sorted points among themselves for these
        radii, built once and shared (densities, grid-ordered view, same-cloud
        convolutions)."""
        key = (_host_values(radii), int(max_neighbors))
        if key not in self._self_neighborhoods:
            self._self_neighborhoods[key] = Neighborhood(self, radii, None, max_neighbors)
        return self._self_neighborhoods[key]

    def known_self_neighborhood(self, radii):
        """The untruncated self-neighbourhood if it has been built, else None."""
        return self._self_neighborhoods.get((_host_values(radii), 0))

    def search_tensors(self):
        """(points, cloud ids, keys, column table or None, num_cells, scaled minimum, inverse
        cell size) of the sorted grid for the host extension.  Small clouds are searched over
        their keys, without the table and the host copy of the grid shape it needs."""
        small = self._shape is None and self._fast_DS is None
        return (self._sorted_points, self._sorted_batch_ids, self._sorted_keys,
                None if small else self.get_DS(), self._num_cells, self._scaled_aabb_min,
                self._inv_cell_sizes)

    def get_DS(self):
        if self._fast_DS is None:
            self._fast_DS = tfg_custom_ops.build_grid_ds(
                self._sorted_keys, self._num_cells, self._num_cells_host, self._batch_size)
        return self._fast_DS


class _SortedView:
    """A neighbourhood with input points and centres both numbered in grid-cell
    order, the layout the layer kernels run on: consecutive centres then share
    their neighbours and every neighbour list is a few contiguous index runs, so
    the feature gathers hit in L2 instead of walking the whole table at random.

    points_in / points_out   coordinates in that order
    point_order [N_in]       position -> original point id (the grid's sort)
    centre_order [N_out]     slot -> original centre id, None if the centres
                             already are the grid's sorted points
    table [M,2], ranges      pairs (point position, centre slot) grouped by slot
    table_t [M,2], ranges_t  pairs (centre slot, point position) grouped by point
    """

    def __init__(self, nbh):
        grid = nbh._grid
        self.points_in = grid._sorted_points
        self.point_rows = grid._sorted_indices           # int32, for kernels
        self._point_order = self._centre_order = None    # their int64 forms, on first use
        if nbh._equal_samples:
            self.centre_rows = None
            self.points_out = grid._sorted_points
            self.table, self.ranges = nbh._neighbors, nbh._samples_neigh_ranges
        else:
            self.centre_rows, self.points_out, self.ranges, self.table = nbh._sorted_search()
        # An untruncated self-neighbourhood is symmetric (the distance test is exact under
        # negation): the rows (x, p) of segment p are at once "x is a neighbour of centre p"
        # and "p is a neighbour of centre x", so the table is its own transpose.
        self._symmetric = (nbh._equal_samples or nbh._self_neighborhood is not None) and \
            nbh.max_neighbors == 0
        self._transposed = (self.table, self.ranges) if self._symmetric else None
        self._search_back = self._search_among_centres(nbh)
        self._pdf_key, self.pdf, self.pdf_t = None, None, None

    @property
    def point_order(self):
        """position -> original point id as int64 (for torch indexing)."""
        if self._point_order is None:
            self._point_order = self.point_rows.long()
        return self._point_order

    @property
    def centre_order(self):
        """slot -> original centre id as int64, None if the centres are the sorted points."""
        if self._centre_order is None and self.centre_rows is not None:
            self._centre_order = self.centre_rows.long()
        return self._centre_order

    def _search_among_centres(self, nbh):
        """Arguments of that search, or None where it does not apply."""
        grid = nbh._grid
        if nbh._sorted_cells is None or self._transposed is not None:
            return None
        bids, cells = nbh._sorted_cells
        return (self.points_in.detach(), grid._sorted_batch_ids, self.points_out, cells,
                grid._num_cells, grid._scaled_aabb_min, grid._inv_cell_sizes, nbh._inv_radii,
                self.table.shape[0])

    def _transpose(self):
        """The pairs grouped by point: needed by gradients only, built on first use."""
        if self._transposed is None and self._search_back is not None:
            ranges_t, table_t = _lib.host().search_known(*self._search_back)
            self._transposed, self._search_back = (table_t, ranges_t), None
        if self._transposed is None:
            ranges_t, pair_order = _lib.host().transpose_neighbors(self.table,
                                                                   self.points_in.shape[0])
            self._transposed = (_lib.host().swapped_pairs(self.table, pair_order), ranges_t)
        return self._transposed

    @property
    def table_t(self):
        return self._transpose()[0]

    @property
    def ranges_t(self):
        return self._transpose()[1]

    def tensors(self, transposed):
        """(points_in, points_out, table, ranges, table_t, ranges_t, point_rows, centre_rows)
        for the host extension; the transposed half is None unless asked for."""
        table_t, ranges_t = self._transpose() if transposed else (None, None)
        return (self.points_in, self.points_out, self.table, self.ranges, table_t, ranges_t,
                self.point_rows, self.centre_rows)

    def pair_pdf(self, nbh, transposed=True):
        """Per-pair densities of `table` and (unless `transposed` is False) `table_t`, the
        neighbour point's."""
        per_point = nbh._pdf_per_point
        # compute_pdf bumps the generation: a key made of the density tensor's address
        # could match a later tensor that the allocator put in the same place
        key = nbh._pdf_generation
        if key != self._pdf_key:
            self._pdf_key, self.pdf, self.pdf_t = key, None, None
        if transposed and self.pdf is None and per_point is not None and not nbh._pdf_normalize:
            self.pdf, self.pdf_t = _lib.host().gather_pdf_both(self.table, self.table_t,
                                                               per_point.detach())
        if self.pdf is None:
            self.pdf = self._pair_values(nbh, per_point, self.table, 0)
        if transposed and self.pdf_t is None:
            self.pdf_t = self.pdf if per_point is None else \
                self._pair_values(nbh, per_point, self.table_t, 1)
        return self.pdf, self.pdf_t


    def _pair_values(self, nbh, per_point, table, column):
        if per_point is None:
            return torch.ones(table.shape[0], dtype=_F32, device=table.device)
        pdf = _lib.host().gather_pdf(table, column, per_point.detach())
        if nbh._pdf_normalize:
            # Neighborhood.py:288-293: divided by the size of the pair's neighbourhood, i.e.
            # the pair count of its centre (column 1 of `table`, column 0 of `table_t`)
            ends = self.ranges.long()
            counts = (ends - torch.cat([ends.new_zeros(1), ends[:-1]])).to(_F32)
            pdf = pdf / counts[table[:, 1 - column].long()]
        return pdf


class Neighborhood:
    """Neighbour pairs of the centres `point_cloud_sample` (default: the grid's
    own sorted points) inside `grid` (pylib/pc/Neighborhood.py:218-311)."""

    # Up to this many points and centres the transposed table of a search without a limit is the
    # search from the points among the centres, three launches: the pairs are the same (cells of a
    # pair are neighbours either way, and the distance test is exact under negation) and so is
    # their order (ascending slots).  Regrouping the pairs by a sort is nine launches: 35 against
    # 24 us of kernels for 16 x 1024 points and their cell averages.  Beyond, a search without a
    # column table of the centres costs more than the sort, and their cells are not kept.  So does
    # one of 81 cell rows and more per point, from five dimensions on (5000 points and a third as many
    # centres, both searches and the transposed table: 174 against 128 us).
    _MOST_SEARCHED_BACK, _MOST_DIMS_SEARCHED_BACK = 16384, 4

    def __init__(self, grid, radius, point_cloud_sample=None, max_neighbors=0, lazy=False):
        """`lazy` puts the search off until the pair table is first read (a hierarchy keeps a
        neighbourhood per level that it never reads itself)."""
        d = grid._point_cloud._dimension
        dev = grid._sorted_points.device
        self._radii = _as_vector(radius, d, dev)
        self._grid = grid
        if point_cloud_sample is None:
            self._equal_samples = True
            self._point_cloud_sampled = PointCloud(grid._sorted_points, grid._sorted_batch_ids,
                                                   grid._batch_size)
        else:
            self._equal_samples = False
            self._point_cloud_sampled = point_cloud_sample
        self.max_neighbors = max_neighbors
        self._inv_radii = _reciprocal(self._radii)
        s = self._point_cloud_sampled
        self._self_neighborhood = None
        self._table = self._ranges = self._original = self._sorted = self._sorted_cells = None
        if point_cloud_sample is grid._point_cloud:
            # The centres are the grid's own points in the caller's order: search once
            # from the sorted points (the same search also serves the densities).
            self._self_neighborhood = grid.self_neighborhood(self._radii, max_neighbors)
        elif not lazy:
            self._search()
        self._pdf = None
        self._pdf_per_point = None
        self._pdf_args = None
        self._pdf_normalize = False
        self._pdf_generation = 0
        # optional visiting order of the centres for the projection kernels
        self._centre_order = self._centre_slots = None
        self._transposed_pairs = None
        self._sorted_view = None
        self._transposed = None

    def _search(self):
        """The pair search.  Centres that are not the grid's sorted points are brought into
        the order of their cells first: consecutive centres then walk the same cells, and the
        table is the grid-ordered view the layers run on.  The table in the caller's centre
        order is the same segments regrouped (the pairs of a centre depend on its coordinates
        only), built column by column when somebody asks for it."""
        s, grid = self._point_cloud_sampled, self._grid
        points, ids, keys, ds, num_cells, smin, inv_cell = grid.search_tensors()
        if self._equal_samples:
            self._ranges, self._table, cut = _lib.host().search(
                points, ids, points, keys, ds, num_cells, smin, inv_cell, self._inv_radii,
                self.max_neighbors)
            if not cut:
                tfg_custom_ops._remember_symmetric(self._table)
            return
        # (an order of few centres is one launch, which does not need the width of the keys)
        one_launch = s._points.shape[0] <= _lib.lib().mccnn_build_grid_single_launch_max()
        back = self.max_neighbors == 0 and points.shape[1] <= self._MOST_DIMS_SEARCHED_BACK and \
            max(points.shape[0], s._points.shape[0]) <= self._MOST_SEARCHED_BACK
        order, pts, bids, cells = _lib.host().order_centres(
            s._points.detach(), s._batch_ids, grid._batch_size, num_cells, smin, inv_cell,
            0 if one_launch else grid._key_bits, back)
        ranges, table, _ = _lib.host().search(pts, bids, points, keys, ds, num_cells, smin,
                                              inv_cell, self._inv_radii, self.max_neighbors)
        self._sorted = (order, pts, ranges, table)
        self._sorted_cells = (bids, cells) if back else None

    def _unsearched_own(self):
        """Whether this is the whole neighbourhood of the grid's own points and its search has been
        put off so far."""
        return self._equal_samples and self.max_neighbors == 0 and self._table is None

    # Dimensions up to which a Poisson-disk sample of cells of one radius is selected from the grid.
    # In more, the cells around one hold more selected points than the registers of a wavefront,
    # and each point is then compared with all of them from memory: 20 000 points of 40 neighbours
    # in five dimensions 0.78 ms with the pair table, 3.1 from the grid; in four (30 000) 0.52 and 0.30.
    _MOST_DIMS_SELECTED_FROM_GRID = 4

    def _selects_from_grid(self):
        """Whether a Poisson-disk sample is selected faster from the grid than from the pair table, which
        has to be searched for it.  Radii well below the cell size have the same effect as more
        dimensions: in four, cells of one radius only (radii of 0.4 cells, as above: 0.44 and 1.8 ms);
        up to three the grid is 1.2 to 1.5 times faster with those as well, but for hundreds of
        points in a cell (0.52 and 0.70 ms)."""
        dims = self._grid._sorted_points.shape[1]
        one_radius = self._radii.data_ptr() == self._grid._cell_sizes.data_ptr()
        return dims <= 3 or (dims <= self._MOST_DIMS_SELECTED_FROM_GRID and one_radius)

    def _sorted_search(self):
        """(centre order, centres, ranges, pairs) with the centres in the order of their cells."""
        if self._sorted is None:
            own = self._self_neighborhood
            if own is None:
                self._search()                   # a search that was put off
            else:
                grid = self._grid
                self._sorted = (grid._sorted_indices, grid._sorted_points,
                                own._samples_neigh_ranges, own._neighbors)
        return self._sorted

    def _slots(self):
        """Position of every centre in the cell order."""
        if self._self_neighborhood is not None:
            return self._grid.sorted_positions()
        if self._centre_slots is None:
            self._centre_slots = _lib.host().invert_order(self._sorted_search()[0])
        return self._centre_slots

    @property
    def _neighbors(self):
        """[M, 2] pairs (sorted point index, centre index), grouped by centre."""
        if self._table is None:
            if self._equal_samples:
                self._search()
            else:
                _, _, ranges, table = self._sorted_search()
                self._table = _lib.host().reorder_pairs(ranges, table, self._slots(),
                                                        self._samples_neigh_ranges, None)
        return self._table

    @property
    def _samples_neigh_ranges(self):
        """[N_out] inclusive end offset of every centre's pairs."""
        if self._ranges is None:
            if self._equal_samples:
                self._search()
            else:
                self._ranges = _lib.host().reorder_ranges(self._sorted_search()[2], self._slots())
        return self._ranges

    @property
    def _original_neigh_ids(self):
        """The pairs addressed by original point ids (Neighborhood.py:246-250);
        built on first use."""
        if self._original is None:
            if self._table is None and not self._equal_samples:
                _, _, ranges, table = self._sorted_search()
                self._original = _lib.host().reorder_pairs(ranges, table, self._slots(),
                                                           self._samples_neigh_ranges,
                                                           self._grid._sorted_indices)
            else:
                self._original = _lib.host().original_neighbor_ids(self._neighbors,
                                                                   self._grid._sorted_indices)
        return self._original

    def transposed_pairs(self):
        """(point_ranges, pair_order): the pairs grouped by neighbour point, used by
        the atomic-free feature gradients; built on first use and kept."""
        if self._transposed_pairs is None:
            self._transposed_pairs = tfg_custom_ops.transpose_neighbors(
                self._original_neigh_ids, self._grid._point_cloud._points.shape[0])
        return self._transposed_pairs

    def get_grid(self):
        """The grid used for the neighbour search (Neighborhood.py:313-316)."""
        return self._grid

    def transpose(self):
        """The neighbourhood with centres and neighbour points switched
        (Neighborhood.py:318-329): itself for a self-neighbourhood, otherwise a
        grid over the centres searched from the original points; built once."""
        if self._transposed is None:
            if self._equal_samples:
                self._transposed = self
            else:
                grid = Grid(self._point_cloud_sampled, self._radii)
                self._transposed = Neighborhood(grid, self._radii, self._grid._point_cloud)
        return self._transposed

    def sorted_view(self):
        """The neighbourhood re-expressed in grid order on both sides (built on
        first use and kept): see `_SortedView`."""
        if self._sorted_view is None:
            self._sorted_view = _SortedView(self)
        return self._sorted_view

    def compute_centre_order(self):
        """Rank the centres by their cell key in the grid (a scheduling hint for
        `basis_proj`; the grid's own sorted points already are in that order)."""
        if not self._equal_samples:
            self._centre_order = self._sorted_search()[0]
        return self._centre_order

    def compute_pdf(self, bandwidth=0.2, mode=KDEMode.constant, normalize=False):
        """Densities of the grid's points from their self-neighbourhood
        (Neighborhood.py:257-293); the per-pair values follow on `get_pdf()`."""
        d = self._grid._point_cloud._dimension
        dev = self._grid._sorted_points.device
        self._pdf = None
        self._pdf_args = (bandwidth, mode)
        self._pdf_normalize = bool(normalize)
        self._pdf_generation += 1
        if mode == KDEMode.no_pdf:
            self._pdf_per_point = None
            return
        grid = self._grid
        inv_bw = _reciprocal(_as_vector(bandwidth, d, dev))
        nbh = self if self._equal_samples else grid.known_self_neighborhood(self._radii)
        if nbh is None and grid._sorted_points.requires_grad:
            nbh = grid.self_neighborhood(self._radii)       # (gradients come from the pairs)
        if nbh is None:          # the points' own pairs are not at hand: densities from the grid
            points, ids, keys, ds, num_cells, smin, inv_cell = grid.search_tensors()
            self._pdf_per_point = _lib.host().grid_density(
                points, ids, keys, ds, num_cells, smin, inv_cell, self._inv_radii, inv_bw,
                mode.value)
            return
        self._pdf_per_point = tfg_custom_ops.compute_pdf_with_pt_grads(
            grid._sorted_points, nbh._neighbors, nbh._samples_neigh_ranges, inv_bw,
            nbh._inv_radii, mode.value,
            symmetric=nbh._equal_samples and nbh.max_neighbors == 0)

    def point_pdf(self, **kwargs):
        """Density per sorted point (None with KDEMode.no_pdf), computed on first use
        with `kwargs` as for `compute_pdf`."""
        if self._pdf_args is None:
            self.compute_pdf(**kwargs)
        return self._pdf_per_point

    def get_pdf(self, **kwargs):
        """Density of the neighbour point of every pair of `_neighbors`
        (Neighborhood.py:287)."""
        per_point = self.point_pdf(**kwargs)
        if self._pdf is None:
            if per_point is None:
                self._pdf = torch.ones(self._neighbors.shape[0], dtype=_F32,
                                       device=self._neighbors.device)
            elif self._table is None and not self._equal_samples:
                _, _, ranges, table = self._sorted_search()
                self._pdf = _lib.host().reorder_pdf(ranges, table, self._slots(),
                                                    self._samples_neigh_ranges,
                                                    per_point.detach())
            else:
                self._pdf = _lib.host().gather_pdf(self._neighbors, 0, per_point.detach())
            if self._pdf_normalize:       # divided by the size of the pair's neighbourhood
                ends = self._samples_neigh_ranges.long()
                counts = (ends - torch.cat([ends.new_zeros(1), ends[:-1]])).to(_F32)
                self._pdf = self._pdf / counts[self._neighbors[:, 1].long()]
        return self._pdf


_SAMPLE_MODES = {"average": 1, "cell average": 1, "cell_average": 1,
                 "poisson": 0, "poisson disk": 0, "poisson_disk": 0}


def sample(neighborhood, sample_mode="poisson"):
    """pylib/pc/sampling.py:123-150 -> (PointCloud, original indices or None)."""
    mode = _SAMPLE_MODES[sample_mode.lower()]
    g = neighborhood._grid
    if mode == 0 and neighborhood._unsearched_own() and not neighborhood._selects_from_grid():
        neighborhood = Neighborhood(g, neighborhood._radii)       # (the caller's stays put off)
    if mode == 0 and neighborhood._unsearched_own():
        # the selection from the grid itself: as from the pair table, which it does not need
        points, ids, keys, ds, num_cells, _, _ = g.search_tensors()
        pts, bids, idx = _lib.host().sampling_grid(points, ids, keys, ds, num_cells,
                                                   neighborhood._inv_radii)
    else:
        if mode == 1:
            # cell averages read the keys only: no reason to run the neighbour search that
            # the (lazily built) pair table of `neighborhood` would cost
            dev = g._sorted_points.device
            pairs = torch.empty((0, 2), dtype=_I32, device=dev)
            ranges = torch.zeros(g._sorted_points.shape[0], dtype=_I32, device=dev)
        else:
            pairs, ranges = neighborhood._neighbors, neighborhood._samples_neigh_ranges
        pts, bids, idx = tfg_custom_ops.sampling(
            g._sorted_points, g._sorted_batch_ids, g._sorted_keys, g._num_cells, pairs, ranges,
            mode)
    original = None
    if mode == 0:
        original = _lib.host().gather_i32(g._sorted_indices, idx)
    return PointCloud(pts, bids, g._batch_size), original


def _sampling_neighborhood(grid, sample_mode):
    """The grid's own neighbourhood for cells of one radius, searched only if sampling reads its pairs."""
    reads = _SAMPLE_MODES[sample_mode.lower()] == 0 and \
        grid._sorted_points.shape[1] > Neighborhood._MOST_DIMS_SELECTED_FROM_GRID
    return Neighborhood(grid, grid._cell_sizes, lazy=not reads)


def poisson_disk_sampling(point_cloud, radius=None, neighborhood=None, return_ids=False):
    """Poisson-disk sample of a point cloud (pylib/pc/sampling.py:31-78) -> PointCloud
    (and the original indices of the kept points).  The reference passes the mode
    of the other sampler here (:67, and :114 below); this follows the names."""
    if radius is None and neighborhood is None:
        raise ValueError("Missing Argument! Either radius or neighborhood must be given!")
    if neighborhood is None:
        radii = _as_vector(radius, point_cloud._dimension, point_cloud._points.device)
        neighborhood = _sampling_neighborhood(Grid(point_cloud, radii), "poisson")
    cloud, ids = sample(neighborhood, "poisson")
    return (cloud, ids) if return_ids else cloud


def cell_average_sampling(point_cloud, cell_sizes=None, grid=None):
    """One point per occupied cell, the mean of the cell's points
    (pylib/pc/sampling.py:81-120) -> PointCloud."""
    if cell_sizes is None and grid is None:
        raise ValueError("Missing Argument! Either cell_sizes or grid must be given!")
    if grid is None:
        grid = Grid(point_cloud, _as_vector(cell_sizes, point_cloud._dimension,
                                            point_cloud._points.device))
    return sample(Neighborhood(grid, grid._cell_sizes, lazy=True), "average")[0]


class PointHierarchy:
    """Successively sampled point clouds (pylib/pc/PointHierarchy.py:40-98)."""

    def __init__(self, point_cloud, cell_sizes, sample_mode="poisson"):
        self._point_clouds = [point_cloud]
        self._cell_sizes = []
        self._neighborhoods = []
        self._sample_indices = []
        cur = point_cloud
        for cs in cell_sizes:
            cs = _as_vector(cs, point_cloud._dimension, point_cloud._points.device)
            self._cell_sizes.append(cs)
            grid = Grid(cur, cs)
            nbh = _sampling_neighborhood(grid, sample_mode)
            cur, idx = sample(nbh, sample_mode)
            self._neighborhoods.append(nbh)
            self._point_clouds.append(cur)
            self._sample_indices.append(idx)

    def get_neighborhood(self, i=None, transposed=False):
        """Neighbourhood between level i and i+1, or all of them
        (PointHierarchy.py:159-183); `transposed` gives level i+1 -> i."""
        if i is None:
            return [nb.transpose() for nb in self._neighborhoods] if transposed \
                else self._neighborhoods
        return self._neighborhoods[i].transpose() if transposed else self._neighborhoods[i]

    def get_points(self, batch_id=None, max_num_points=None):
        """Per level: the points of cloud `batch_id`, or all of them padded
        (PointHierarchy.py:100-122)."""
        return [c.get_points(batch_id, max_num_points) for c in self._point_clouds]

    def get_sizes(self):
        """Per level: points per cloud (PointHierarchy.py:124-138)."""
        return [c.get_sizes() for c in self._point_clouds]

    def set_batch_shape(self, batch_shape):
        """PointHierarchy.py:140-157."""
        for c in self._point_clouds:
            c.set_batch_shape(batch_shape)

    def __getitem__(self, index):
        return self._point_clouds[index]

    def __len__(self):
        return len(self._point_clouds)
