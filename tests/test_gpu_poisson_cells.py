"""Poisson-disk selection in cells of more points than one batch or one wavefront holds, with several
selections in a cell, and with lists longer than the registers of a wavefront."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,cell,radius", [(3, 1, 0.3, 0.3), (3, 5, 2.0, 0.05), (3, 3000, 0.3, 0.3),
                                             (3, 3000, 0.4, 0.1), (2, 2500, 0.4, 0.1),
                                             (2, 2500, 0.25, 0.25), (4, 1500, 0.6, 0.2)])
def test_poisson_selection_in_crowded_cells(oracle, d, n, cell, radius):
    from tensorflow_graphics_point_clouds_amd import tfg_custom_ops as ops
    rng = np.random.default_rng(n + d)
    pts = rng.random((2 * n, d)).astype(np.float32)
    bids = np.repeat(np.arange(2, dtype=np.int32), n)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()
    g = oracle.Grid(pts, bids, 2, np.float32(cell))
    nbh = oracle.Neighborhood(g, np.float32(radius))
    _, _, expect = oracle.sampling(g.sorted_points, g.sorted_batch_ids, g.sorted_keys, g.num_cells,
                                   nbh.neighbors, nbh.ranges, 0)
    _, _, got = ops.sampling(dev(g.sorted_points), dev(g.sorted_batch_ids), dev(g.sorted_keys),
                             dev(g.num_cells), dev(nbh.neighbors), dev(nbh.ranges), 0)
    assert np.array_equal(got.cpu().numpy(), expect)


@pytest.mark.parametrize("d,n,cell,radius", [
    (3, 1, 0.3, 0.3), (3, 5, 2.0, 0.05), (3, 3000, 0.3, 0.3), (3, 3000, 0.4, 0.1),
    (3, 1500, 2.0, 0.07), (3, 3000, 0.4, 0.04), (3, 20000, 0.09, 0.09), (3, 20000, 0.2, 0.05),
    (3, 3000, 0.1, 0.25), (2, 2500, 0.4, 0.1), (2, 2500, 0.25, 0.25), (2, 30000, 0.02, 0.02),
    (4, 1500, 0.6, 0.2), (4, 1500, 0.5, 0.5), (5, 800, 0.7, 0.7)])
def test_selection_from_the_grid_is_that_from_the_table(d, n, cell, radius):
    """Selected points around a cell that fit the registers, do not, or stop fitting at a point of
    the cell; with and without a column table; points that coincide or are no numbers."""
    from tensorflow_graphics_point_clouds_amd import pc
    gen = torch.Generator(device="cuda").manual_seed(n + d)
    pts = torch.rand((2 * n, d), device="cuda", generator=gen)
    pts[n // 2] = pts[0]
    if n > 1000:
        pts[n + 3, 0] = float("nan")
    bids = torch.arange(2, device="cuda").repeat_interleave(n).int()
    grid = pc.Grid(pc.PointCloud(pts, bids, 2), cell)
    own = pc.Neighborhood(grid, radius, lazy=True)
    assert own._unsearched_own()
    got, ids = pc.sample(own, "poisson")
    assert own._unsearched_own()
    expect, expect_ids = pc.sample(pc.Neighborhood(grid, radius), "poisson")
    assert torch.equal(ids, expect_ids)
    assert torch.equal(got._points.nan_to_num(7.0), expect._points.nan_to_num(7.0))
    assert torch.equal(got._batch_ids, expect._batch_ids)


@pytest.mark.parametrize("d,n,cell,radius", [(4, 1500, 0.6, 0.2), (4, 1500, 0.5, 0.5), (5, 800, 0.7, 0.7),
                                             (5, 800, 0.7, 0.3), (6, 300, 0.8, 0.8)])
def test_selection_by_the_grid_kernels_in_more_dimensions(d, n, cell, radius):
    """The kernels themselves, also where sampling takes the pair table as the faster one."""
    from tensorflow_graphics_point_clouds_amd import _lib, pc
    gen = torch.Generator(device="cuda").manual_seed(n + d)
    pts = torch.rand((2 * n, d), device="cuda", generator=gen)
    grid = pc.Grid(pc.PointCloud(pts, torch.arange(2, device="cuda").repeat_interleave(n).int(), 2),
                   cell)
    nbh = pc.Neighborhood(grid, radius)
    _, _, expect = _lib.host().sampling(grid._sorted_points, grid._sorted_batch_ids,
                                        grid._sorted_keys, grid._num_cells, nbh._neighbors,
                                        nbh._samples_neigh_ranges, 0)
    points, ids, keys, ds, num_cells, _, _ = grid.search_tensors()
    _, _, got = _lib.host().sampling_grid(points, ids, keys, ds, num_cells, nbh._inv_radii)
    assert torch.equal(got, expect)


@pytest.mark.parametrize("d,from_grid", [(2, True), (3, True), (4, True), (5, False)])
def test_which_samples_are_selected_from_the_grid(d, from_grid, monkeypatch):
    """Hierarchies and samples of one radius leave their neighbourhoods unsearched where the grid is
    the faster one; radii of their own in four dimensions go to the pair table."""
    from tensorflow_graphics_point_clouds_amd import pc
    searched = []
    search = pc.Neighborhood._search
    monkeypatch.setattr(pc.Neighborhood, "_search", lambda self: (searched.append(self), search(self)))
    gen = torch.Generator(device="cuda").manual_seed(d)
    cloud = pc.PointCloud(torch.rand(700, d, device="cuda", generator=gen),
                          torch.zeros(700, dtype=torch.int32, device="cuda"), 1)
    hierarchy = pc.PointHierarchy(cloud, [0.3, torch.full((d,), 0.5)], "poisson")
    assert [n._unsearched_own() for n in hierarchy._neighborhoods] == [from_grid] * 2
    pc.poisson_disk_sampling(cloud, 0.3)
    assert len(searched) == (0 if from_grid else 3)
    own = pc.Neighborhood(pc.Grid(cloud, 0.5), 0.2, lazy=True)
    pc.sample(own, "poisson")
    assert own._unsearched_own()
    assert len(searched) == (0 if d <= 3 else 1 if d == 4 else 4)
    pc.PointHierarchy(cloud, [0.3], "cell average")
    assert len(searched) == (0 if d <= 3 else 1 if d == 4 else 4)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 4096, 4097, 16383, 16384, 16385])
@pytest.mark.parametrize("cell", [0.04, 0.4, 3.0])
def test_cells_of_points_on_either_side_of_one_block(n, cell):
    """One point per occupied cell: cells of one point, of tens and of all, as many as a block lists in
    one launch and one more."""
    from tensorflow_graphics_point_clouds_amd import pc
    gen = torch.Generator(device="cuda").manual_seed(n)
    pts = torch.rand((n, 3), device="cuda", generator=gen)
    bids = (torch.arange(n, device="cuda") * 3 // n).int()
    grid = pc.Grid(pc.PointCloud(pts, bids, 3), cell)
    got = pc.cell_average_sampling(None, grid=grid)
    _, owner, counts = torch.unique_consecutive(grid._sorted_keys, return_inverse=True,
                                                return_counts=True)
    sums = torch.zeros(len(counts), 3, device="cuda", dtype=torch.float64)
    sums.index_add_(0, owner, grid._sorted_points.double())
    want = sums / counts[:, None]
    # n - 1 float32 additions of values up to 1 and a division
    assert got._points.shape == want.shape
    assert bool(((got._points.double() - want).abs() <= (counts[:, None] + 1) * 2.0 ** -24).all())
    firsts = torch.cumsum(counts, 0) - counts
    assert torch.equal(got._batch_ids, grid._sorted_batch_ids[firsts])
