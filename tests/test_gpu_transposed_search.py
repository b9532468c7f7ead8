"""The transposed pair table found by searching back from the points among the centres is the one a
sort of the pairs gives: dimensions, radii beyond the cell size, centres outside the grid's box,
clouds without points or centres, and the largest sizes that are searched back."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,n_out,cell,radius,spread", [
    (3, 900, 400, 0.1, 0.1, 1.0), (3, 900, 400, 0.1, 0.23, 1.0), (3, 900, 400, 0.2, 0.07, 1.0),
    (3, 2000, 1, 0.15, 0.15, 1.0), (3, 1, 2000, 0.15, 0.15, 1.0), (3, 900, 700, 0.1, 0.15, 1.6),
    (2, 1500, 600, 0.05, 0.05, 1.3), (2, 1500, 600, 0.05, 0.09, 1.0), (4, 1200, 500, 0.3, 0.3, 1.2),
    (3, 16384, 3000, 0.06, 0.06, 1.0), (3, 3000, 16384, 0.06, 0.09, 1.0),
    (3, 16385, 50, 0.06, 0.06, 1.0)])
def test_transposed_table_of_a_search_back(d, n, n_out, cell, radius, spread):
    from tensorflow_graphics_point_clouds_amd import _lib, pc
    gen = torch.Generator(device="cuda").manual_seed(n + n_out + d)
    rand = lambda *shape: torch.rand(shape, device="cuda", generator=gen)
    batch = 4                                       # clouds 1 (points) and 3 (centres) stay empty
    ids = torch.sort(torch.randint(0, 3, (n,), device="cuda", generator=gen) + 1)[0] % 4
    ids = torch.sort(torch.where(ids == 1, 0, ids))[0].int()
    cids = torch.randint(0, 3, (n_out,), device="cuda", generator=gen).int()
    centres = (rand(n_out, d) - 0.5) * spread + 0.5
    grid = pc.Grid(pc.PointCloud(rand(n, d), ids, batch), cell)
    nbh = pc.Neighborhood(grid, radius, pc.PointCloud(centres, cids, batch))
    view = nbh.sorted_view()
    assert (view._search_back is not None) == (max(n, n_out) <= 16384)
    ranges_t, order = _lib.host().transpose_neighbors(view.table, n)
    assert torch.equal(view.ranges_t, ranges_t)
    assert torch.equal(view.table_t, _lib.host().swapped_pairs(view.table, order))
    limited = pc.Neighborhood(grid, radius, pc.PointCloud(centres, cids, batch), max_neighbors=2)
    assert limited.sorted_view()._search_back is None


def test_search_back_checks_dimensions():
    from tensorflow_graphics_point_clouds_amd import _lib
    f = lambda *s: torch.zeros(*s, device="cuda")
    i = lambda *s: torch.ones(*s, dtype=torch.int32, device="cuda")
    keys = torch.zeros(5, dtype=torch.int64, device="cuda")
    with pytest.raises(_lib.InvalidArgumentError, match="dimensions"):
        _lib.host().search_known(f(4, 3), i(4), f(5, 2), keys, i(3), f(1, 3), f(3), f(3), 7)
    with pytest.raises(_lib.InvalidArgumentError, match="keys"):
        _lib.host().search_known(f(4, 3), i(4), f(5, 3), keys[:4], i(3), f(1, 3), f(3), f(3), 7)


@pytest.mark.parametrize("d,n,n_out,limit,kept", [
    (3, 16384, 300, 0, True), (3, 300, 16384, 0, True), (3, 16385, 300, 0, False),
    (3, 300, 16385, 0, False), (3, 300, 200, 4, False), (4, 300, 200, 0, True),
    (5, 300, 200, 0, False), (6, 300, 200, 0, False)])
def test_cells_of_centres_are_kept_where_they_are_searched(d, n, n_out, limit, kept):
    """Neighbourhoods that are never searched back hold no cell keys or cloud ids of their centres."""
    from tensorflow_graphics_point_clouds_amd import pc
    cloud = lambda m: pc.PointCloud(torch.rand(m, d, device="cuda"),
                                    torch.zeros(m, dtype=torch.int32, device="cuda"), 1)
    r = 0.1 if d == 3 else 0.3
    nbh = pc.Neighborhood(pc.Grid(cloud(n), r), r, cloud(n_out), max_neighbors=limit)
    assert (nbh._sorted_cells is not None) == kept
    if kept:
        assert nbh._sorted_cells[1].shape == (n_out,)
    view = nbh.sorted_view()
    assert (view._search_back is not None) == kept
    # the pairs by point, each list in ascending slots
    order = torch.argsort(view.table[:, 0].long() * n_out + view.table[:, 1].long())
    assert torch.equal(view.table_t, view.table[order][:, [1, 0]])
