"""Neighbour search where a centre's candidates end at the edges of what the search lists and
remembers at a time: trips of 8, windows of 32 trips, two windows of remembered hits; in two to five
dimensions, with a limit on the list, and beyond the size up to which the count finds its slices."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def crowd(d, n, others, seed):
    """n points inside one cell of edge 0.25, `others` in the unit cube, in mixed order."""
    rng = np.random.default_rng(seed)
    pts = np.concatenate([0.5 + 0.249 * rng.random((n, d)), rng.random((others, d))])
    return np.ascontiguousarray(pts[rng.permutation(len(pts))], dtype=np.float32)


@pytest.mark.parametrize("d,n,others,limit", [
    (3, 1, 0, 0), (3, 7, 0, 0), (3, 8, 0, 0), (3, 9, 3, 0), (3, 255, 0, 0), (3, 256, 0, 0),
    (3, 257, 5, 0), (3, 511, 40, 0), (3, 512, 0, 0), (3, 513, 0, 0), (3, 1100, 300, 0),
    (3, 600, 100, 37), (3, 300, 16300, 0), (2, 513, 200, 0), (4, 513, 200, 0), (5, 300, 50, 0),
    (4, 700, 0, 300)])
def test_search_at_the_edges_of_its_windows(d, n, others, limit):
    from oracle import mccnn_oracle as oracle
    from tensorflow_graphics_point_clouds_amd import pc
    pts = crowd(d, n, others, 10 * n + d)
    ids = np.zeros(len(pts), np.int32)
    grid = pc.Grid(pc.PointCloud(torch.as_tensor(pts).cuda(), torch.as_tensor(ids).cuda(), 1), 0.25)
    expect = oracle.Neighborhood(oracle.Grid(pts, ids, 1, np.float32(0.25)), np.float32(0.25),
                                 pts, ids, limit)
    centres = pc.PointCloud(torch.as_tensor(pts).cuda(), torch.as_tensor(ids).cuda(), 1)
    nbh = pc.Neighborhood(grid, 0.25, centres, limit)
    assert np.array_equal(nbh._samples_neigh_ranges.cpu().numpy(), expect.ranges)
    assert np.array_equal(nbh._neighbors.cpu().numpy(), expect.neighbors)
