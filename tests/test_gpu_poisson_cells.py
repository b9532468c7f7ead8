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
