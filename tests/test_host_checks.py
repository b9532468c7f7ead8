"""What the host path refuses before anything reaches the GPU: calls that the kernels behind it
would answer wrongly or read out of range for.  Needs the built libraries, no GPU."""
import pytest
import torch

from tensorflow_graphics_point_clouds_amd import _lib, blocks


def test_norm_act_takes_only_activations_that_keep_signs():
    """The gradient reads the side of 0 off the result, which a negative slope turns round."""
    x = torch.linspace(-2.0, 3.0, 24).reshape(8, 3).requires_grad_()
    norm = torch.nn.BatchNorm1d(3)
    args = (norm.weight, norm.bias, norm.running_mean, norm.running_var, None, True, 0.1, 1e-3)
    for slope in (-0.3, float("nan")):
        with pytest.raises(_lib.InvalidArgumentError):
            _lib.host().norm_act(x, *args, slope)
        assert blocks._leaky_slope(torch.nn.LeakyReLU(slope)) is None
    assert blocks._leaky_slope(torch.nn.LeakyReLU(0.3)) == 0.3
    _lib.host().norm_act(x, *args, 0.3)


def _layer_arguments(points=40, dims=3):
    """Operands of a layer pass on host memory: what is checked is checked before the GPU."""
    pts = torch.zeros(points, dims)
    table, ranges = torch.zeros(4, 2, dtype=torch.int32), torch.zeros(points, dtype=torch.int32)
    rows = torch.zeros(points, dtype=torch.int32)
    return (pts, pts, table, ranges, None, None, rows, None), torch.ones(dims)


@pytest.mark.parametrize("features,dims,kernel,final", [
    ((40, 7), 3, (1, 3, 16), (1, 96, 32)), ((40, 5), 3, (1, 3, 16), (1, 96, 32)),
    ((39, 6), 3, (1, 3, 16), (1, 96, 32)), ((40, 6), 2, (1, 3, 16), (1, 96, 32)),
    ((40, 6), 3, (1, 3, 8), (1, 96, 32)), ((40, 6), 3, (1, 3, 16), (1, 96, 16))])
def test_monte_carlo_layer_checks_its_operands(features, dims, kernel, final):
    """Surplus feature columns are not dropped in silence, and no kernel reads past an operand."""
    from tensorflow_graphics_point_clouds_amd import layers
    geometry, inv_radii = _layer_arguments(dims=dims)
    plan = layers._layer_plan(3, 6, 32, 1, 16, 0)
    with pytest.raises(_lib.InvalidArgumentError):
        _lib.host().mc_conv(torch.zeros(features), torch.zeros(kernel), torch.zeros(1, 16),
                            torch.zeros(final), plan, False, *geometry, torch.zeros(4), None,
                            inv_radii, None)


@pytest.mark.parametrize("features,dims,weights,kernel_points", [
    ((40, 7), 3, (90, 32), 15), ((40, 5), 3, (90, 32), 15), ((39, 6), 3, (90, 32), 15),
    ((40, 6), 2, (90, 32), 15), ((40, 6), 3, (90, 16), 15), ((40, 6), 3, (90, 32), 14)])
def test_kernel_point_layer_checks_its_operands(features, dims, weights, kernel_points):
    from tensorflow_graphics_point_clouds_amd import layers
    geometry, inv_radii = _layer_arguments(dims=dims)
    plan = layers._kp_plan(3, 6, 32, 15, 16)
    with pytest.raises(_lib.InvalidArgumentError):
        _lib.host().kp_conv(torch.zeros(features), torch.zeros(weights),
                            torch.zeros(kernel_points, 3), plan, 0, 1.0, False, *geometry,
                            inv_radii, None)


def _grid_arguments(dims, points=8):
    """(points, cloud ids, keys, column table, num_cells, scaled minimum, inverse cell size)."""
    return (torch.zeros(points, dims), torch.zeros(points, dtype=torch.int32),
            torch.zeros(points, dtype=torch.int64), None, torch.ones(dims, dtype=torch.int32),
            torch.zeros(1, dims), torch.ones(dims))


@pytest.mark.parametrize("samples,grid,radii", [(2, 3, 3), (3, 2, 2), (3, 2, 3), (3, 3, 2), (2, 2, 3)])
def test_searches_check_dimensions(samples, grid, radii):
    """Centres, grid and radii of different dimensions are refused as find_neighbors refuses
    them: the kernels would read past the shorter one."""
    host = _lib.host()
    centres, ids = torch.zeros(5, samples), torch.zeros(5, dtype=torch.int32)
    args = _grid_arguments(grid)
    with pytest.raises(_lib.InvalidArgumentError, match="dimensions"):
        host.search(centres, ids, *args[:1], *args[2:], torch.ones(radii), 0)
    with pytest.raises(_lib.InvalidArgumentError, match="dimensions"):
        host.grid_density(*args, torch.ones(radii), torch.ones(5 - grid), 0)
    if samples != grid:
        with pytest.raises(_lib.InvalidArgumentError, match="dimensions"):
            host.order_centres(centres, ids, 1, *args[4:], 0)
    with pytest.raises(_lib.InvalidArgumentError, match="batch ids"):
        host.search(torch.zeros(5, grid), ids[:4], *args[:1], *args[2:], torch.ones(grid), 0)
    with pytest.raises(_lib.InvalidArgumentError, match="cell size"):
        host.build_grid(torch.zeros(5, 3), ids, 1, torch.ones(2))
