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
