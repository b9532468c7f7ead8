"""The final-weight gradient at the edges of its steps and slices: fewer points than a step, a
last step of one point, slices without points, one and several column blocks."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,r", [(32, 256), (32, 4096), (64, 256), (64, 1024), (128, 256),
                                 (128, 2048)])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 4097, 12319])
def test_weight_grads_at_step_edges(n, c, r):
    from tensorflow_graphics_point_clouds_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n + c + r)
    x = torch.randn(n, c, device="cuda", generator=gen)
    y = torch.randn(n, r, device="cuda", generator=gen)
    got = _lib.host().weight_grad_product(x, y)
    # a sum of n products in any order is off by at most (n + 1) 2^-24 times the sum of their
    # absolute values; the parts of the three-way split left out add one rounding per product
    mag = x.double().abs().t() @ y.double().abs()
    err = (got.double() - x.double().t() @ y.double()).abs()
    assert bool((err <= (n + 2) * 2.0 ** -24 * mag).all())
