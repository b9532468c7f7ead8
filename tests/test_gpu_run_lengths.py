"""Convolution kernels where the number of centres per wavefront changes: last runs that are not
full, counts just below and at each change, and enough blocks for the folded reduction."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _table(n, mean, gen):
    """A pair table of n centres with 0 to 2 * mean neighbours each, in ascending order."""
    counts = torch.randint(0, 2 * mean + 1, (n,), device="cuda", generator=gen)
    ranges = torch.cumsum(counts, 0).int()
    centres = torch.repeat_interleave(torch.arange(n, device="cuda"), counts)
    ids = torch.randint(0, n, (centres.shape[0],), device="cuda", generator=gen)
    return torch.stack([ids, centres], dim=1).int().contiguous(), ranges


# runs of 1 | 2 | 4 | 8 centres of the projection change at 20 000, 64 000 and 160 000 centres (16 to
# 128 channels are one chunk), those of the gradients at 16 000 / 32 000 (short lists) and at 24 000 /
# 128 000; 131 073 centres in runs of 8 are more than 4096 blocks
@pytest.mark.parametrize("n,mean,c", [(1, 20, 16), (9, 3, 64), (15999, 3, 16), (16003, 20, 16),
                                      (20001, 20, 16), (24001, 20, 16), (32001, 3, 16), (64001, 20, 16),
                                      (160001, 3, 16), (131073, 17, 16), (16003, 3, 128)])
def test_projection_and_gradients_at_changes_of_the_run_length(n, mean, c):
    from tensorflow_graphics_point_clouds_amd import layers, tfg_custom_ops
    gen = torch.Generator(device="cuda").manual_seed(n + mean + c)
    rand = lambda *shape: torch.rand(shape, device="cuda", generator=gen)
    nbrs, ranges = _table(n, mean, gen)
    points = rand(n, 3)
    inv_radii = torch.full((3,), 2.0, device="cuda")
    weights = (rand(1, 3, 16) - 0.5).requires_grad_(True)
    biases = (rand(1, 1, 16) - 0.5).requires_grad_(True)
    pdf = rand(nbrs.shape[0]) + 0.5
    feats = rand(n, c) - 0.5
    upstream = rand(n, c, 16) - 0.5
    got = layers._MCConvProject.apply(weights, biases, feats, points, points, nbrs, ranges,
                                      inv_radii, pdf, 1, None)
    basis = layers._MCBasis.apply(weights, biases, points, points, nbrs, inv_radii, pdf, 1)
    expect = tfg_custom_ops.basis_proj(basis, feats, nbrs, ranges)
    # both are float32 sums of at most 2 * mean products: off by that many roundings of their
    # absolute values, the basis functions (|z| <= 4, 1 / pdf <= 2) by a few roundings each
    mag = tfg_custom_ops.basis_proj(basis.detach().abs(), feats.abs(), nbrs, ranges)
    assert bool(((got - expect).abs() <= (2 * mean + 16) * 2.0 ** -23 * (mag + 8 * mean)).all())
    dw, db = torch.autograd.grad(got, [weights, biases], upstream)
    # the gradients of the basis in float64 by hand
    ids, ctr = nbrs[:, 0].long(), nbrs[:, 1].long()
    delta = (points[ids] - points[ctr]) * inv_radii
    z = delta.double() @ weights[0].detach().double() + biases[0].detach().double()
    dw64 = torch.zeros(3, 16, dtype=torch.float64, device="cuda")
    db64, mag_w, mag_b = torch.zeros_like(dw64[0]), torch.zeros_like(dw64), torch.zeros_like(dw64[0])
    for part in torch.split(torch.arange(ids.shape[0], device="cuda"), 1 << 17):
        dbasis = (feats[ids[part]].double().unsqueeze(1) @ upstream[ctr[part]].double()).squeeze(1)
        dz = dbasis * torch.where(z[part] > 0, 1.0, 0.2) / pdf[part].double().unsqueeze(1)
        dw64 += delta[part].double().t() @ dz
        db64 += dz.sum(0)
        mag_w += delta[part].double().abs().t() @ dz.abs()
        mag_b += dz.abs().sum(0)
    # a pair's term has c products; the sums over pairs run in chains of some hundred terms that are
    # added pairwise, and a few z within a rounding of the kink take the other slope
    tol = (c + 256) * 2.0 ** -23
    assert bool(((dw[0].double() - dw64).abs() <= tol * (mag_w + 8 * c)).all())
    assert bool(((db.reshape(-1).double() - db64).abs() <= tol * (mag_b + 8 * c)).all())
