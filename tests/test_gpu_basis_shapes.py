"""The basis projection at the edges of its tiles: channel counts around sixteens, chunks and the
32 where eight columns change kernels; centres without pairs, with one, with more than a wavefront
fetches at once, and an infinite feature beside them."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [8, 16, 32, 64])
@pytest.mark.parametrize("c", [1, 3, 7, 8, 16, 24, 32, 40, 64, 72, 96, 128, 136, 200])
def test_projection_at_tile_edges(c, k):
    from tensorflow_graphics_point_clouds_amd import tfg_custom_ops as ops
    gen = torch.Generator(device="cuda").manual_seed(100 * c + k)
    n, n_out = 300, 211
    counts = torch.randint(0, 30, (n_out,), device="cuda", generator=gen)
    counts[::9], counts[1::9], counts[5], counts[6], counts[-1] = 0, 1, 64, 65, 133
    ranges = torch.cumsum(counts, 0).int()
    seg = torch.repeat_interleave(torch.arange(n_out, device="cuda"), counts)
    ids = torch.randint(1, n, (seg.shape[0],), device="cuda", generator=gen)
    basis = torch.randn(seg.shape[0], k, device="cuda", generator=gen)
    feat = torch.randn(n, c, device="cuda", generator=gen)
    feat[0] = float("inf")                            # a row that no pair lists
    pairs = torch.stack([ids, seg], dim=1).int().contiguous()
    out = ops.basis_proj(basis, feat, pairs, ranges)
    term = feat.double()[ids][:, :, None] * basis.double()[:, None, :]
    want = torch.zeros(n_out, c, k, dtype=torch.float64, device="cuda").index_add(0, seg, term)
    mag = torch.zeros_like(want).index_add(0, seg, term.abs())
    # sums of at most 133 rounded products, each added with one rounding
    assert bool(((out.double() - want).abs() <= 134 * 2.0 ** -24 * mag).all())
