"""Maximum pooling where its kernels branch: channel counts on either side of the row-wise ones,
many equal maxima, rows that are not 16-byte aligned, centres without and with long lists."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [1, 2, 3, 4, 5, 12, 48, 100, 256, 260])
@pytest.mark.parametrize("values", ["distinct", "ties", "unaligned"])
def test_max_pooling_with_ties(c, values, most=39):
    from tensorflow_graphics_point_clouds_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(c)
    n, n_out = 500, 301
    counts = torch.randint(0, most + 1, (n_out,), device="cuda", generator=gen)
    counts[::7], counts[5], counts[6] = 0, 200, 64
    ranges = torch.cumsum(counts, 0).int()
    seg = torch.repeat_interleave(torch.arange(n_out, device="cuda"), counts)
    # (a point at most once per list: unequal strides through the points)
    first = torch.cumsum(counts, 0) - counts
    ids = (torch.arange(seg.shape[0], device="cuda") - first[seg] + 13 * seg) % n
    pairs = torch.stack([ids, seg], dim=1).int().contiguous()
    feat = torch.randn(n, c, device="cuda", generator=gen)
    if values == "ties":
        feat = (feat * 2).round() / 2
    if values == "unaligned":
        feat = torch.cat([feat.new_zeros(1), feat.reshape(-1)])[1:].reshape(n, c)
    feat.requires_grad_(True)
    out = _lib.host().local_pool(feat, pairs, ranges, 0)
    up = torch.randn(n_out, c, device="cuda", generator=gen)
    grad, = torch.autograd.grad(out, feat, up)
    lowest = torch.finfo(torch.float32).min
    expect = torch.full((n_out, c), lowest, device="cuda").scatter_reduce(
        0, seg[:, None].expand(-1, c), feat.detach()[ids], "amax")
    assert torch.equal(out, expect)
    top = feat.detach()[ids] == expect[seg]
    ties = torch.zeros(n_out, c, dtype=torch.float64, device="cuda").index_add(0, seg, top.double())
    share = torch.where(top, (up.double() / ties.clamp(min=1))[seg], 0.0)
    want = torch.zeros(n, c, dtype=torch.float64, device="cuda").index_add(0, ids, share)
    mag = torch.zeros(n, c, dtype=torch.float64, device="cuda").index_add(0, ids, share.abs())
    # a point is in at most 301 lists: as many float32 additions of rounded shares
    assert bool(((grad.double() - want).abs() <= 302 * 2.0 ** -24 * mag).all())


# lists of fewer than 12 pairs are walked by a lane per channel from 32 channels on: nothing but such
# lists, lists on either side, mostly longer ones; the last 64 channels not full
@pytest.mark.parametrize("c", [4, 12, 28, 32, 64, 96, 256])
@pytest.mark.parametrize("values", ["distinct", "ties"])
@pytest.mark.parametrize("most", [2, 11, 24, 90])
def test_max_pooling_of_short_and_long_lists(c, values, most):
    test_max_pooling_with_ties(c, values, most)


@pytest.mark.parametrize("c", [4, 16, 32])
@pytest.mark.parametrize("n_out,k", [(127999, 5), (128000, 5), (128000, 6)])
def test_max_pooling_of_many_short_lists(c, n_out, k):
    """Either side of the number of centres from which short lists of few channels are packed."""
    from tensorflow_graphics_point_clouds_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(c + k)
    seg = torch.repeat_interleave(torch.arange(n_out, device="cuda"), k)
    ids = (7 * seg + torch.arange(k, device="cuda").repeat(n_out)) % n_out
    pairs = torch.stack([ids, seg], dim=1).int().contiguous()
    ranges = (k * torch.arange(1, n_out + 1, device="cuda")).int()
    feat = torch.randint(0, 40, (n_out, c), device="cuda", generator=gen).float().requires_grad_(True)
    up = torch.randn(n_out, c, device="cuda", generator=gen)
    out = _lib.host().local_pool(feat, pairs, ranges, 0)
    grad, = torch.autograd.grad(out, feat, up)
    rows = feat.detach()[ids].reshape(n_out, k, c)
    assert torch.equal(out, rows.amax(1))
    top = rows == rows.amax(1, keepdim=True)
    share = (top * (up / top.sum(1)).double()[:, None, :]).reshape(-1, c)
    want = torch.zeros(n_out, c, dtype=torch.float64, device="cuda").index_add(0, ids, share)
    mag = torch.zeros_like(want).index_add(0, ids, share.abs())
    # a point is in at most k lists: as many float32 additions of rounded shares
    assert bool(((grad.double() - want).abs() <= (k + 2) * 2.0 ** -24 * mag).all())
