"""Gradients of layers with few input and more output channels, which go through the gradient of the
projection: channel counts at the edges of the gathered 4 / 8 / 16, output columns that are padded,
several kernel MLPs, points without neighbours, runs of every length; and which layers go there."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layer", ["mc", "mc_two", "mc_2d", "kp"])
@pytest.mark.parametrize("c,f", [(1, 32), (3, 64), (4, 48), (5, 96), (8, 128), (9, 112), (16, 32),
                                 (16, 128)])
def test_gradients_of_narrow_layers(layer, c, f, n_in=700, n_out=431, edge=0.0):
    from tensorflow_graphics_point_clouds_amd import layers, pc
    gen = torch.Generator(device="cuda").manual_seed(100 * c + f)
    rand = lambda *shape: torch.rand(shape, device="cuda", generator=gen)
    d = 2 if layer == "mc_2d" else 3
    r = 0.16
    pts, ctr = rand(n_in, d), rand(n_out, d)
    pts[-20:] += 3.0                                        # points that no centre reaches
    ids = torch.arange(n_in, device="cuda").mul(2).div(n_in, rounding_mode="floor").int()
    cids = torch.arange(n_out, device="cuda").mul(2).div(n_out, rounding_mode="floor").int()
    cin, cout = pc.PointCloud(pts, ids, 2), pc.PointCloud(ctr, cids, 2)
    nbh = pc.Neighborhood(pc.Grid(cin, r), r, cout)
    if layer == "kp":
        conv = layers.KPConv(c, f, num_kernel_points=15, num_dims=3, seed=c)
    else:
        mlps = 2 if layer == "mc_two" else 1
        conv = layers.MCConv(c, f, d, num_mlps=mlps, mlp_size=[16], non_linearity_type="elu", seed=c)
        with torch.no_grad():
            conv.biases.add_(rand(*conv.biases.shape) - 0.5)
    feats = (rand(n_in, c) - 0.5).requires_grad_(True)
    up = rand(n_out, f) - 0.5
    out = conv(feats, cin, cout, r, neighborhood=nbh)
    out.backward(up)

    pairs = nbh._original_neigh_ids.long()
    delta = (pts.double()[pairs[:, 0]] - ctr.double()[pairs[:, 1]]) / r
    if layer == "kp":            # linear influence of sigma = 1 radius (KPConv.py:193-213)
        dist = (delta[:, None, :] - conv._kernel_points.double()[None]).norm(dim=2)
        basis, finals = [(1.0 - dist).clamp(min=0.0)], [conv.weights.double()]
        near = edge
    else:
        pdf = nbh.get_pdf().double().reshape(-1, 1)
        basis = [torch.nn.functional.elu(delta @ w + b) / pdf
                 for w, b in zip(conv.weights.double(), conv.biases.double())]
        finals = list(conv.final_weights.double())
        near = edge / pdf
    g = f // len(finals)
    dfeat = torch.zeros(n_in, c, dtype=torch.float64, device="cuda")
    mag = torch.zeros_like(dfeat)
    for m, (b, w) in enumerate(zip(basis, finals)):
        k = b.shape[1]
        dproj = up[:, m * g:(m + 1) * g].double() @ w.detach().t()
        big = up[:, m * g:(m + 1) * g].double().abs() @ w.detach().t().abs()
        part = lambda basis, grad: (basis[:, None, :] * grad.reshape(n_out, c, k)[pairs[:, 1]]).sum(2)
        dfeat.index_add_(0, pairs[:, 0], part(b.detach(), dproj))
        mag.index_add_(0, pairs[:, 0], part(b.detach().abs() + near, big))
        proj = torch.zeros(n_out, c, k, dtype=torch.float64, device="cuda").index_add(
            0, pairs[:, 1], feats.detach().double()[pairs[:, 0]][:, :, None] * b.detach()[:, None, :])
        dw = proj.reshape(n_out, c * k).t() @ up[:, m * g:(m + 1) * g].double()
        got = conv.weights.grad if layer == "kp" else conv.final_weights.grad[m]
        assert float((got.double().reshape(dw.shape) - dw).norm()) <= 2e-6 * float(dw.norm())
    # f products per entry of G, 16 basis values and some hundred pairs per sum, a float32 density or
    # correlation (a few roundings) in each
    assert bool(((feats.grad.double() - dfeat).abs() <= 400 * 2.0 ** -24 * mag).all())
    assert feats.grad.shape == (n_in, c) and float(feats.grad[-20:].abs().max()) == 0.0


# runs of 1 | 2 | 4 | 8 points change at 20 000, 64 000 and 160 000 points; with 101 centres a point is
# in 0.9 lists on average, in none often, and the last run of each is not full.  Where a point has one
# pair its basis value can be the difference of two numbers near 1 (1 - dist, dist <= 2; z = 0 of three
# products below 2), which float32 has to some 32 * 2^-24 beside the value's own rounding: that over
# the 400 * 2^-24 of the sums is `edge`
@pytest.mark.parametrize("layer", ["mc", "mc_two", "kp"])
@pytest.mark.parametrize("c,f", [(3, 64), (5, 96), (16, 128)])
@pytest.mark.parametrize("n_in", [20001, 64003, 160005])
def test_gradients_of_narrow_layers_in_longer_runs(layer, c, f, n_in):
    from tensorflow_graphics_point_clouds_amd import _lib
    _lib.start_timing()
    try:
        test_gradients_of_narrow_layers(layer, c, 2 * f if layer == "mc_two" else f, n_in, 101,
                                        edge=32 / 400)
    finally:
        timed = _lib.collect_timing()
    assert any("gather_grads" in name for name in timed)


# through the gradient of the projection from five columns per gathered channel (4, 8 or 16) on, from
# three on where lists have 16 pairs or fewer on average
@pytest.mark.parametrize("c,f,short,longer", [
    (1, 32, True, True), (4, 32, True, True), (5, 32, True, False), (8, 32, True, False),
    (8, 48, True, True), (9, 32, False, False), (16, 32, False, False), (9, 48, True, False),
    (16, 64, True, False), (16, 80, True, True)])
@pytest.mark.parametrize("layer", ["mc", "kp"])
def test_layers_that_gather_gradients(layer, c, f, short, longer):
    from tensorflow_graphics_point_clouds_amd import _lib, layers, pc
    gen = torch.Generator(device="cuda").manual_seed(c + f)
    cloud = pc.PointCloud(torch.rand(1500, 3, device="cuda", generator=gen),
                          torch.zeros(1500, dtype=torch.int32, device="cuda"), 1)
    conv = layers.KPConv(c, f, num_kernel_points=15, num_dims=3, seed=c) if layer == "kp" else \
        layers.MCConv(c, f, 3, num_mlps=1, mlp_size=[16], seed=c)
    for r, expected in ((0.1, short), (0.2, longer)):
        nbh = pc.Neighborhood(pc.Grid(cloud, r), r, cloud)
        assert (nbh._neighbors.shape[0] <= 16 * 1500) == (r < 0.15)
        x = torch.rand(1500, c, device="cuda", generator=gen).requires_grad_(True)
        _lib.start_timing()
        try:
            conv(x, cloud, cloud, r, neighborhood=nbh).sum().backward()
        finally:
            timed = _lib.collect_timing()
        assert any("gather_grads" in name for name in timed) == expected


@pytest.mark.parametrize("d", [2, 3])
@pytest.mark.parametrize("c", [1, 3, 4, 5, 7, 9, 13, 15, 16])
def test_gathered_rows_of_any_width(d, c):
    """A gradient of the projection that holds no more channels than there are gives the bits that
    one padded to 16 channels gives, and nothing behind its last row is asked for."""
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cfloat, cint, i64, ptr, stream
    gen = torch.Generator(device="cuda").manual_seed(c)
    rand = lambda *shape: torch.rand(shape, device="cuda", generator=gen)
    n_pts, n_ctr, per = 37, 21, 9
    pts, ctr, inv_radii = rand(n_pts, d), rand(n_ctr, d), -torch.ones(d, device="cuda")
    pairs = torch.randint(0, n_ctr, (n_pts * per, 2), device="cuda", generator=gen).int()
    pairs[-1, 0] = n_ctr - 1                                # the last row is among those read
    ranges = per * torch.arange(1, n_pts + 1, device="cuda", dtype=torch.int32)
    w, b, pdf, kpts = rand(1, d, 16), rand(16), rand(n_pts * per) + 0.5, rand(15, d)
    padded = torch.zeros(n_ctr, 16, 16, device="cuda")
    padded[:, :c] = rand(n_ctr, c, 16) - 0.5
    out = {}
    for width in (c, 16):
        grads = padded[:, :width].contiguous()
        geometry = (stream(), cint(d), i64(n_ctr), ptr(ctr), cint(c), cint(width), ptr(grads),
                    i64(n_pts), ptr(pts), i64(n_pts * per), ptr(pairs), ptr(ranges), ptr(inv_radii))
        mc, kp = torch.empty(n_pts, c, device="cuda"), torch.empty(n_pts, c, device="cuda")
        _lib.call("mc_conv_gather_grads", *geometry, cint(1), cint(0), ptr(w), ptr(b), ptr(pdf),
                  ptr(None), cint(0), ptr(mc))
        _lib.call("kp_conv_gather_grads", *geometry, cint(15), ptr(kpts), cint(0), cfloat(1.0),
                  ptr(None), ptr(kp))
        out[width] = mc, kp
    for exact, whole in zip(out[c], out[16]):
        assert float(whole.abs().max()) > 0.0 and torch.equal(exact, whole)
