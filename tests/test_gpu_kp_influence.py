"""The linear influence of a kernel point as the projection kernel evaluates it: points on the
kernel points and next to them, at the edge of the influence, and small and large ones."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [0.02, 0.3, 1.0 / 3.0, 0.7, 40.0])
def test_influence_matches_float64(sigma):
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cfloat, cint, i64, ptr, stream
    gen = torch.Generator(device="cuda").manual_seed(int(100 * sigma))
    n, kp = 4096, 15
    kpts = (torch.rand(kp, 3, device="cuda", generator=gen) - 0.5) * sigma
    # around a kernel point at distances from 0 and 1e-12 up to the influence and a last place beyond
    near = kpts[torch.randint(0, kp, (n,), device="cuda", generator=gen)]
    way = torch.nn.functional.normalize(torch.randn(n, 3, device="cuda", generator=gen), dim=1)
    step = sigma * 10.0 ** (-12.0 * torch.rand(n, 1, device="cuda", generator=gen))
    step[::5], step[1::5] = 0.0, sigma
    points = (near + way * step).contiguous()
    centres = torch.zeros(n, 3, device="cuda")
    pairs = torch.arange(n, device="cuda", dtype=torch.int32)[:, None].expand(-1, 2).contiguous()
    ranges = torch.arange(1, n + 1, device="cuda", dtype=torch.int32)
    ones, feat = torch.ones(3, device="cuda"), torch.zeros(n, 16, device="cuda")
    feat[:, 0] = 1.0
    out = torch.empty(n, 16, 16, device="cuda")
    _lib.call("kp_conv_project", stream(), cint(3), i64(n), ptr(points), cint(16), ptr(feat), i64(n),
              ptr(centres), i64(n), ptr(pairs), ptr(ranges), ptr(ones), cint(kp), ptr(kpts), cint(0),
              cfloat(sigma), ptr(None), ptr(out))
    s = torch.tensor(sigma, dtype=torch.float32).double().item()
    dist = (points.double()[:, None] - kpts.double()[None]).norm(dim=2)
    want = (1.0 - dist / s).clamp(min=0.0)
    # rounded: the difference of the coordinates (half a last place of it), three squares and
    # two sums, root, quotient, 1 - quotient: below 5 of dist / sigma and one of the result
    bound = 2.0 ** -24 * (10 * dist / s + 2)
    assert bool(((out[:, 0, :kp].double() - want).abs() <= bound).all())
    assert float(out[:, 1:].abs().max()) == 0.0 and float(out[:, 0, kp:].abs().max()) == 0.0


@pytest.mark.parametrize("sigma", [1e29, 2e30, 3e38, float("inf")])
def test_influence_without_an_edge(sigma):
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cfloat, cint, i64, ptr, stream
    gen = torch.Generator(device="cuda").manual_seed(3)
    n, kp = 64, 15
    kpts = torch.rand(kp, 3, device="cuda", generator=gen)
    points = torch.rand(n, 3, device="cuda", generator=gen)
    points[:kp] = kpts
    pairs = torch.arange(n, device="cuda", dtype=torch.int32)[:, None].expand(-1, 2).contiguous()
    ranges = torch.arange(1, n + 1, device="cuda", dtype=torch.int32)
    out = torch.empty(n, 16, 16, device="cuda")
    feat, centres = torch.ones(n, 16, device="cuda"), torch.zeros(n, 3, device="cuda")
    ones = torch.ones(3, device="cuda")
    _lib.call("kp_conv_project", stream(), cint(3), i64(n), ptr(points), cint(16), ptr(feat), i64(n),
              ptr(centres), i64(n), ptr(pairs), ptr(ranges), ptr(ones), cint(kp), ptr(kpts), cint(0),
              cfloat(sigma), ptr(None), ptr(out))
    assert bool((out[:, :, :kp] == 1.0).all())


@pytest.mark.parametrize("step,expect", [(1e-12, -2.0), (3e-16, -2.0), (1e-18, -2.0), (0.0, 0.0),
                                         (0.4, -2.0), (0.6, 0.0), (1e20, 0.0)])
def test_offset_gradient_of_any_distance(step, expect):
    """d influence / d distance is -1 / sigma inside the influence, at any distance but none."""
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cfloat, cint, i64, ptr, stream
    n, kp, sigma = 40, 15, 0.5
    zeros = torch.zeros(n, 3, device="cuda")
    pairs = torch.arange(n, device="cuda", dtype=torch.int32)[:, None].expand(-1, 2).contiguous()
    ranges = torch.arange(1, n + 1, device="cuda", dtype=torch.int32)
    offsets = torch.zeros(n, kp, 3, device="cuda")
    offsets[:, :, 0] = -step                         # the points lie at +step of the kernel points
    feat = torch.zeros(n, 16, device="cuda")
    feat[:, 0] = 1.0
    upstream = torch.ones(n, 16, 16, device="cuda")
    out = torch.empty(n, kp, 3, device="cuda")
    ones, kpts = torch.ones(3, device="cuda"), torch.zeros(kp, 3, device="cuda")
    _lib.call("kp_deform_offset_grads", stream(), cint(3), i64(n), ptr(zeros), cint(16), ptr(feat),
              i64(n), ptr(zeros), i64(n), ptr(pairs), ptr(ranges), ptr(ones), cint(kp), ptr(kpts),
              cint(0), cfloat(sigma), ptr(offsets), ptr(upstream), ptr(out))
    # moving a kernel point towards the point (+x) raises the influence by 1 / sigma
    want = torch.zeros_like(out)
    want[:, :, 0] = -expect
    assert torch.allclose(out, want, rtol=4 * 2.0 ** -23, atol=0.0)



@pytest.mark.parametrize("up", [1.0, -3.0, 1e38, float("inf")])
def test_offset_gradient_beside_the_corrections(up):
    """Distances whose square is subnormal, and gradients that are infinite or become so by the
    division: as sqrtf and the division give them."""
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cfloat, cint, i64, ptr, stream
    sigma = np.float32(0.5)
    x = np.float32([0.0, 1e-24, 3e-23, 1e-20, -7e-20, 1e-19, 2e-19, 1e-17, 1e-15, -1.1e-15, 1e-6, -0.3,
                    0.4, 0.499, 0.5, 0.7, 1e19, 3e19])
    n, kp = len(x), 15
    zeros, ones = torch.zeros(n, 3, device="cuda"), torch.ones(3, device="cuda")
    # each pair sixteen times, which fills a tile (empty places are multiplied by 0)
    pairs = torch.arange(16 * n, device="cuda").div(16, rounding_mode="floor").int()
    pairs = pairs[:, None].expand(-1, 2).contiguous()
    ranges = 16 * torch.arange(1, n + 1, device="cuda", dtype=torch.int32)
    offsets = torch.zeros(n, kp, 3, device="cuda")
    offsets[:, :, 0] = -torch.from_numpy(x).cuda()[:, None]
    feat, kpts = torch.ones(n, 16, device="cuda"), torch.zeros(kp, 3, device="cuda")
    upstream = torch.zeros(n, 16, 16, device="cuda")
    upstream[:, 0] = up
    out = torch.empty(n, kp, 3, device="cuda")
    _lib.call("kp_deform_offset_grads", stream(), cint(3), i64(n), ptr(zeros), cint(16), ptr(feat),
              i64(n), ptr(zeros), i64(16 * n), ptr(pairs), ptr(ranges), ptr(ones), cint(kp), ptr(kpts),
              cint(0), cfloat(sigma), ptr(offsets), ptr(upstream), ptr(out))
    with np.errstate(all="ignore"):
        dist = np.sqrt(x * x)
        slope = np.where(dist < sigma, -1 / sigma, np.float32(0.0))
        coef = np.where(dist > 0, -np.float32(up) * slope / dist, np.float32(0.0)).astype(np.float32)
        want = np.broadcast_to((16 * (coef * x))[:, None], (n, kp))
    got = out[:, :, 0].cpu().numpy()
    # (a quotient and a product, each rounded once; sixteen times it is exact)
    assert np.allclose(got, want, rtol=2 * 2.0 ** -23, atol=0.0, equal_nan=True)
    finite = np.isfinite(coef)                       # (infinite: times 0 in the other coordinates)
    assert float(out[:, :, 1:].cpu()[finite].abs().max()) == 0.0


@pytest.mark.parametrize("deformed", [False, True])
@pytest.mark.parametrize("sigma", [1.0, 1.0 / 3.0, 0.07, 1e30, 2e30, 1.01e-7, 0.99e-7, 1e-8, 1e-15, 1e-16,
                                   1e-20, 1e-39])
def test_influence_has_the_bits_of_root_and_quotient(sigma, deformed):
    """1 - sqrt(sq) / sigma with root and quotient correctly rounded, for random mantissas of the
    distance and for influences as small as any that is accepted."""
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cfloat, cint, i64, ptr, stream
    gen = torch.Generator().manual_seed(7)
    n = 1 << 16
    s = torch.tensor(sigma, dtype=torch.float32)
    x = (s.double() * torch.rand(n, generator=gen, dtype=torch.float64)).float()
    # down to a millionth of the influence, none, its edge, and fixed small ones
    x[::3] = (x[::3].double() * 10.0 ** (-6.0 * torch.rand(x[::3].numel(), generator=gen,
                                                           dtype=torch.float64))).float()
    x[:6] = torch.tensor([0.0, 5e-16, 1e-15, 1e-18, sigma, 2.0 * sigma])
    # (numpy: torch's root on the CPU is off by a last place now and then)
    want = np.maximum(np.float32(1.0) - np.sqrt(x.numpy() * x.numpy()) / s.numpy(), np.float32(0.0))
    points = torch.zeros(n, 3, device="cuda")
    points[:, 0] = x.cuda()
    pairs = torch.arange(n, device="cuda", dtype=torch.int32)[:, None].expand(-1, 2).contiguous()
    ranges = torch.arange(1, n + 1, device="cuda", dtype=torch.int32)
    ones, zeros = torch.ones(3, device="cuda"), torch.zeros(n, 3, device="cuda")
    feat, out = torch.zeros(n, 16, device="cuda"), torch.empty(n, 16, 16, device="cuda")
    feat[:, 0] = 1.0
    kernel_point = torch.zeros(1, 3, device="cuda")
    geometry = (stream(), cint(3), i64(n), ptr(points), cint(16), ptr(feat), i64(n), ptr(zeros), i64(n),
                ptr(pairs), ptr(ranges), ptr(ones), cint(1), ptr(kernel_point), cint(0), cfloat(sigma))
    if deformed:
        _lib.call("kp_deform_project", *geometry, ptr(zeros), cint(0), ptr(None), ptr(out))
    else:
        _lib.call("kp_conv_project", *geometry, ptr(None), ptr(out))
    assert np.array_equal(out[:, 0, 0].cpu().numpy(), want)
