"""Normalisation + activation and the per-point linear map at the edges of their kernels (a point
more or less than a slab or tile, widths that are no multiple of 4 or 64), against float64."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _rand(*shape, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=gen)


@pytest.mark.parametrize("n,c,training,slope", [
    (2, 3, True, 1.0), (64, 64, True, 0.3), (65, 6, True, 0.0), (1025, 68, True, 0.3),
    (16384, 16, True, 0.3), (16385, 130, True, 0.0), (140001, 20, True, 0.3), (1, 8, False, 0.3),
    (777, 65, False, 0.0)])
def test_norm_act(n, c, training, slope):
    from tensorflow_graphics_point_clouds_amd import blocks
    x, g = _rand(n, c, seed=n) * 2 + 3, _rand(n, c, seed=c)
    norm = blocks.BatchNorm(c)
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5)
        norm.bias.normal_()
        norm.running_mean.normal_()
        norm.running_var.uniform_(0.5, 2.0)
    ref = torch.nn.BatchNorm1d(c, eps=norm.eps, momentum=norm.momentum, device="cuda")
    ref.load_state_dict(norm.state_dict())
    ref = ref.double().train(training)
    a, b = x.clone().requires_grad_(), x.double().requires_grad_()
    out = norm(a, training, slope)
    out.backward(g)
    z = ref(b)
    z.retain_grad()
    # the activation of the float32 pass decides on which side of 0 a point lies
    expect = torch.where(out.detach() > 0, z, slope * z)
    expect.backward(g.double())
    # A result is a handful of float32 roundings of terms of the size of |x| inv w (forward) and
    # |g| inv w (backward): x, mean and inv are off by 2^-24 each and meet twice.
    inv = 1 / torch.sqrt((b.detach().var(0, unbiased=False) if training else
                          norm.running_var.double()) + norm.eps)
    size = (b.detach().abs() + 3) * inv * norm.weight.double().detach() + norm.bias.double().abs()
    assert torch.all((out.double() - expect).abs() <= 16 * EPS * size)
    gsize = (g.double().abs() + 3) * inv * norm.weight.double().detach() * (1 + z.detach().abs())
    assert torch.all((a.grad.double() - b.grad).abs() <= 64 * EPS * gsize)
    for p, q in ((norm.weight.grad, ref.weight.grad), (norm.bias.grad, ref.bias.grad)):
        # n terms of |g| (1 + |xhat|), at most 64 of them added one after the other per lane
        bound = 64 * EPS * (g.double().abs() * (4 + (b.detach().abs() + 3) * inv)).sum(0)
        assert torch.all((p.double() - q).abs() <= bound)
    for name in ("running_mean", "running_var"):
        p, q = getattr(norm, name).double(), getattr(ref, name)
        assert torch.all((p - q).abs() <= 16 * EPS * (q.abs() + 4))
    assert int(norm.num_batches_tracked) == int(ref.num_batches_tracked) == int(training)


@pytest.mark.parametrize("form", ["no bias", "strided"])
def test_norm_act_with_parameters_that_only_torch_takes(form):
    from tensorflow_graphics_point_clouds_amd import blocks
    norm = blocks.BatchNorm(6)
    ref = torch.nn.BatchNorm1d(6, eps=norm.eps, momentum=norm.momentum, device="cuda")
    if form == "no bias":
        norm.bias = ref.bias = None
    else:
        norm.weight = torch.nn.Parameter(_rand(6, 2, seed=1)[:, 0])
        ref.weight = torch.nn.Parameter(norm.weight.detach().clone())
    x, g = _rand(50, 6, seed=2).requires_grad_(), _rand(50, 6, seed=3)
    results = []
    for out in (blocks._norm_act(norm, torch.relu, x), torch.relu(ref(x))):
        wanted = [x] + list((norm if not results else ref).parameters())
        results.append([out.detach(), *torch.autograd.grad(out, wanted, g)])
    for a, b in zip(*results):       # (torch has two kernels of its own: sums of 50 terms)
        assert (a - b).norm() <= 64 * EPS * b.norm()


@pytest.mark.parametrize("n,r,f,bias", [
    (1, 1, 1, True), (31, 8, 16, True), (33, 36, 60, False), (127, 64, 64, True),
    (129, 65, 67, True), (4097, 256, 72, True), (5000, 3, 130, True), (0, 8, 4, True)])
def test_linear(n, r, f, bias):
    from tensorflow_graphics_point_clouds_amd import _lib
    x, w, b, g = (_rand(n, r, seed=1), _rand(r, f, seed=2), _rand(1, f, seed=3),
                  _rand(n, f, seed=4))
    leaves = [t.clone().requires_grad_() for t in (x, w, b)]
    out = _lib.host().linear(leaves[0], leaves[1], leaves[2] if bias else None)
    out.backward(g)
    # a sum of m products is off by less than (m + 2) 2^-24 times the sum of their sizes
    def close(got, expect, size, terms):
        assert torch.all((got.double() - expect).abs() <= (terms + 2) * EPS * size)
    x, w, b, g = (t.double() for t in (x, w, b, g))
    shift = b if bias else torch.zeros_like(b)
    close(out, x @ w + shift, x.abs() @ w.abs() + shift.abs(), r)
    close(leaves[0].grad, g @ w.t(), g.abs() @ w.abs().t(), f)
    close(leaves[1].grad, x.t() @ g, x.abs().t() @ g.abs(), n)
    if bias:
        close(leaves[2].grad, g.sum(0, keepdim=True), g.abs().sum(0, keepdim=True), n)


def test_second_derivatives():
    """The layers stay differentiable twice."""
    from tensorflow_graphics_point_clouds_amd import _lib, blocks
    norm = blocks.BatchNorm(5)
    x, w = _rand(40, 5).requires_grad_(), _rand(5, 4, seed=1).requires_grad_()
    out = _lib.host().linear(norm(x, True, 0.3), w, None)
    first, = torch.autograd.grad(out.square().sum(), x, create_graph=True)
    second, = torch.autograd.grad(first.square().sum(), w)
    y = torch.nn.functional.leaky_relu(torch.nn.functional.batch_norm(
        x, None, None, norm.weight, norm.bias, True, 0.0, norm.eps), 0.3) @ w
    expect, = torch.autograd.grad(y.square().sum(), x, create_graph=True)
    second_expect, = torch.autograd.grad(expect.square().sum(), w)
    assert torch.allclose(first, expect, rtol=1e-4, atol=1e-4)
    assert torch.allclose(second, second_expect, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("slope", [-0.3, -1.0, 0.0, 0.3])
def test_activation_of_any_slope(slope):
    """An activation that does not keep signs (a negative slope) has its gradient taken from its
    input: first and second derivatives against torch's operations in float64."""
    from tensorflow_graphics_point_clouds_amd import blocks
    x, g = _rand(300, 6, seed=1) * 2 + 1, _rand(300, 6, seed=2)
    norm, act = blocks.BatchNorm(6), torch.nn.LeakyReLU(slope)
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5)
        norm.bias.normal_()

    def derivatives(x, weight, bias, result):
        first = torch.autograd.grad(result, (x, weight, bias), g.to(result.dtype),
                                    create_graph=True)
        return list(first) + list(torch.autograd.grad(first[0].square().sum(), (x, weight)))
    a = x.clone().requires_grad_()
    got = derivatives(a, norm.weight, norm.bias, blocks._norm_act(norm, act, a, True))
    b, w, c = (t.detach().double().requires_grad_() for t in (x, norm.weight, norm.bias))
    expect = derivatives(b, w, c, torch.nn.functional.leaky_relu(torch.nn.functional.batch_norm(
        b, None, None, w, c, True, 0.0, norm.eps), slope))
    for p, q in zip(got, expect):
        # chains of some ten float32 roundings, the second derivatives of sums of 300 terms
        assert (p.double() - q).norm() <= 1e-5 * q.norm()


def test_transforms_see_torch_operations():
    """Forward-mode derivatives and torch.func transforms through the layers, against the same on
    the CPU."""
    from tensorflow_graphics_point_clouds_amd import blocks, pc
    x, t = _rand(50, 6, seed=1), _rand(50, 6, seed=2)

    def derivatives(device):
        norm, lin = blocks.BatchNorm(6, device=device), blocks.Conv1x1(6, 4, device=device, seed=3)
        points = torch.zeros(50, 3, device=device)
        cloud = pc.PointCloud(points, torch.zeros(50, dtype=torch.int32, device=device), 1)
        f = lambda v: lin(blocks._norm_act(norm, torch.nn.LeakyReLU(0.3), v, False), cloud)
        a, b = x.to(device), t.to(device)
        _, tangent = torch.func.jvp(f, (a,), (b,))
        gradient = torch.func.grad(lambda v: f(v).square().sum())(a)
        with torch.autograd.forward_ad.dual_level():
            dual = f(torch.autograd.forward_ad.make_dual(a, b))
            again = torch.autograd.forward_ad.unpack_dual(dual).tangent
        many = torch.func.vmap(f)(torch.stack([a, b]))
        return [v.detach().cpu() for v in (tangent, gradient, again, many)]
    for got, expect in zip(derivatives("cuda"), derivatives("cpu")):
        assert torch.allclose(got, expect, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("act", [torch.relu, torch.nn.ReLU(), torch.nn.LeakyReLU(0.3),
                                 torch.nn.LeakyReLU(0.0)])
@pytest.mark.parametrize("training", [False, True])
def test_infinities_and_nan_take_the_gradient_of_torch(act, training):
    """Against torch's own operations on the same float32 values; with given statistics a point
    that is not finite leaves the gradients of the others alone."""
    from tensorflow_graphics_point_clouds_amd import blocks
    x, g = _rand(70, 8, seed=1), _rand(70, 8, seed=2)
    x[3, 0], x[4, 1], x[5, 2] = float("nan"), float("inf"), -float("inf")
    norm = blocks.BatchNorm(8)
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5)
        norm.running_mean.normal_()
        norm.running_var.uniform_(0.5, 2.0)
    plain = torch.nn.BatchNorm1d(8, eps=norm.eps, device="cuda")
    plain.load_state_dict(norm.state_dict())
    results = []
    for module, call in ((norm, lambda v: blocks._norm_act(norm, act, v, training)),
                         (plain, lambda v: act(plain.train(training)(v)))):
        a = x.clone().requires_grad_()
        out = call(a)
        out.backward(g)
        results.append((out.detach(), a.grad, module.weight.grad, module.bias.grad))
    for got, expect in zip(*results):       # sums of 70 terms in float32, elsewhere a few roundings
        assert torch.allclose(got, expect, rtol=1e-5, atol=1e-4, equal_nan=True)
