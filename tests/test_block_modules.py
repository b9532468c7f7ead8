"""Normalisation and activation of the residual blocks as modules of the caller's: hooks, subclasses
and forwards of their own are not passed by.  No GPU."""
import pytest
import torch

from tensorflow_graphics_point_clouds_amd import blocks


class _Shifted(blocks.BatchNorm):
    def forward(self, features, training=None):
        return super().forward(features, training) - 1.0


class _Clipped(torch.nn.LeakyReLU):
    def forward(self, x):
        return super().forward(x).clamp(max=0.5)


def _norm(kind=blocks.BatchNorm):
    return kind(3, device="cpu")


def _x():
    return torch.randn(20, 3, generator=torch.Generator().manual_seed(1))


def _expected(x):
    return torch.nn.functional.batch_norm(x, None, None, training=True, eps=1e-3)


def test_hooks_of_the_two_modules_fire_where_they_are():
    norm, act, x, seen = _norm(), torch.nn.LeakyReLU(0.3), _x().requires_grad_(), {}
    keep = lambda name, value: seen.update({name: value})             # (None: nothing changes)
    norm.register_forward_hook(lambda m, args, out: keep("norm", out))
    act.register_forward_hook(lambda m, args, out: keep("act", out))
    act.register_full_backward_hook(lambda m, gin, gout: keep("gradient", gin[0]))
    blocks._norm_act(norm, act, x, True).sum().backward()
    assert torch.allclose(seen["norm"], _expected(x), atol=1e-6)          # before the activation
    assert torch.allclose(seen["act"], torch.nn.functional.leaky_relu(seen["norm"], 0.3))
    assert torch.equal(seen["gradient"], torch.where(seen["norm"] > 0, 1.0, 0.3))


@pytest.mark.parametrize("norm,act,expect", [
    (_Shifted, torch.nn.ReLU(), lambda z: torch.relu(z - 1.0)),
    (blocks.BatchNorm, _Clipped(0.3), lambda z: torch.nn.functional.leaky_relu(z, 0.3).clamp(max=0.5)),
    (blocks.BatchNorm, torch.nn.LeakyReLU(-0.3), lambda z: torch.where(z > 0, z, -0.3 * z)),
    (blocks.BatchNorm, torch.relu, torch.relu)])
def test_forwards_of_subclasses_run(norm, act, expect):
    x = _x()
    assert torch.allclose(blocks._norm_act(_norm(norm), act, x, True), expect(_expected(x)), atol=1e-6)


@pytest.mark.parametrize("act", [torch.relu, torch.nn.ReLU()])
def test_relu_of_infinities_without_the_kernels(act):
    """Where torch's operations run instead of the kernels they are a ReLU's too: 0 at -inf, and
    the gradient of NaN passes."""
    norm = _norm().eval()
    x = torch.tensor([[-float("inf"), -1.0, 2.0], [float("nan"), float("inf"), 0.0]],
                     requires_grad=True)
    expect = act(norm(x))
    got = blocks._norm_act(norm, act, x)
    assert torch.equal(torch.nan_to_num(got, nan=-7.0), torch.nan_to_num(expect, nan=-7.0))
    want = torch.autograd.grad(expect.sum(), x)[0]
    assert torch.equal(torch.autograd.grad(got.sum(), x)[0], want)


def test_forward_of_an_instance_runs():
    act = torch.nn.ReLU()
    act.forward = lambda z: z * 2.0
    x = _x()
    assert torch.allclose(blocks._norm_act(_norm(), act, x, True), 2.0 * _expected(x), atol=1e-6)
