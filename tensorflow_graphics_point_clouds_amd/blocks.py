"""Feature-space layers and residual blocks around the point convolutions
(pylib/pc/layers/Conv1x1.py:24-101, pylib/pc/layers/network_blocks.py:27-465).
Dense per-point work (a product, batch normalisation, an activation) on the
kernels of csrc/point_dense.hip where they cover the input, else on stock torch;
the spatial convolutions inside the blocks are the layers of `layers.py`."""
import math

import torch
from torch.autograd import forward_ad
from torch.nn.modules.module import _has_any_global_hook

from . import _lib, layers, pc

_F32 = torch.float32

layer_types = {"mcconv": layers.MCConv, "mc": layers.MCConv, "mc_conv": layers.MCConv,
               "kpconv": layers.KPConv, "kp": layers.KPConv, "kp_conv": layers.KPConv,
               "pointconv": layers.PointConv, "point_conv": layers.PointConv}


def _eager():
    """Whether nothing looks at the operations themselves: forward-mode derivatives, torch.func
    transforms, tracing and compilation see torch's operations, not the kernels' nodes."""
    return not (forward_ad._current_level >= 0 or torch._C._are_functorch_transforms_active() or
                torch.compiler.is_compiling() or torch.jit.is_tracing())


def _plain_rows(features):
    """float32 rows on the GPU that the per-point kernels take."""
    return (features.is_cuda and features.dtype == _F32 and features.dim() == 2 and
            features.is_contiguous() and type(features) in (torch.Tensor, torch.nn.Parameter) and
            not torch.is_autocast_enabled("cuda") and _eager())


def _bare(module, kind):
    """Whether calling the module is calling `kind`'s forward and nothing else: no hooks, no
    forward of a subclass or of the instance's own."""
    return (type(module).forward is kind.forward and "forward" not in module.__dict__ and
            not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or
                 module._backward_pre_hooks or _has_any_global_hook()))


def _leaky_slope(activation):
    """The slope for negative inputs of a leaky activation (0: ReLU) that keeps signs, as the
    gradients of the kernels need it, else None (a LeakyReLU of slope 0 is not a ReLU: infinities
    and NaN differ)."""
    if activation is torch.relu:
        return 0.0
    if isinstance(activation, torch.nn.ReLU) and _bare(activation, torch.nn.ReLU):
        return 0.0
    if (isinstance(activation, torch.nn.LeakyReLU) and _bare(activation, torch.nn.LeakyReLU) and
            activation.negative_slope > 0):
        return activation.negative_slope
    return None


def _norm_act(norm, activation, features, training=None):
    """activation(norm(features)), in the kernel of the normalisation if nothing looks between
    the two or at either of them."""
    slope = _leaky_slope(activation)
    if slope is None or not (isinstance(norm, BatchNorm) and _bare(norm, BatchNorm)):
        return activation(norm(features, training))
    return norm(features, training, slope)


def _identity(features, *args, **kwargs):
    return features


class BatchNorm(torch.nn.BatchNorm1d):
    """Batch normalisation over the points with Keras' defaults (moving-average
    momentum 0.99, epsilon 1e-3; torch counts the momentum from the other side).
    `training`, when given, overrides the module's train/eval mode, as the
    reference passes it per call.  `negative_slope` applies a leaky ReLU of that
    slope (0: ReLU) to the result."""

    def __init__(self, num_features, momentum=0.99, eps=1e-3, device="cuda"):
        super().__init__(num_features, eps=eps, momentum=1.0 - momentum, device=device)

    def forward(self, features, training=None, negative_slope=None):
        training = self.training if training is None else bool(training)
        weight, bias = self.weight, self.bias
        if (_plain_rows(features) and features.shape[1] == self.num_features and
                features.shape[0] > 1 and weight is not None and bias is not None and
                self.momentum is not None and self.running_mean is not None and
                weight.dtype == bias.dtype == self.running_mean.dtype == _F32 and
                weight.device == features.device and
                weight.is_contiguous() and bias.is_contiguous() and
                (negative_slope is None or negative_slope >= 0)):
            return _lib.host().norm_act(features, weight, bias, self.running_mean,
                                        self.running_var, self.num_batches_tracked, training,
                                        self.momentum, self.eps,
                                        1.0 if negative_slope is None else negative_slope)
        out = self._forward(features, training)
        if negative_slope is None:
            return out
        if negative_slope == 0:                    # (a leaky ReLU of slope 0 makes NaN of -inf)
            return torch.relu(out)
        return torch.nn.functional.leaky_relu(out, negative_slope)

    def _forward(self, features, training):
        if training == self.training:
            return super().forward(features)
        mode = self.training
        self.train(training)
        try:
            return super().forward(features)
        finally:
            self.train(mode)


class Conv1x1(torch.nn.Module):
    """Per-point linear map features [N, C_in] -> [N, C_out] with a bias
    (Conv1x1.py:24-101): truncated-normal weights of scale sqrt(2 / C_in), zero
    bias."""

    def __init__(self, num_features_in, num_features_out, use_bias=True, device="cuda", seed=0):
        super().__init__()
        gen = torch.Generator().manual_seed(seed)
        w = layers._truncated_normal((num_features_in, num_features_out),
                                     math.sqrt(2.0 / float(num_features_in)), gen, device)
        self.weights = torch.nn.Parameter(w)
        self.bias = torch.nn.Parameter(torch.zeros((1, num_features_out), dtype=_F32,
                                                   device=device)) if use_bias else None

    def forward(self, features, point_cloud, return_sorted=False, return_padded=False):
        features = point_cloud.flatten_features(features)
        if (_plain_rows(features) and features.shape[1] == self.weights.shape[0] and
                self.weights.dtype == _F32 and self.weights.device == features.device and
                self.weights.is_contiguous()):
            out = _lib.host().linear(features, self.weights, self.bias)
        else:
            out = features @ self.weights
            if self.bias is not None:
                out = out + self.bias
        return point_cloud.format_output(out, return_sorted, return_padded)


def _own_neighborhood(point_cloud, radius, num_dims):
    radii = pc._as_vector(radius, num_dims, point_cloud._points.device)
    return pc.Neighborhood(pc.Grid(point_cloud, radii), radii, point_cloud)


class PointResNet(torch.nn.Module):
    """Pre-activation residual blocks of two point convolutions on one cloud
    (network_blocks.py:27-151).  `kwargs` go to the convolution layers."""

    def __init__(self, num_features, num_blocks, num_dims, layer_type="MCConv",
                 projection_shortcuts=False, activation=torch.relu, device="cuda", **kwargs):
        super().__init__()
        self._num_dims, self._num_blocks, self._activation = num_dims, num_blocks, activation
        conv = layer_types[layer_type.lower()]
        self._batch_norm_layers = torch.nn.ModuleList(
            BatchNorm(num_features, device=device) for _ in range(2 * num_blocks))
        self._conv_layers = torch.nn.ModuleList(
            conv(num_features, num_features, num_dims=num_dims, device=device, seed=i, **kwargs)
            for i in range(2 * num_blocks))
        self._projection_layers = torch.nn.ModuleList(
            Conv1x1(num_features, num_features, device=device, seed=100 + i)
            for i in range(num_blocks)) if projection_shortcuts else None

    def forward(self, features, point_cloud, radius, training=None, neighborhood=None,
                return_sorted=False, return_padded=False, **kwargs):
        features = point_cloud.flatten_features(features)
        if neighborhood is None:
            neighborhood = _own_neighborhood(point_cloud, radius, self._num_dims)
        for i in range(self._num_blocks):
            skip = features
            for j in (2 * i, 2 * i + 1):
                features = _norm_act(self._batch_norm_layers[j], self._activation, features, training)
                features = self._conv_layers[j](features, point_cloud, point_cloud, radius,
                                                neighborhood, **kwargs)
            if self._projection_layers is not None:
                skip = self._projection_layers[i](skip, point_cloud)
            features = features + skip
        return point_cloud.format_output(features, return_sorted, return_padded)


class PointResNetBottleNeck(torch.nn.Module):
    """Residual blocks whose point convolution runs on fewer channels: 1x1 down,
    convolution, 1x1 up, each after batch normalisation and the activation
    (network_blocks.py:153-298)."""

    def __init__(self, num_features, bottle_neck_num_features, num_blocks, num_dims,
                 layer_type="MCConv", projection_shortcuts=False, activation=torch.relu,
                 device="cuda", **kwargs):
        super().__init__()
        self._num_dims, self._num_blocks, self._activation = num_dims, num_blocks, activation
        conv = layer_types[layer_type.lower()]
        inner = bottle_neck_num_features
        widths = (num_features, inner, inner)
        self._batch_norm_layers = torch.nn.ModuleList(
            BatchNorm(widths[j % 3], device=device) for j in range(3 * num_blocks))
        self._downsampling_layers = torch.nn.ModuleList(
            Conv1x1(num_features, inner, device=device, seed=200 + i) for i in range(num_blocks))
        self._conv_layers = torch.nn.ModuleList(
            conv(inner, inner, num_dims=num_dims, device=device, seed=i, **kwargs)
            for i in range(num_blocks))
        self._upsampling_layers = torch.nn.ModuleList(
            Conv1x1(inner, num_features, device=device, seed=300 + i) for i in range(num_blocks))
        self._projection_layers = torch.nn.ModuleList(
            Conv1x1(num_features, num_features, device=device, seed=100 + i)
            for i in range(num_blocks)) if projection_shortcuts else None

    def forward(self, features, point_cloud, radius, training=None, neighborhood=None,
                return_sorted=False, return_padded=False, **kwargs):
        features = point_cloud.flatten_features(features)
        if neighborhood is None:
            neighborhood = _own_neighborhood(point_cloud, radius, self._num_dims)
        bn, act = self._batch_norm_layers, self._activation
        for i in range(self._num_blocks):
            skip = features
            features = self._downsampling_layers[i](
                _norm_act(bn[3 * i], act, features, training), point_cloud)
            features = self._conv_layers[i](_norm_act(bn[3 * i + 1], act, features, training),
                                            point_cloud, point_cloud, radius, neighborhood,
                                            **kwargs)
            features = self._upsampling_layers[i](
                _norm_act(bn[3 * i + 2], act, features, training), point_cloud)
            if self._projection_layers is not None:
                skip = self._projection_layers[i](skip, point_cloud)
            features = features + skip
        return point_cloud.format_output(features, return_sorted, return_padded)


class PointResNetSpatialBottleNeck(torch.nn.Module):
    """Residual blocks with a bottleneck in space: a convolution onto a
    down-sampled cloud, one inside it, one back onto the full cloud
    (network_blocks.py:300-465).  `conv_radii` holds the three radii in that
    order; `neighborhoods`, when given, the three matching neighbourhoods.  When
    the first and the last radius agree the way back is the transpose of the way
    down and no third search is made."""

    def __init__(self, num_features, num_blocks, num_dims, layer_type="MCConv",
                 projection_shortcuts=False, activation=torch.relu, device="cuda", **kwargs):
        super().__init__()
        self._num_dims, self._num_blocks, self._activation = num_dims, num_blocks, activation
        conv = layer_types[layer_type.lower()]
        self._batch_norm_layers = torch.nn.ModuleList(
            BatchNorm(num_features, device=device) for _ in range(3 * num_blocks))
        self._stage_layers = torch.nn.ModuleList(
            conv(num_features, num_features, num_dims=num_dims, device=device, seed=i, **kwargs)
            for i in range(3 * num_blocks))
        self._projection_layers = torch.nn.ModuleList(
            Conv1x1(num_features, num_features, device=device, seed=100 + i)
            for i in range(num_blocks)) if projection_shortcuts else None

    def forward(self, features, point_cloud, point_cloud_downsampled, conv_radii, training=None,
                neighborhoods=None, return_sorted=False, return_padded=False, **kwargs):
        features = point_cloud.flatten_features(features)
        radii = [float(r) for r in torch.as_tensor(conv_radii).reshape(-1).tolist()]
        if len(radii) != 3:
            raise ValueError("conv_radii holds three radii: down, inside, up")
        d, dev = self._num_dims, features.device
        if neighborhoods is None:
            vec = [pc._as_vector(r, d, dev) for r in radii]
            down = pc.Neighborhood(pc.Grid(point_cloud, vec[0]), vec[0], point_cloud_downsampled)
            inside = pc.Neighborhood(pc.Grid(point_cloud_downsampled, vec[1]), vec[1],
                                     point_cloud_downsampled)
            if radii[0] == radii[2]:
                up = down.transpose()
            else:
                up = pc.Neighborhood(pc.Grid(point_cloud_downsampled, vec[2]), vec[2],
                                     point_cloud)
            neighborhoods = [down, inside, up]
        clouds = [(point_cloud, point_cloud_downsampled),
                  (point_cloud_downsampled, point_cloud_downsampled),
                  (point_cloud_downsampled, point_cloud)]
        for i in range(self._num_blocks):
            skip = features
            for stage in range(3):
                j = 3 * i + stage
                features = _norm_act(self._batch_norm_layers[j], self._activation, features, training)
                features = self._stage_layers[j](features, clouds[stage][0], clouds[stage][1],
                                                 radii[stage], neighborhoods[stage], **kwargs)
            if self._projection_layers is not None:
                skip = self._projection_layers[i](skip, point_cloud)
            features = features + skip
        return point_cloud.format_output(features, return_sorted, return_padded)
