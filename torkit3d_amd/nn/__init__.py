"""The ``torkit3d.nn`` helpers the layers and models are built from: shared MLPs as
1x1 convolutions or linear layers with batch norm and ReLU
(torkit3d/nn/modules/conv.py, torkit3d/nn/modules/linear.py, torkit3d/nn/modules/mlp.py)
and ``batch_index_select`` (torkit3d/nn/functional.py:34-69). Modules and sub-module names
are the reference's, so that its checkpoints load; the shared MLPs run on fused kernels where
these take them (``SharedMLP``).
"""
import torch
from torch import nn
from torch.nn.modules.module import _has_any_global_hook

from .. import _native

__all__ = ["Conv1dBNReLU", "Conv2dBNReLU", "LinearBNReLU", "SharedMLP", "mlp_bn_relu", "mlp1d_bn_relu",
           "mlp2d_bn_relu", "batch_index_select"]


class _ConvBNReLU(nn.Module):
    conv_type = None
    bn_type = None

    def __init__(self, in_channels, out_channels, kernel_size, relu=True, bn=True, **kwargs):
        super().__init__()
        self.in_channels = in_channels
        self.out_channels = out_channels
        self.conv = self.conv_type(in_channels, out_channels, kernel_size, bias=(not bn),
                                   **kwargs)
        self.bn = self.bn_type(out_channels) if bn else None
        self.relu = nn.ReLU(inplace=True) if relu else None

    def forward(self, x):
        x = self.conv(x)
        if self.bn is not None:
            x = self.bn(x)
        if self.relu is not None:
            x = self.relu(x)
        return x


class Conv1dBNReLU(_ConvBNReLU):
    conv_type = nn.Conv1d
    bn_type = nn.BatchNorm1d
    ones, no_padding = (1,), (0,)


class Conv2dBNReLU(_ConvBNReLU):
    conv_type = nn.Conv2d
    bn_type = nn.BatchNorm2d
    ones, no_padding = (1, 1), (0, 0)


class LinearBNReLU(nn.Module):
    """``nn.Linear`` (named ``fc``), then optional batch norm and ReLU
    (torkit3d/nn/modules/linear.py:6-27); the bias is dropped when batch norm follows."""

    def __init__(self, in_channels, out_channels, relu=True, bn=True):
        super().__init__()
        self.in_channels = in_channels
        self.out_channels = out_channels
        self.fc = nn.Linear(in_channels, out_channels, bias=(not bn))
        self.bn = nn.BatchNorm1d(out_channels) if bn else None
        self.relu = nn.ReLU(inplace=True) if relu else None

    def forward(self, x):
        x = self.fc(x)
        if self.bn is not None:
            x = self.bn(x)
        if self.relu is not None:
            x = self.relu(x)
        return x


class SharedMLP(nn.Sequential):
    """The layers of ``mlp1d_bn_relu`` / ``mlp2d_bn_relu`` (an ``nn.Sequential`` to its
    checkpoints and to anything that walks its modules), run as one chain of fused kernels
    (csrc/mlp.hip) on float32 GPU tensors: in evaluation mode the products with their norms and
    maxima, in training mode the backward and what it needs of the forward (the activations stay
    those of the stock modules, bit by bit). Whatever is not plain - hooks, other modules in place
    of the blocks', frozen layers among training ones, autocast - runs layer by layer in stock
    torch."""

    def forward(self, input):
        if not torch.jit.is_scripting():
            out = self._chain(input)
            if out is not None:
                return out
        for module in self:
            input = module(input)
        return input

    def forward_cat(self, x, x2):
        """``self(torch.cat([x, x2], dim=1))`` without the concatenation."""
        out = self._chain(x, x2)
        return self(torch.cat([x, x2], dim=1)) if out is None else out

    def forward_max(self, x):
        """``self(x).max(dim=3)[0]`` for x [B, C, M, S]."""
        out = self._chain(x, pool=x.size(-1))
        return torch.max(self(x), dim=3)[0] if out is None else out

    def forward_points_max(self, x):
        """``torch.max(self(x), 2)`` for x [B, C, N]: values and places, [B, C'] each."""
        plan = self._plan(x)
        out = _native.mlp_max(x, *plan) if plan is not None and plan[-1] else None
        return (out[0], out[1]) if out else torch.max(self(x), 2)

    def forward_grouped_max(self, feature, xyz, centre, index):
        """``self(group_points_with_xyz(feature, xyz, centre, index)).max(dim=3)[0]``, or None
        where the fused chain does not take it."""
        if torch.is_grad_enabled() and (xyz.requires_grad or centre.requires_grad):
            return None
        return self._chain(feature, None, xyz, centre, index, pool=index.size(2))

    def forward_edges_max(self, x, index, lists=None):
        """A single layer on the edge features of x's graph with itself, then the maximum over
        the neighbours: x [B, C, N], index [B, N, K] -> [B, C', N]; ``lists`` is
        ``edge_lists(index, N)``. None where the fused kernels do not take it."""
        plan = self._plan(x) if len(self) == 1 else None
        if plan is None:
            return None
        params, buffers, (eps,), (momentum,), training = plan
        return _native.edge_conv(x, index, lists, params, buffers, eps, momentum, training)

    def _chain(self, x, x2=None, xyz=None, centre=None, index=None, pool=0):
        plan = self._plan(xyz if x is None else x)
        if plan is None:
            return None
        return _native.mlp(x, x2, xyz, centre, index, *plan, pool)

    def _plan(self, like):
        """(parameters, buffers, eps, momentum, training) of plain layers, or None."""
        if (type(like) not in _TENSORS  # (a tracer's proxy, a subclass)
                or not like.is_cuda or like.dtype != torch.float32 or torch.is_autocast_enabled()
                or torch.compiler.is_compiling() or torch.jit.is_tracing()
                or _has_any_global_hook() or type(self) is not SharedMLP or not _plain(self)):
            return None
        params, buffers, eps, momentum = [], [], [], []
        training = None
        for block in self._modules.values():
            if type(block) not in (Conv1dBNReLU, Conv2dBNReLU) or not _plain(block):
                return None
            conv, bn, relu = (block._modules.get(name) for name in ("conv", "bn", "relu"))
            if (type(conv) not in (nn.Conv1d, nn.Conv2d) or not _plain(conv)
                    or type(bn) not in (nn.BatchNorm1d, nn.BatchNorm2d) or not _plain(bn)
                    or type(relu) is not nn.ReLU or not _plain(relu)
                    or conv.groups != 1 or conv.padding != block.no_padding
                    or conv.kernel_size != block.ones or conv.stride != block.ones
                    or conv._parameters.get("bias") is not None or bn.momentum is None
                    # (the flag may be off although the buffers are there: training leaves them)
                    or (bn.training and not bn.track_running_stats)):
                return None
            if training is None:
                training = bn.training
            # (a replica of DataParallel holds its tensors as attributes: get() finds none)
            weight = conv._parameters.get("weight")
            gamma, beta = (bn._parameters.get(name) for name in ("weight", "bias"))
            mean, var, count = (bn._buffers.get(name) for name in
                                ("running_mean", "running_var", "num_batches_tracked"))
            if (training != bn.training or weight is None or gamma is None or beta is None
                    or mean is None or var is None):
                return None
            params += (weight, gamma, beta)
            buffers += (mean, var, count)
            eps.append(bn.eps)
            momentum.append(bn.momentum)
        return params, buffers, eps, momentum, bool(training)


_TENSORS = (torch.Tensor, nn.Parameter)


def _plain(module):
    return not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                or module._backward_pre_hooks or "forward" in module.__dict__)


# The forms of a shared MLP that layers call. A layer's MLP may also be a plain nn.Sequential: put
# there by hand, or from a model that was pickled as a whole before SharedMLP was there.

def forward_cat(mlp, x, x2):
    if isinstance(mlp, SharedMLP):
        return mlp.forward_cat(x, x2)
    return mlp(torch.cat([x, x2], dim=1))


def forward_max(mlp, x):
    if isinstance(mlp, SharedMLP):
        return mlp.forward_max(x)
    return torch.max(mlp(x), dim=3)[0]


def forward_points_max(mlp, x):
    if isinstance(mlp, SharedMLP):
        return mlp.forward_points_max(x)
    return torch.max(mlp(x), 2)


def forward_grouped_max(mlp, feature, xyz, centre, index):
    if isinstance(mlp, SharedMLP):
        return mlp.forward_grouped_max(feature, xyz, centre, index)
    return None


def forward_edges_max(mlp, x, index, lists=None):
    if isinstance(mlp, SharedMLP):
        return mlp.forward_edges_max(x, index, lists)
    return None


def _mlp(block, in_channels, out_channels_list):
    layers = []
    for out_channels in out_channels_list:
        layers.append(block(in_channels, out_channels, 1, relu=True))
        in_channels = out_channels
    return SharedMLP(*layers)


def mlp_bn_relu(in_channels, out_channels_list):
    layers = []
    for out_channels in out_channels_list:
        layers.append(LinearBNReLU(in_channels, out_channels, relu=True, bn=True))
        in_channels = out_channels
    return nn.Sequential(*layers)


def mlp1d_bn_relu(in_channels, out_channels_list):
    return _mlp(Conv1dBNReLU, in_channels, out_channels_list)


def mlp2d_bn_relu(in_channels, out_channels_list):
    return _mlp(Conv2dBNReLU, in_channels, out_channels_list)


def batch_index_select(input, index, dim):
    """Batched ``torch.index_select``: input [B, ...], index [B, N] or [B]."""
    squeeze = index.dim() == 1
    if squeeze:
        index = index.unsqueeze(1)
    assert index.dim() == 2, "index is expected to be 2-dim (or 1-dim), but %d received." % index.dim()
    assert input.size(0) == index.size(0), "Mismatched batch size: %d vs %d" % (
        input.size(0), index.size(0))
    view = [1] * input.dim()
    view[0], view[dim] = index.size(0), index.size(1)
    shape = list(input.shape)
    shape[dim] = -1
    out = torch.gather(input, dim, index.view(view).expand(shape))
    return out.squeeze(1) if squeeze else out
