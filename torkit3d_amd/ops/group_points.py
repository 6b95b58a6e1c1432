"""Group (gather) point features by neighbour index (API of torkit3d/ops/group_points.py)."""
import torch

from .. import _C, _native


class GroupPointsFunction(torch.autograd.Function):
    """forward(points, index) -> grouped; backward -> (grad_points, None)
    (torkit3d/ops/group_points.py:6-19)."""

    @staticmethod
    def forward(ctx, points, index):
        ctx.save_for_backward(index)
        ctx.num_points = points.size(2)
        return _C.group_points_forward_cuda(points.contiguous(), index.contiguous())

    @staticmethod
    def backward(ctx, *grad_output):
        (index,) = ctx.saved_tensors
        grad_input = _C.group_points_backward_cuda(
            grad_output[0].contiguous(), index.contiguous(), ctx.num_points)
        return grad_input, None


def group_points(points, index):
    """points [B, C, N1], index [B, N2, K] -> [B, C, N2, K] with
    out[b, c, m, s] = points[b, c, index[b, m, s]]."""
    if not _native.direct(points, index):
        return GroupPointsFunction.apply(points, index)
    return _native.group_points(points, index)


def group_points_with_xyz(feature, xyz, centre, index):
    """The grouping step of the reference's SetAbstraction with ``use_xyz``
    (torkit3d/layers/pointnet2.py:46-58) as one op: equal to
    ``torch.cat([group_points(feature, index), group_points(xyz, index) -
    centre.unsqueeze(-1)], dim=1)``, written once.

    Args:
        feature: [B, C, N1] or None; xyz: [B, 3, N1]; centre: [B, 3, N2];
        index: [B, N2, K] int64.
    """
    if not _native.direct(feature, xyz, centre, index):
        grouped = GroupPointsFunction.apply(xyz, index) - centre.unsqueeze(-1)
        if feature is None:
            return grouped
        return torch.cat([GroupPointsFunction.apply(feature, index), grouped], dim=1)
    return _native.group_points_with_xyz(feature, xyz, centre, index)

gather_points = group_points  # the spelling common elsewhere
