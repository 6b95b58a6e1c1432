"""Entry points of ``include/tk3d.h`` that have no counterpart among the nine
``torkit3d._C`` functions: they fuse steps the reference performs in Python
around those functions (layout copies, coordinate gathers, concatenation, weight
arithmetic). Same conventions as ``_C``; the work is in the extension module ``_native``.
"""
import torch  # noqa: F401

from . import _native

__all__ = [
    "sample_farthest_points_gather",
    "ball_query_bcn",
    "knn_distance_bcn",
    "chamfer_forward_bcn",
    "group_points_concat_forward",
    "group_points_concat_backward",
    "three_nn",
]


def sample_farthest_points_gather(points, num_samples, channels_first, want_xyz=True):
    """points [B,N,3] (or [B,3,N] with ``channels_first``) -> (index [B,K] int64,
    sampled [B,K,3] (or [B,3,K]) or None). ``index`` equals
    ``_C.sample_farthest_points_cuda`` on the [B,N,3] cloud."""
    return _native.sample_farthest_points(points, int(num_samples), bool(channels_first),
                                          bool(want_xyz))


def ball_query_bcn(query, key, radius, max_neighbors):
    """query [B,3,N1], key [B,3,N2] -> index [B,N1,max_neighbors] int64; equals
    ``_C.ball_query_cuda`` on the transposed clouds."""
    return _native.ball_query(query, key, float(radius), int(max_neighbors), True)


def knn_distance_bcn(query, key, k, version):
    """query [B,3,N1], key [B,3,N2] -> [distance [B,N1,k], index [B,N1,k]]; equals
    ``_C.knn_distance_cuda`` on the transposed clouds. Returns None when the library
    declines this k and launch size on this layout (it has a faster kernel that reads
    [B,N,3] only, or none at all for k > 64): the caller then copies to [B,N,3]."""
    return _native.knn(query, key, int(k), int(version), True) or None


def group_points_concat_forward(feature, xyz, centre, index):
    """feature [B,C,N1] or None, xyz [B,3,N1], centre [B,3,N2], index [B,N2,K] ->
    [B,C+3,N2,K]: grouped features, then grouped coordinates minus their centre."""
    return _native.group_concat_forward(feature, xyz, centre, index)


def group_points_concat_backward(grad_output, index, n1, want_feature, want_xyz):
    """grad_output [B,C+3,N2,K], index [B,N2,K] -> (grad_feature [B,C,n1] or None,
    grad_xyz [B,3,n1] or None)."""
    return _native.group_concat_backward(grad_output, index, int(n1), bool(want_feature),
                                         bool(want_xyz))


def three_nn(query, key, channels_first, eps=1e-10):
    """3 nearest keys of every query with inverse-squared-distance weights ->
    (distance [B,N1,3], index [B,N1,3] int64, weight [B,N1,3]); distance and index
    equal ``_C.knn_distance_cuda(query, key, 3, 1)`` on [B,N,3] clouds."""
    return _native.three_nn(query, key, bool(channels_first), float(eps))


def chamfer_forward_bcn(xyz1, xyz2):
    """xyz1 [B,3,N1], xyz2 [B,3,N2] -> [dist1, idx1, dist2, idx2], the clouds read in place
    (the reference copies them to [B,N,3] first, torkit3d/ops/chamfer_distance.py:52-55)."""
    return _native.chamfer_forward(xyz1, xyz2, True)
