"""Drop-in for the reference's compiled extension ``torkit3d._C``.

The reference registers nine functions in a pybind11 module
(torkit3d/csrc/torkit3d.cpp:13-21). This module exposes the same nine names with
the same positional arguments and return values. The work is in the extension module
``_native`` (csrc/native.cpp): it validates the tensors the way the reference's host code
does (TORCH_CHECK -> RuntimeError), allocates the outputs with torch and hands raw device
pointers to the C ABI in ``include/tk3d.h``. Kernels are enqueued on torch's current
stream for the tensors' device.

Placing this file (plus ``_native.py``, ``_host.so`` and ``libtk3d.so``) inside a checkout of the
reference as ``torkit3d/_C.py`` makes the reference's own ``torkit3d.ops`` run on
MI355X unchanged.
"""
import torch  # noqa: F401  (loads the libraries the extension resolves against)

from . import _native

__all__ = [
    "sample_farthest_points_cuda",
    "ball_query_cuda",
    "group_points_forward_cuda",
    "group_points_backward_cuda",
    "interpolate_forward_cuda",
    "interpolate_backward_cuda",
    "knn_distance_cuda",
    "chamfer_distance_forward_cuda",
    "chamfer_distance_backward_cuda",
]


def sample_farthest_points_cuda(points, num_samples):
    """points [B,N,3] -> index [B,num_samples] int64
    (sample_farthest_points_kernel.cu:106-165)."""
    return _native.sample_farthest_points(points, int(num_samples), False, False)[0]


def ball_query_cuda(query, key, radius, max_neighbors):
    """query [B,N1,3], key [B,N2,3] -> index [B,N1,max_neighbors] int64
    (ball_query_kernel.cu:105-173)."""
    return _native.ball_query(query, key, float(radius), int(max_neighbors), False)


def group_points_forward_cuda(input, index):
    """input [B,C,N1], index [B,N2,K] -> [B,C,N2,K] (group_points_kernel.cu:8-31).
    Like the reference (which goes through at::gather) this accepts
    non-contiguous tensors; they are made contiguous first."""
    return _native.group_forward(input, index)


def group_points_backward_cuda(grad_output, index, n1):
    """grad_output [B,C,N2,K], index [B,N2,K], n1 -> grad_input [B,C,n1]
    (group_points_kernel.cu:67-114)."""
    return _native.group_backward(grad_output, index, int(n1))


def interpolate_forward_cuda(input, index, weight):
    """input [B,C,N1], index [B,N2,3], weight [B,N2,3] -> [B,C,N2]
    (interpolate_kernel.cu:49-103)."""
    return _native.interpolate_forward(input, index, weight)


def interpolate_backward_cuda(grad_output, index, weight, n1):
    """grad_output [B,C,N2], index, weight [B,N2,3], n1 -> grad_input [B,C,n1]
    (interpolate_kernel.cu:147-201)."""
    return _native.interpolate_backward(grad_output, index, weight, int(n1))


def knn_distance_cuda(query, key, k, version):
    """query [B,N1,3], key [B,N2,3] -> [distance [B,N1,k], index [B,N1,k] int64],
    squared distances in MinK slot order (knn_distance_kernel.cu:187-298)."""
    return _native.knn(query, key, int(k), int(version), False)


def chamfer_distance_forward_cuda(xyz1, xyz2):
    """xyz1 [B,N1,3], xyz2 [B,N2,3] -> [dist1, idx1, dist2, idx2]
    (chamfer_distance_kernel.cu:91-151)."""
    return _native.chamfer_forward(xyz1, xyz2, False)


def chamfer_distance_backward_cuda(grad_dist1, grad_dist2, xyz1, xyz2, idx1, idx2):
    """-> [grad_xyz1 [B,N1,3], grad_xyz2 [B,N2,3]] (chamfer_distance_kernel.cu:200-274)."""
    return _native.chamfer_backward(grad_dist1, grad_dist2, xyz1, xyz2, idx1, idx2)
