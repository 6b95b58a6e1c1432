"""The operators under what has to see them: tracing records them as calls (a trace that held only the
outputs' allocation would return memory that nobody fills), and forward-mode tangents and function
transforms, for which they have no rule, are refused and not dropped in silence."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.func import grad, vmap

from torkit3d_amd.ops.ball_query import ball_query
from torkit3d_amd.ops.chamfer_distance import chamfer_distance
from torkit3d_amd.ops.group_points import group_points, group_points_with_xyz
from torkit3d_amd.ops.interpolate_feature import interpolate_feature
from torkit3d_amd.ops.knn_points import knn_points
from torkit3d_amd.ops.sample_farthest_points import sample_farthest_points

pytestmark = pytest.mark.gpu


def cloud(n, channels=3):
    return torch.rand(2, channels, n, device="cuda")


def neighbours():
    return (torch.arange(2 * 64 * 3, device="cuda") * 7 % 48).view(2, 64, 3)


CASES = {
    "chamfer": (lambda a, b: chamfer_distance(a, b, transpose=True), (3, 64), (3, 48)),
    "chamfer_roots": (lambda a, b: chamfer_distance(a, b, transpose=True, sqrt=True), (3, 64), (3, 48)),
    "chamfer_rows": (lambda a, b: chamfer_distance(a.transpose(1, 2), b.transpose(1, 2)), (3, 64), (3, 48)),
    "group": (lambda f: group_points(f, neighbours()), (5, 48)),
    "group_with_xyz": (lambda f, x, c: group_points_with_xyz(f, x, c, neighbours()),
                       (5, 48), (3, 48), (3, 64)),
    "group_xyz_alone": (lambda x, c: group_points_with_xyz(None, x, c, neighbours()), (3, 48), (3, 64)),
    "interpolate": (lambda f, w: interpolate_feature(f, neighbours(), w.transpose(1, 2).contiguous()),
                    (5, 48), (3, 64)),
    "ball": (lambda a, b: ball_query(a, b, 0.3, 8), (3, 64), (3, 48)),
    "ball_rows": (lambda a, b: ball_query(a.transpose(1, 2), b.transpose(1, 2), 0.3, 8, transpose=False),
                  (3, 64), (3, 48)),
    "knn": (lambda a, b: knn_points(a, b, 4, transpose=True), (3, 64), (3, 48)),
    "knn_sorted_roots": (lambda a, b: knn_points(a, b, 4, sorted=True, sqrt_distance=True, transpose=True),
                         (3, 64), (3, 48)),
    "knn_rows": (lambda a, b: knn_points(a.transpose(1, 2), b.transpose(1, 2), 4), (3, 64), (3, 48)),
    "fps": (lambda a: sample_farthest_points(a, 8, transpose=True), (3, 64)),
}


def made(name):
    call, *shapes = CASES[name]
    return call, tuple(cloud(n, c) for c, n in shapes)


def as_list(out):
    return list(out) if isinstance(out, (tuple, list)) else [out]


@pytest.mark.parametrize("name", CASES)
def test_traced(cuda, name):
    call, example = made(name)
    traced = torch.jit.trace(call, example, check_trace=False)
    _, other = made(name)
    for got, want in zip(as_list(traced(*other)), as_list(call(*other))):
        assert torch.equal(got, want)


@pytest.mark.parametrize("name", CASES)
def test_forward_mode_is_refused(cuda, name):
    call, clouds = made(name)
    with forward_ad.dual_level():
        duals = [forward_ad.make_dual(c, torch.ones_like(c)) for c in clouds]
        with pytest.raises((RuntimeError, NotImplementedError)):
            call(*duals)


@pytest.mark.parametrize("name", ["chamfer", "chamfer_roots", "chamfer_rows", "group", "group_with_xyz",
                                  "interpolate"])
def test_saved_tensors_come_back_in_another_layout(cuda, name):
    """What hooks on saved tensors return need not lie in memory as what they were given."""

    def unpack(t):
        return t.transpose(-1, -2).contiguous().transpose(-1, -2) if t.dim() > 1 else t

    call, clouds = made(name)
    if name == "interpolate":
        clouds = (clouds[0], clouds[1].requires_grad_(False))
    grads = []
    for hooked in (False, True):
        leaves = [c.clone().requires_grad_(name != "interpolate" or i == 0) for i, c in enumerate(clouds)]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack if hooked else lambda t: t):
            out = call(*leaves)
        total = sum((o * o).sum() for o in as_list(out))
        grads.append(torch.autograd.grad(total, [x for x in leaves if x.requires_grad]))
    for a, b in zip(*grads):
        torch.testing.assert_close(a, b, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("name", CASES)
def test_function_transforms_are_refused(cuda, name):
    call, clouds = made(name)
    with pytest.raises(RuntimeError):
        vmap(lambda c: as_list(call(c, *clouds[1:]))[0])(torch.stack([clouds[0], clouds[0]]))
    with pytest.raises(RuntimeError):
        grad(lambda c: as_list(call(c, *clouds[1:]))[0].sum())(clouds[0])
