"""What surrounds the chamfer op: the copy to padded rows, one gradient alone, square roots."""
import numpy as np
import pytest
import torch

import oracle
from torkit3d_amd.ops.chamfer_distance import chamfer_distance, nn_distance, safe_sqrt

pytestmark = pytest.mark.gpu


def clouds(b, n1, n2, dtype=torch.float32):
    g = torch.Generator().manual_seed(n1 + n2)
    return [torch.rand(b, n, 3, generator=g, dtype=dtype) for n in (n1, n2)]


# lengths on either side of a multiple of four, of the shortest cloud that is copied, and of the
# matrix kernel's shortest
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("b,n1,n2", [(2, 255, 256), (3, 256, 257), (2, 259, 1000), (2, 1021, 1023),
                                     (2, 1024, 1025), (3, 1027, 300), (8, 2500, 3001), (2, 4099, 1),
                                     (1, 1025, 1025), (16, 1025, 1027), (32, 489, 1130), (8, 5001, 300)])
def test_copied_clouds(cuda, b, n1, n2, transpose):
    x, y = clouds(b, n1, n2)
    a, c = [(t.transpose(1, 2) if transpose else t).contiguous().to(cuda) for t in (x, y)]
    for got, want in zip(nn_distance(a, c, transpose=transpose),
                         oracle.chamfer_forward(x.numpy(), y.numpy())):
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("which", [(True, False), (False, True), (True, True)])
def test_gradients_that_are_wanted(cuda, which, transpose, dtype):
    x, y = [(t.transpose(1, 2) if transpose else t).contiguous().to(cuda)
            for t in clouds(2, 700, 5001, dtype)]
    g1, g2 = torch.randn(2, 700, device=cuda, dtype=dtype), torch.randn(2, 5001, device=cuda, dtype=dtype)
    both = [t.clone().requires_grad_() for t in (x, y)]
    some = [t.clone().requires_grad_(w) for t, w in zip((x, y), which)]
    for leaves in (both, some):
        torch.autograd.backward(chamfer_distance(*leaves, transpose=transpose), (g1, g2))
    for a, c, w in zip(both, some, which):
        if not w:
            assert c.grad is None
        elif dtype == torch.float32:
            assert torch.equal(a.grad, c.grad)
        else:  # (float64 sums through atomics)
            torch.testing.assert_close(a.grad, c.grad, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("transpose", [False, True])
def test_square_roots(cuda, transpose, dtype):
    x, y = [(t.transpose(1, 2) if transpose else t).contiguous().to(cuda)
            for t in clouds(2, 300, 513, dtype)]
    eps = 1e-4  # above some of the squared distances, below others
    leaves = [[t.clone().requires_grad_() for t in (x, y)] for _ in range(2)]
    fused = chamfer_distance(*leaves[0], transpose=transpose, sqrt=True, eps=eps)
    plain = [safe_sqrt(d, eps) for d in chamfer_distance(*leaves[1], transpose=transpose)]
    low = sum(int((d * d <= eps * 1.0001).sum()) for d in plain)
    assert 0 < low < 2 * (300 + 513)
    grads = [torch.randn(2, n, device=cuda, dtype=dtype) for n in (300, 513)]
    for f, p in zip(fused, plain):
        assert torch.equal(f, p)
    torch.autograd.backward(fused, grads)
    torch.autograd.backward(plain, grads)
    for a, c in zip(*leaves):
        if dtype == torch.float32:
            assert torch.equal(a.grad, c.grad)
        else:
            torch.testing.assert_close(a.grad, c.grad, rtol=1e-12, atol=1e-12)
    with torch.no_grad():
        for f, p in zip(chamfer_distance(x, y, transpose=transpose, sqrt=True, eps=eps), plain):
            assert torch.equal(f, p)


# lengths on either side of a range of the backward kernel and of the longest cloud whose layout and roots it takes itself
@pytest.mark.parametrize("sqrt", [False, True])
@pytest.mark.parametrize("b,n1,n2", [(2, 1, 3), (2, 1023, 1025), (3, 4095, 4097), (1, 4097, 5001), (2, 8192, 5), (1, 8193, 700)])
def test_backward_of_planes_and_roots(cuda, b, n1, n2, sqrt):
    rows = [t.to(cuda).requires_grad_() for t in clouds(b, n1, n2)]
    planes = [t.detach().transpose(1, 2).contiguous().requires_grad_() for t in rows]
    grads = [torch.randn(b, n, device=cuda) for n in (n1, n2)]
    eps = 1e-6
    dists = chamfer_distance(*rows)
    want = torch.autograd.grad([safe_sqrt(d, eps) for d in dists] if sqrt else dists, rows, grads)
    roots = chamfer_distance(*rows, sqrt=sqrt, eps=eps)
    for got, w in zip(torch.autograd.grad(roots, rows, grads), want):
        assert torch.equal(got, w)
    for some in ((0, 1), (0,), (1,)):  # (both gradients, or one)
        leaves = [p.detach().requires_grad_(i in some) for i, p in enumerate(planes)]
        out = chamfer_distance(*leaves, transpose=True, sqrt=sqrt, eps=eps)
        for i, got in zip(some, torch.autograd.grad(out, [leaves[i] for i in some], grads)):
            assert torch.equal(got, want[i].transpose(1, 2))


def test_backward_of_planes_and_roots_with_infinite_gradients(cuda):
    x, y = [t.to(cuda).transpose(1, 2).contiguous().requires_grad_() for t in clouds(2, 300, 513)]
    grads = [torch.randn(2, n, device=cuda) for n in (300, 513)]
    grads[1][0, 7] = float("inf")  # (a batch element with sums through atomics)
    rows = [t.detach().transpose(1, 2).contiguous().requires_grad_() for t in (x, y)]
    plain = [safe_sqrt(d) for d in chamfer_distance(*rows)]
    want = torch.autograd.grad(plain, rows, grads)
    got = torch.autograd.grad(chamfer_distance(x, y, transpose=True, sqrt=True), (x, y), grads)
    # (the distances' gradients agree to the bit; sums of the same float32 terms in another order: a few of them a point)
    for g, w in zip(got, want):
        torch.testing.assert_close(g.transpose(1, 2), w, rtol=1e-5, atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("sqrt", [False, True])
@pytest.mark.parametrize("n1,n2", [(300, 700), (4097, 4097), (8193, 600)])
def test_backward_allocates_no_more_than_it_needs(cuda, n1, n2, transpose, sqrt):
    """Both gradients, and one piece for copies of planes and gradients of distances only where launches of their own
    make them: what is allocated for a path that is then not taken is host time of every call."""
    from torkit3d_amd import _lib

    x, y = [(t.transpose(1, 2) if transpose else t).contiguous().to(cuda).requires_grad_() for t in clouds(1, n1, n2)]
    grads = [torch.randn(1, n, device=cuda) for n in (n1, n2)]
    out = chamfer_distance(x, y, transpose=transpose, sqrt=sqrt)
    torch.autograd.grad(out, (x, y), grads, retain_graph=True)
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    result = torch.autograd.grad(out, (x, y), grads, retain_graph=True)
    taken = torch.cuda.memory_stats()["allocation.all.allocated"] - before
    alone = not (transpose or sqrt) or _lib.lib().tk3d_chamfer_distance_backward_takes_forms(
        int(transpose), int(sqrt), _lib.i64(n1), _lib.i64(n2))
    assert len(result) == 2 and taken == (2 if alone else 3)
