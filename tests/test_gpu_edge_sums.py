"""The sums over the edges whose value is the maximum (EdgeConv's backward), through the C ABI."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
i32 = ctypes.c_int


class Norm(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("mean", "var", "gamma", "beta")] + [("eps", ctypes.c_float)]


def sums(g, place, index):
    """The sparse part of du [B, O, N], which lies in the workspace, and dx: the other terms' coefficients are zero."""
    from torkit3d_amd import _lib
    from torkit3d_amd._lib import ptr, stream_of

    lib, dev = _lib.lib(), g.device
    (b, o, n), k, c = g.shape, index.size(2), 3
    size = lib.tk3d_mlp_edge_backward_bytes
    size.restype = ctypes.c_int64
    x, w, dw = (torch.ones(s, device=dev) for s in ((b, c, n), (o, 2 * c), (o, 2 * c)))
    dx, extreme = torch.empty_like(x), torch.ones_like(g)
    one, zero = torch.ones(o, device=dev), torch.zeros(o, device=dev)
    norm = Norm(zero.data_ptr(), one.data_ptr(), one.data_ptr(), zero.data_ptr(), 1e-5)
    coef = torch.zeros(o, 4, device=dev)
    coef[:, 0] = 1
    lists = torch.empty(b, n + 1 + n * k, dtype=torch.int32, device=dev)
    work = torch.zeros(size(i32(b), i32(n), i32(o), i32(c)), dtype=torch.uint8, device=dev)
    assert lib.tk3d_mlp_edge_lists(ptr(index), i32(b), i32(n), i32(k), ptr(lists), stream_of(x)) == 0
    assert lib.tk3d_mlp_edge_backward_f32(
        ptr(g), ptr(extreme), ptr(place), ptr(x), ptr(index), ptr(lists), ptr(w), i32(b), i32(n), i32(k), i32(c), i32(o),
        ctypes.byref(norm), ptr(coef), ptr(work), ptr(dx), ptr(dw), stream_of(x)) == 0
    behind = b * n * 4 * (2 * o + 3 * c)  # duv, rows and st are the last three
    duv = work[work.numel() - behind:][: b * n * 2 * o * 4].view(torch.float32).view(b, 2 * o, n)
    return duv[:, :o].clone(), dx


@pytest.mark.parametrize("hot", [1, 3, 17, None])  # so many points are everybody's neighbours
@pytest.mark.parametrize("b,n,k,o", [(2, 2047, 4, 8), (1, 4096, 8, 5), (300, 300, 4, 2)])
def test_sums_come_in_the_order_of_the_points(cuda, b, n, k, o, hot):
    """Terms of 2^-45 to 2^45: a sum in float64 depends on the order of its terms, which is the same in every call."""
    g = torch.Generator().manual_seed(n + k)
    index = torch.randint(0, hot or n, (b, n, k), generator=g)
    place = torch.randint(0, k, (b, o, n), generator=g)
    grad = torch.randn(b, o, n, generator=g) * torch.exp2(torch.randint(-45, 46, (b, o, n), generator=g).float())
    args = grad.to(cuda), place.to(torch.uint8).to(cuda), index.to(cuda)
    first = sums(*args)
    for _ in range(3):
        assert all(torch.equal(a, f) for a, f in zip(sums(*args), first))
    owner = torch.gather(index.view(b, 1, n, k).expand(b, o, n, k), 3, place.unsqueeze(3))[..., 0].numpy()
    got = first[0].cpu().numpy()
    for bi in {0, b - 1}:
        for oi in range(o):
            want = np.zeros(n)
            np.add.at(want, owner[bi, oi], grad[bi, oi].numpy().astype(np.float64))  # one after the other
            assert np.array_equal(got[bi, oi], want.astype(np.float32))
