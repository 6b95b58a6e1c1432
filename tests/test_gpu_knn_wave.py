"""The wave-per-query KNN kernel (launches of few queries, k <= 64) and the rows put in order on
the way out, against the oracle's literal MinK: slot for slot, bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from debug_abi import knn_wave
from torkit3d_amd.ops.interpolate_feature import three_nn_interpolation
from torkit3d_amd.ops.knn_points import knn_points

pytestmark = pytest.mark.gpu


def cloud(kind, seed, b, n):
    g = np.random.default_rng(seed)
    p = g.random((b, n, 3), dtype=np.float32)
    if kind == "lattice":  # equal distances everywhere
        p = np.floor(p * 4).astype(np.float32)
    elif kind == "far to near":  # every key is inserted
        order = np.argsort(-((p - 0.5) ** 2).sum(-1), axis=1)
        p = np.take_along_axis(p, order[:, :, None], 1)
    elif kind == "broken":
        p[:, g.integers(0, n, max(1, n // 5)), 0] = np.nan
        p[:, g.integers(0, n, max(1, n // 7)), 1] = np.inf
        p[0, 0, 2] = np.nan  # MinK starts with a NaN maximum on this cloud
    return p


def same(got, want):
    assert np.array_equal(got[0].cpu().numpy(), want[0], equal_nan=True)
    assert np.array_equal(got[1].cpu().numpy(), want[1])


# k around the 16, 32 and 64 lanes of the maximum, keys around the chunks of 64 and 256.
@pytest.mark.parametrize("channels_first", [False, True])
@pytest.mark.parametrize("kind", ["uniform", "lattice", "far to near", "broken"])
@pytest.mark.parametrize("n2,k", [(1, 1), (2, 2), (16, 16), (63, 17), (64, 64), (65, 33), (255, 32),
                                  (256, 3), (257, 15), (300, 64), (1000, 20), (2049, 63)])
def test_slots(cuda, kind, n2, k, channels_first):
    q, c = cloud("uniform", 1, 2, 37), cloud(kind, n2 + k, 2, n2)
    a, b = torch.from_numpy(q).to(cuda), torch.from_numpy(c).to(cuda)
    if channels_first:
        a, b = a.transpose(1, 2).contiguous(), b.transpose(1, 2).contiguous()
    want = oracle.knn(q, c, k)
    same(knn_wave(a, b, k, channels_first), want)
    same(knn_points(a, b, k, transpose=channels_first), want)


# The first k keys put in order by networks of 2, 4, 8, 16, 32 and 64 lanes, full and not, on clouds of one chunk of
# keys to more than eight.
@pytest.mark.parametrize("kind", ["uniform", "lattice", "broken"])
@pytest.mark.parametrize("n2", [64, 65, 128, 129, 256, 257, 512, 513])
def test_order_of_the_first_keys(cuda, kind, n2):
    q, c = cloud("uniform", n2, 2, 19), cloud(kind, n2, 2, n2)
    a, b = torch.from_numpy(q).to(cuda), torch.from_numpy(c).to(cuda)
    for k in (1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 48, 63, 64):
        same(knn_wave(a, b, k, False), oracle.knn(q, c, k))
        few = np.ascontiguousarray(c[:, : k + 1])
        same(knn_wave(a, torch.from_numpy(few).to(cuda), k, False), oracle.knn(q, few, k))


def in_order(want, root):
    """A stable sort of the slots, NaNs last (numpy sorts NaNs last)."""
    order = np.argsort(want[0], axis=2, kind="stable")
    d = np.take_along_axis(want[0], order, 2)
    return (np.sqrt(d) if root else d), np.take_along_axis(want[1], order, 2)


# few queries: in the wave kernel; many, or float64: a kernel over the rows (8, 16, 32, 64 lanes)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("kind", ["uniform", "lattice", "broken"])
@pytest.mark.parametrize("n1,k", [(5, 1), (37, 7), (37, 16), (33, 24), (40, 64), (19001, 8),
                                  (19000, 20), (37001, 33)])
def test_rows_in_order(cuda, kind, n1, k, dtype):
    few = 40 if n1 > 1000 else n1
    q = np.tile(cloud("uniform", 2, 1, few), (1, n1 // few + 1, 1))[:, :n1]
    c = cloud(kind, k, 1, 300)
    if dtype == torch.float64:
        q, c = q.astype(np.float64), c.astype(np.float64)
    want = oracle.knn(q, c, k)
    a, b = torch.from_numpy(q).to(cuda), torch.from_numpy(c).to(cuda)
    same(knn_points(a, b, k, sorted=True), in_order(want, False))
    same(knn_points(a, b, k, sorted=True, sqrt_distance=True), in_order(want, True))
    with np.errstate(invalid="ignore"):
        same(knn_points(a, b, k, sqrt_distance=True), (np.sqrt(want[0]), want[1]))


@pytest.mark.parametrize("kind", ["uniform", "lattice"])
@pytest.mark.parametrize("n2", [3, 64, 700])
def test_three_nn_weights(cuda, kind, n2):
    q, c = cloud("uniform", 3, 2, 50), cloud(kind, n2, 2, n2)
    d, i, w = three_nn_interpolation(torch.from_numpy(q).to(cuda), torch.from_numpy(c).to(cuda))
    want = oracle.knn(q, c, 3)
    same((d, i), want)
    # one division and one sum of three: the same float32 operations in the same order
    assert np.allclose(w.cpu().numpy(), oracle.three_nn_weights(want[0]), rtol=1e-6, atol=0)


@pytest.mark.parametrize("k,n2", [(3, 200), (8, 300), (12, 400), (24, 300), (48, 200)])
def test_launches_of_many_queries_keep_their_kernels(cuda, k, n2):
    """Beyond the wave kernel's launches: a lane per query, short clouds."""
    q, c = cloud("uniform", 5, 2, 20000), cloud("lattice", 6, 2, n2)
    same(knn_points(torch.from_numpy(q).to(cuda), torch.from_numpy(c).to(cuda), k),
         oracle.knn(q, c, k))


@pytest.mark.parametrize("b,n1,n2,k", [  # either side of the lines up to which a query has a wave
    (18, 1024, 1024, 3), (18, 1025, 1024, 3), (100, 256, 1025, 8), (100, 257, 1025, 8),
    (50, 512, 4096, 16), (40, 512, 4097, 16), (40, 513, 4097, 16), (50, 513, 4096, 16), (100, 256, 4097, 17), (100, 257, 4097, 17),
    (48, 1024, 200, 33), (48, 1025, 200, 33), (128, 1024, 2047, 64), (128, 1024, 2048, 64), (128, 1025, 2048, 64)])
def test_both_sides_of_the_limits(cuda, b, n1, n2, k):
    """A batch as a whole and a few clouds of it at a time, which have a wave per query, agree bit for bit; some of
    the distances are equal (coordinates in steps of 1/16)."""
    from torkit3d_amd import _C

    g = torch.Generator().manual_seed(b + n1 + n2)
    query = (torch.rand(b, n1, 3, generator=g) * 16).round().div(16).to(cuda)
    key = (torch.rand(b, n2, 3, generator=g) * 16).round().div(16).to(cuda)
    distance, index = _C.knn_distance_cuda(query, key, k, 1)
    few = max(1, 8192 // n1)
    for i in (0, b // 2, b - few):
        d, j = _C.knn_distance_cuda(query[i:i + few].contiguous(), key[i:i + few].contiguous(), k, 1)
        assert torch.equal(distance[i:i + few], d) and torch.equal(index[i:i + few], j)
