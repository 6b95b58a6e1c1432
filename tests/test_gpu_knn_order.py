"""The pre-filtered KNN kernel on keys in an order, which launches of few workgroups look for: they then sweep every
key instead of those in reach of a wave's box, half of the queries to a workgroup where CUs are free. Against the
oracle's literal MinK, bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from debug_abi import knn_filter, knn_wave_queries
from torkit3d_amd.ops.knn_points import knn_points

pytestmark = pytest.mark.gpu


def cloud(kind, b, n, seed):
    g = np.random.default_rng(seed)
    p = g.random((b, n, 3), dtype=np.float32)
    if kind == "lattice by x":  # and equal distances everywhere
        p = np.floor(p * 6).astype(np.float32)
    if kind in ("by x", "lattice by x", "mixed", "not numbers"):
        p = np.take_along_axis(p, np.argsort(p[:, :, :1], axis=1, kind="stable"), 1)
    if kind == "mixed":  # ordered clouds and others in a launch
        p[::2] = p[::2, g.permutation(n)]
    elif kind == "flat":  # an axis without extent, keys by another
        p = np.take_along_axis(p, np.argsort(p[:, :, 1:2], axis=1), 1)
        p[:, :, 0] = 0.25
    elif kind == "far key":  # in random order, but one key makes the cloud's box large
        p[:, -1] = 1e3
    elif kind == "not numbers":
        p[:, : n // 3, 0] = np.nan
        p[0, n - 2, 1] = np.nan
    return p


# k: the smallest and largest of 4, 8 and 16 slots; keys: the fewest that have boxes, a stage's edge, a remainder;
# queries: around 256, 512 and their sums (the halves of a workgroup)
@pytest.mark.parametrize("kind", ["by x", "lattice by x", "mixed", "flat", "far key", "not numbers"])
@pytest.mark.parametrize("b,n1,n2,k", [
    (2, 257, 2048, 1), (3, 511, 2049, 4), (2, 512, 2560, 3), (2, 513, 2048, 3), (3, 769, 2100, 4), (2, 1280, 2047, 4),
    (2, 300, 4096, 5), (2, 768, 4097, 8), (1, 1025, 4095, 8), (2, 256, 4096, 8), (2, 129, 16384, 2), (2, 128, 16384, 2),
    (1, 300, 8192, 9), (2, 770, 8705, 16), (2, 513, 8191, 16)])
def test_few_workgroups(cuda, kind, b, n1, n2, k):
    q, key = cloud("random", b, n1, n1), cloud(kind, b, n2, n2)
    if kind == "not numbers":
        q[0, 3, 2], q[-1, n1 - 1, 0] = np.nan, np.inf
    got = knn_filter(torch.from_numpy(q).to(cuda), torch.from_numpy(key).to(cuda), k)
    with np.errstate(invalid="ignore"):
        want = oracle.knn(q, key, k)
    assert np.array_equal(got[0].cpu().numpy(), want[0], equal_nan=True)
    assert np.array_equal(got[1].cpu().numpy(), want[1])


# either side of a workgroup to two CUs, and of one to one (256 CUs), beyond which order makes no difference
@pytest.mark.parametrize("b,n2,k", [(128, 2048, 3), (129, 2048, 3), (256, 2048, 3), (257, 2048, 3), (257, 1024, 4),
                                    (129, 3584, 16), (129, 3583, 16), (256, 2560, 8), (257, 1023, 12)])
def test_workgroups_to_a_cu(cuda, b, n2, k):
    q, key = cloud("random", b, 257, b), cloud("mixed", b, n2, n2)
    got = knn_filter(torch.from_numpy(q).to(cuda), torch.from_numpy(key).to(cuda), k)
    some = sorted({0, 1, b // 2, b - 2, b - 1})
    want = oracle.knn(q[some], key[some], k)
    assert np.array_equal(got[0].cpu().numpy()[some], want[0])
    assert np.array_equal(got[1].cpu().numpy()[some], want[1])
    # the rest against the same clouds a few at a time
    few = 16
    for at in range(0, b, few):
        part = knn_filter(torch.from_numpy(q[at:at + few]).to(cuda), torch.from_numpy(key[at:at + few]).to(cuda), k)
        assert torch.equal(got[0][at:at + few], part[0]) and torch.equal(got[1][at:at + few], part[1])


# ---- either side of the lines up to which a query has a wave, whatever they are ----

@pytest.mark.parametrize("n2,k", [(64, 2), (512, 3), (512, 8), (513, 8), (1024, 16), (1025, 1), (2048, 8), (4096, 5), (4097, 3),
                                  (8192, 16), (8193, 9), (1024, 20), (4096, 32), (4097, 17), (32769, 24)])
def test_both_sides_of_a_wave_to_a_query(cuda, n2, k):
    """A cloud of as many queries as have a wave each, and of one more, which do not: the same rows."""
    limit = knn_wave_queries(n2, k)
    query, key = (torch.from_numpy(cloud(kind, 1, n, n)).to(cuda) for kind, n in (("random", limit + 1), ("by x", n2)))
    few = knn_points(query[:, :limit].contiguous(), key, k)
    many = knn_points(query, key, k)
    assert torch.equal(few[0], many[0][:, :limit]) and torch.equal(few[1], many[1][:, :limit])
    some = slice(limit - 40, limit + 1)
    d, i = oracle.knn(query[:, some].cpu().numpy(), key.cpu().numpy(), k)
    assert np.array_equal(many[0][:, some].cpu().numpy(), d) and np.array_equal(many[1][:, some].cpu().numpy(), i)


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("kind", ["random", "lattice by x"])
@pytest.mark.parametrize("n2,k", [(40, 33), (200, 48), (300, 64), (2100, 40)])
def test_more_than_32_neighbours_beyond_a_wave_to_a_query(cuda, kind, n2, k, transpose):
    """The tree in LDS, rows and planes, and the kernel that puts its rows in order: the sizes follow the line."""
    limit, b = knn_wave_queries(n2, k), 3
    n1 = limit // b + 7
    assert b * n1 > limit
    few = cloud("random", b, 50, 5)
    q, key = np.tile(few, (1, n1 // 50 + 1, 1))[:, :n1], cloud(kind, b, n2, n2)
    d, i = (np.tile(t, (1, n1 // 50 + 1, 1))[:, :n1] for t in oracle.knn(few, key, k))
    clouds = [torch.from_numpy(np.ascontiguousarray(t.transpose(0, 2, 1) if transpose else t)).to(cuda) for t in (q, key)]
    got = knn_points(*clouds, k, transpose=transpose)
    assert np.array_equal(got[0].cpu().numpy(), d) and np.array_equal(got[1].cpu().numpy(), i)
    order = np.argsort(d, axis=2, kind="stable")
    got = knn_points(*clouds, k, transpose=transpose, sorted=True, sqrt_distance=True)
    assert np.array_equal(got[0].cpu().numpy(), np.sqrt(np.take_along_axis(d, order, 2)))
    assert np.array_equal(got[1].cpu().numpy(), np.take_along_axis(i, order, 2))
