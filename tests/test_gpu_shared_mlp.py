"""The fused chains of ``SharedMLP`` (csrc/mlp.hip) against the same modules in stock torch.

The oracle is the stock chain in float64. A float32 implementation may differ from it by what
float32 gives, so every output, gradient and running statistic of the fused chain has to be
about as close to float64 (2-norm of the difference over 2-norm of the result) as stock
float32 is: within four times its error plus 2e-6 (a few rounding errors of 2^-24 through up
to four layers)."""
import copy
import ctypes

import pytest
import torch
from torch import nn

from torkit3d_amd import _lib, _native
from torkit3d_amd.nn import SharedMLP, mlp1d_bn_relu, mlp2d_bn_relu
from torkit3d_amd.ops.edge_conv import edge_lists
from torkit3d_amd.ops.group_points import group_points_with_xyz

pytestmark = pytest.mark.gpu


def make(build, cin, widths, training, cuda):
    torch.manual_seed(1)
    mlp = build(cin, widths)
    for m in mlp.modules():
        if isinstance(m, (nn.BatchNorm1d, nn.BatchNorm2d)):
            nn.init.uniform_(m.weight, -1.0, 1.5)  # both signs: maxima become minima
            nn.init.uniform_(m.bias, -0.5, 0.5)
            nn.init.uniform_(m.running_mean, -0.5, 0.5)
            nn.init.uniform_(m.running_var, 0.5, 2.0)
    return mlp.to(cuda).train(training)


def stock(mlp, dtype):
    """The same layers as a plain nn.Sequential."""
    return nn.Sequential(*copy.deepcopy(mlp).to(dtype).children()).train(mlp.training)


def everything(module, fn, inputs):
    """Outputs, gradients (inputs that float, parameters) and buffers after one pass."""
    if not module.training:  # (evaluation with gradients runs in the stock modules)
        with torch.no_grad():
            return [fn(module, *[t for t, _ in inputs])]
    leaves = [t.clone().requires_grad_() if t.is_floating_point() and g else t for t, g in inputs]
    out = fn(module, *leaves)
    grad = torch.linspace(-1.0, 1.0, out.numel(), device=out.device, dtype=torch.float64)
    grad = grad[torch.randperm(out.numel(), generator=torch.Generator().manual_seed(3)).to(out.device)]
    wanted = [t for t in leaves if t.requires_grad] + list(module.parameters())
    grads = torch.autograd.grad(out, wanted, grad.view_as(out).to(out.dtype))
    return [out.detach(), *grads, *[b.clone() for b in module.buffers()]]


def check(mlp, fused, reference, inputs, monkeypatch):
    used = []
    real = SharedMLP._chain
    monkeypatch.setattr(SharedMLP, "_chain",
                        lambda self, *a, **k: used.append(real(self, *a, **k)) or used[-1])
    compare_forms(mlp, fused, reference, inputs)
    assert len(used) == 1 and used[0] is not None, "the fused chain did not run"


def compare_forms(mlp, fused, reference, inputs):
    plain32, plain64 = stock(mlp, torch.float32), stock(mlp, torch.float64)
    got = everything(mlp, fused, inputs)
    single = everything(plain32, reference, inputs)
    exact = everything(plain64, reference, [(t.double() if t.is_floating_point() else t, g)
                                            for t, g in inputs])
    for i, (a, s, e) in enumerate(zip(got, single, exact)):
        assert a.shape == e.shape
        if not e.is_floating_point():
            assert torch.equal(a, e)
            continue
        norm = float(e.norm()) + 1e-30
        mine, theirs = float((a.double() - e).norm()) / norm, float((s.double() - e).norm()) / norm
        assert mine <= 4 * theirs + 2e-6, (i, tuple(e.shape), mine, theirs)


def randn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).cuda()


# Positions and channels around the tiles (32 channels, 32/64/128 positions, 8 input channels a
# step, weights in one piece or in several), row lengths that are multiples of 4 and not.
@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("b,p,widths", [
    (2, 1, (5, 7)), (1, 37, (3, 33, 65)), (3, 64, (8, 32)), (2, 130, (64, 31, 64)),
    (1, 4, (9, 16, 8)), (5, 1000, (131, 128, 128)), (2, 1024, (16, 32, 64, 32)),
    (1, 129, (300, 257)), (4, 36, (768, 256, 40)), (40, 4096, (6, 32, 64, 40)),
])
def test_dense(cuda, monkeypatch, b, p, widths, training):
    mlp = make(mlp1d_bn_relu, widths[0], widths[1:], training, cuda)
    check(mlp, lambda m, x: m(x), lambda m, x: m(x), [(randn(b + p, b, widths[0], p), True)],
          monkeypatch)


@pytest.mark.parametrize("c1,c2,p", [(5, 3, 37), (128, 3, 512), (64, 96, 1000)])
def test_concatenated_input(cuda, monkeypatch, c1, c2, p):
    mlp = make(mlp1d_bn_relu, c1 + c2, (32, 48), True, cuda)
    check(mlp, lambda m, x, y: m.forward_cat(x, y), lambda m, x, y: m(torch.cat([x, y], 1)),
          [(randn(1, 2, c1, p), True), (randn(2, 2, c2, p), True)], monkeypatch)


# Groups of 32 and 64 in the three tile shapes; one and several channel tiles.
@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("b,m,s,widths", [
    (2, 5, 32, (6, 32, 32)), (1, 3, 32, (4, 20, 70)), (2, 2, 64, (9, 64, 33)),
    (2, 1600, 32, (3, 32, 32)), (4, 600, 64, (16, 64, 96)), (8, 1024, 32, (7, 40, 64)),
    (4, 1025, 32, (5, 70, 130)),  # (runs of four groups, the last one cut short)
])
def test_maximum_over_neighbours(cuda, monkeypatch, b, m, s, widths, training):
    mlp = make(mlp2d_bn_relu, widths[0], widths[1:], training, cuda)
    check(mlp, lambda n, x: n.forward_max(x), lambda n, x: n(x).max(dim=3)[0],
          [(randn(m, b, widths[0], m, s), True)], monkeypatch)


# Input and weight gradient of a layer in one launch: every shape in tiles of 32 channels on either side (the
# widths' neighbours), widths and positions off the tiles, one tile in all, a few tiles a workgroup and many.
@pytest.mark.parametrize("b,p", [(2, 4), (3, 36), (2, 1000), (5, 20004)])
@pytest.mark.parametrize("widths", [(64, 128, 128, 64, 64, 32, 32), (100, 30, 128, 40, 128), (33, 65, 33, 20, 64)])
def test_both_gradients_of_a_layer(cuda, monkeypatch, b, p, widths):
    mlp = make(mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    check(mlp, lambda m, x: m(x), lambda m, x: m(x), [(randn(p, b, widths[0], p), True)], monkeypatch)


@pytest.mark.parametrize("b,m,s,widths", [(1, 3, 32, (64, 128, 128)), (4, 1025, 32, (70, 100, 64, 40)),
                                          (3, 700, 64, (128, 128, 32, 128)),
                                          # (more than 128 outputs: waves share a group; 9000 groups: sums first)
                                          (3, 70, 64, (6, 33, 300)), (9, 1000, 32, (3, 20, 24))])
def test_both_gradients_under_a_maximum(cuda, monkeypatch, b, m, s, widths):
    mlp = make(mlp2d_bn_relu, widths[0], widths[1:], True, cuda)
    check(mlp, lambda n, x: n.forward_max(x), lambda n, x: n(x).max(dim=3)[0],
          [(randn(m, b, widths[0], m, s), True)], monkeypatch)


# Layers too wide for that, in tiles in LDS: three, four and five tiles of channels a workgroup with remainders
# of all of them, of 128 positions and of 32 input channels; rows in parts of a block of 128; two inputs.
@pytest.mark.parametrize("b,p,widths", [(6, 4100, (330, 160, 384, 260, 140)), (200, 36, (129, 70, 300)),
                                        (1, 24580, (65, 129, 512, 66))])
def test_wide_layers(cuda, monkeypatch, b, p, widths):
    mlp = make(mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    check(mlp, lambda m, x: m(x), lambda m, x: m(x), [(randn(p, b, widths[0], p), True)], monkeypatch)


def test_wide_layers_of_two_inputs(cuda, monkeypatch):
    mlp = make(mlp1d_bn_relu, 100 + 35, (140,), True, cuda)
    check(mlp, lambda m, x, y: m.forward_cat(x, y), lambda m, x, y: m(torch.cat([x, y], 1)),
          [(randn(1, 4, 100, 8200), True), (randn(2, 4, 35, 8200), True)], monkeypatch)


@pytest.mark.parametrize("b,m,s,widths", [(4, 225, 32, (20, 200, 300)), (3, 150, 64, (9, 256, 96))])
def test_wide_layers_under_a_maximum(cuda, monkeypatch, b, m, s, widths):
    mlp = make(mlp2d_bn_relu, widths[0], widths[1:], True, cuda)
    check(mlp, lambda n, x: n.forward_max(x), lambda n, x: n(x).max(dim=3)[0],
          [(randn(m, b, widths[0], m, s), True)], monkeypatch)


# A maximum over all points behind the last layer: on the layer's own input (tiles of it as for wide layers) and on
# activations of up to 128 channels and more, several and single clouds, rows off the tiles of 64 positions, channels
# whose maximum is negative, equal maxima; sizes that stay with the dense backward.
@pytest.mark.parametrize("b,p,widths", [
    (6, 4100, (330, 700)), (13, 2048, (70, 160)), (3, 1400, (9, 64, 128)), (1, 5000, (40, 33, 70)), (2, 2084, (6, 160, 330)),
    (5, 1028, (3, 30, 100)), (40, 128, (12, 65, 140)),
    (2, 2048, (64, 100)), (3, 37, (8, 16, 40)), (2, 512, (320, 1024))])
def test_maximum_over_points(cuda, monkeypatch, b, p, widths):
    mlp = make(mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    with torch.no_grad():
        mlp[-1].bn.bias[0::5] = -40.0  # (nothing passes the ReLU)
    x = randn(p, b, widths[0], p)
    x[:, :, 1::3] = x[:, :, 0:1]  # copies of a point
    reference = stock(mlp, torch.float32)
    values, places = mlp.forward_points_max(x.clone().requires_grad_())
    want = torch.max(reference(x), 2)
    assert torch.equal(values, want[0]) and torch.equal(places, want[1])
    used = []
    real = _native.mlp_max
    monkeypatch.setattr(_native, "mlp_max", lambda *a: used.append(real(*a)) or used[-1])
    mlp2 = make(mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    compare_forms(mlp2, lambda m, x: m.forward_points_max(x)[0], lambda m, x: m(x).max(dim=2)[0],
                  [(randn(p + 1, b, widths[0], p), True)])
    assert bool(used[0]) == (widths[-1] >= 2 * widths[-2] and b * p >= 4096 and p % 4 == 0)


# A first layer under a maximum over all points, its input `far` deviations from zero. The rounding of the saved
# statistics is most of the error then, in the stock modules too; of the weight gradient, which is made of second
# moments, counting from the mean leaves 0.41 to 0.74 of theirs, counting from zero 1.1 to 1.2. The bound lies between.
# About zero it is what is left of the sums: 0.1 to 0.2 of theirs, 0.7 with 1024 clouds in one float32 chain.
@pytest.mark.parametrize("far", [0.0, 8.0, -8.0, 30.0, -30.0])
@pytest.mark.parametrize("b,p,widths", [(13, 2048, (70, 160)), (6, 4100, (330, 700)), (1024, 128, (70, 160))])
def test_maximum_over_points_far_from_zero(cuda, b, p, widths, far):
    mlp = mlp1d_bn_relu(widths[0], widths[1:]).to(cuda).train()
    single, exact = stock(mlp, torch.float32), stock(mlp, torch.float64)
    x, g = randn(p, b, widths[0], p) + far, randn(3, b, widths[-1])
    with torch.no_grad():  # (the places and signs of the float32 activations)
        top, place = torch.max(single[0].bn(single[0].conv(x)), 2, keepdim=True)
    grads = []
    for module in (mlp, single, exact):
        leaf = x.to(torch.float64 if module is exact else torch.float32).requires_grad_()
        if module is mlp:
            out = mlp.forward_points_max(leaf)[0]
            assert "Node" in out.grad_fn.name()
        else:
            out = (module[0].bn(module[0].conv(leaf)) * (top > 0)).gather(2, place)[..., 0]
        grads.append(torch.autograd.grad(out, [leaf, module[0].conv.weight], g.to(out.dtype)))
    for mine, theirs, e, bound in zip(*grads, (1.25, 0.8 if far else 0.4)):
        errors = [float((t.double() - e).norm() / e.norm()) for t in (mine, theirs)]
        assert errors[0] <= bound * errors[1], (tuple(e.shape), errors)


# What is left to the dense backward: a first layer on rows under 128, and fewer positions than one for every 32
# weights, except in rows under 16.
@pytest.mark.parametrize("b,p,widths,taken", [
    (512, 64, (70, 160), False), (512, 124, (70, 160), False), (300, 128, (70, 160), True), (1024, 4, (9, 64, 128), True),
    (32, 128, (70, 256, 1024), False), (64, 128, (70, 256, 1024), True), (512, 12, (9, 200, 800), True),
    (280, 16, (9, 200, 800), False)])
def test_maximum_over_few_positions(cuda, b, p, widths, taken):
    mlp = make(mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    out = mlp.forward_points_max(randn(p, b, widths[0], p).requires_grad_())[0]
    assert ("Max" not in out.grad_fn.name()) == taken
    compare_forms(mlp, lambda m, x: m.forward_points_max(x)[0], lambda m, x: m(x).max(dim=2)[0],
                  [(randn(p + 1, b, widths[0], p), True)])


# Products whose waves share a tile: groups of 32 and
# of 64 in evaluation (one channel tile and two), channels that leave waves without a group of eight.
@pytest.mark.parametrize("b,p,widths,pool,training", [
    (4, 4100, (260, 256, 140), 0, True), (2, 8252, (131, 192, 128), 0, True), (3, 130, (20, 9, 200), 0, True),
    (1, 32, (16, 64, 128), 64, False), (4, 65, (9, 40, 130), 64, False), (1, 100, (6, 33, 70), 32, False),
    (1, 260, (200, 128, 64), 32, False), (2, 3, (7, 8, 9), 64, False),
    # more tiles than SIMDs: in eight stretches of unequal lengths, channel blocks that are no multiple of eight
    (41, 130, (140, 200, 131), 0, True), (17, 510, (24, 136, 150), 0, True), (171, 33, (136, 264, 96), 0, False),
    (64, 33, (131, 256, 1024), 0, False), (67, 4, (24, 128, 130), 32, False)])
def test_products_of_shared_tiles(cuda, monkeypatch, b, p, widths, pool, training):
    mlp = make(mlp2d_bn_relu if pool else mlp1d_bn_relu, widths[0], widths[1:], training, cuda)
    x = randn(p, b, widths[0], p, *([pool] if pool else []))
    fused = (lambda m, x: m.forward_max(x)) if pool else (lambda m, x: m(x))
    reference = (lambda m, x: m(x).max(dim=3)[0]) if pool else (lambda m, x: m(x))
    check(mlp, fused, reference, [(x, True)], monkeypatch)
    if not training:  # infinities and NaN stay where they are
        x[0, 0, 0], x[-1, -1, -1] = float("inf"), float("nan")
        with torch.no_grad():
            # (on the CPU: of the convolutions that the library picks between, some mix neighbouring positions,
            # and a NaN then reaches those of a whole tile)
            got, want = fused(mlp, x).cpu(), reference(stock(mlp, torch.float32).cpu(), x.cpu())
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


# Grouped input: with features (gradient wanted or not, few or many), without, indices outside.
@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("features,tracked,n,m,s", [
    (0, False, 100, 7, 64), (3, False, 333, 40, 32), (5, True, 333, 40, 32), (61, True, 64, 33, 64),
    (64, False, 500, 30, 32), (64, True, 2048, 512, 32),
])
def test_grouped(cuda, monkeypatch, features, tracked, n, m, s, training):
    g = torch.Generator().manual_seed(n)
    mlp = make(mlp2d_bn_relu, features + 3, (36, 32, 64), training, cuda)
    xyz, centre = randn(1, 2, 3, n), randn(2, 2, 3, m)
    index = torch.randint(0, n, (2, m, s), generator=g)
    index[0, 0] = -1
    index = index.cuda()
    inputs = [(xyz, False), (centre, False), (index, False)]
    if features:
        inputs.append((randn(3, 2, features, n), tracked))

    def fused(mod, xyz, centre, index, f=None):
        return mod.forward_grouped_max(f, xyz, centre, index)

    def reference(mod, xyz, centre, index, f=None):
        return mod(group_points_with_xyz(f, xyz, centre, index)).max(dim=3)[0]

    check(mlp, fused, reference, inputs, monkeypatch)


# Three layers behind a grouping in one launch, in evaluation: tiles of 32 and of 64 positions, with half a tile left
# over; four waves and eight, with fewer channel blocks than waves and with more; the last layer's channels in one part
# and in several; activations that nearly fill LDS.
class GroupedPool(ctypes.Structure):  # tk3d_mlp_grouped_pool
    _fields_ = [("pointers", ctypes.c_void_p * 7), ("norms", ctypes.c_void_p * 15), ("out", ctypes.c_void_p),
                ("sizes", ctypes.c_int32 * 8)]


@pytest.mark.parametrize("b,features,n,m,s,widths", [
    (1, 0, 100, 7, 32, (32, 32, 32)), (1, 64, 100, 1, 64, (96, 128, 160)), (2, 3, 333, 257, 32, (64, 96, 32)),
    (3, 0, 40, 50, 32, (64, 128, 96)), (2, 5, 64, 64, 64, (128, 160, 256)), (9, 12, 50, 61, 32, (256, 256, 512)),
    (2, 3, 70, 80, 64, (32, 480, 64)), (5, 1, 300, 999, 32, (32, 64, 288)),
])
def test_grouped_in_one_launch(cuda, monkeypatch, b, features, n, m, s, widths):
    sizes = GroupedPool(sizes=(features + 3, b, n, m, s, *widths))
    assert _lib.lib().tk3d_mlp_grouped_pool_supported(ctypes.byref(sizes)) == 1
    for other in ((30, *widths[1:]), (widths[0], 4096, widths[2])):  # (the general chain's)
        sizes = GroupedPool(sizes=(features + 3, b, n, m, s, *other))
        assert _lib.lib().tk3d_mlp_grouped_pool_supported(ctypes.byref(sizes)) == 0
    mlp = make(mlp2d_bn_relu, features + 3, widths, False, cuda)
    xyz, centre = randn(1, b, 3, n), randn(2, b, 3, m)
    index = torch.randint(0, n, (b, m, s), generator=torch.Generator().manual_seed(n))
    index[0, 0] = -1
    inputs = [(xyz, False), (centre, False), (index.cuda(), False)]
    if features:
        inputs.append((randn(3, b, features, n), False))

    def fused(mod, xyz, centre, index, f=None):
        return mod.forward_grouped_max(f, xyz, centre, index)

    def reference(mod, xyz, centre, index, f=None):
        return mod(group_points_with_xyz(f, xyz, centre, index)).max(dim=3)[0]

    check(mlp, fused, reference, inputs, monkeypatch)
    xyz[0, 0, 0], xyz[-1, 2, -1] = float("inf"), float("nan")
    # (these stay where they are. In float64: a float32 convolution of the library's carries them over to the
    # positions beside.)
    with torch.no_grad():
        args = [t for t, _ in inputs]
        got = fused(mlp, *args)
        want = reference(stock(mlp, torch.float64), *[t.double() if t.is_floating_point() else t for t in args])
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


# Products in evaluation add up in several chains. Roundings of at most u = 2^-24 to numbers that grow as a
# random walk over n terms make an error of about 0.21 u sqrt(n) of the result (one chain over all K:
# 1.9 u at 64 channels, 3.4 u at 256, 6.9 u at 1024), in four chains half of it, in chains of 16 or
# 32 less; the norm adds less than u. (The library runs in one chain or in up to four, depending on the size.)
@pytest.mark.parametrize("b,p", [(1, 128), (1, 129), (8, 2048), (8, 16384)])
@pytest.mark.parametrize("k,c", [(64, 64), (72, 128), (256, 40), (768, 256), (1024, 64)])
def test_evaluation_adds_up_in_short_chains(cuda, b, p, k, c):
    if b * p * max(k, c) > 3 << 25:
        b = 1
    mlp = mlp1d_bn_relu(k, [c]).to(cuda).eval()
    x = torch.relu(randn(k, b, k, p))
    with torch.no_grad():
        got, exact = mlp(x), stock(mlp, torch.float64)(x.double())
    error = float((got.double() - exact).norm() / exact.norm())
    assert error <= 2.0 ** -24 * (1.0 + 0.11 * k ** 0.5), error


# The gradient of the input, where the tiles are 32 x 32: four chains over the output channels too. What
# dy itself brings along (products, statistics and coefficients in float32) is below 2 u.
@pytest.mark.parametrize("k,c,p", [(64, 256, 128), (96, 512, 100), (32, 1024, 64)])
def test_input_gradients_add_up_in_short_chains(cuda, k, c, p):
    mlp = mlp1d_bn_relu(k, [c]).to(cuda).train()
    single, exact = stock(mlp, torch.float32), stock(mlp, torch.float64)
    x, g = randn(k, 4, k, p), randn(c, 4, c, p)
    leaf, leaf64 = x.clone().requires_grad_(), x.double().requires_grad_()
    (got,) = torch.autograd.grad(mlp(leaf), leaf, g)
    with torch.no_grad():  # (the signs of the float32 activations)
        sign = single[0].bn(single[0].conv(x)) > 0
    (want,) = torch.autograd.grad(exact[0].bn(exact[0].conv(leaf64)) * sign, leaf64, g.double())
    error = float((got.double() - want).norm() / want.norm())
    assert error <= 2.0 ** -24 * (2.0 + 0.11 * c ** 0.5), error / 2.0 ** -24


# In training mode the activations and statistics are the stock modules' own, bit by bit, and so are
# the signs the backward takes: gradients differ by sums in another order alone, 1.5e-6 over 40
# steps of whole networks (four times that is the bound), where a single sign gave 1e-2.
@pytest.mark.parametrize("b,p,widths,pool", [(3, 1000, (6, 64, 33), 0), (2, 512, (67, 64, 128), 32),
                                             (1, 130, (20, 128, 40), 64), (2, 4096, (9, 32, 32), 0)])
def test_training_is_that_of_the_stock_modules(cuda, b, p, widths, pool):
    mlp = make(mlp2d_bn_relu if pool else mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    plain = stock(mlp, torch.float32)
    x = randn(p, b, widths[0], p, *([pool] if pool else []))
    results = []
    for module in (mlp, plain):
        leaf = x.clone().requires_grad_()
        if pool:
            out = mlp.forward_max(leaf) if module is mlp else module(leaf).max(dim=3)[0]
        else:
            out = module(leaf)
        grads = torch.autograd.grad(out, [leaf, *module.parameters()], torch.sin(out.detach() * 50))
        results.append((out.detach(), [t.clone() for t in module.buffers()], grads))
    assert torch.equal(results[0][0], results[1][0])
    assert all(torch.equal(a, c) for a, c in zip(results[0][1], results[1][1]))
    for a, c in zip(results[0][2], results[1][2]):
        assert float((a - c).norm()) <= 6e-6 * float(c.norm())


def pinned(single, exact, x, x64):
    """The maxima over neighbours of the float64 chain `exact`, with the signs and places of the
    float32 chain `single` (the same layers): what differs in its gradients is arithmetic alone."""
    for a, b in zip(single, exact):
        with torch.no_grad():
            z = a.bn(a.conv(x))
            x = torch.relu(z)
        x64 = b.bn(b.conv(x64)) * (z > 0)
    return x64.gather(3, z.max(dim=3, keepdim=True)[1]).squeeze(3)


# Activations in front of a pooled layer at up to `far` deviations from zero. The weight gradient is
# made of second moments there: about zero they give 2.1 times the stock modules' error at 3 and
# at 8, about the activations' mean 0.6 times. (The error of one draw is good to a tenth: a quarter is
# left for it.)
@pytest.mark.parametrize("far", [0, 3, 8])
@pytest.mark.parametrize("b,m,s,widths", [(8, 128, 64, (131, 128, 256)), (4, 513, 32, (9, 40, 33)),
                                          (2, 512, 32, (6, 64, 64, 128))])
def test_pooled_layer_far_from_zero(cuda, b, m, s, widths, far):
    mlp = make(mlp2d_bn_relu, widths[0], widths[1:], True, cuda)
    with torch.no_grad():
        for block in mlp:
            block.bn.weight.abs_().add_(0.5)
            block.bn.bias.add_(far * block.bn.weight)
    single, again, exact = stock(mlp, torch.float32), stock(mlp, torch.float32), stock(mlp, torch.float64)
    x, g = randn(m, b, widths[0], m, s), randn(3, b, widths[-1], m)
    grads = []
    for module, dtype in ((mlp, torch.float32), (single, torch.float32), (exact, torch.float64)):
        leaf = x.to(dtype).requires_grad_()
        if module is exact:
            out = pinned(again, exact, x, leaf)
        else:
            out = mlp.forward_max(leaf) if module is mlp else module(leaf).max(dim=3)[0]
        wanted = [leaf, *[p for block in module for p in (block.conv.weight, block.bn.weight)]]
        grads.append(torch.autograd.grad(out, wanted, g.to(dtype)))
    for mine, theirs, e in zip(*grads):
        errors = [float((t.double() - e).norm() / e.norm()) for t in (mine, theirs)]
        assert errors[0] <= 1.25 * errors[1] + 2e-7, (tuple(e.shape), errors)


# Short and long rows, few and many of them, one value a row: the library has a kernel for each.
@pytest.mark.parametrize("b,c,p", [
    (2, 5, 1), (3, 7, 33), (32, 64, 20), (2, 64, 510), (64, 32, 512), (1, 16, 516), (8, 3, 1000),
    (16, 64, 1024), (2, 64, 1028), (40, 33, 2048), (8, 64, 4096), (1, 8, 65536), (16, 32, 16384),
    (8, 64, 40960), (4, 32, 131072),
])
def test_the_backward_takes_the_signs_of_the_library(cuda, b, c, p):
    """The activations as the backward works them out are those of the library's batch norm, bit by
    bit."""
    class Norm(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in ("mean", "var", "gamma", "beta")] + [("eps", ctypes.c_float)]

    y = randn(p, b, c, p) * 3 + randn(1, c, 1) * 5
    gamma, beta = randn(2, c), randn(3, c)
    z, mean, inv_std, _, backend = torch._batch_norm_impl_index(
        y, gamma, beta, torch.zeros_like(gamma), torch.ones_like(gamma), True, 0.1, 1e-5, True)
    assert backend == 2  # MIOpen
    out = torch.empty_like(y)
    norm = Norm(*(t.data_ptr() for t in (mean, inv_std, gamma, beta)), -1.0)
    code = _lib.lib().tk3d_mlp_activate_f32(
        ctypes.c_void_p(y.data_ptr()), ctypes.c_int64(b * c), ctypes.c_int(c), ctypes.c_int(p),
        ctypes.byref(norm), ctypes.c_void_p(out.data_ptr()),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert code == 0 and torch.equal(out, torch.relu(z))


# Rows around the two orders of summation (4096 values), batches whose last thread chains are shorter
# than the others, one row, a group that is no power of two; a constant channel (a variance that rounds
# below zero), one with a NaN and one with an infinity.
@pytest.mark.parametrize("b,c,m,size", [
    (2, 5, 257, 4), (3, 4, 33, 32), (1, 64, 64, 64), (7, 33, 100, 20), (5, 6, 1023, 4), (2, 7, 128, 32),
    (3, 8, 1025, 4), (16, 33, 512, 32), (4, 5, 84, 63), (1, 2048, 64, 32), (512, 3, 128, 32),
    # (2^21 values a channel, the most that it takes, and just under them; rows of a segmentation step)
    (8, 64, 2048, 32), (32, 4, 2048, 32), (512, 3, 1023, 4), (1, 3, 32768, 64), (511, 3, 1026, 4),
])
def test_batch_norm_is_the_librarys_bit_by_bit(cuda, b, c, m, size):
    class Norm(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in
                    ("partial", "gamma", "beta", "running_mean", "running_var", "mean", "inv_std")] + [
                        ("eps", ctypes.c_double), ("momentum", ctypes.c_float),
                        ("B", ctypes.c_int32), ("C", ctypes.c_int32), ("P", ctypes.c_int32)]

    def pointers(*tensors):
        return [ctypes.c_void_p(t.data_ptr()) for t in tensors]

    y = randn(m, b, c, m, size) * (1 + randn(1, c, 1, 1).abs()) + randn(2, c, 1, 1) * 3
    y[:, 0] = 0.1
    y[0, 1, 1, 1] = float("nan")
    y[b - 1, 2 % c, 0, 3] = float("inf")
    gamma, beta = randn(3, c), randn(4, c)
    mine, theirs = ([randn(5, c), randn(6, c).abs()] for _ in range(2))
    z, mean, inv_std, _, backend = torch._batch_norm_impl_index(y, gamma, beta, *theirs, True, 0.3, 1e-3, True)
    assert backend == 2  # MIOpen
    lib, p, stream = _lib.lib(), m * size, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    lib.tk3d_mlp_batch_norm_partial_bytes.restype = ctypes.c_int64
    size_of = [ctypes.c_int64(v) for v in (b, c, p)]
    assert lib.tk3d_mlp_batch_norm_supported(*size_of) == 1
    partial = torch.empty(lib.tk3d_mlp_batch_norm_partial_bytes(size_of[1]), dtype=torch.uint8, device=cuda)
    got = [torch.empty(c, device=cuda) for _ in range(2)]
    norm = Norm(*(t.data_ptr() for t in (partial, gamma, beta, *mine, *got)), 1e-3, 0.3, b, c, p)
    assert lib.tk3d_mlp_batch_sums_f32(*pointers(y), b, c, p, *pointers(partial), stream) == 0
    out = torch.empty_like(y)
    assert lib.tk3d_mlp_batch_relu_f32(*pointers(y), ctypes.byref(norm), *pointers(out), stream) == 0
    for a, e in zip((out, *got, *mine), (z.relu(), mean, inv_std, *theirs)):
        assert torch.equal(a.isnan(), e.isnan()) and torch.equal(a.nan_to_num(7.0), e.nan_to_num(7.0))
    best, extreme = torch.empty(b, c, m, device=cuda), torch.empty(b, c, m, device=cuda)
    arg = torch.empty(b, c, m, dtype=torch.uint8, device=cuda)
    assert lib.tk3d_mlp_batch_pool_f32(*pointers(y), ctypes.byref(norm), size,
                                       *pointers(best, extreme, arg), stream) == 0
    top, where = z.max(dim=3)
    assert torch.equal(best.nan_to_num(7.0), top.relu().nan_to_num(7.0))
    there = z.gather(3, arg.long()[..., None])[..., 0]
    assert torch.equal(there.nan_to_num(7.0), top.nan_to_num(7.0))
    assert torch.equal(extreme.nan_to_num(7.0), y.gather(3, arg.long()[..., None])[..., 0].nan_to_num(7.0))
    # what it is not made for
    for shape in ((2, 8, 1024), (2, 8, 1030), (513, 8, 2048), (600, 1, 4096), (2, 2049, 2048)):
        assert lib.tk3d_mlp_batch_norm_supported(*(ctypes.c_int64(v) for v in shape)) == 0


@pytest.mark.parametrize("form", ["relu", "pool", "rows"])
def test_batches_are_counted(cuda, form):
    # by the pass that normalises, once a call and layer; where the count is not beside the values, or no int64, as before
    mlp = make(mlp2d_bn_relu if form == "pool" else mlp1d_bn_relu, 16, (32, 64, 32), True, cuda)
    norms = [m for m in mlp.modules() if isinstance(m, (nn.BatchNorm1d, nn.BatchNorm2d))]
    norms[0]._buffers["num_batches_tracked"] = torch.tensor(3)
    norms[1]._buffers["num_batches_tracked"] = torch.tensor(5, dtype=torch.int32, device=cuda)
    x = randn(4, 4, 16, 64, 32) if form == "pool" else randn(4, 4, 16, 2048)
    versions = [m.num_batches_tracked._version for m in norms]
    for call in (1, 2):
        if form == "pool":
            mlp.forward_max(x.requires_grad_())
        elif form == "rows":
            mlp.forward_points_max(x.requires_grad_())
        else:
            mlp(x.requires_grad_())
        assert [int(m.num_batches_tracked) for m in norms] == [3 + call, 5 + call, call]
        assert [m.num_batches_tracked._version for m in norms] == [v + call for v in versions]


@pytest.mark.parametrize("size", [20, 32, 64])
def test_a_maximum_is_the_first_of_equals(cuda, size):
    # quantised values (and their order is that of their norm: ascending or, with gamma < 0, descending), a
    # channel of one value, NaNs above all
    class Norm(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in
                    ("partial", "gamma", "beta", "running_mean", "running_var", "mean", "inv_std")] + [
                        ("eps", ctypes.c_double), ("momentum", ctypes.c_float),
                        ("B", ctypes.c_int32), ("C", ctypes.c_int32), ("P", ctypes.c_int32)]

    def pointers(*tensors):
        return [ctypes.c_void_p(t.data_ptr()) for t in tensors]

    b, c, m = 2, 6, 103
    y = (randn(size, b, c, m, size) * 1.5).round() / 2
    y[:, 3] = 0.25
    gamma, beta = torch.tensor([1.0, -1.0, 0.5, 2.0, 1.0, -2.0], device=cuda), randn(4, c)
    lib, p, stream = _lib.lib(), m * size, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    lib.tk3d_mlp_batch_norm_partial_bytes.restype = ctypes.c_int64
    partial = torch.empty(lib.tk3d_mlp_batch_norm_partial_bytes(ctypes.c_int64(c)), dtype=torch.uint8, device=cuda)
    state = [randn(5, c), randn(6, c).abs(), torch.empty(c, device=cuda), torch.empty(c, device=cuda)]
    norm = Norm(*(t.data_ptr() for t in (partial, gamma, beta, *state)), 1e-3, 0.3, b, c, p)
    assert lib.tk3d_mlp_batch_sums_f32(*pointers(y), b, c, p, *pointers(partial), stream) == 0
    y[0, :, ::5, 7] = float("nan")      # (behind the sums: the other values keep their norm)
    y[0, :, ::10, size - 1] = float("nan")
    out, extreme = torch.empty(b, c, m, device=cuda), torch.empty(b, c, m, device=cuda)
    arg = torch.empty(b, c, m, dtype=torch.uint8, device=cuda)
    assert lib.tk3d_mlp_batch_pool_f32(*pointers(y), ctypes.byref(norm), size, *pointers(out, extreme, arg),
                                       stream) == 0
    order = (y * gamma.sign()[:, None, None]).nan_to_num(float("inf"))
    first = (order == order.max(dim=3, keepdim=True)[0]).int().argmax(dim=3)
    assert torch.equal(arg.long(), first)
    there = y.gather(3, first[..., None])[..., 0]
    assert torch.equal(extreme.nan_to_num(7.0), there.nan_to_num(7.0)) and torch.equal(out.isnan(), there.isnan())


@pytest.mark.parametrize("b,m,s", [(1, 4097, 32), (3, 2731, 32), (5, 3277, 32), (1, 2049, 64), (3, 1366, 64), (3, 2731, 64)])
def test_scatter_of_several_groups_a_wave(cuda, b, m, s):
    # around the numbers of groups from which a wave takes two and four in a row, numbers that neither divides
    o, i = 5, 3
    place = torch.randint(0, s, (b, o, m), device=cuda, dtype=torch.int32)
    value, w = randn(m, b, o, m), randn(s, o, i)
    sel = torch.stack([value.view(torch.int32), place], dim=3).contiguous()
    out = torch.full((b, i, m, s), 7.0, device=cuda)
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in (sel, w)]
    assert _lib.lib().tk3d_mlp_pool_scatter_f32(*ptr, b, o, i, m, s, ctypes.c_void_p(out.data_ptr()),
                                                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    e = torch.zeros(b, o, m, s, dtype=torch.float64, device=cuda).scatter_(3, place.long()[..., None],
                                                                           value.double()[..., None])
    want = torch.einsum("oi,bop->bip", w.double(), e.flatten(2)).view_as(out)
    # (up to five terms of one sum, each rounded once, and the sum after each)
    assert ((out - want).abs() <= 6 * 2.0 ** -24 * torch.einsum(
        "oi,bop->bip", w.double().abs(), e.abs().flatten(2)).view_as(out) + 1e-30).all()


@pytest.mark.parametrize("form", ["dense", "edges"])
def test_without_the_library_training_is_left_to_stock(cuda, form):
    """torch's own batch norm rounds in another order than the backward takes its signs by."""
    from torkit3d_amd.ops.edge_conv import EdgeConvBlock

    index = torch.randint(0, 40, (2, 40, 5), generator=torch.Generator().manual_seed(0)).to(cuda)
    block = EdgeConvBlock(6, (8,)).to(cuda).train()
    mlp = make(mlp1d_bn_relu, 6, (8, 5), True, cuda)
    x = randn(1, 2, 6, 40).requires_grad_()

    def ran():
        if form == "dense":
            return "Node" in mlp(x).grad_fn.name()
        return block.convs.forward_edges_max(x, index) is not None

    assert ran()
    with torch.backends.cudnn.flags(enabled=False):
        assert not ran()


@pytest.mark.parametrize("p", [514, 1030])
def test_rows_on_which_the_library_differs_run_in_stock(cuda, p):
    mlp = make(mlp1d_bn_relu, 6, (8, 5), True, cuda)
    out = mlp(randn(1, 2, 6, p).requires_grad_())
    assert "Relu" in out.grad_fn.name()
    assert "Node" in mlp(randn(1, 2, 6, p + 2).requires_grad_()).grad_fn.name()


def test_gradient_of_a_gradient(cuda):
    mlp = make(mlp1d_bn_relu, 6, (8, 5), True, cuda)
    results = []
    for module in (mlp, stock(mlp, torch.float32)):
        x = randn(4, 2, 6, 20).requires_grad_()
        out = module(x)
        (first,) = torch.autograd.grad(out.square().sum(), x, create_graph=True)
        results.append((first.detach(), *torch.autograd.grad(first.square().sum(),
                                                             [x, *module.parameters()])))
    for a, b in zip(*results):
        assert float((a - b).norm()) <= 1e-4 * float(b.norm()) + 1e-6


# The same of a maximum over all points, on the layer's own input and on activations.
@pytest.mark.parametrize("b,p,widths", [(13, 2048, (70, 160)), (3, 1400, (9, 64, 128))])
def test_gradient_of_a_gradient_of_a_maximum_over_points(cuda, b, p, widths):
    mlp = make(mlp1d_bn_relu, widths[0], widths[1:], True, cuda)
    results = []
    for module in (mlp, stock(mlp, torch.float32)):
        x = randn(4, b, widths[0], p).requires_grad_()
        if module is mlp:
            out = mlp.forward_points_max(x)[0]
            assert "Node" in out.grad_fn.name()
        else:
            out = torch.max(module(x), 2)[0]
        (first,) = torch.autograd.grad(out.square().sum(), x, create_graph=True)
        results.append((first.detach(), *torch.autograd.grad(first.square().sum(),
                                                             [x, *module.parameters()])))
    for a, b in zip(*results):
        assert float((a - b).norm()) <= 1e-4 * float(b.norm()) + 1e-6


def test_what_is_not_plain_runs_layer_by_layer(cuda):
    mlp = make(mlp1d_bn_relu, 6, (8, 5), True, cuda)
    x = randn(5, 2, 6, 20)
    seen = []
    handle = mlp[0].bn.register_forward_hook(lambda *a: seen.append(1))
    mlp(x)
    assert seen == [1]
    handle.remove()
    mlp[1].bn.eval()  # a frozen layer among training ones
    assert torch.allclose(mlp(x), stock_forward(mlp, x), atol=1e-5)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        mlp(x)
    nan = x.clone()
    nan[0, 0, 0] = float("nan")
    mlp.eval()
    assert torch.equal(mlp(nan).isnan(), nn.Sequential.forward(mlp, nan).isnan())


def stock_forward(mlp, x):
    return nn.Sequential.forward(mlp, x)


# EdgeConv on a graph of a cloud with itself: points around the workgroup's 16, 32 and 64, channels
# around its 64 and around the 16 of a step, neighbours around the eight rows requested at once; lists
# given or not.
@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("b,c,n,k,o,lists", [
    (1, 3, 5, 2, 5, False), (2, 3, 33, 7, 64, False), (3, 64, 100, 20, 65, True),
    (2, 70, 31, 9, 130, True), (8, 64, 2048, 20, 64, True), (1, 6, 5000, 40, 128, False),
    (2, 15, 65, 5, 70, False), (2, 16, 64, 20, 64, False), (3, 130, 17, 3, 40, True),
])
def test_edge_conv(cuda, b, c, n, k, o, lists, training):
    from torkit3d_amd.ops.edge_conv import EdgeConvBlock, get_edge_feature_builtin

    torch.manual_seed(1)
    block = EdgeConvBlock(c, [o])
    block.convs = make(mlp2d_bn_relu, 2 * c, [o], training, cuda)
    index = torch.randint(0, n, (b, n, k), generator=torch.Generator().manual_seed(n)).to(cuda)
    x = randn(7, b, c, n)
    results = []
    for dtype in (None, torch.float32, torch.float64):
        leaf = x.clone().to(dtype or torch.float32).requires_grad_()
        if dtype is None:
            module = block.convs
            extra = {"lists": edge_lists(index, n)} if lists else {}
            with torch.set_grad_enabled(training):
                out = module.forward_edges_max(leaf, index, **extra)
            assert out is not None, "the fused kernels did not run"
        else:
            module = saved if dtype == torch.float32 else saved64
            out = module(get_edge_feature_builtin(leaf, leaf, index)).max(dim=3)[0]
        grad = torch.sin(torch.arange(out.numel(), device=cuda, dtype=torch.float64) * 1.7)
        grads = torch.autograd.grad(out, [leaf, *module.parameters()],
                                    grad.view_as(out).to(out.dtype)) if training else ()
        results.append([out.detach(), *grads, *[t.clone() for t in module.buffers()]])
        if dtype is None:
            # (statistics as they were before this pass)
            fresh = make(mlp2d_bn_relu, 2 * c, [o], training, cuda)
            saved, saved64 = stock(fresh, torch.float32), stock(fresh, torch.float64)
    for i, (a, s, e) in enumerate(zip(*results)):
        assert a.shape == e.shape
        if not e.is_floating_point():
            assert torch.equal(a, e)
            continue
        norm = float(e.norm()) + 1e-30
        mine, theirs = float((a.double() - e).norm()) / norm, float((s.double() - e).norm()) / norm
        assert mine <= 4 * theirs + 2e-6, (i, tuple(e.shape), mine, theirs)


# The sums over the edges whose value is the maximum, in LDS: rows around the 2048 points of a part, the last channel
# alone in its workgroup of two, rows that fit LDS once but not twice, few rows just beyond those that are added there
# (four neighbours: the fused training takes more than 512 edges of a cloud only in multiples of four).
@pytest.mark.parametrize("b,c,n,k,o", [
    (2, 4, 2047, 4, 5), (1, 4, 2049, 4, 6), (1, 3, 4096 + 511, 4, 3), (172, 3, 40, 3, 3), (104, 3, 2049, 4, 5),
    (64, 3, 7168, 4, 8), (64, 3, 7169, 4, 8), (1, 3, 6144, 4, 6), (1, 3, 6145, 4, 6),
])
def test_edge_sums_of_maxima(cuda, b, c, n, k, o):
    test_edge_conv(cuda, b, c, n, k, o, False, True)


# On a graph of near neighbours, with the cloud at `far` from the origin: y taken apart into a term
# of the neighbour and one of the point loses what their difference keeps, unless the products are more
# exact than float32 (with float32 products the error of the activations was 1.1 to 1.7 times the stock
# modules' here, that of the weights' first half 1.1 to 2.7 times). The bound as for pooled layers.
@pytest.mark.parametrize("far", [0.0, 0.5, 3.0])
@pytest.mark.parametrize("c,o", [(3, 64), (6, 64), (16, 64), (64, 128)])
def test_edge_conv_is_as_exact_as_the_stock_modules(cuda, c, o, far):
    from torkit3d_amd.ops.edge_conv import EdgeConvBlock, get_edge_feature_builtin
    from torkit3d_amd.ops.knn_points import knn_points

    xyz = torch.rand(4, 3, 1024, generator=torch.Generator().manual_seed(c)).to(cuda) - 0.5
    index = knn_points(xyz, xyz, 20, transpose=True)[1]
    x = xyz + far
    if c > 3:
        x = torch.relu(torch.matmul(randn(1, c, 3), xyz)) + far
    block = EdgeConvBlock(c, [o])
    block.convs = make(mlp2d_bn_relu, 2 * c, [o], True, cuda)
    single, again, exact = (stock(block.convs, t) for t in (torch.float32, torch.float32, torch.float64))
    g = randn(2, 4, o, 1024)
    results = []
    for module in (block, single, exact):
        leaf = x.to(g.dtype if module is not exact else torch.float64).requires_grad_()
        if module is block:
            out = block(leaf, leaf, index)
        elif module is single:
            out = single(get_edge_feature_builtin(leaf, leaf, index)).max(dim=3)[0]
        else:
            out = pinned(again, exact, get_edge_feature_builtin(x, x, index),
                         get_edge_feature_builtin(leaf, leaf, index))
        chain = block.convs if module is block else module
        dx, dw = torch.autograd.grad(out, [leaf, chain[0].conv.weight], g.to(out.dtype))
        chain.eval()
        with torch.no_grad():
            z = (block(x, x, index) if module is block else
                 chain(get_edge_feature_builtin(*(leaf.detach(),) * 2, index)).max(dim=3)[0])
        results.append([dx, dw[:, :c], dw[:, c:], z])
    for mine, theirs, e in zip(*results):
        errors = [float((t.double() - e).norm() / e.norm()) for t in (mine, theirs)]
        assert errors[0] <= 1.25 * errors[1] + 2e-8, (tuple(e.shape), errors)


def test_edge_conv_lists_are_checked(cuda):
    """What is not the inverse of a graph of this size is refused, and whatever such a tensor holds,
    the backward stays inside it and inside the cloud."""
    from torkit3d_amd.ops.edge_conv import EdgeConvBlock

    block = EdgeConvBlock(4, [8]).to(cuda).train()
    b, n, k = 2, 50, 6
    index = torch.randint(0, n, (b, n, k), generator=torch.Generator().manual_seed(0)).to(cuda)
    x = randn(8, b, 4, n).requires_grad_()
    lists = edge_lists(index, n)
    shorter = edge_lists(index[:, :40, :].clamp(max=39).contiguous(), 40)
    for wrong in (shorter, edge_lists(index[:, :, :5].contiguous(), n), lists[:1], lists.long(),
                  lists.cpu(), lists.view(-1), lists.t().contiguous().t()):
        with pytest.raises(RuntimeError, match="lists"):
            block(x, x, index, lists=wrong)
    block(x, x, index, lists=lists).sum().backward()
    low, high = torch.iinfo(torch.int32).min, torch.iinfo(torch.int32).max
    noise = torch.randint(low, high, tuple(lists.shape), dtype=torch.int32,
                          generator=torch.Generator().manual_seed(1)).to(cuda)
    noise[1, : n + 1] = torch.arange(n + 1, dtype=torch.int32, device=cuda) * k
    for any_lists in (noise, torch.full_like(lists, low), torch.full_like(lists, high)):
        x.grad = None
        block(x, x, index, lists=any_lists).sum().backward()
        assert torch.isfinite(x.grad).all()


def test_edge_conv_with_indices_outside(cuda):
    """A neighbour outside the cloud reads as zeros, as ``group_points`` reads it."""
    from torkit3d_amd.ops.edge_conv import EdgeConvBlock, get_edge_feature_custom

    block = EdgeConvBlock(4, [8])
    block.convs = make(mlp2d_bn_relu, 8, [8], True, cuda)
    index = torch.randint(0, 50, (2, 50, 6), generator=torch.Generator().manual_seed(0)).to(cuda)
    index[0, :, 2], index[1, 3, :] = -1, 50
    x, y = randn(8, 2, 4, 50).requires_grad_(), randn(8, 2, 4, 50).requires_grad_()
    out = block(x, x, index)
    ref = stock(make(mlp2d_bn_relu, 8, [8], True, cuda), torch.float32)(
        get_edge_feature_custom(y, y, index)).max(dim=3)[0]
    torch.testing.assert_close(out, ref, rtol=1e-5, atol=1e-5)
    weight = randn(9, *out.shape)
    (out * weight).sum().backward()
    (ref * weight).sum().backward()
    torch.testing.assert_close(x.grad, y.grad, rtol=1e-4, atol=1e-4)


# The inverse of a graph: several slices of a cloud and one, points without edges, a cloud whose edges all go to one
# point, indices outside.
@pytest.mark.parametrize("b,n,k", [(8, 2048, 20), (3, 1000, 20), (2, 32768, 4), (300, 70, 2), (1, 129, 3), (1, 1, 1)])
def test_edge_lists(cuda, b, n, k):
    index = torch.randint(-1, n + 1, (b, n, k), generator=torch.Generator().manual_seed(n))
    index[0] = n // 2
    lists = edge_lists(index.to(cuda), n).cpu()
    for i in range(b):
        counts = torch.bincount(index[i][(index[i] >= 0) & (index[i] < n)], minlength=n)
        assert torch.equal(lists[i, :n + 1], torch.cat([counts.new_zeros(1), counts.cumsum(0)]).int())
        edges = lists[i, n + 1:n + 1 + int(counts.sum())].long()
        assert torch.equal(index[i][edges >> 8, edges & 255], torch.repeat_interleave(torch.arange(n), counts))
        assert len(set(edges.tolist())) == len(edges)
