"""Workloads by which the performance of this package is measured.

A case is a dict of plain values. ``listed()`` gives the fixed ones, ``draw(rng)`` another one
of the same ranges, ``prepare(case, seed)`` what a user's program holds before the call, and
``run(state)`` one pass through the public entry points. Five families:

  chamfer      ``chamfer_distance`` forward and backward (the loss of a completion or
               reconstruction network), or ``nn_distance`` (the same as a metric, no gradients)
  abstraction  one or more PointNet++ levels without their MLPs: farthest point sampling, ball
               query, grouping with centred coordinates, and the grouping's backward
  propagation  3-NN weights and feature interpolation, forward and backward
  knn          ``knn_points``
  model        a forward pass in evaluation mode, or a forward and backward pass in training
               mode, of a model of ``torkit3d_amd.models`` with its default constructor

Everything is float32, the type the models train and serve in: float64 exists for gradient
checks, and no entry point takes a shorter type. Clouds are [B, 3, N] where the call says
``channels_first`` and in the model family, else [B, N, 3].
"""
import torch
from torch import nn

from torkit3d_amd.models.classification.dgcnn import DGCNN
from torkit3d_amd.models.classification.pointnet import PointNet
from torkit3d_amd.models.classification.pointnet2 import PN2SSG as PN2Classification
from torkit3d_amd.models.segmentation.pointnet2 import PN2SSG as PN2Segmentation
from torkit3d_amd.ops.ball_query import ball_query
from torkit3d_amd.ops.chamfer_distance import chamfer_distance, nn_distance
from torkit3d_amd.ops.group_points import group_points_with_xyz
from torkit3d_amd.ops.interpolate_feature import interpolate_feature, three_nn_interpolation
from torkit3d_amd.ops.knn_points import knn_points
from torkit3d_amd.ops.sample_farthest_points import sample_farthest_points_gather

MODELS = {"pointnet": PointNet, "pn2_cls": PN2Classification, "pn2_seg": PN2Segmentation,
          "dgcnn": DGCNN}
NUM_CLASSES = {"pointnet": 40, "pn2_cls": 40, "pn2_seg": 20, "dgcnn": 40}


# ---- cases --------------------------------------------------------------------------------


def chamfer(batch, n1, n2, cloud, channels_first=False, sqrt=False, grads="both"):
    return {"family": "chamfer", "batch": batch, "n1": n1, "n2": n2, "cloud": cloud,
            "channels_first": channels_first, "sqrt": sqrt, "grads": grads}


def abstraction(batch, n, channels, levels, radius, neighbors, cloud):
    return {"family": "abstraction", "batch": batch, "n": n, "channels": channels,
            "levels": levels, "radius": radius, "neighbors": neighbors, "cloud": cloud}


def propagation(batch, n1, n2, channels, channels_first):
    return {"family": "propagation", "batch": batch, "n1": n1, "n2": n2, "channels": channels,
            "channels_first": channels_first}


def knn(batch, n1, n2, k, channels_first=False, ordered=False, sqrt=False):
    return {"family": "knn", "batch": batch, "n1": n1, "n2": n2, "k": k,
            "channels_first": channels_first, "ordered": ordered, "sqrt": sqrt}


def model(which, batch, n, features, train):
    return {"family": "model", "model": which, "batch": batch, "n": n, "features": features,
            "train": train}


def listed():
    cases = {
        # The loss of a small reconstruction head: launches and host time are all of it.
        "chamfer_small": chamfer(2, 1024, 1024, "uniform"),
        # A completion network's loss: predicted cloud against a ground truth of another, odd
        # length, channel-first as the network's last layer leaves it, only the prediction has
        # a gradient, distances instead of their squares.
        "chamfer_ragged": chamfer(8, 2500, 3001, "sphere", True, True, "first"),
        # The largest: dense surface clouds.
        "chamfer_large": chamfer(32, 16384, 16384, "sphere"),
        # One encoder level at a training batch.
        "abstraction_level": abstraction(16, 4096, 64, 1, 0.2, 32, "uniform"),
        # A whole encoder on large clouds: each level samples the previous level's picks.
        "abstraction_chain": abstraction(8, 16384, 32, 3, 0.1, 32, "uniform"),
        # A decoder's last level: features carried from 2048 points back to 8192.
        "propagation": propagation(32, 8192, 2048, 128, False),
        # Neighbourhoods of a whole batch.
        "knn_k16": knn(32, 8192, 2048, 16),
        # A few queries with many neighbours on a long cloud, sorted.
        "knn_k64_sorted": knn(4, 512, 10000, 64, False, True, True),
        # Serving one cloud: the latency of a whole network's forward pass.
        "model_cls_serve": model("pn2_cls", 1, 1024, 0, False),
        # Training steps of the three networks built on the ops.
        "model_cls_train": model("pn2_cls", 16, 4096, 3, True),
        "model_seg_train": model("pn2_seg", 8, 16384, 3, True),
        "model_dgcnn_train": model("dgcnn", 8, 2048, 0, True),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_uniform(rng, low, high):
    """A whole number from ``low`` to ``high``, spread over its logarithm."""
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw(rng):
    family = rng.choice(["chamfer", "abstraction", "propagation", "knn", "model", "model"])
    if family == "chamfer":
        n1 = _log_uniform(rng, 512, 16384)
        n2 = min(16384, max(256, round(n1 * 2.0 ** rng.uniform(-2, 2))))
        batch = _log_uniform(rng, 1, min(32, 2 ** 19 // max(n1, n2)))
        return chamfer(batch, n1, n2, rng.choice(["uniform", "sphere", "clusters"]),
                       rng.random() < 0.5, rng.random() < 0.25,
                       rng.choice(["both", "first", "none"]))
    if family == "abstraction":
        n = _log_uniform(rng, 512, 16384)
        return abstraction(_log_uniform(rng, 1, min(16, 2 ** 17 // n)), n, rng.choice([16, 32, 61, 64]),
                           rng.choice([1, 2, 3]), round(rng.uniform(0.1, 0.3), 3),
                           rng.choice([16, 24, 32, 64]), rng.choice(["uniform", "sphere", "clusters"]))
    if family == "propagation":
        n1 = _log_uniform(rng, 128, 16384)
        return propagation(_log_uniform(rng, 1, min(32, 2 ** 18 // n1)), n1,
                           max(16, round(n1 / rng.uniform(2, 8))), rng.choice([64, 128, 131, 256]),
                           rng.random() < 0.5)
    if family == "knn":
        n1, n2 = _log_uniform(rng, 256, 8192), _log_uniform(rng, 256, 16384)
        return knn(_log_uniform(rng, 1, max(1, min(32, 2 ** 29 // (n1 * n2)))), n1, n2,
                   rng.choice([1, 3, 8, 16, 20, 32, 64]), rng.random() < 0.5, rng.random() < 0.25,
                   rng.random() < 0.25)
    which = rng.choice(sorted(MODELS))
    low, points = {"pointnet": (512, 2 ** 16), "pn2_cls": (600, 2 ** 16), "pn2_seg": (2048, 2 ** 17),
                   "dgcnn": (256, 2 ** 14)}[which]
    n = _log_uniform(rng, low, {"pn2_seg": 16384, "dgcnn": 4096}.get(which, 8192))
    train = rng.random() < 0.6
    batch = _log_uniform(rng, 2 if train else 1, max(2, min(32, points // n)))
    features = rng.choice([0, 3]) if which.startswith("pn2") else 0
    return model(which, batch, n, features, train)


# ---- what a user's program holds ----------------------------------------------------------


def _cloud(gen, kind, batch, n, channels_first):
    dev = gen.device
    if kind == "uniform":  # a volume: the unit cube
        cloud = torch.rand(batch, n, 3, generator=gen, device=dev)
    elif kind == "sphere":  # a scanned surface: a sphere with measurement noise
        cloud = torch.randn(batch, n, 3, generator=gen, device=dev)
        cloud = cloud / cloud.norm(dim=2, keepdim=True)
        cloud = cloud + 0.01 * torch.randn(batch, n, 3, generator=gen, device=dev)
    else:  # objects in a scene: eight Gaussian blobs
        centres = torch.rand(batch, 8, 3, generator=gen, device=dev) * 2 - 1
        which = torch.randint(0, 8, (batch, n, 1), generator=gen, device=dev)
        cloud = torch.gather(centres, 1, which.expand(-1, -1, 3))
        cloud = cloud + 0.1 * torch.randn(batch, n, 3, generator=gen, device=dev)
    return (cloud.transpose(1, 2) if channels_first else cloud).contiguous()


def _level_sizes(case):
    """(points, samples, channels, radius, neighbours) of every abstraction level."""
    n, radius, sizes = case["n"], case["radius"], []
    for level in range(case["levels"]):
        m = max(1, n // 4)
        sizes.append((n, m, case["channels"] << level, radius * 2 ** level,
                      case["neighbors"] * (2 if level == 2 else 1)))
        n = m
    return sizes


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    family, b = case["family"], case["batch"]
    state = dict(case)
    if family == "chamfer":
        for name in ("1", "2"):
            n = case["n" + name]
            state["xyz" + name] = _cloud(gen, case["cloud"], b, n, case["channels_first"])
            state["grad" + name] = randn(b, n) / n  # of a loss that averages over the points
        state["xyz1"].requires_grad_(case["grads"] != "none")
        state["xyz2"].requires_grad_(case["grads"] == "both")
    elif family == "abstraction":
        state["points"] = _cloud(gen, case["cloud"], b, case["n"], True)
        state["features"] = [randn(b, c, n).requires_grad_()
                             for n, _, c, _, _ in _level_sizes(case)]
        state["grads"] = [randn(b, c + 3, m, k) for _, m, c, _, k in _level_sizes(case)]
    elif family == "propagation":
        state["query"] = _cloud(gen, "uniform", b, case["n1"], case["channels_first"])
        state["key"] = _cloud(gen, "uniform", b, case["n2"], case["channels_first"])
        state["feature"] = randn(b, case["channels"], case["n2"]).requires_grad_()
        state["grad"] = randn(b, case["channels"], case["n1"])
    elif family == "knn":
        state["query"] = _cloud(gen, "uniform", b, case["n1"], case["channels_first"])
        state["key"] = _cloud(gen, "uniform", b, case["n2"], case["channels_first"])
    else:
        which = case["model"]
        with torch.random.fork_rng(devices=[dev]):
            torch.manual_seed(seed)
            if which in ("pointnet", "dgcnn"):
                net = MODELS[which]()
            else:
                net = MODELS[which](case["features"])
            classes = NUM_CLASSES[which]
            head = (nn.Conv1d(net.out_channels - case["features"], classes, 1)
                    if which == "pn2_seg" else nn.Linear(net.out_channels, classes))
        state["net"], state["head"] = net.to(dev).train(case["train"]), head.to(dev).train(case["train"])
        state["points"] = _cloud(gen, "uniform", b, case["n"], True)
        state["feature"] = randn(b, case["features"], case["n"]) if case["features"] else None
        if which == "pn2_seg":  # a point's class follows from where it is: 5 by 4 columns
            x, y = state["points"][:, 0], state["points"][:, 1]
            state["labels"] = (x * 5).long().clamp(0, 4) * 4 + (y * 4).long().clamp(0, 3)
        else:
            state["labels"] = torch.randint(0, classes, (b,), generator=gen, device=dev)
    return state


# ---- one pass -----------------------------------------------------------------------------


def _run_chamfer(s):
    x, y, transpose = s["xyz1"], s["xyz2"], s["channels_first"]
    if s["grads"] == "none":
        return nn_distance(x, y, transpose=transpose)
    dist1, dist2 = chamfer_distance(x, y, transpose=transpose, sqrt=s["sqrt"])
    wanted = (x, y) if s["grads"] == "both" else (x,)
    return [dist1, dist2, *torch.autograd.grad((dist1, dist2), wanted, (s["grad1"], s["grad2"]))]


def _run_abstraction(s):
    points, out = s["points"], []
    for (_, m, _, radius, k), feature, grad in zip(_level_sizes(s), s["features"], s["grads"]):
        index, centres = sample_farthest_points_gather(points, m, transpose=True)
        neighbours = ball_query(centres, points, radius, k)
        grouped = group_points_with_xyz(feature, points, centres, neighbours)
        (grad_feature,) = torch.autograd.grad(grouped, feature, grad)
        out += [index, centres, neighbours, grouped, grad_feature]
        points = centres
    return out


def _run_propagation(s):
    distance, index, weight = three_nn_interpolation(s["query"], s["key"], s["channels_first"])
    carried = interpolate_feature(s["feature"], index, weight)
    (grad_feature,) = torch.autograd.grad(carried, s["feature"], s["grad"])
    return distance, index, weight, carried, grad_feature


def _run_model(s):
    net, head = s["net"], s["head"]
    inputs = (s["points"],) if s["feature"] is None else (s["points"], s["feature"])
    if not s["train"]:
        with torch.no_grad():
            return head(net(*inputs)["feature"])
    logits = head(net(*inputs)["feature"])
    loss = nn.functional.cross_entropy(logits, s["labels"])
    weights = [*net.parameters(), *head.parameters()]
    grads = torch.autograd.grad(loss, weights, allow_unused=True)
    # (the gradients as clipping or an all-reduce takes them: one flat vector)
    flat = torch.cat([g.reshape(-1) for g in grads if g is not None])
    statistics = torch.cat([t for name, t in net.named_buffers() if name.endswith(("_mean", "_var"))])
    return {"logits": logits, "loss": loss, "grads": flat, "statistics": statistics}


def run(state):
    family = state["family"]
    if family == "chamfer":
        return _run_chamfer(state)
    if family == "abstraction":
        return _run_abstraction(state)
    if family == "propagation":
        return _run_propagation(state)
    if family == "knn":
        return knn_points(state["query"], state["key"], state["k"], sorted=state["ordered"],
                          sqrt_distance=state["sqrt"], transpose=state["channels_first"])
    return _run_model(state)


# ---- what it takes, and how exact it is ----------------------------------------------------

DISTANCE_FLOPS = 8  # three differences, three products, two sums


def _mlp_flops(widths, positions):
    return sum(2 * a * b * positions for a, b in zip(widths, widths[1:]))


def _model_work(case):
    """(parameters, operations of the matrix products of a forward pass). A neighbourhood's
    first layer is linear in the neighbour's features, so its product with them is counted once
    per point of the level, not once per neighbour."""
    which, b, n, f = case["model"], case["batch"], case["n"], case["features"]
    classes, params, flops = NUM_CLASSES[which], 0, 0

    def mlp(widths, positions):
        nonlocal params, flops
        params += sum(a * c + 2 * c for a, c in zip(widths, widths[1:]))
        flops += _mlp_flops(widths, positions)

    if which == "pointnet":
        mlp((3, 64, 64, 64, 128, 1024), b * n)
        mlp((1024, 512, 256, classes), b)
    elif which == "dgcnn":
        width = 3
        for out in (64, 64, 64, 128):
            mlp((2 * width, out), b * n)
            width = out
        mlp((320, 1024), b * n)
        mlp((1024, 512, 256, classes), b)
    else:
        if which == "pn2_cls":
            levels = ((512, 32, (64, 64, 128)), (128, 64, (128, 128, 256)))
        else:
            levels = ((2048, 32, (32, 32, 64)), (512, 32, (64, 64, 128)),
                      (128, 32, (128, 128, 256)), (32, 32, (256, 256, 512)))
        width, points, sizes = f, n, [n]
        for m, k, channels in levels:
            if width:
                mlp((width, channels[0]), b * points)
            mlp((3, channels[0]), b * m * k)
            mlp(channels, b * m * k)
            width, points = channels[-1], m
            sizes.append(m)
        if which == "pn2_cls":
            mlp((256, 256, 512, 1024), b * sizes[-1])
            mlp((1024, classes), b)
        else:
            mlp((768, 256, 256), b * sizes[3])
            mlp((384, 256, 256), b * sizes[2])
            mlp((320, 256, 128), b * sizes[1])
            mlp((128 + f, 128, 128, 128), b * n)
            mlp((128, classes), b * n)
    return params, flops


def work(case):
    family, b = case["family"], case["batch"]
    if family == "chamfer":
        n1, n2 = case["n1"], case["n2"]
        own, other = 12 * b * n1, 12 * b * n2
        dists = 4 * b * (n1 + n2)
        flops = DISTANCE_FLOPS * b * (n1 + n2)
        if case["grads"] == "none":
            return {"bytes": own + other + 3 * dists, "flops": flops}  # (and an int64 index each)
        back = own + (other if case["grads"] == "both" else 0)
        return {"bytes": own + other + 2 * dists + back, "flops": 2 * flops}
    if family == "abstraction":
        size = flops = 0
        for n, m, c, _, k in _level_sizes(case):
            size += b * (12 * n + 12 * m + 8 * m + 8 * m * k + 4 * c * n)  # clouds, picks, indices
            size += b * (2 * 4 * (c + 3) * m * k + 4 * c * n)  # grouped, its gradient, the sum
            flops += b * ((c + 3) * m * k + DISTANCE_FLOPS * (n + m * k))
        return {"bytes": size, "flops": flops}
    if family == "propagation":
        n1, n2, c = case["n1"], case["n2"], case["channels"]
        return {"bytes": b * (12 * (n1 + n2) + 48 * n1 + 2 * 4 * c * (n1 + n2)),
                "flops": b * n1 * (DISTANCE_FLOPS * 3 + 2 * 6 * c)}
    if family == "knn":
        n1, n2, k = case["n1"], case["n2"], case["k"]
        return {"bytes": b * (12 * (n1 + n2) + 12 * n1 * k), "flops": DISTANCE_FLOPS * b * n1 * k}
    params, flops = _model_work(case)
    b, n, f = case["batch"], case["n"], case["features"]
    outputs = NUM_CLASSES[case["model"]] * (b * n if case["model"] == "pn2_seg" else b)
    size = 4 * (b * n * (3 + f) + params + outputs)
    if case["train"]:
        return {"bytes": size + 4 * params, "flops": 3 * flops}
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # Indices and the distances that decide them are the same for every implementation: the
    # arithmetic of a distance is fixed. Sums of float32 terms may come in another order.
    if case["family"] != "model":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if not case["train"]:
        return {"rel": 1e-5, "max": 1e-3}
    # A training step divides by batch statistics and selects by maxima and signs: last-bit
    # differences in a few of millions of activations send their gradients elsewhere, and the
    # gradient in front of a batch norm is what remains of a large cancelling sum. Two stock
    # float32 back ends (with and without MIOpen) differ by up to 9e-3 (largest entry 0.5) of
    # the flat gradient on the segmentation network, 3e-3 (0.13) on the others.
    if case["model"] == "pn2_seg":
        return {"rel": 0.03, "max": 0.99}
    return {"rel": 0.01, "max": 0.5}
