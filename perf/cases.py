"""What users of this framework have it do, as cases whose speed is measured.

A case is a dict of plain values.  Its "kind" names the path:

  layer     one steerable convolution on a voxelised batch, as a training loop (rulebook,
            kernel synthesis, convolution, optionally the backward pass) or an inference loop
            (filters synthesised once) calls it
  down      a strided convolution followed by the sparse max and average pool
  backbone  points -> voxels -> blocks of [convolution, batch norm, gated activation] ->
            pooled descriptor and point features, evaluation mode
  train     the same blocks in training mode, forward and backward to every parameter
  points    points -> voxels -> points (Point2Voxel, Voxel2Point) without a network

The clouds are surfaces of boxes and ellipsoids with noise (synth.py), features N(0, 1), the
parameters the layers' own initialisation.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "ss-conv_amd"))

import synth  # noqa: E402
from ss_conv.activation import Activation  # noqa: E402
from ss_conv.batchnorm import BatchNorm  # noqa: E402
from ss_conv.convolution import Convolution  # noqa: E402
from ss_conv.fused import BatchNormActivation, ConvBatchNormActivation  # noqa: E402
from ss_conv.pool import AvgPool, GlobalAvgPool, MaxPool  # noqa: E402
from ss_conv.sp_ops.tensor import SparseTensor  # noqa: E402
from ss_conv.sp_ops.voxelize import Point2Voxel, Voxel2Point  # noqa: E402


# ---- the cases ----------------------------------------------------------------------------
def _layer(name=None, clouds=2, points=1024, ragged=False, shapes=1, grid=32, fields_in="2222",
           fields_out="2222", kernel=3, stride=1, dtype="f32", mode="train"):
    """fields_in / fields_out: multiplicities of the orders 0, 1, 2, ... as hexadecimal digits
    ("8888": eight fields each of orders 0 to 3).  mode: "train" (forward of a training
    step, no gradient asked for), "grad" (forward and backward), "eval"."""
    case = dict(kind="layer", clouds=clouds, points=points, ragged=ragged, shapes=shapes, grid=grid,
                fields_in=fields_in, fields_out=fields_out, kernel=kernel, stride=stride,
                dtype=dtype, mode=mode)
    if name is not None:
        case["name"] = name
    return case


def _network(kind, name=None, clouds=32, points=1024, ragged=False, grid=64, channels=3, width=8,
             strides="1221", dtype="f32"):
    """width: multiplicity of the first block's fields; it doubles at every block up to four
    times the first one.  strides: one digit per block."""
    case = dict(kind=kind, clouds=clouds, points=points, ragged=ragged, grid=grid,
                channels=channels, width=width, strides=strides, dtype=dtype)
    if name is not None:
        case["name"] = name
    return case


def _points(name=None, clouds=8, points=16384, ragged=False, shapes=5, grid=128, channels=64, mode=4):
    case = dict(kind="points", clouds=clouds, points=points, ragged=ragged, shapes=shapes,
                grid=grid, channels=channels, mode=mode)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # a layer of a small network on two clouds: the smallest call, where launches and the
        # host count (the first benchmark configuration)
        _layer("layer small", 2, 1024, False, 1, 32, "2222", "2222"),
        # the benchmark layer: 32 clouds, 64 -> 128 channels (the second configuration)
        _layer("layer", 32, 2048, False, 1, 64, "4444", "8888"),
        # the same layer with its backward pass, as a training step runs it
        _layer("layer backward", 32, 2048, False, 1, 64, "4444", "8888", mode="grad"),
        # half-precision rows and filters, inference
        _layer("layer half", 32, 2048, False, 1, 64, "4444", "8888", dtype="f16", mode="eval"),
        # half precision forward and backward, a middle layer of equal widths
        _layer("layer half backward", 16, 2048, False, 1, 64, "8888", "8888", dtype="f16",
               mode="grad"),
        # clouds of different sizes, a grid that is no power of two, channel counts that are
        # no multiple of four: 14 -> 31 channels, inference
        _layer("layer ragged", 7, 1900, True, 2, 50, "321", "5321", mode="eval"),
        # orders up to 4, kernel 5, fine grid: the stress layer (the fifth configuration)
        _layer("layer kernel 5", 8, 16384, False, 5, 128, "88888", "88888", kernel=5),
        # strided convolution and both sparse pools (the third configuration)
        dict(_layer("down", 32, 2048, False, 1, 64, "8888", "gggg", stride=2), kind="down"),
        # the whole backbone in evaluation mode (the fourth configuration)
        _network("backbone", "backbone", 32, 1024, False, 64, 3, 8, "1221"),
        # a narrower backbone serving a few clouds in half precision
        _network("backbone", "backbone half", 6, 1500, True, 64, 3, 4, "122", "f16"),
        # a training step of a three-block network, gradients of every parameter
        _network("train", "train step", 16, 1024, False, 64, 3, 4, "122"),
        # points to voxels and back on clouds of a scene's size
        _points("points", 8, 16384, False, 5, 128, 64),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _flops_bound(case):
    """About the operations of a case's convolutions, rather too many than too few."""
    n = case["clouds"] * case["points"]
    if case["kind"] in ("layer", "down"):
        k = 27 if case["kernel"] == 3 else 125
        per = 2.0 * n * k * _channels(case["fields_in"]) * _channels(case["fields_out"])
        return per / case["stride"] ** 3 * {"grad": 3}.get(case["mode"], 1)
    if case["kind"] in ("backbone", "train"):
        total, c, grown = 0.0, case["channels"], False
        for (co, gates), s in zip(_widths(case), case["strides"]):
            total += 2.0 * n * 27 / int(s) ** 3 * c * (co + gates)
            # a surface's rows after a dilation, after halving, and of rows that already are
            # a thick layer
            n *= (2.0 if grown else 15.0) if s == "1" else (0.3 if grown else 1.5)
            grown, c = True, co
        return total * (3 if case["kind"] == "train" else 1)
    return 0.0


def draw(rng):
    most = 5.0e11
    while True:
        kind = rng.choice(["layer", "layer", "layer", "layer", "layer", "down", "backbone", "train",
                           "points"])
        ragged = rng.random() < 0.5
        if kind in ("layer", "down"):
            grid = rng.choice([32, 64, 64, 128, rng.randrange(20, 120)])
            case = _layer(None, _log(rng, 1, 40), _log(rng, 200, 4096), ragged, rng.choice([1, 1, 3]),
                          grid, rng.choice(["2222", "4444", "8888", "88888", "321", "642", "4321", "9753"]),
                          rng.choice(["2222", "4444", "8888", "gggg", "88888", "321", "5321", "864"]),
                          5 if kind == "layer" and rng.random() < 0.15 else 3,
                          2 if kind == "down" or rng.random() < 0.2 else 1,
                          rng.choice(["f32", "f32", "f32", "f16"]) if kind == "layer" else "f32",
                          rng.choice(["train", "train", "grad", "grad", "eval"])
                          if kind == "layer" else "train")
            case["kind"] = kind
        elif kind in ("backbone", "train"):
            half = kind == "backbone" and rng.random() < 0.4
            case = _network(kind, None, _log(rng, 1, 32), _log(rng, 256, 2048), ragged,
                            rng.choice([32, 64, 64, rng.randrange(32, 100)]), rng.choice([1, 3, 3, 6]),
                            rng.choice([2, 4, 4, 6, 8]), rng.choice(["12", "122", "122", "1221", "212"]),
                            "f16" if half else "f32")
        else:
            case = _points(None, _log(rng, 1, 40), _log(rng, 500, 16384), ragged, rng.choice([1, 5]),
                           rng.choice([32, 64, 128, rng.randrange(20, 128)]),
                           rng.choice([3, 16, 37, 64, 128]), rng.choice([3, 4, 4]))
            if case["clouds"] * case["points"] > 131072:
                continue
        if _flops_bound(case) <= most and case["clouds"] * case["grid"] ** 3 <= 6.8e7:
            return case


# ---- their inputs -------------------------------------------------------------------------
def _irreps(fields):
    """"8841" -> [(8, 0), (8, 1), (4, 2), (1, 3)]; the digits up to g = 16."""
    return [("0123456789abcdefg".index(m), order) for order, m in enumerate(fields)]


def _channels(fields):
    return sum(m * (2 * order + 1) for m, order in _irreps(fields))


def _widths(case):
    """(field channels, gates) of every block of a network."""
    got, m = [], case["width"]
    for _ in case["strides"]:
        got.append((16 * m, 3 * m))
        m = min(2 * m, 4 * case["width"])
    return got


def _clouds(case, seed):
    """points [N, 3] float32 and batch ids [N] int64 (host).  The shapes of the clouds belong
    to the case; the seed puts the clouds into another order, turns each of them (the axes
    change places) and shuffles its points: other rows throughout, as many of them."""
    rng = np.random.default_rng([case["clouds"], case["points"], case["grid"]])
    clouds = []
    for _ in range(case["clouds"]):
        n = case["points"]
        if case["ragged"]:
            n = max(1, int(n * rng.uniform(0.3, 1.0)))
        clouds.append(synth.surface_cloud(rng, n, True, (1, case.get("shapes", 1))))
    rng = np.random.default_rng(seed)
    clouds = [clouds[i] for i in rng.permutation(len(clouds))]
    clouds = [c[rng.permutation(len(c))][:, rng.permutation(3)] for c in clouds]
    ids = np.repeat(np.arange(len(clouds), dtype=np.int64), [len(c) for c in clouds])
    return np.ascontiguousarray(np.concatenate(clouds)), ids


def _layers(case, dev):
    """The blocks of a network."""
    blocks, rs_in = [], [(case["channels"], 0)]
    m = case["width"]
    for stride in case["strides"]:
        rs = synth.irreps(m, 3)
        gated = rs + [(sum(mult for mult, _ in rs[1:]), 0)]
        conv = Convolution(rs_in, gated, 3, stride=int(stride), padding=1)
        block = ConvBatchNormActivation(conv, BatchNorm(gated),
                                        Activation(rs, (torch.relu, torch.sigmoid)))
        blocks.append(block.to(dev))
        rs_in, m = rs, min(2 * m, 4 * case["width"])
    return torch.nn.ModuleList(blocks)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    torch.manual_seed(seed)
    gen = torch.Generator(device=dev).manual_seed(seed)
    pts, ids = _clouds(case, seed)
    grid, kind = case["grid"], case["kind"]
    state = dict(case=case, shape=[grid] * 3, batch=case["clouds"])
    half = case.get("dtype") == "f16"
    if kind in ("layer", "down"):
        idx = torch.from_numpy(synth.voxel_indices(pts, ids, grid)).to(dev)
        rs_in, rs_out = _irreps(case["fields_in"]), _irreps(case["fields_out"])
        conv = Convolution(rs_in, rs_out, case["kernel"], stride=case["stride"],
                           padding=case["kernel"] // 2).to(dev)
        conv.train(case["mode"] != "eval")
        feats = torch.randn(idx.shape[0], _channels(case["fields_in"]), device=dev, generator=gen)
        state.update(indices=idx, conv=conv, feats=feats.half() if half else feats)
        if case["mode"] == "grad":
            # the gradient that arrives from the rest of the network: its rows are drawn for
            # the layer's outputs, whose number the geometry decides
            n_out = _geometry(idx, [(case["kernel"], case["stride"])], grid, case["clouds"])[0][1]
            dy = torch.randn(n_out, _channels(case["fields_out"]), device=dev, generator=gen)
            state["dy"] = dy.half() if half else dy
        if kind == "down":
            state["pools"] = (MaxPool(2, 2), AvgPool(2, 2))
    else:
        state.update(points=torch.from_numpy(pts).to(dev), ids=torch.from_numpy(ids).to(dev),
                     p2v=Point2Voxel([grid] * 3, [2.0 / grid] * 3,
                                     voxelization_mode=case.get("mode", 4)),
                     feats=torch.randn(pts.shape[0], case["channels"], device=dev, generator=gen))
    if kind in ("backbone", "train"):
        state["blocks"] = _layers(case, dev).train(kind == "train")
        state["pool"] = GlobalAvgPool()
        if kind == "train":
            state["dy"] = torch.randn(case["clouds"], _widths(case)[-1][0], device=dev,
                                      generator=gen)
    return state


# ---- one pass -----------------------------------------------------------------------------
def run(state):
    kind = state["case"]["kind"]
    return {"layer": _run_layer, "down": _run_down, "backbone": _run_backbone,
            "train": _run_train, "points": _run_points}[kind](state)


def _run_layer(state):
    if state["case"]["mode"] != "grad":
        with torch.no_grad():
            y = state["conv"](SparseTensor(state["feats"], state["indices"], state["shape"],
                                           state["batch"]))
        return {"features": y.features, "indices": y.indices}
    feats = state["feats"].detach().requires_grad_(True)
    conv = state["conv"]
    conv.zero_grad(set_to_none=True)
    y = conv(SparseTensor(feats, state["indices"], state["shape"], state["batch"]))
    y.features.backward(state["dy"])
    return {"features": y.features.detach(), "d_features": feats.grad,
            "d_weight": conv.kernel.weight.grad}


def _run_down(state):
    with torch.no_grad():
        y = state["conv"](SparseTensor(state["feats"], state["indices"], state["shape"],
                                       state["batch"]))
        most, mean = [pool(y) for pool in state["pools"]]
    return {"features": y.features, "indices": y.indices, "max": most.features,
            "max_indices": most.indices, "mean": mean.features}


def _run_backbone(state):
    half = state["case"]["dtype"] == "f16"
    with torch.no_grad():
        pts, x, ids, _ = state["p2v"](state["points"], state["feats"], state["ids"])
        if half:
            x.features = x.features.half()
        for block in state["blocks"]:
            x = block(x)
        if half:
            x.features = x.features.float()
        pooled = state["pool"](x)
        back = Voxel2Point(unit_voxel_extent=[2.0 / s for s in x.spatial_shape])
        return {"pooled": pooled, "points": back(x, pts, ids), "indices": x.indices}


def _run_train(state):
    blocks = state["blocks"]
    blocks.zero_grad(set_to_none=True)
    _, x, _, _ = state["p2v"](state["points"], state["feats"], state["ids"])
    for block in blocks:
        x = block(x)
    pooled = state["pool"](x)
    pooled.backward(state["dy"])
    out = {n: p.grad for n, p in blocks.named_parameters() if p.grad is not None}
    out["features"], out["pooled"] = x.features.detach(), pooled.detach()
    return out


def _run_points(state):
    with torch.no_grad():
        pts, x, ids, flag = state["p2v"](state["points"], state["feats"], state["ids"])
        grid = state["case"]["grid"]
        back = Voxel2Point(unit_voxel_extent=[2.0 / grid] * 3)
        return {"voxels": x.features, "indices": x.indices, "back": back(x, pts, ids),
                "flags": flag}


# ---- what a pass cannot do without, and how far two right answers may lie apart ------------
def _geometry(indices, layers, grid, batch):
    """[(N_in, N_out, pairs), ...] of a stack of convolutions [(kernel, stride), ...] with
    padding kernel // 2, from the voxel rows `indices` [N, 4]."""
    got, x, size = [], indices.long(), grid
    for k, s in layers:
        p = k // 2
        out = (size + 2 * p - k) // s + 1
        t = torch.arange(k, device=x.device)
        taps = torch.stack(torch.meshgrid(t, t, t, indexing="ij"), -1).reshape(-1, 3)
        keys, pairs = None, 0
        for part in taps.split(9):
            to = x[:, None, 1:] + p - part[None]
            ok = ((to >= 0) & (to % s == 0) & (to // s < out)).all(-1)
            to = to // s
            key = ((x[:, None, 0] * out + to[..., 0]) * out + to[..., 1]) * out + to[..., 2]
            key = key[ok]
            pairs += key.numel()
            keys = torch.unique(key if keys is None else torch.cat([keys, key]))
        got.append((x.shape[0], keys.numel(), pairs))
        x = torch.stack([keys // out ** 3, keys // out ** 2 % out, keys // out % out, keys % out], -1)
        size = out
    return got


def work(case):
    """Rows, filters and indices read once and written once; two operations per multiply-add
    of every (input, output) pair."""
    pts, ids = _clouds(case, 1)
    grid, kind = case["grid"], case["kind"]
    idx = torch.from_numpy(synth.voxel_indices(pts, ids, grid))
    if torch.cuda.is_available():
        idx = idx.cuda()
    n_pts, n_vox = pts.shape[0], idx.shape[0]
    size = 2 if case.get("dtype") == "f16" else 4
    nbytes = flops = 0.0
    if kind in ("layer", "down"):
        layers = [(case["kernel"], case["stride"], _channels(case["fields_in"]),
                   _channels(case["fields_out"]))]
    elif kind in ("backbone", "train"):
        c, layers = case["channels"], []
        for (co, gates), s in zip(_widths(case), case["strides"]):
            layers.append((3, int(s), c, co + gates))
            c = co
    else:
        layers = []
    geometry = _geometry(idx, [l[:2] for l in layers], grid, case["clouds"])
    back = case.get("mode") == "grad" or kind == "train"
    for (k, s, cin, cout), (n_in, n_out, pairs) in zip(layers, geometry):
        written = cout if kind in ("layer", "down") else cout * 16 // 19  # (the gates end here)
        rows = n_in * cin + n_out * written
        nbytes += size * (rows + k ** 3 * cin * cout) + 16 * (n_in + n_out)
        flops += 2.0 * pairs * cin * cout
        if back:  # both inputs again, the arriving gradient, both gradients
            nbytes += size * (2 * rows + 2 * k ** 3 * cin * cout)
            flops += 4.0 * pairs * cin * cout
    if kind == "down":
        n = geometry[0][1]
        c = layers[0][3]
        pooled = _pooled(idx, case)
        nbytes += 2 * (4 * c * (n + pooled) + 16 * (n + pooled))
    if kind in ("backbone", "train", "points"):
        c = case["channels"]
        nbytes += n_pts * (12 + 8 + 4 * c) + n_vox * (16 + 4 * c)
    if kind in ("backbone", "points"):  # pooled rows aside: the points read three voxel rows
        c = layers[-1][3] * 16 // 19 if layers else case["channels"]
        n = geometry[-1][1] if layers else n_vox
        nbytes += n_pts * (12 + 8 + 4 * c) + n * (16 + 4 * c)
    return {"bytes": nbytes, "flops": flops}


def _pooled(idx, case):
    """Rows that a pool of size 2 and stride 2 leaves of a strided layer's output."""
    s, p, k = case["stride"], case["kernel"] // 2, case["kernel"]
    out = (case["grid"] + 2 * p - k) // s + 1
    keys = None
    for dx in range(k):
        for dy in range(k):
            for dz in range(k):
                to = idx[:, 1:].long() + p - torch.tensor([dx, dy, dz], device=idx.device)
                ok = ((to >= 0) & (to % s == 0) & (to // s < out)).all(-1)
                to = torch.div(to, s, rounding_mode="floor")
                ok &= (to // 2 < out // 2).all(-1)
                to = to[ok] // 2
                b = idx[:, 0].long()[ok]
                key = ((b * out + to[:, 0]) * out + to[:, 1]) * out + to[:, 2]
                keys = torch.unique(key if keys is None else torch.cat([keys, key]))
    return keys.numel()


def tolerance(case):
    if case["kind"] == "points":
        # sums of a few float32 rows and three weighted rows, always in the same order; the
        # three nearest of equally far voxels are the first ones
        return {"rel": 1e-6, "max": 1e-4}
    if case.get("dtype") == "f16":
        # results rounded to half (2^-11) once per layer: 3e-4 of a layer's norm where two
        # right sums round differently everywhere, and a few times that behind several
        # layers
        return {"rel": 2e-3 if case["kind"] == "layer" else 4e-3}
    if case["kind"] == "train":
        # float32 sums through three blocks and their batch statistics, there and back
        return {"rel": 1e-4}
    return {"rel": 1e-5}
