"""What this framework's speed is measured on: a dozen uses of its public entry points, and draws from their ranges.

Each case is one of four kinds of work.

* ``conv``     a point convolution layer: inference or a training step, on a neighborhood that the program keeps (several
               layers of one level share it) or with everything built on the way (cloud, density, search);
* ``search``   bounding box, grid and radius neighbors of a cloud;
* ``density``  the kernel density estimate of a cloud;
* ``encoder``  several levels of Poisson-disk pooling, density, search and convolution, and the mean of the last features
               over each cloud (a classifier's body); inference or a training step.

Sizes are those of the repository's benchmark and tests, and sizes around them.  A case states the mean number of
neighbors beside its radius: ``work`` counts pairs with it without building them.
"""
import math

import numpy as np
import torch

import pccnn_lib_amd as lib
from pccnn_lib_amd import synthetic

_DEVICE = "cuda:0"
# surface that the generators of ``synthetic`` spread their points over: a primitive scaled into the unit cube, and
# the room with its boxes (square metres); a radius r then holds about neighbors = points * pi r^2 / area points
_AREA = {"object": 2.25, "room": 417.0, "room_unit": 4.17}

_LAYERS = {"kpconv": "KPConv", "kpconvn": "KPConvN", "pccnn": "PCCNN", "mcconv": "MCConv", "pointconv": "PointConv",
           "sphconv": "SPHConv"}
_NEEDS_DENSITY = ("kpconvn", "pccnn", "mcconv", "pointconv")
_BANDWIDTH = 0.2                    # of the radius, as in the benchmark's workloads


def _conv(name=None, layer="mcconv", cloud="object", clouds=1, points=1024, ragged=False, radius=0.1, neighbors=10.0,
          c_in=32, c_out=64, basis=16, contraction="f32", mode="train", keep=True, direction="same", coarse=0):
    """``mode``: "infer" (no gradients), "train" (features and parameters), "train_points" (also positions and
    densities).  ``keep``: the neighborhood (and density) is in hand before the call.  ``direction``: "same" (samples
    are the points), "down" (samples are ``coarse`` of each cloud's points, spread by a Poisson-disk pooling; of a smaller
    cloud proportionally fewer), "up" (points are the coarse ones, samples all)."""
    case = dict(kind="conv", layer=layer, cloud=cloud, clouds=clouds, points=points, ragged=ragged, radius=radius,
                neighbors=neighbors, c_in=c_in, c_out=c_out, basis=basis, contraction=contraction, mode=mode, keep=keep,
                direction=direction, coarse=coarse)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call: inference on two small clouds, everything built on the way (latency, launches, read-backs)
        _conv("kpconv_infer_2x1024", layer="kpconv", cloud="sphere", clouds=2, points=1024, radius=0.1, neighbors=3.6,
              c_in=32, c_out=32, basis=15, mode="infer", keep=False),
        # a small training step on a minibatch of objects of uneven sizes, built anew from the points each time
        _conv("mcconv_train_ragged_objects", clouds=7, points=1500, ragged=True, radius=0.1, neighbors=16.0, c_in=3,
              c_out=33, basis=8, mode="train", keep=False),
        # the benchmark's headline step: every gradient, positions and densities included, one kept neighborhood
        _conv("mcconv_train_points_16x4096", clouds=16, points=4096, radius=0.05, neighbors=14.4, c_in=64, c_out=128,
              basis=16, mode="train_points"),
        # the same layer inside a network, with the bf16 contraction that the layer offers
        _conv("mcconv_train_bf16_16x4096", clouds=16, points=4096, radius=0.05, neighbors=14.4, c_in=64, c_out=128,
              basis=16, contraction="bf16", mode="train"),
        # kernel points, wide channels, gradients of the positions too
        _conv("kpconv_train_points_8x8192", layer="kpconv", clouds=8, points=8192, radius=0.04, neighbors=18.1, c_in=128,
              c_out=256, basis=15, mode="train_points"),
        # a deployed network's layer: inference on one kept neighborhood, odd channel counts
        _conv("pccnn_infer_ragged", layer="pccnn", clouds=5, points=9001, ragged=True, radius=0.045, neighbors=21.5,
              c_in=48, c_out=96, basis=15, mode="infer"),
        # explicit basis: the layer evaluates it with torch operations around the native ops
        _conv("pointconv_train_ragged", layer="pointconv", clouds=6, points=3001, ragged=True, radius=0.07,
              neighbors=17.4, c_in=32, c_out=64, basis=16, mode="train"),
        # the way back up: features of few coarse points to all points of the scene (decoder of a segmentation network)
        _conv("kpconv_train_up_4x30000", layer="kpconv", cloud="room_unit", clouds=4, points=30000, radius=0.1,
              neighbors=13.5, c_in=128, c_out=64, basis=15, mode="train", direction="up", coarse=1200),
        # a scene's neighbor lists
        dict(name="search_room_1000000", kind="search", cloud="room", clouds=1, points=1000000, ragged=False, radius=0.05,
             neighbors=19.6, max_neighbors=0),
        # densities of uneven room scans
        dict(name="density_rooms_3x90001", kind="density", cloud="room", clouds=3, points=90001, ragged=True, radius=0.12,
             neighbors=9.4, bandwidth=0.03),
        # a small scene through two levels, inference, fp32
        dict(name="encoder_infer_2x6000", kind="encoder", cloud="room_unit", clouds=2, points=6000, ragged=True,
             radius=0.05, neighbors=62.0, c_in=6, channels=24, levels=2, basis=8, contraction="f32", mode="infer"),
        # the benchmark's encoder: four levels, training, bf16 contraction
        dict(name="encoder_train_bf16_8x100000", kind="encoder", cloud="room_unit", clouds=8, points=100000, ragged=False,
             radius=0.025, neighbors=234.0, c_in=8, channels=32, levels=4, basis=8, contraction="bf16", mode="train"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _radius(cloud, points, neighbors):
    return math.sqrt(neighbors * _AREA[cloud] / (math.pi * points))


def draw(rng):
    kind = rng.choice(["conv", "conv", "conv", "conv", "search", "density", "encoder"])
    if kind == "conv":
        layer = rng.choice(sorted(_LAYERS) + ["mcconv", "kpconv"])
        direction = rng.choice(["same", "same", "same", "down", "up"])
        clouds = rng.randint(1, 16)
        points = max(256, _log_int(rng, 2000, 90000 if layer != "pointconv" else 30000) // clouds)
        cloud = rng.choice(["object", "room_unit"])
        neighbors = rng.uniform(6.0, 30.0)
        c_in, c_out = _log_int(rng, 3, 160), _log_int(rng, 16, 260)
        basis = {"mcconv": rng.choice([8, 16]), "pointconv": rng.choice([8, 16, 32]), "sphconv": 16}.get(
            layer, rng.choice([13, 15]))
        # no more multiplications than the widest listed layer's
        while clouds * points * basis * c_in * c_out > 3.2e10:
            c_in, c_out = max(3, c_in * 3 // 4), max(16, c_out * 3 // 4)
        coarse = 0 if direction == "same" else max(64, points // rng.randint(6, 30))
        radius = _radius(cloud, coarse if direction == "up" else points, neighbors)
        mode = rng.choice(["infer", "train", "train", "train_points"])
        if mode == "train_points" and (direction != "same" or layer in ("pointconv", "sphconv")):
            mode = "train"
        keep = rng.choice([True, True, False]) if direction == "same" else True
        contraction = rng.choice(["f32", "f32", "bf16"]) if layer in ("mcconv", "kpconv") else "f32"
        return _conv(None, layer, cloud, clouds, points, rng.choice([True, False]), radius, neighbors, c_in, c_out, basis,
                     contraction, mode, keep or mode == "train_points", direction, coarse)
    clouds = rng.randint(1, 8)
    if kind == "search":
        points = max(500, _log_int(rng, 3000, 900000) // clouds)
        neighbors = rng.uniform(6.0, 40.0) if clouds * points < 300000 else rng.uniform(6.0, 18.0)
        cloud = rng.choice(["object", "room"])
        return dict(kind="search", cloud=cloud, clouds=clouds, points=points, ragged=rng.choice([True, False]),
                    radius=_radius(cloud, points, neighbors), neighbors=neighbors,
                    max_neighbors=rng.choice([0, 0, rng.randint(16, 64)]))
    if kind == "density":
        points = max(500, _log_int(rng, 3000, 800000) // clouds)
        neighbors = rng.uniform(5.0, 40.0)
        cloud = rng.choice(["object", "room"])
        radius = _radius(cloud, points, neighbors)
        return dict(kind="density", cloud=cloud, clouds=clouds, points=points, ragged=rng.choice([True, False]),
                    radius=radius, neighbors=neighbors, bandwidth=radius / 4.0)
    clouds = rng.randint(1, 8)
    points = _log_int(rng, 3000, 400000) // clouds
    cloud = rng.choice(["object", "room_unit"])
    neighbors = rng.uniform(30.0, 160.0)
    return dict(kind="encoder", cloud=cloud, clouds=clouds, points=points, ragged=rng.choice([True, False]),
                radius=_radius(cloud, points, neighbors) / 2.0, neighbors=neighbors, c_in=rng.randint(3, 16),
                channels=rng.choice([16, 24, 32]), levels=rng.randint(2, 3), basis=8,
                contraction=rng.choice(["f32", "bf16"]), mode=rng.choice(["infer", "train"]))


# ------------------------------------------------------------------------------------------------------- preparation

def _cloud_sizes(case):
    """Points of every cloud: all alike, or between two fifths and all of the stated number."""
    n = case["points"]
    if not case["ragged"]:
        return [n] * case["clouds"]
    rng = np.random.default_rng(n)
    return [n] + [int(rng.integers(max(1, 2 * n // 5), n + 1)) for _ in range(case["clouds"] - 1)]


def _make_cloud(case, seed):
    # A pair list is as long as its cloud has pairs: a search's clouds have the same points for every seed, and the
    # seed says in which order they stand in memory.
    fixed = case["kind"] == "search"
    rng, order = np.random.default_rng(case["points"] if fixed else seed), np.random.default_rng(seed)
    parts, ids = [], []
    for b, n in enumerate(_cloud_sizes(case)):
        own = int(rng.integers(1 << 31))
        if case["cloud"] == "object":
            pts = synthetic.primitives(own, 1, n)[0]
        elif case["cloud"] == "sphere":
            pts = synthetic.sphere_surface(np.random.default_rng(own), n)
        else:
            pts = synthetic.room(own, n)
            if case["cloud"] == "room_unit":
                pts = pts / np.float32(10.0)
        parts.append(pts[order.permutation(n)] if fixed else pts)
        ids.append(np.full(n, b, np.int32))
    return (torch.as_tensor(np.concatenate(parts), device=_DEVICE),
            torch.as_tensor(np.concatenate(ids), device=_DEVICE))


def _coarse_points(case, cloud):
    """``coarse`` points of every full cloud, in its order: a Poisson-disk pooling that keeps somewhat more, thinned."""
    # such a pooling of radius r keeps about 0.64 A / r^2 points of a densely sampled surface A
    spacing = math.sqrt(0.64 * _AREA[case["cloud"]] / (1.3 * case["coarse"]))
    chosen = lib.pc.PointPooling(cloud, spacing).pooling_ids_
    score = torch.rand(cloud.pts_.shape[0], device=_DEVICE)
    score[chosen] += 1.0
    kept, first = [], 0
    for n in _cloud_sizes(case):
        few = max(1, case["coarse"] * n // case["points"])
        kept.append(first + torch.topk(score[first:first + n], few).indices.sort().values)
        first += n
    kept = torch.cat(kept)
    return lib.pc.Pointcloud(cloud.pts_[kept], cloud.batch_ids_[kept])


def _new_layer(case, c_in, c_out):
    cls = getattr(lib.pc.layers, _LAYERS[case.get("layer", "mcconv")])
    if case.get("layer") == "sphconv":
        layer = cls(3, c_in, c_out, 1, 5, 3)
    else:
        layer = cls(3, c_in, c_out, case["basis"])
    if case.get("layer") in ("kpconvn", "pccnn"):
        # these two draw the rotation of their kernel points from the clock; a fixed rotation instead
        layer.kernel_pts_.copy_(lib.pc.layers.KPConv(3, 1, 1, case["basis"]).kernel_pts_)
    layer = layer.to(_DEVICE)
    if case["contraction"] != "f32":
        layer.contraction_ = case["contraction"]
    return layer


def _density(case, cloud):
    if case.get("layer", "mcconv") in _NEEDS_DENSITY:
        cloud.compute_pdf(_BANDWIDTH * case["radius"])


def _prepare_conv(case, seed, state):
    pts, ids = state["pts"], state["ids"]
    train = case["mode"] != "infer"
    layer = _new_layer(case, case["c_in"], case["c_out"])
    fine = lib.pc.Pointcloud(pts, ids)
    cloud_in = cloud_out = fine
    if case["direction"] != "same":
        few = _coarse_points(case, fine)
        cloud_in, cloud_out = (few, fine) if case["direction"] == "up" else (fine, few)
    _density(case, cloud_in)
    generator = torch.Generator(device=_DEVICE).manual_seed(seed)
    feats = torch.randn(cloud_in.pts_.shape[0], case["c_in"], device=_DEVICE, generator=generator)
    if train:
        state["upstream"] = torch.randn(cloud_out.pts_.shape[0], case["c_out"], device=_DEVICE, generator=generator)
    neighborhood = None
    if case["keep"]:
        with torch.no_grad():
            _, neighborhood = layer(cloud_in, cloud_out, feats, case["radius"])
    wanted = []
    if train:
        feats.requires_grad_(True)
        wanted = [feats] + [p for p in layer.parameters() if p.requires_grad]
    if case["mode"] == "train_points":
        cloud_in.pts_.requires_grad_(True)
        wanted.append(cloud_in.pts_)
        if cloud_in.pts_unnorm_pdf_ is not None:
            cloud_in.pts_unnorm_pdf_.requires_grad_(True)
            # KPConvN hands no gradient to the densities
            wanted += [cloud_in.pts_unnorm_pdf_] if case["layer"] != "kpconvn" else []
    state.update(layer=layer, cloud_in=cloud_in, cloud_out=cloud_out, feats=feats, neighborhood=neighborhood,
                 wanted=wanted)


def _prepare_encoder(case, seed, state):
    layers, c_in = [], case["c_in"]
    for level in range(case["levels"]):
        c_out = case["channels"] << level
        layers.append(_new_layer(case, c_in, c_out))
        c_in = c_out
    generator = torch.Generator(device=_DEVICE).manual_seed(seed)
    feats = torch.randn(state["pts"].shape[0], case["c_in"], device=_DEVICE, generator=generator)
    wanted = []
    if case["mode"] == "train":
        feats.requires_grad_(True)
        wanted = [feats] + [p for layer in layers for p in layer.parameters()]
        state["upstream"] = torch.randn(case["clouds"], c_in, device=_DEVICE, generator=generator)
    state.update(layers=layers, feats=feats, wanted=wanted)


def prepare(case, seed):
    torch.manual_seed(seed)
    pts, ids = _make_cloud(case, seed)
    state = dict(case=case, pts=pts, ids=ids)
    if case["kind"] == "conv":
        _prepare_conv(case, seed, state)
    elif case["kind"] == "encoder":
        _prepare_encoder(case, seed, state)
    return state


# ---------------------------------------------------------------------------------------------------------- one pass

def _run_conv(state):
    case, cloud_in, cloud_out = state["case"], state["cloud_in"], state["cloud_out"]
    args = (state["feats"], case["radius"])
    if case["mode"] == "infer":
        with torch.no_grad():
            if case["keep"]:
                return state["layer"](cloud_in, cloud_out, *args, p_neighborhood=state["neighborhood"])
            cloud = lib.pc.Pointcloud(state["pts"], state["ids"])
            _density(case, cloud)
            return state["layer"](cloud, cloud, *args)[0]
    if case["keep"]:
        out = state["layer"](cloud_in, cloud_out, *args, p_neighborhood=state["neighborhood"])
    else:
        cloud = lib.pc.Pointcloud(state["pts"], state["ids"])
        _density(case, cloud)
        out = state["layer"](cloud, cloud, *args)[0]
    return (out,) + torch.autograd.grad(out, state["wanted"], state["upstream"])


def _run_search(state):
    case = state["case"]
    cloud = lib.pc.Pointcloud(state["pts"], state["ids"])
    grid = lib.pc.Grid(cloud, lib.pc.BoundingBox(cloud), case["radius"])
    found = lib.pc.Neighborhood(grid, cloud, case["max_neighbors"])
    return found.neighbors_, found.start_ids_


def _run_density(state):
    cloud = lib.pc.Pointcloud(state["pts"], state["ids"])
    cloud.compute_pdf(state["case"]["bandwidth"])
    return cloud.pts_unnorm_pdf_, cloud.pts_pdf_


def _encoder_forward(state):
    """The last features' mean over each cloud, and the densities of the input points."""
    case = state["case"]
    cloud = first = lib.pc.Pointcloud(state["pts"], state["ids"])
    feats, radius = state["feats"], case["radius"]
    for layer in state["layers"]:
        pool = lib.pc.PointPooling(cloud, radius)
        cloud.compute_pdf(_BANDWIDTH * radius)
        pooled = lib.pc.Pointcloud(pool.pool_tensor(cloud.pts_), pool.pool_tensor(cloud.batch_ids_))
        feats, _ = layer(cloud, pooled, feats, 2.0 * radius)
        feats = torch.nn.functional.leaky_relu(feats, 0.2)
        cloud, radius = pooled, 2.0 * radius
    return cloud.global_pooling(feats), first.pts_pdf_


def _run_encoder(state):
    if state["case"]["mode"] == "infer":
        with torch.no_grad():
            return _encoder_forward(state)
    out, density = _encoder_forward(state)
    return (out, density) + torch.autograd.grad(out, state["wanted"], state["upstream"])


def run(state):
    return {"conv": _run_conv, "search": _run_search, "density": _run_density,
            "encoder": _run_encoder}[state["case"]["kind"]](state)


# ------------------------------------------------------------------------------------------------- work and tolerance

def _total_points(case):
    # ragged clouds have seven tenths of the stated number on average, the first one all of it
    n = case["points"] * case["clouds"]
    return n if not case["ragged"] else case["points"] * (0.7 * (case["clouds"] - 1) + 1.0)


def _search_bytes(n, m, pairs):
    # points and cloud ids in, pair list and segment ends out
    return 16.0 * n + (16.0 * m if m != n else 0.0) + 8.0 * pairs + 4.0 * m


def _conv_work(n, m, pairs, basis, c_in, c_out, mode):
    """Bytes and operations of a convolution on a pair list: the gather by basis value and the product with the
    weights, and in a training step the two transposed products and the way back through the gather."""
    rows = 4.0 * n * c_in + 4.0 * m * c_out + 4.0 * basis * c_in * c_out
    geometry = 8.0 * pairs + 4.0 * m + 12.0 * n + (12.0 * m if m != n else 0.0) + 4.0 * n
    product, gather = 2.0 * m * basis * c_in * c_out, 2.0 * pairs * basis * c_in
    if mode == "infer":
        return rows + geometry, product + gather
    # features, weights and the output's gradient in again, their gradients out
    moved = 2.0 * (rows + geometry) + 4.0 * n * c_in + 4.0 * basis * c_in * c_out
    if mode == "train_points":
        moved += 16.0 * n
    return moved, 3.0 * product + 3.0 * gather


def work(case):
    n = _total_points(case)
    pairs = n * case["neighbors"]
    if case["kind"] == "search":
        if case["max_neighbors"]:
            pairs = n * min(case["neighbors"], case["max_neighbors"])
        return {"bytes": _search_bytes(n, n, pairs), "flops": 8.0 * pairs}
    if case["kind"] == "density":
        return {"bytes": 16.0 * n + 8.0 * n, "flops": 10.0 * pairs}
    if case["kind"] == "conv":
        m = n
        if case["direction"] != "same":
            few = case["coarse"] * (n / case["points"])
            n, m = (few, n) if case["direction"] == "up" else (n, few)
            pairs = m * case["neighbors"]
        moved, flops = _conv_work(n, m, pairs, case["basis"], case["c_in"], case["c_out"], case["mode"])
        if not case["keep"]:
            # the pair list is made and used inside the pass; what has to move is the points
            moved += 16.0 * n - (12.0 * n + 4.0 * n + 4.0 * m + 8.0 * pairs) * (1.0 if case["mode"] == "infer" else 2.0)
            flops += 8.0 * pairs
        return {"bytes": moved, "flops": flops}
    moved = flops = 0.0
    c_in = case["c_in"]
    for level in range(case["levels"]):
        c_out = case["channels"] << level
        m = max(n / (case["neighbors"] / 4.0 * 0.4) if level == 0 else n / 4.7, 1.0)
        level_pairs = m * (case["neighbors"] if level == 0 else 41.0)
        # points and densities of the level in, those of the next out, and the convolution without its pair list
        b, f = _conv_work(n, m, 0.0, case["basis"], c_in, c_out, case["mode"])
        moved += b + 16.0 * n + 4.0 * n
        flops += f + level_pairs * case["basis"] * c_in * (2.0 if case["mode"] == "infer" else 6.0) + 8.0 * level_pairs
        n, c_in = m, c_out
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times what the path differs by from itself in 64 bits (sums of products; bf16 operands rounded as
    the path rounds them).  Seen, largest of all outputs: 1.1e-6 and 1e-5 (the layers), 4e-8 and 2e-7 (densities),
    2.1e-5 and 4e-3 (bf16: a projection on a rounding boundary)."""
    if case["kind"] == "search":
        return "exact"
    if case["kind"] == "density":
        return {"rel": 2e-7, "max": 1e-6}
    if case["kind"] == "encoder":
        # A feature within rounding of zero takes the other slope of the activation, and all its gradients with it.
        # In 64 bits: 7.4e-3 and 0.53 (four levels, bf16).
        if case["contraction"] == "bf16":
            return {"rel": 2e-2, "max": 0.9}
        return {"rel": 5e-6, "max": 4e-5} if case["mode"] == "infer" else {"rel": 2e-3, "max": 0.5}
    if case["contraction"] == "bf16":
        return {"rel": 1e-4, "max": 2e-2}
    if case["mode"] == "train_points" and case["layer"] in ("kpconv", "kpconvn", "mcconv"):
        # The position gradients jump where an offset lies on a kink of the basis, and the last bit says on which side.
        # In 64 bits: 5.9e-4 and 0.14.
        return {"rel": 2e-3, "max": 0.6}
    if case["layer"] == "pointconv" and case["mode"] != "infer":
        # its basis has a kink at zero: in 64 bits 3.2e-4 and 1.6e-3 on the gradients of the basis' parameters
        return {"rel": 1.3e-3, "max": 6e-3}
    return {"rel": 5e-6, "max": 4e-5}
