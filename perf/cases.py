"""What this framework is measured on: the passes a perception program has it run on every frame, through the public
entry points, from one scan line's worth of points to a batch of four full scans.

Five kinds of pass, which between them call every entry point a user's program calls per frame:

* ``voxelize``  simple_mean_encoder: points -> voxels with mean features
* ``layer``     spconv_index + spconv_mm: one sparse convolution by the two functions of the reference's surface, the
                index tensor between them in the caller's hands
* ``backbone``  layers.SparseBackbone: a network of sparse convolutions (VoxelNet, a Cylinder3D block, an
                encoder-decoder with inverse convolutions), enqueued call by call (``eager``), through the native
                schedule (``scheduled``) or captured once in a HIP graph and replayed (``replay``)
* ``pipeline``  onnx_graph.GraphExecutor: points -> voxels -> VoxelNet backbone -> dense bird's-eye-view map
* ``densify``   bev_densify: sparse rows -> dense map

Coordinates and features are drawn from the seed with this package's generators of LiDAR-like and cylindrical clouds;
weights are fixed, as a deployed network's are.  Row capacities are fixed too: they come from a sizing pass over another
cloud of the same kind, times ``room``, as an engine is sized on a recording before it serves a sensor.
"""
import functools

import numpy as np
import torch

import deploy3d_amd
from deploy3d_amd import layers as L
from deploy3d_amd import onnx_graph, synth

DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16, "int8": torch.int8}
BYTES = {"float32": 4, "float16": 2, "bfloat16": 2, "int8": 1}
SCENE = (41, 1440, 1440)        # detection grid (z, y, x), voxels of 0.1 x 0.1 x 0.15 m
SCENE_ORIGIN = (-72.0, -72.0, -2.0)
CYLINDER = (480, 360, 32)       # segmentation grid (rho, phi, z)
WIDE = (41, 1536, 1536)         # the voxeliser test's grid, from (-76.8, -76.8, -2)
WIDE_ORIGIN = (-76.8, -76.8, -2.0)
VOXEL = (0.1, 0.1, 0.15)
SIZING_SEED = 77                # the recording that capacities are planned on
# per-tensor activation scales of the VoxelNet backbone (99.99th percentile over 127 of a floating-point pass)
INT8_SCALES = {"input": 0.0305, "conv_input": 0.0123, "conv1_0": 0.00394, "conv1_1": 0.00281, "down1": 0.00286,
               "conv2_0": 0.00566, "conv2_1": 0.00436, "down2": 0.00393, "conv3_0": 0.00434, "conv3_1": 0.00426,
               "down3": 0.00427, "conv4_0": 0.00448, "conv4_1": 0.00444, "conv_out": 0.0073}


def listed():
    return [
        # a sparse sensor's packet of points: launch and call latency
        dict(name="voxelize 3k points", kind="voxelize", points=3001, channels=4, batch=1),
        # two full sweeps of a spinning LiDAR (the size of the reference's voxeliser test)
        dict(name="voxelize 200k points", kind="voxelize", points=200000, channels=4, batch=2),
        # one submanifold layer called by itself, fp32, uniform cloud
        dict(name="layer subm fp32 20k", kind="layer", voxels=20000, cin=16, cout=16, stride=1, dtype="float32",
             cloud="uniform"),
        # one downsampling layer called by itself, fp16, LiDAR-like cloud
        dict(name="layer down fp16 60k", kind="layer", voxels=60000, cin=32, cout=64, stride=2, dtype="float16",
             cloud="lidar"),
        # a far or filtered scan through the detection backbone, call by call
        dict(name="scan 9k fp16 eager", kind="backbone", net="voxelnet", voxels=9001, batch=1, dtype="float16",
             room=1.05, mode="eager"),
        # a full scan through the detection backbone, served from a graph; head-room as a stream of scans needs it
        dict(name="scan 120k fp16", kind="backbone", net="voxelnet", voxels=120000, batch=1, dtype="float16", room=1.05,
             mode="replay"),
        # the quantized engine of the same network, with head-room in every capacity
        dict(name="scan 120k int8 room", kind="backbone", net="voxelnet", voxels=120000, batch=1, dtype="int8",
             room=1.25, mode="replay"),
        # offline labelling: four scans per pass, bf16
        dict(name="scan 4x120k bf16", kind="backbone", net="voxelnet", voxels=480000, batch=4, dtype="bfloat16",
             room=1.05, mode="replay"),
        # segmentation block on a cylindrical grid: asymmetric kernels, two branches and their sum
        dict(name="cylinder 250k fp16", kind="backbone", net="cylinder", voxels=250000, batch=1, dtype="float16",
             room=1.05, mode="replay"),
        # encoder-decoder with inverse convolutions in full precision, as an export is validated
        dict(name="unet 40k fp32", kind="backbone", net="unet", voxels=40009, batch=1, dtype="float32", room=1.05,
             mode="eager"),
        # the whole sparse part of a detector as one imported graph: points in, dense map out
        dict(name="points to map 100k fp16", kind="pipeline", points=100000, dtype="float16", mode="eager"),
        # the map the detection backbone hands to its 2-D head
        dict(name="map 38k fp16", kind="densify", rows=38000, channels=128, batch=1, z=2, y=180, x=180,
             dtype="float16"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["voxelize", "layer", "backbone", "backbone", "backbone", "pipeline", "densify"])
    if kind == "voxelize":
        return dict(kind=kind, points=_log_uniform(rng, 2000, 400000), channels=rng.choice([3, 4, 5, 6]),
                    batch=rng.choice([1, 1, 2, 4]))
    if kind == "layer":
        stride = rng.choice([1, 2])
        cin, cout = rng.choice([(16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (5, 16)])
        return dict(kind=kind, voxels=_log_uniform(rng, 2000, 120000), cin=cin, cout=cout, stride=stride,
                    dtype=rng.choice(["float32", "float16", "bfloat16"]), cloud=rng.choice(["uniform", "lidar"]))
    if kind == "backbone":
        net = rng.choice(["voxelnet", "voxelnet", "voxelnet", "cylinder", "unet"])
        dtype = rng.choice(["float16", "float16", "bfloat16", "float32"] + (["int8", "int8"] if net == "voxelnet" else []))
        batch = rng.choice([1, 1, 2, 4]) if net == "voxelnet" else 1
        most = 30000 if dtype == "float32" else 250000 if net == "cylinder" else 120000 * batch
        voxels = _log_uniform(rng, 6000, most)
        modes = ["replay", "eager"] if net != "voxelnet" else ["replay", "eager", "scheduled"]
        return dict(kind=kind, net=net, voxels=voxels, batch=batch, dtype=dtype, room=rng.choice([1.05, 1.25, 1.5]),
                    mode=rng.choice(modes))
    if kind == "pipeline":
        return dict(kind=kind, points=_log_uniform(rng, 10000, 200000), dtype=rng.choice(["float16", "bfloat16"]),
                    mode=rng.choice(["eager", "replay"]))
    z, side = rng.choice([1, 2, 2, 4]), _log_uniform(rng, 60, 400)
    batch = rng.choice([1, 2])
    return dict(kind=kind, rows=_log_uniform(rng, 1000, min(80000, batch * z * side * side)),
                channels=rng.choice([32, 64, 128, 128, 256]), batch=batch, z=z, y=side, x=side + rng.choice([0, 1, 16]),
                dtype=rng.choice(["float32", "float16", "bfloat16", "int8"]))


# ---- networks ---------------------------------------------------------------------------------------------------
def _unet_layers():
    """Two levels down by strided convolutions, two up by the inverse convolutions of the same keys, with skip sums."""
    p = (1, 1, 1)
    k = (3, 3, 3)
    return [
        synth.layer("enc0", "s0", True, k, 5, 16, padding=p),
        synth.layer("enc0b", "s0", True, k, 16, 16, padding=p),
        synth.layer("down1", "d1", False, k, 16, 32, stride=(2, 2, 2), padding=p),
        synth.layer("enc1", "s1", True, k, 32, 32, padding=p),
        synth.layer("down2", "d2", False, k, 32, 64, stride=(2, 2, 2), padding=p),
        synth.layer("mid", "s2", True, k, 64, 64, padding=p),
        dict(synth.layer("up2", "d2", False, k, 64, 32, stride=(2, 2, 2), padding=p), inverse=True),
        synth.layer("dec1", "s1", True, k, 32, 32, padding=p, src="up2+enc1"),
        dict(synth.layer("up1", "d1", False, k, 32, 16, stride=(2, 2, 2), padding=p), inverse=True),
        synth.layer("dec0", "s0", True, k, 16, 16, padding=p, src="up1+enc0b"),
    ]


@functools.lru_cache(maxsize=None)
def _network(net, dtype):
    """(layer table, weights, grid) of a network: fixed, like a deployed model's."""
    specs = {"voxelnet": synth.voxelnet_layers, "cylinder": synth.cylinder_block_layers, "unet": _unet_layers}[net]()
    config = {"voxelnet": 3, "cylinder": 5, "unet": 6}[net]
    weights = [synth.layer_weights(config, i, s) for i, s in enumerate(specs)]
    if dtype == "int8":
        prev = "input"
        for s in specs:
            s.update(s_in=INT8_SCALES[prev], s_out=INT8_SCALES[s["name"]])
            prev = s["name"]
    return specs, weights, CYLINDER if net == "cylinder" else SCENE


# ---- inputs -----------------------------------------------------------------------------------------------------
def _cloud(seed, grid, n, batch=1, cloud="lidar"):
    """int32 [n, 4] rows (b, z, y, x): one cloud per sample, samples in order."""
    make = {"lidar": synth.coords_lidar, "uniform": synth.coords_uniform, "cylinder": synth.coords_cylinder}[cloud]
    parts = []
    for b in range(batch):
        rows = make(1000003 * (seed + 1) + b, grid, n // batch + (1 if b < n % batch else 0))
        rows[:, 0] = b
        parts.append(rows)
    return np.concatenate(parts)


def _normal(seed, shape):
    return np.random.default_rng(seed).standard_normal(shape, dtype=np.float32)


def _scan_points(seed, n):
    """n points (x y z intensity time) of a LiDAR-like scan of SCENE on the device: five points to three voxels, each
    well inside its cell, in random order."""
    coords = torch.from_numpy(_cloud(seed, SCENE, 3 * n // 5)).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(seed)
    pick = torch.cat([torch.arange(len(coords), device=DEV),
                      torch.randint(0, len(coords), (n - len(coords),), generator=g, device=DEV)])
    pick = pick[torch.randperm(n, generator=g, device=DEV)]
    at = coords[pick][:, [3, 2, 1]].float() + 0.1 + 0.8 * torch.rand((n, 3), generator=g, device=DEV)
    xyz = at * torch.tensor(VOXEL, device=DEV) + torch.tensor(SCENE_ORIGIN, device=DEV)
    return torch.cat([xyz, torch.rand((n, 2), generator=g, device=DEV)], dim=1).contiguous()


def _shape(batch, grid):
    return torch.empty((batch, 0) + tuple(grid), dtype=torch.int32, device=DEV)


@functools.lru_cache(maxsize=None)
def _planned(net, voxels, batch, room):
    """(input rows, output rows of every layer) the network's buffers are made for."""
    specs, _, grid = _network(net, "float32")
    coords = _cloud(SIZING_SEED, grid, voxels, batch, "cylinder" if net == "cylinder" else "lidar")
    counts = L.measure_output_counts(specs, coords, grid, batch)
    n_in = int(len(coords) * room)
    return n_in, L.plan_capacities(specs, n_in, {k: int(v * room) for k, v in counts.items()})


@functools.lru_cache(maxsize=None)
def _layer_rows(voxels, cloud):
    """Output rows of a downsampling layer called by itself: a limit the scan exceeds a little, so every row is live."""
    spec = synth.layer("layer", "layer", False, (3, 3, 3), 16, 16, stride=(2, 2, 2), padding=(1, 1, 1))
    return int(0.95 * L.measure_output_counts([spec], _cloud(SIZING_SEED, SCENE, voxels, cloud=cloud), SCENE)["layer"])


def _clear_tail(coors, num_act):
    """Coordinate rows past the live count are left as they are by every operator: set once, they stay."""
    coors[int(num_act.item()):] = 0


def _captured(fn):
    """fn's kernels in a HIP graph, as a serving program captures them: two passes, then the capture."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            fn()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = fn()
    torch.cuda.current_stream().wait_stream(stream)
    return graph, out


# ---- prepare ----------------------------------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_voxelize(case, seed):
    n, c = case["points"], case["channels"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    pts = torch.randn((n, c), generator=g, device=DEV)
    pts[:, :2] *= 50.0
    pts[:, 2] = pts[:, 2] * 2.0 + 1.0
    batch = torch.randint(0, case["batch"], (n,), dtype=torch.int32, generator=g, device=DEV)
    # points within 1e-3 of a cell boundary fall on either side with the last bit of a division: left out, as in the
    # voxeliser's test
    config = torch.tensor(WIDE_ORIGIN + VOXEL, dtype=torch.float32, device=DEV)
    at = (pts[:, :3] - config[:3]) / config[3:]
    batch[(at - at.round()).abs().amin(-1) < 1e-3] = -1
    # two points in three fall into cells of the grid, nearly all into cells of their own: the limit on voxels is
    # reached, as on a scan that is denser than the network takes
    return dict(kind="voxelize", args=(pts, batch, config, _shape(case["batch"], WIDE), 3 * n // 5))


def _prepare_layer(case, seed):
    cin, cout, stride = case["cin"], case["cout"], (case["stride"],) * 3
    subm = case["stride"] == 1
    coords = _cloud(seed, SCENE, case["voxels"], cloud=case["cloud"])
    n = len(coords)
    spec = synth.layer("layer", "layer", subm, (3, 3, 3), cin, cout, stride=stride, padding=(1, 1, 1), relu=False)
    weight, bias = synth.layer_weights(2, 0, spec)
    cap = n if subm else _layer_rows(case["voxels"], case["cloud"])
    x = L.make_input(coords, _normal(seed, (n, cin)), SCENE, dtype=DTYPES[case["dtype"]])
    return dict(kind="layer", x=x, shape=_shape(1, SCENE), cap=cap, spec=spec, weight=weight.reshape(-1), bias=bias)


def _prepare_backbone(case, seed):
    specs, weights, grid = _network(case["net"], case["dtype"])
    dtype, batch = DTYPES[case["dtype"]], case["batch"]
    coords = _cloud(seed, grid, case["voxels"], batch, "cylinder" if case["net"] == "cylinder" else "lidar")
    feats = _normal(seed, (len(coords), specs[0]["cin"]))
    if case["dtype"] == "int8":
        feats = synth.quantize_activations(feats, INT8_SCALES["input"])
    n_in, caps = _planned(case["net"], case["voxels"], batch, case["room"])
    net = L.SparseBackbone(specs, weights, caps, dtype=dtype)
    x = L.make_input(coords, feats, grid, dtype=dtype, capacity=n_in, batch=batch)
    state = dict(kind="backbone", net=net, x=x, graph=None, step=net.forward)
    if case["mode"] == "replay":
        state["graph"], state["y"] = _captured(lambda: net.forward(x))
    elif case["mode"] == "scheduled":
        state["step"] = net.forward_scheduled
    y = state["y"] if case["mode"] == "replay" else state["step"](x)
    _clear_tail(y.coors, y.num_act)
    return state


def _prepare_pipeline(case, seed):
    dtype = DTYPES[case["dtype"]]
    specs, weights, grid = _network("voxelnet", case["dtype"])
    n = case["points"]
    points = _scan_points(seed, n)
    config = torch.tensor(SCENE_ORIGIN + VOXEL, dtype=torch.float32, device=DEV)
    batch = torch.zeros(n, dtype=torch.int32, device=DEV)
    # _scan_points makes three voxels of five points; the voxeliser's rows are sized like the layers' behind it
    n_in, caps = _planned("voxelnet", 3 * n // 5, 1, 1.1)
    model = onnx_graph.backbone_model(specs, weights, caps, n_in, 5, grid, dtype=dtype, densify=True, points=n)
    executor = onnx_graph.GraphExecutor(model)
    inputs = dict(points=points, batch_indices=batch, voxel_config=config, spatial_shape=_shape(1, grid))
    state = dict(kind="pipeline", executor=executor, inputs=inputs, graph=None)
    if case["mode"] == "replay":
        state["graph"], state["y"] = _captured(lambda: executor.run(**inputs))
    y = state["y"] if case["mode"] == "replay" else executor.run(**inputs)
    state["names"] = [v.name for v in model.outputs]  # features, coordinates, live count, dense map
    _clear_tail(y[state["names"][1]], y[state["names"][2]])
    return state


def _prepare_densify(case, seed):
    b, z, y, x = case["batch"], case["z"], case["y"], case["x"]
    c, rows, dtype = case["channels"], case["rows"], DTYPES[case["dtype"]]
    g = torch.Generator(device=DEV).manual_seed(seed)
    # rows of a strided layer come sorted by cell
    cells = torch.randperm(b * z * y * x, generator=g, device=DEV)[:rows].sort().values
    coords = torch.stack([cells // (z * y * x), cells // (y * x) % z, cells // x % y, cells % x], dim=1).int()
    feats = torch.randn((rows, c), generator=g, device=DEV)
    feats = (feats * 40).round().clamp(-128, 127).to(dtype) if dtype == torch.int8 else feats.to(dtype)
    num = torch.tensor([rows], dtype=torch.int32, device=DEV)
    return dict(kind="densify", args=(feats, coords.contiguous(), num, _shape(b, (z, y, x)), c * z))


_PREPARE = dict(voxelize=_prepare_voxelize, layer=_prepare_layer, backbone=_prepare_backbone,
                pipeline=_prepare_pipeline, densify=_prepare_densify)


# ---- run --------------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "voxelize":
        return deploy3d_amd.simple_mean_encoder(*state["args"])
    if kind == "layer":
        x, s = state["x"], state["spec"]
        rb = deploy3d_amd.spconv_index(x.coors, x.num_act, state["shape"], s["ksize"], s["stride"], s["padding"],
                                       s["dilation"], (0, 0, 0), state["cap"], s["subm"], False)
        num_out = x.num_act if s["subm"] else rb[3]
        y = deploy3d_amd.spconv_mm(x.feats, x.num_act, num_out, rb[0], rb[1], s["ksize"], s["cin"], s["cout"],
                                   state["cap"], s["subm"], False, state["weight"], state["bias"])
        return (y,) + tuple(rb[:4])
    if kind == "backbone":
        if state["graph"] is not None:
            state["graph"].replay()
            y = state["y"]
        else:
            y = state["step"](state["x"])
        return y.feats, y.coors, y.num_act
    if kind == "pipeline":
        if state["graph"] is not None:
            state["graph"].replay()
            y = state["y"]
        else:
            y = state["executor"].run(**state["inputs"])
        return [y[name] for name in state["names"]]
    return deploy3d_amd.bev_densify(*state["args"])


# ---- work and tolerance -----------------------------------------------------------------------------------------
def _index_pairs(index, num_index):
    return int((index[2, :int(num_index.item())] >= 0).sum().item())


@functools.lru_cache(maxsize=None)
def _counted(items):
    """(bytes, operations) of one pass, from the live rows and pairs of one cloud of the case's ranges."""
    case = dict(items)
    kind = case["kind"]
    if kind == "voxelize":
        n, c = case["points"], case["channels"]
        return n * (4 * c + 4) + (3 * n // 5) * (4 * c + 16), n * (c + 6)
    state = prepare(case, 0)
    if kind == "layer":
        es, s, out = BYTES[case["dtype"]], state["spec"], run(state)
        x = state["x"]
        nbytes = (x.coors.numel() * 4 + x.feats.numel() * es + state["weight"].size * es + out[0].numel() * es +
                  out[1].numel() * 4 + (0 if s["subm"] else 16 * state["cap"]))
        return nbytes, 2 * _index_pairs(out[1], out[2]) * s["cin"] * s["cout"]
    if kind in ("backbone", "pipeline"):
        dtype = case["dtype"]
        es = BYTES[dtype]
        if kind == "backbone":
            net, x = state["net"], state["x"]
            specs, weights, _ = _network(case["net"], dtype)
            y = net.forward(x)
            nbytes = x.coors.numel() * 4 + x.feats.numel() * es + y.feats.numel() * es + y.coors.numel() * 4
        else:
            # the executor leaves index tensors between its own nodes unwritten: the pairs are counted by the runner
            specs, weights, grid = _network("voxelnet", dtype)
            points, batch, config, _ = state["inputs"].values()
            feats, coords, num = deploy3d_amd.simple_mean_encoder(points, batch, config, _shape(1, grid), len(points))
            n = int(num.item())
            _, caps = _planned("voxelnet", n, 1, 1.1)
            caps = L.plan_capacities(specs, n, dict(zip((s["name"] for s in specs), caps)))
            net = L.SparseBackbone(specs, weights, caps, dtype=DTYPES[dtype])
            net.forward(L.SparseTensor(feats[:n].to(DTYPES[dtype]), coords[:n].contiguous(), num, grid))
            out = run(state)
            nbytes = points.numel() * 4 + batch.numel() * 4 + sum(t.numel() * t.element_size() for t in out)
        nbytes += sum(w.size for w, _ in weights) * es
        pairs = {k: _index_pairs(rb.index, rb.num_index) for k, rb in net.rulebooks.items()}
        return nbytes, sum(2 * pairs[s["key"]] * s["cin"] * s["cout"] for s in specs)
    feats, coords, _, _, channels = state["args"]
    cells = case["batch"] * case["y"] * case["x"]
    return feats.numel() * feats.element_size() + coords.numel() * 4 + cells * channels * feats.element_size(), 0


def work(case):
    nbytes, flops = _counted(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Whole numbers and the dense map of given rows are exact; floating results differ by the order of their sums and,
    through a network, by the storage type's rounding of each layer."""
    if case["kind"] == "densify" or case.get("dtype") == "int8":
        return "exact"
    return {"rel": {"float32": 1e-5, "float16": 2e-3, "bfloat16": 1e-2}[case.get("dtype", "float32")]}
