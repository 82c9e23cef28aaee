"""What users of this library have it do, as measurable cases.

An application hands the library device tensors through the C ABI (nnforge_amd.capi: what a layer tester's
enqueue_forward_propagation calls) or whole networks on host arrays (nnforge_amd.backend.run_schema: forward_propagation::run
of the hip backend). The cases are the layer groups that inference of a convolutional network puts between and behind its
convolutions: batch normalisation with its activation and residual add, activation chains with exponentials, softmax over
class scores, subsampling in planes and volumes, the global average that ends a residual network, Inception branches written
side by side, statistics that refresh batch normalisation weights, and one whole network from and to host memory.
A case is a dict: "kind", sizes, and what the kind chooses from. All tensors are fp32 in [entry][feature map][y][x].
"""

import ctypes
import math

import numpy as np
import torch

from nnforge_amd import backend, capi, schemas, workloads

# A drawn case's tensors hold at most as many values as the largest listed case's (128 x 256 planes of 56 x 56); exp chains
# cost several times more per value, so they stop earlier.
MAX_ELEMENTS = 128 * 256 * 56 * 56
MAX_EXP_ELEMENTS = 64 * 1024 * 1024


def listed():
    return [
        # One image through one bottleneck block of a residual network (56 x 56, 64 -> 64 -> 256 feature maps): three small
        # groups one after the other, as in serving with a batch of one. Latency and launches.
        {"name": "block_one_entry", "kind": "block", "entries": 1, "maps": 64, "side": 56},
        # BatchNorm -> ReLU behind a convolution at an ordinary batch: the benchmark's headline configuration.
        {"name": "bn_relu_batch", "kind": "chain", "group": "bn_relu", "entries": 32, "maps": 64, "side": 56},
        # The last group of a bottleneck at a large batch: BatchNorm, residual add, PReLU. The largest tensors.
        {"name": "bn_add_prelu_large", "kind": "chain", "group": "bn_add_prelu", "entries": 128, "maps": 256, "side": 56},
        # BatchNorm -> ELU -> Sigmoid -> TanH with saturating inputs: networks of the older kind, bound by expf.
        {"name": "bn_elu_sigmoid_tanh", "kind": "chain", "group": "bn_elu_sigmoid_tanh", "entries": 64, "maps": 512, "side": 28},
        # Late feature maps of an odd side, planes that are no multiple of four floats (13 x 13).
        {"name": "bn_relu_odd_planes", "kind": "chain", "group": "bn_relu", "entries": 100, "maps": 384, "side": 13},
        # Class scores of a classifier's test set: 1000-way softmax, one row per image.
        {"name": "softmax_rows", "kind": "softmax", "entries": 2048, "maps": 1000, "side": 1},
        # Per-pixel class scores of dense prediction: 21 classes at every position of an odd-sided map.
        {"name": "softmax_per_pixel", "kind": "softmax", "entries": 16, "maps": 21, "side": 129},
        # The stem of a residual network: BatchNorm -> ReLU -> 3 x 3 max subsampling every 2, rounded up.
        {"name": "bn_relu_max_pool", "kind": "pool", "fused": True, "dims": 2, "entries": 64, "maps": 64, "side": 112, "window": 3, "stride": 2},
        # 2 x 2 x 2 max subsampling of volumes (video clips, scans).
        {"name": "max_pool_volumes", "kind": "pool", "fused": False, "dims": 3, "entries": 16, "maps": 64, "side": 28, "window": 2, "stride": 2},
        # The last block of a residual network folded into the global average behind it.
        {"name": "block_global_average", "kind": "average", "entries": 64, "maps": 2048, "side": 7},
        # Statistics of a layer's output over a batch, from which batch normalisation weights are refreshed.
        {"name": "map_statistics", "kind": "statistics", "entries": 128, "maps": 192, "side": 35},
        # Everything behind the convolutions of ResNet-50 as a network on host arrays, from the schema's text to the results:
        # forward_propagation::run with its copies to and from the device.
        {"name": "resnet50_from_host", "kind": "network", "network": "resnet50", "entries": 4, "maps": 0, "side": 0},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _fit_entries(rng, per_entry, limit, most):
    """An entry count that keeps the tensor below `limit` values, spread over the logarithm."""
    return _log_int(rng, 1, max(1, min(most, limit // per_entry)))


def draw(rng):
    kind = rng.choice(["block", "chain", "chain", "chain", "softmax", "softmax", "pool", "pool", "average", "statistics", "network"])
    if kind == "block":
        maps, side = 4 * _log_int(rng, 8, 128), _log_int(rng, 7, 64)
        return {"kind": kind, "entries": _fit_entries(rng, 4 * maps * side * side, 4 << 20, 16), "maps": maps, "side": side}
    if kind == "chain":
        group = rng.choice(["bn_relu", "bn_add_prelu", "bn_elu_sigmoid_tanh"])
        maps, side = _log_int(rng, 16, 2048), _log_int(rng, 4, 128)
        limit = MAX_EXP_ELEMENTS if group == "bn_elu_sigmoid_tanh" else MAX_ELEMENTS
        entries = _fit_entries(rng, maps * side * side, limit, 256)
        return {"kind": kind, "group": group, "entries": entries, "maps": maps, "side": side}
    if kind == "softmax":
        if rng.random() < 0.5:
            maps = _log_int(rng, 10, 5000)
            return {"kind": kind, "entries": max(64, _fit_entries(rng, maps, 16 << 20, 65536)), "maps": maps, "side": 1}
        maps, side = _log_int(rng, 2, 1000), _log_int(rng, 5, 192)
        return {"kind": kind, "entries": _fit_entries(rng, maps * side * side, 32 << 20, 64), "maps": maps, "side": side}
    if kind == "pool":
        if rng.random() < 0.5:
            window, stride = rng.choice([(2, 2), (3, 2), (3, 3)])
            maps, side = _log_int(rng, 16, 512), _log_int(rng, 8, 224)
            return {"kind": kind, "fused": rng.random() < 0.5, "dims": 2, "entries": _fit_entries(rng, maps * side * side, MAX_ELEMENTS // 2, 128),
                    "maps": maps, "side": side, "window": window, "stride": stride}
        window, stride = rng.choice([(2, 2), (2, 2), (3, 2)])
        maps, side = _log_int(rng, 8, 256), _log_int(rng, 7, 64)
        return {"kind": kind, "fused": False, "dims": 3, "entries": _fit_entries(rng, maps * side ** 3, MAX_ELEMENTS // 2, 64),
                "maps": maps, "side": side, "window": window, "stride": stride}
    if kind == "average":
        maps, side = _log_int(rng, 64, 2048), rng.randint(4, 15)
        return {"kind": kind, "entries": _fit_entries(rng, maps * side * side, MAX_ELEMENTS // 2, 256), "maps": maps, "side": side}
    if kind == "statistics":
        maps, side = _log_int(rng, 16, 1024), _log_int(rng, 4, 128)
        return {"kind": kind, "entries": max(2, _fit_entries(rng, maps * side * side, MAX_ELEMENTS, 256)), "maps": maps, "side": side}
    network = rng.choice(["stem", "stage"])
    maps, side = _log_int(rng, 8, 256), _log_int(rng, 7, 112)
    per_entry = maps * side * side if network == "stem" else 15 * maps * side * side
    return {"kind": kind, "network": network, "entries": _fit_entries(rng, per_entry, 24 << 20, 512), "maps": maps, "side": side}


# ---- inputs ---------------------------------------------------------------------------------------------


class _Device:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.device = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.device)
        self.gen.manual_seed(seed)

    def normal(self, count, std=1.0):
        t = torch.randn(count, generator=self.gen, device=self.device, dtype=torch.float32)
        return t if std == 1.0 else t.mul_(std)

    def uniform(self, count, lo, hi):
        return torch.rand(count, generator=self.gen, device=self.device, dtype=torch.float32).mul_(hi - lo).add_(lo)

    def bn(self, maps):
        """gamma, beta, mean, inverse sigma: the weight chunks of a batch normalisation layer"""
        variance = self.uniform(maps, 0.5, 2.0)
        return [self.uniform(maps, 0.5, 1.5), self.normal(maps, math.sqrt(0.1)), self.normal(maps, math.sqrt(0.1)),
                torch.rsqrt(variance + workloads.BN_EPSILON)]

    def empty(self, count):
        return torch.empty(count, device=self.device, dtype=torch.float32)


def _host_bn(gen, maps):
    variance = gen.random(maps, dtype=np.float32) * np.float32(1.5) + np.float32(0.5)
    return [gen.random(maps, dtype=np.float32) + np.float32(0.5), gen.standard_normal(maps, dtype=np.float32) * np.float32(0.3),
            gen.standard_normal(maps, dtype=np.float32) * np.float32(0.3),
            (np.float32(1.0) / np.sqrt(variance + np.float32(workloads.BN_EPSILON))).astype(np.float32)]


def _scatter_(tensor, gen, share, values):
    """A `share` of the tensor's values set to one of `values`, at random places."""
    at = torch.randint(tensor.numel(), (max(1, int(tensor.numel() * share)),), generator=gen, device=tensor.device)
    tensor[at] = values[torch.arange(at.numel(), device=tensor.device) % values.numel()]


def _group(case):
    n, c, plane = case["entries"], case["maps"], case["side"] ** 2
    if case["group"] == "bn_relu":
        return workloads.bn_relu("bn_relu", n, c, plane)
    if case["group"] == "bn_add_prelu":
        return workloads.Group("bn_add_prelu", n, c, plane, [[], [(capi.OP_BATCH_NORM, 0)]], [(capi.OP_PRELU, 4)], [("bn", c), ("prelu", c)])
    return workloads.Group("bn_elu_sigmoid_tanh", n, c, plane,
                           [[(capi.OP_BATCH_NORM, 0), (capi.OP_ELU,), (capi.OP_SIGMOID,),
                             (capi.OP_TANH, 0, workloads.TANH_SCALE, workloads.TANH_STEEPNESS)]], [], [("bn", c)])


def _block_groups(case):
    n, c, plane = case["entries"], case["maps"], case["side"] ** 2
    return [workloads.bn_relu("reduce", n, c, plane), workloads.bn_relu("bottleneck", n, c, plane), workloads.bn_add_relu("restore", n, 4 * c, plane)]


def _prepare_groups(dev, groups):
    launches = []
    for g in groups:
        elements = workloads.group_elements(g)
        inputs = [dev.normal(elements) for _ in g.arms]
        if any(op[0] == capi.OP_ELU for arm in g.arms for op in arm):
            inputs[0].mul_(math.sqrt(2.0))
            _scatter_(inputs[0], dev.gen, 0.001, torch.tensor([50.0, -50.0], device=dev.device))
        chunks = []
        for what, maps in g.chunks:
            chunks += dev.bn(maps) if what == "bn" else [dev.uniform(maps, 0.0, 0.25)]
        desc = capi.make_desc(g.entry_count, g.feature_map_count, g.plane, g.arms, g.tail)
        launches.append((desc, dev.empty(elements), inputs, chunks))
    return launches


def _u32(values):
    return (ctypes.c_uint32 * len(values))(*values)


def _pool_output_side(case):
    side, window, stride = case["side"], case["window"], case["stride"]
    round_up = window - 1 if window != stride else 0
    return (side + stride - window + round_up) // stride


def _network(case):
    """-> (layers, {data layer: (feature maps, [width, height])}, {output layer: values per entry})"""
    c, side = case["maps"], case["side"]
    L = schemas.L
    if case["network"] == "resnet50":
        layers, inputs, outputs = schemas.resnet50_post_convolution(with_pool1=True)
    elif case["network"] == "stage":
        # two bottleneck blocks of a residual network, the first with a shortcut of its own
        layers, inputs, outputs, last = [], {}, [], None
        for block in ("a", "b"):
            for name, maps in [("shortcut", 4 * c)] * (last is None) + [("reduce", c), ("bottleneck", c), ("restore", 4 * c)]:
                inputs[name + block] = (maps, [side, side])
                layers += [L("Data", name + block), L("BatchNorm", name + block + "_bn", [name + block], feature_map_count=maps)]
                if name in ("reduce", "bottleneck"):
                    layers.append(L("ReLU", name + block + "_relu", [name + block + "_bn"]))
                    outputs.append(name + block + "_relu")
            layers += [L("Add", "add" + block, [last or "shortcut" + block + "_bn", "restore" + block + "_bn"]), L("ReLU", "relu" + block, ["add" + block])]
            last = "relu" + block
            outputs.append(last)
    else:
        # what surrounds the convolutions of a small classifier: a subsampled stem and the class probabilities
        layers = [L("Data", "conv1"), L("BatchNorm", "conv1_bn", ["conv1"], feature_map_count=c), L("ReLU", "relu1", ["conv1_bn"]),
                  L("MaxSubsampling", "pool1", ["relu1"], windows=[2, 2]), L("Data", "logits"), L("Softmax", "prob", ["logits"])]
        inputs, outputs = {"conv1": (c, [side, side]), "logits": (100, [1, 1])}, ["pool1", "prob"]
    shapes = {}
    by_name = {l["name"]: l for l in layers}

    def shape(name):
        if name in shapes:
            return shapes[name]
        layer = by_name[name]
        if layer["type"] == "Data":
            maps, (w, h) = inputs[name]
        else:
            maps, h, w = shape(layer["inputs"][0])
            if layer["type"] == "MaxSubsampling":
                p = layer["params"]
                window, stride = p["windows"][0], p.get("strides", p["windows"])[0]
                extra = window - 1 if p.get("round_ups", [False])[0] else 0
                h, w = (h + stride - window + extra) // stride, (w + stride - window + extra) // stride
            elif layer["type"] == "AverageSubsampling":
                h, w = h // layer["params"]["windows"][1], w // layer["params"]["windows"][0]
        shapes[name] = (maps, h, w)
        return shapes[name]

    return layers, inputs, {name: shape(name) for name in outputs}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "network":
        gen = np.random.Generator(np.random.SFC64(seed))
        layers, inputs, outputs = _network(case)
        n = case["entries"]
        return {"case": case, "schema": schemas.schema_text(layers),
                "weights": {l["name"]: _host_bn(gen, l["params"]["feature_map_count"]) for l in layers if l["type"] == "BatchNorm"},
                "inputs": {name: gen.standard_normal((n, maps, h, w), dtype=np.float32) for name, (maps, (w, h)) in inputs.items()},
                "output_shapes": {name: (n,) + shape for name, shape in outputs.items()}}

    dev = _Device(seed)
    state = {"case": case, "lib": capi.load()}
    n, c, side = case["entries"], case["maps"], case["side"]
    if kind == "block":
        state["launches"] = _prepare_groups(dev, _block_groups(case))
    elif kind == "chain":
        state["launches"] = _prepare_groups(dev, [_group(case)])
    elif kind == "softmax":
        x = dev.normal(n * c * side * side, 2.0)
        _scatter_(x, dev.gen, 0.01, torch.tensor([30.0], device=dev.device))
        state.update(input=x, output=torch.empty_like(x))
    elif kind == "pool":
        dims, out_side = case["dims"], _pool_output_side(case)
        overlapping = int(case["window"] != case["stride"])
        state.update(input=dev.normal(n * c * side ** dims), output=dev.empty(n * c * out_side ** dims),
                     sizes=(_u32([side] * dims), _u32([case["window"]] * dims), _u32([case["stride"]] * dims), _u32([overlapping] * dims)))
        if case["fused"]:
            state["chunks"] = dev.bn(c)
            state["desc"] = capi.make_desc(n, c, side ** dims, [[(capi.OP_BATCH_NORM, 0), (capi.OP_RELU, 0, 0.0)]])
    elif kind == "average":
        state.update(inputs=[dev.normal(n * c * side * side) for _ in range(2)], output=dev.empty(n * c), chunks=dev.bn(c),
                     desc=capi.make_desc(n, c, side * side, [[], [(capi.OP_BATCH_NORM, 0)]], [(capi.OP_RELU, 0, 0.0)]))
    elif kind == "statistics":
        # values as behind a convolution: every feature map has a mean and a spread of its own
        x = dev.normal(n * c * side * side).view(n, c, side * side)
        x.mul_(dev.uniform(c, 0.5, 2.0).view(1, c, 1)).add_(dev.normal(c).view(1, c, 1))
        workspace_bytes = ctypes.c_size_t()
        capi.check(state["lib"].nnf_hip_feature_map_stat_workspace_bytes(n, c, side * side, ctypes.byref(workspace_bytes)))
        state.update(input=x, states=torch.zeros((c, 4), device=dev.device, dtype=torch.float64), workspace_bytes=workspace_bytes.value,
                     workspace=torch.empty(workspace_bytes.value, device=dev.device, dtype=torch.uint8))
    else:
        raise ValueError(kind)
    return state


# ---- one pass -------------------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "network":
        return backend.run_schema(state["schema"], state["weights"], state["inputs"], state["output_shapes"])[0]

    lib, stream = state["lib"], torch.cuda.current_stream().cuda_stream
    n, c, side = case["entries"], case["maps"], case["side"]
    if kind in ("block", "chain"):
        for desc, output, inputs, chunks in state["launches"]:
            capi.chain_forward(desc, output.data_ptr(), [t.data_ptr() for t in inputs], [t.data_ptr() for t in chunks], stream)
        return [output for _, output, _, _ in state["launches"]]
    if kind == "softmax":
        capi.check(lib.nnf_hip_softmax_forward(stream, state["output"].data_ptr(), state["input"].data_ptr(), n, c, side * side))
        return state["output"]
    if kind == "pool":
        if case["fused"]:
            chunks = capi.pointer_array([t.data_ptr() for t in state["chunks"]])
            capi.check(lib.nnf_hip_max_subsampling_fused_forward(stream, state["output"].data_ptr(), state["input"].data_ptr(), ctypes.byref(state["desc"]),
                                                                 chunks, n, c, case["dims"], *state["sizes"], 1, 1, 0))
        else:
            capi.check(lib.nnf_hip_max_subsampling_forward(stream, state["output"].data_ptr(), state["input"].data_ptr(), n, c, case["dims"],
                                                           *state["sizes"], 1, 1, 0))
        return state["output"]
    if kind == "average":
        inputs = capi.pointer_array([t.data_ptr() for t in state["inputs"]])
        chunks = capi.pointer_array([t.data_ptr() for t in state["chunks"]])
        capi.check(lib.nnf_hip_average_subsampling_joined_forward(stream, state["output"].data_ptr(), inputs, ctypes.byref(state["desc"]), chunks, n, c,
                                                                  side, side, side, side, 1.0 / (side * side)))
        return state["output"]
    states = state["states"]
    capi.check(lib.nnf_hip_feature_map_stat_init(stream, states.data_ptr(), c))
    capi.check(lib.nnf_hip_feature_map_stat_accumulate(stream, states.data_ptr(), state["workspace"].data_ptr(), state["workspace_bytes"],
                                                       state["input"].data_ptr(), n, c, side * side))
    # count, mean, sum of squared deviations in double; smallest and largest value in the fourth double's two floats
    return {"count": states[:, 0], "mean": states[:, 1], "m2": states[:, 2], "range": states.view(torch.float32)[:, 6:8]}


def work(case):
    kind = case["kind"]
    n, c, side = case["entries"], case["maps"], case["side"]
    if kind in ("block", "chain"):
        groups = _block_groups(case) if kind == "block" else [_group(case)]
        # BatchNorm and the activation 4 operations a value, the add 1; an exponential about 10, a division about 5
        per_value = 47 if case.get("group") == "bn_elu_sigmoid_tanh" else 5
        return {"bytes": sum(workloads.group_algorithmic_bytes(g) for g in groups), "flops": per_value * sum(workloads.group_elements(g) for g in groups)}
    if kind == "softmax":
        elements = n * c * side * side
        return {"bytes": 8 * elements, "flops": 14 * elements}
    if kind == "pool":
        inputs, outputs = n * c * side ** case["dims"], n * c * _pool_output_side(case) ** case["dims"]
        fused = bool(case["fused"])
        return {"bytes": 4 * (inputs + outputs) + 16 * c * fused, "flops": outputs * case["window"] ** case["dims"] + 3 * inputs * fused}
    if kind == "average":
        elements = n * c * side * side
        return {"bytes": 4 * (2 * elements + n * c + 4 * c), "flops": 5 * elements}
    if kind == "statistics":
        elements = n * c * side * side
        return {"bytes": 4 * elements + 32 * c, "flops": 5 * elements}
    layers, inputs, outputs = _network(case)
    values_in = n * sum(maps * w * h for maps, (w, h) in inputs.values())
    values_out = n * sum(maps * h * w for maps, h, w in outputs.values())
    return {"bytes": 4 * (values_in + values_out), "flops": 5 * values_in}


def tolerance(case):
    if case["kind"] == "softmax":
        return {"rel": 3e-7}   # the sum of the exponentials in another order; against 64 bits the path shows 3e-8 to 7e-8
    if case["kind"] == "statistics":
        return {"rel": 1e-14}  # sums in double in another order; against two passes in 64 bits the path shows 1e-16 to 7e-16
    if case["kind"] == "network":
        return {"rel": 3e-7}   # the softmax at its end; everything else is the same bits
    return "exact"  # one rounding per operation in the reference's order, however the layers are fused
