"""Performance cases: the work that a user of this framework has it do, through its Python entry points.

Families and where their sizes come from:

* ``mlp``       identity-encoded networks: the tiny network of configuration 1, the 16-to-64-wide networks of the
                reference's benchmark (2 or 4 hidden layers, 10^6 points), wide networks of 128 channels (inference)
* ``siren``     configuration 4: heterogeneous widths with sine, CELU and bias
* ``hash``      configurations 2 and 3: multiresolution hash grid (16 levels x 2 features, 2^19 entries) in front of
                64 -> 64 -> 1, tables in half or (the default of the specification) in single precision
* ``dense4d``   configuration 5: dense 4-D grid with 8 features and identity in front of 32 -> 32 -> 32 -> 2
* ``encoding``  the hash grid alone, as a differentiable module in front of other PyTorch code
* ``pullpush``  differentiable inpainting of images

A case is a dict of plain values; ``op`` is ``inference`` (no gradients) or ``train`` (the forward pass and the
gradients of everything that is trained, for a given gradient of the output).
"""
import json
import math
import os
import sys

import torch

# the working folder is the root of the tree that is measured
sys.path.insert(0, os.path.abspath("quick-mlp_amd"))
import qmlp  # noqa: E402

BUILTIN = "qmlp/builtin-activations.json"
SINE30 = {
    "id": "sine30",
    "forward": "z = hsin(__hmul(__float2half(30.0f), x))",
    "adjoint": "adjx = __hmul(__hmul(__float2half(30.0f), hcos(__hmul(__float2half(30.0f), x))), adjz)",
}
HASH_LEVELS, HASH_FEATURES = 16, 2
DENSE_RESOLUTION, DENSE_FEATURES = 32, 8


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # a handful of coordinates per call, as an interactive viewer or a solver asks: latency and the host's path
        {"name": "mlp_tiny_inference", "family": "mlp", "op": "inference", "points": 1000, "inputs": 3, "width": 16,
         "hidden": 1, "outputs": 1, "bias": False, "activation": "relu"},
        # a training step on a batch of the unit tests' size: launches and the host's path again
        {"name": "mlp_small_train", "family": "mlp", "op": "train", "points": 513, "inputs": 16, "width": 32,
         "hidden": 2, "outputs": 4, "bias": True, "activation": "relu", "input_gradients": False},
        # the largest network of the reference's benchmark, trained on 10^6 points
        {"name": "mlp_64x4_train", "family": "mlp", "op": "train", "points": 1000000, "inputs": 16, "width": 64,
         "hidden": 4, "outputs": 4, "bias": False, "activation": "relu", "input_gradients": True},
        # a wide network evaluated on an image of a megapixel: the matrix cores
        {"name": "mlp_128x3_inference", "family": "mlp", "op": "inference", "points": 1 << 20, "inputs": 16,
         "width": 128, "hidden": 3, "outputs": 16, "bias": False, "activation": "relu"},
        # fitting an image or a field with sines
        {"name": "siren_train", "family": "siren", "op": "train", "points": 1 << 20, "input_gradients": True},
        # rendering a field stored in a hash grid: the headline of the benchmark
        {"name": "hash_inference", "family": "hash", "op": "inference", "points": 1 << 20, "tables": "half"},
        # fitting such a field, positions differentiated too (camera or geometry optimisation)
        {"name": "hash_train", "family": "hash", "op": "train", "points": 1 << 18, "tables": "half",
         "input_gradients": True},
        # a smaller, ragged batch on the tables that a specification gets by default
        {"name": "hash_train_ragged", "family": "hash", "op": "train", "points": 20011, "tables": "float",
         "input_gradients": False},
        # a time-dependent volume in a dense grid: a ragged batch of samples to evaluate ...
        {"name": "dense4d_inference_ragged", "family": "dense4d", "op": "inference", "points": 700001,
         "tables": "half"},
        # ... and the largest batch to train on
        {"name": "dense4d_train", "family": "dense4d", "op": "train", "points": 1 << 21, "tables": "half",
         "input_gradients": True},
        # the encoding as a module of its own, in front of layers that are not this framework's
        {"name": "encoding_train", "family": "encoding", "op": "train", "points": 1 << 17, "tables": "float",
         "input_gradients": False},
        # inpainting inside an optimisation: an image and its gradient
        {"name": "pullpush_train", "family": "pullpush", "op": "train", "batch": 1, "channels": 4, "height": 2048,
         "width": 2048, "dtype": "float32", "density": 0.2},
    ]


def _log_uniform(rng, low, high):
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    return max(low, min(high, n))


def draw(rng):
    family = rng.choice(["mlp", "mlp", "siren", "hash", "hash", "dense4d", "encoding", "pullpush"])
    op = rng.choice(["inference", "train"])
    case = {"family": family, "op": op}
    if family == "pullpush":
        case.update(batch=rng.choice([1, 1, 2]), channels=rng.randint(1, 4), height=_log_uniform(rng, 32, 2048),
                    width=_log_uniform(rng, 32, 1024), dtype=rng.choice(["float32", "float32", "float64"]),
                    density=rng.choice([0.05, 0.2, 0.5]))
        return case
    if family == "mlp":
        widths = [16, 32, 48, 64] if op == "train" else [16, 32, 48, 64, 128]
        case.update(points=_log_uniform(rng, 16, 1000000), inputs=rng.randint(2, 16), width=rng.choice(widths),
                    hidden=rng.choice([1, 2, 3, 4]), outputs=rng.randint(1, 4), bias=rng.random() < 0.5,
                    activation=rng.choice(["relu", "relu", "celu", "sine"]))
    elif family == "siren":
        case.update(points=_log_uniform(rng, 64, 1 << 20))
    elif family == "dense4d":
        case.update(points=_log_uniform(rng, 64, 1 << 21), tables="half")
    elif family == "hash":
        case.update(points=_log_uniform(rng, 64, 1 << 20 if op == "inference" else 1 << 18),
                    tables=rng.choice(["half", "float"]))
    else:
        case.update(points=_log_uniform(rng, 1024, 1 << 17), tables=rng.choice(["half", "float"]))
    if op == "train":
        case["input_gradients"] = rng.random() < 0.5
    return case


# ------------------------------------------------------------------------------------------------ specifications
def _hash_grid(precision):
    return {"id": "HashGrid", "start_in": 0, "n_in": 3, "n_levels": HASH_LEVELS,
            "n_features_per_level": HASH_FEATURES, "log2_hashmap_size": 19, "min_resolution": 16,
            "max_resolution": 4096, "combination_mode": "concat", "bounding_box_min": [0.0] * 3,
            "bounding_box_size": [1.0] * 3, "parameter_precision": precision}


def _dense_grid(precision):
    return {"id": "HashGrid", "start_in": 0, "n_in": 4, "n_levels": 1, "n_features_per_level": DENSE_FEATURES,
            "log2_hashmap_size": -1, "min_resolution": DENSE_RESOLUTION, "max_resolution": DENSE_RESOLUTION,
            "combination_mode": "concat", "bounding_box_min": [0.0] * 4, "bounding_box_size": [1.0] * 4,
            "parameter_precision": precision}


def _shape(case):
    """(input channels, encodings, widths of the layers, activations, biases, channels behind the encodings)"""
    family = case["family"]
    if family == "mlp":
        hidden = case["hidden"]
        return (case["inputs"], [{"id": "Identity", "start_in": 0, "n_in": case["inputs"]}],
                [case["width"]] * hidden + [case["outputs"]], [case["activation"]] * hidden + ["identity"],
                [case["bias"]] * (hidden + 1), case["inputs"])
    if family == "siren":
        return (4, [{"id": "Identity", "start_in": 0, "n_in": 4}], [128, 64, 48, 4],
                ["sine30", "sine", "celu", "identity"], [True] * 4, 4)
    if family == "hash":
        return (3, [_hash_grid(case["tables"])], [64, 64, 1], ["relu", "relu", "identity"], [False] * 3,
                HASH_LEVELS * HASH_FEATURES)
    return (4, [_dense_grid(case["tables"]), {"id": "Identity", "start_in": 0, "n_in": 4}], [32, 32, 32, 2],
            ["relu"] * 4, [True] * 4, DENSE_FEATURES + 4)


def _specification(case):
    inputs, encodings, widths, activations, biases, _ = _shape(case)
    return json.dumps({"num_inputs": inputs, "num_outputs": widths[-1], "activation_specification": [BUILTIN, SINE30],
                       "encodings": encodings,
                       "network": [{"n_out": w, "bias": b, "activation": a}
                                   for w, a, b in zip(widths, activations, biases)]})


# ------------------------------------------------------------------------------------------------ state and pass
def prepare(case, seed):
    qmlp.set_log_level("error")
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    uniform = lambda low, high, *shape: torch.rand(shape, generator=g, device="cuda") * (high - low) + low  # noqa: E731
    train = case["op"] == "train"
    state = {"family": case["family"], "train": train}
    if case["family"] == "pullpush":
        dtype = getattr(torch, case["dtype"])
        b, c, h, w = case["batch"], case["channels"], case["height"], case["width"]
        # sparse samples of an image: known pixels and holes
        state["mask"] = (uniform(0, 1, b, h, w) < case["density"]).to(dtype).requires_grad_(train)
        state["data"] = uniform(0, 1, b, c, h, w).to(dtype).requires_grad_(train)
        state["gradient"] = uniform(-1, 1, b, c, h, w).to(dtype)
        return state
    n = case["points"]
    if case["family"] == "encoding":
        encoding = qmlp.FusedEncoding(json.dumps(_hash_grid(case["tables"])))
        table = encoding.create_parameter_tensor()
        table.copy_(uniform(-0.1, 0.1, table.numel()))
        state.update(encoding=encoding, table=table.requires_grad_(train), x=uniform(0, 1, n, 3),
                     gradient=uniform(-1, 1, n, encoding.num_output_channels()))
        state["wanted"] = [table]
    else:
        torch.manual_seed(seed)   # the network's own initialisation of its weights
        # single-precision master weights where an optimizer steps them, half where they are only used
        net = qmlp.FusedNetwork(_specification(case), weight_dtype=torch.float32 if train else torch.float16)
        low, high = (-1, 1) if case["family"] in ("siren", "mlp") else (0, 1)
        with torch.no_grad():
            if case["family"] == "siren":
                _, _, widths, _, _, fan_in = _shape(case)
                for layer, fan_in in enumerate([fan_in] + widths[:-1]):
                    w = net.get_weight(layer, False, False)
                    bound = math.sqrt(6.0 / fan_in) / 30.0
                    net.set_weight(layer, False, False, uniform(-bound, bound, *w.shape).to(w.dtype))
            for table in net.encoding_parameters:
                if table.requires_grad:   # features of a field that has been fitted for a while
                    table.copy_(uniform(-0.1, 0.1, table.numel()))
            if case["family"] == "dense4d":   # ends in a ReLU: outputs that are alive
                bias = net.get_weight(3, True, False)
                net.set_weight(3, True, False, torch.full_like(bias, 0.5))
        if not train:
            net.requires_grad_(False)
        state.update(net=net, x=uniform(low, high, n, net.channels_in()),
                     gradient=uniform(-1, 1, n, net.channels_out()))
        state["wanted"] = [p for p in net.parameters() if p.requires_grad]
    if train and case["input_gradients"]:
        state["x"].requires_grad_(True)
        state["wanted"] = state["wanted"] + [state["x"]]
    return state


def run(state):
    train = state["train"]
    if state["family"] == "pullpush":
        if not train:
            return qmlp.pullpush.pullpush(state["mask"], state["data"])
        out = qmlp.pullpush.pullpush(state["mask"], state["data"])
        return [out.detach(), *torch.autograd.grad(out, [state["mask"], state["data"]], state["gradient"])]
    if state["family"] == "encoding":
        evaluate = lambda: state["encoding"](state["x"], state["table"])  # noqa: E731
    else:
        evaluate = lambda: state["net"](state["x"])  # noqa: E731
    if not train:
        with torch.no_grad():
            return evaluate()
    out = evaluate()
    return [out.detach(), *torch.autograd.grad(out, state["wanted"], state["gradient"])]


# ------------------------------------------------------------------------------------------------ floors and limits
def _table_entries(case):
    """Entries of the tables, and how many of them a batch touches at most."""
    if case["family"] == "dense4d":
        return DENSE_RESOLUTION ** 4, 16 * case["points"]
    total = 0
    growth = math.exp((math.log(4096) - math.log(16)) / (HASH_LEVELS - 1))
    touched = 0
    for level in range(HASH_LEVELS):
        entries = min(1 << 19, int(16 * growth ** level) ** 3)
        total += entries
        touched += min(entries, 8 * case["points"])
    return total, touched


def work(case):
    train = case["op"] == "train"
    if case["family"] == "pullpush":
        item = 8 if case["dtype"] == "float64" else 4
        pixels = case["batch"] * case["height"] * case["width"]
        planes = (1 + case["channels"]) + case["channels"]                      # mask and data in, data out
        if train:
            planes += (1 + 2 * case["channels"]) + (1 + case["channels"])       # both again and dL/dout in, both gradients out
        # the pyramid is 1/3 of the finest level; a handful of operations per pixel and channel
        return {"bytes": item * pixels * planes, "flops": pixels * (1 + case["channels"]) * (60 if train else 20)}
    n = case["points"]
    flops, byts = 0, 0
    if case["family"] == "encoding":
        inputs, outputs, weights = 3, HASH_LEVELS * HASH_FEATURES, 0
    else:
        inputs, _, widths, _, _, encoded = _shape(case)
        outputs, weights = widths[-1], 0
        for a, b in zip([encoded] + widths[:-1], widths):
            weights += a * b
        flops += 2 * weights * n * (3 if train else 1)
    byts += 4 * n * (inputs + outputs) + weights * (4 if train else 2)
    if train:
        byts += 4 * n * outputs + (4 * n * inputs if case["input_gradients"] else 0) + 4 * weights
    if case["family"] in ("hash", "encoding", "dense4d"):
        features = DENSE_FEATURES if case["family"] == "dense4d" else HASH_FEATURES
        item = 4 if case["tables"] == "float" else 2
        entries, touched = _table_entries(case)
        byts += min(entries, touched) * features * item
        if train:
            byts += entries * features * item       # the gradient is dense: zeros are written too
        corners = 16 if case["family"] == "dense4d" else 8 * HASH_LEVELS
        flops += 2 * corners * features * n * (2 if train else 1)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    if case["family"] == "pullpush":
        # sums of a few terms per pixel and level, and divisions by their weights
        return {"rel": 1e-12, "max": 1e-9} if case["dtype"] == "float64" else {"rel": 2e-5, "max": 5e-3}
    if case["family"] == "encoding":
        # single-precision sums; what is stored in half precision is rounded once
        return {"rel": 1e-3, "max": 5e-2} if case["tables"] == "half" else {"rel": 1e-5, "max": 2e-3}
    if case["op"] == "inference":
        return {"rel": 5e-3, "max": 0.1}            # activations are rounded to half precision after every layer
    # half-precision adjoints; a ReLU whose argument rounds to the other side of zero switches a point's unit
    return {"rel": 1e-2, "max": 0.9}
