"""The work that a user of this framework has it do, as cases that can be timed and compared.

Every case goes through the public entry points: ``native.gemm``, ``native.conv2d_forward`` and
``conv2d_backward``, ``native.maxpool2d_forward`` and ``maxpool2d_backward``, small networks of layers
(``Dense``, ``BasicBlock``, ResNet18's stem) under a ``Graph``, whole ResNet18 training steps and ResNet18
inference. Everything is float32, the only data type that the framework computes in.

``listed()`` gives the cases by name, ``draw(rng)`` one more of the same ranges, ``prepare`` makes the
inputs and what a program keeps (the model, its graph), ``run`` is one pass, ``work`` what the pass
cannot do without, ``tolerance`` how far another correct float32 implementation may be off and
``exact`` the same pass in 64 bits by plain torch.
"""

from __future__ import annotations

import numpy as np
import torch
import torch.nn.functional as F

import myflows_amd as mf
from myflows_amd import native

DEVICE = "cuda"


def listed():
    return [
        # A small product, such as one head or one projection of a small batch: the launch counts.
        {"name": "gemm_small_odd", "kind": "gemm", "m": 100, "n": 130, "k": 257, "layout": "NN", "bias": True},
        # The square product that bench.py prices the GEMM engine by.
        {"name": "gemm_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "layout": "NN", "bias": False},
        # A ragged product with a transposed right operand (an activation times a stored weight).
        {"name": "gemm_ragged_nt", "kind": "gemm", "m": 1531, "n": 1000, "k": 777, "layout": "NT", "bias": False},
        # A classifier head's training pass: forward, dX, dW and db of a Linear.
        {"name": "dense_train", "kind": "dense", "batch": 256, "n_in": 512, "n_out": 1000},
        # The layer1 convolution of ResNet18 at batch 64 (3x120x160 images), forward and backward.
        {"name": "conv3x3_train", "kind": "conv", "batch": 64, "ci": 64, "co": 64, "h": 29, "w": 39, "size": 3,
         "stride": 1, "bias": True},
        # A strided convolution that halves odd planes and widens, with channel counts off the tiles.
        {"name": "conv_stride2_odd", "kind": "conv", "batch": 33, "ci": 96, "co": 160, "h": 27, "w": 35, "size": 3,
         "stride": 2, "bias": True},
        # The last residual block of ResNet18 at batch 64: deep products over few pixels, batch norm.
        {"name": "block_deep_train", "kind": "block", "batch": 64, "ci": 512, "co": 512, "h": 4, "w": 5, "stride": 1},
        # ResNet18's stem on a batch of 3x120x160 images: 7x7/2 convolution, batch norm, ReLU, max-pool.
        {"name": "stem_train", "kind": "stem", "batch": 64, "co": 64, "h": 120, "w": 160},
        # A default max-pool, forward and backward: memory traffic only.
        {"name": "maxpool_train", "kind": "pool", "batch": 32, "c": 64, "h": 30, "w": 40, "size": 2, "stride": 2},
        # The training step that bench.py reports: batch 64, recorded once and replayed, then Adam.
        {"name": "resnet18_train_64", "kind": "train", "batch": 64, "h": 120, "w": 160, "recorded": True},
        # One camera image through the deployed network: latency.
        {"name": "resnet18_infer_1", "kind": "infer", "batch": 1, "h": 120, "w": 160},
        # A bulk scoring pass over 224x224 images.
        {"name": "resnet18_infer_256", "kind": "infer", "batch": 256, "h": 224, "w": 224},
    ]


def _spread(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return max(low, min(high, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "dense", "conv", "conv", "conv", "conv", "block", "block", "stem", "pool",
                       "train", "infer", "infer"])
    if kind == "gemm":
        m, n, k = (_spread(rng, 64, 4096) for _ in range(3))
        if rng.random() < 0.25:  # a weight gradient: a small output over a long inner dimension
            m, n, k = _spread(rng, 32, 600), _spread(rng, 32, 600), _spread(rng, 4096, 65536)
        return {"kind": kind, "m": m, "n": n, "k": k, "layout": rng.choice(["NN", "NT", "TN"]),
                "bias": rng.random() < 0.5}
    if kind == "dense":
        return {"kind": kind, "batch": _spread(rng, 16, 2048), "n_in": _spread(rng, 64, 2048),
                "n_out": _spread(rng, 10, 2048)}
    if kind == "conv":
        c = 32 if rng.random() < 0.75 else 1  # most networks' widths are multiples of 32
        ci, co = (c * _spread(rng, 32 // c, 512 // c) for _ in range(2))
        area = _spread(rng, 16, 3000)
        h = max(4, min(60, int(round((area * rng.uniform(0.6, 1.0)) ** 0.5))))
        w = max(4, min(80, area // h))
        size, stride = rng.choice([(3, 1), (3, 1), (3, 2), (1, 1), (1, 2), (5, 1)])
        largest = 60e9 / (2.0 * ci * co * size * size * h * w / stride ** 2)  # at most 60 GFLOP forward
        return {"kind": kind, "batch": _spread(rng, 1, max(1, min(128, int(largest)))), "ci": ci, "co": co, "h": h,
                "w": w, "size": size, "stride": stride, "bias": rng.random() < 0.7}
    if kind == "block":
        ci, side = rng.choice([(64, 40), (128, 20), (256, 12), (512, 7)])
        stride = rng.choice([1, 2]) if ci < 512 else 1
        return {"kind": kind, "batch": _spread(rng, 2, 96), "ci": ci, "co": ci * stride,
                "h": rng.randint(max(4, side // 2), side), "w": rng.randint(max(4, side // 2), side), "stride": stride}
    if kind == "stem":
        return {"kind": kind, "batch": _spread(rng, 2, 64), "co": 64, "h": rng.randint(60, 160), "w": rng.randint(60, 224)}
    if kind == "pool":
        size, stride = rng.choice([(2, 2), (2, 2), (3, 2)])
        return {"kind": kind, "batch": _spread(rng, 1, 128), "c": _spread(rng, 16, 256), "h": rng.randint(7, 60),
                "w": rng.randint(7, 80), "size": size, "stride": stride}
    if kind == "train":
        return {"kind": kind, "batch": _spread(rng, 2, 64), "h": rng.randint(64, 120), "w": rng.randint(64, 160),
                "recorded": rng.random() < 0.5}
    return {"kind": kind, "batch": _spread(rng, 1, 128), "h": rng.randint(64, 224), "w": rng.randint(64, 224)}


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device=DEVICE) * scale


def _inputs(case, seed):
    """The data of a case in float32, made from the seed alone (both the float32 and the 64-bit pass
    start from these): activations of unit variance, after a ReLU where a ReLU comes before the layer in
    a network, Kaiming-scaled weights, small biases, targets of the outputs' scale."""
    g, kind = _generator(seed), case["kind"]
    if kind == "gemm":
        m, n, k, layout = case["m"], case["n"], case["k"], case["layout"]
        return {"a": _normal(g, *((k, m) if layout == "TN" else (m, k))),
                "b": _normal(g, *((n, k) if layout == "NT" else (k, n))),
                "bias": _normal(g, n) if case["bias"] else None}
    if kind == "dense":
        return {"x": _normal(g, case["batch"], case["n_in"]).relu(),
                "w": _normal(g, case["n_in"], case["n_out"], scale=(2.0 / case["n_in"]) ** 0.5),
                "b": _normal(g, 1, case["n_out"], scale=0.1), "t": _normal(g, case["batch"], case["n_out"])}
    if kind == "conv":
        pad = case["size"] // 2
        oh, ow = ((case[d] + 2 * pad - case["size"]) // case["stride"] + 1 for d in ("h", "w"))
        fan = case["ci"] * case["size"] ** 2
        return {"x": _normal(g, case["batch"], case["ci"], case["h"], case["w"]).relu(),
                "w": _normal(g, case["co"], case["ci"], case["size"], case["size"], scale=(2.0 / fan) ** 0.5),
                "b": _normal(g, case["co"], scale=0.1) if case["bias"] else None,
                "dy": _normal(g, case["batch"], case["co"], oh, ow)}
    if kind == "block":
        s = case["stride"]
        weights = [(case["co"], case["ci"], 3), (case["co"], case["co"], 3)]
        if s != 1 or case["ci"] != case["co"]:
            weights.append((case["co"], case["ci"], 1))
        return {"x": _normal(g, case["batch"], case["ci"], case["h"], case["w"]).relu(),
                "weights": [_normal(g, co, ci, f, f, scale=(2.0 / (ci * f * f)) ** 0.5) for co, ci, f in weights],
                **_head(g, case)}
    if kind == "stem":
        return {"x": _normal(g, case["batch"], 3, case["h"], case["w"]),
                "w": _normal(g, case["co"], 3, 7, 7, scale=(2.0 / 147) ** 0.5), **_head(g, case)}
    if kind == "pool":
        oh, ow = ((case[d] - case["size"]) // case["stride"] + 1 for d in ("h", "w"))
        return {"x": _normal(g, case["batch"], case["c"], case["h"], case["w"]).relu(),
                "dy": _normal(g, case["batch"], case["c"], oh, ow)}
    return {"x": _normal(g, case["batch"], 3, case["h"], case["w"]),
            "t": torch.rand((case["batch"], 2), generator=g, device=DEVICE) * 2 - 1}


def _head(g, case):
    """The classifier over a block's pooled features, and its targets."""
    return {"head": _normal(g, case["co"], 10, scale=(2.0 / case["co"]) ** 0.5), "t": _normal(g, case["batch"], 10)}


def _graph(out, target):
    """The training graph of these outputs under a mean-squared-error loss."""
    return mf.Graph(mf.MSELoss(out, mf.Variable(target, requires_grad=False)), optimize=True)


def _classifier(features, data):
    """Global average pooling and a Dense head over a block's output."""
    layer = mf.Dense(*data["head"].shape, backend="hip_native", initializer="constant")
    layer.W.value = data["head"]
    return layer(mf.GlobalAvgPool2d()(features)), layer.params


def _weights(seed):
    """An initializer: Kaiming-scaled normal weights of a seeded sequence of shapes."""
    rng = np.random.default_rng(seed)
    return lambda shape: rng.standard_normal(shape) * (2.0 / np.prod(shape[1:] if len(shape) == 4 else shape[:1])) ** 0.5


def _resnet(seed):
    """ResNet18, with running statistics as after some training."""
    model = mf.ResNet18(output_dim=2, initializer=_weights(seed), conv_backend="hip_native")
    rng = np.random.default_rng(seed)
    for layer in model.sub_layers:
        if isinstance(layer, mf.BatchNorm2d):
            layer.running_mean.copy_(torch.as_tensor(rng.normal(0, 0.1, layer.num_features)))
            layer.running_var.copy_(torch.as_tensor(rng.uniform(0.5, 1.5, layer.num_features)))
    return model


def prepare(case, seed):
    mf.set_device(DEVICE)
    kind, data = case["kind"], _inputs(case, seed)
    if kind in ("gemm", "conv", "pool"):
        return {"case": case, **data}
    if kind == "dense":
        layer = mf.Dense(case["n_in"], case["n_out"], backend="hip_native", initializer="constant")
        layer.W.value, layer.b.value = data["w"], data["b"]
        x = mf.Variable(data["x"], requires_grad=True)
        out = layer(x)
        return {"case": case, "graph": _graph(out, data["t"]), "out": out, "grads": [x, *layer.params]}
    if kind == "block":
        block = mf.BasicBlock(case["ci"], case["co"], case["stride"], conv_backend="hip_native", compat="torchvision",
                              initializer="constant")
        for layer, w in zip([block.conv1, block.conv2] + ([block.downsample_conv] if block.downsample else []),
                            data["weights"]):
            layer.kernel.value = w
        x = mf.Variable(data["x"], requires_grad=True)
        out, head = _classifier(block(x), data)
        return {"case": case, "graph": _graph(out, data["t"]), "out": out, "grads": [x, *block.params, *head]}
    if kind == "stem":
        conv = mf.Conv2D(3, case["co"], kernel_size=7, stride=2, padding=3, backend="hip_native", bias=False,
                         fuse_activation=False, initializer="constant")
        conv.kernel.value = data["w"]
        bn = mf.BatchNorm2d(case["co"])
        x = mf.Variable(data["x"], requires_grad=False)  # images: the network's input has no gradient
        out, head = _classifier(mf.MaxPool2d(3, 2, backend="hip_native")(mf.ReLU(bn(conv(x)))), data)
        return {"case": case, "graph": _graph(out, data["t"]), "out": out, "grads": [*conv.params, *bn.params, *head]}
    model = _resnet(seed)
    x = mf.Variable(data["x"], requires_grad=False)
    if kind == "train":
        out = model(x)
        optimizer = mf.Adam(_graph(out, data["t"]), learning_rate=1e-4)
        step = mf.RecordedStep(optimizer, warmup=2) if case["recorded"] else optimizer
        # Without the convolutions' biases: ahead of a batch norm their gradients are zero but for rounding.
        biases = {id(layer.b) for layer in model.sub_layers if isinstance(layer, mf.Conv2D)}
        for block in model.blocks():
            biases |= {id(layer.b) for layer in block.sub_layers if isinstance(layer, mf.Conv2D)}
        return {"case": case, "step": step, "out": out, "grads": [p for p in model.params if id(p) not in biases]}
    model.eval()
    root, _ = mf.apply_graph_optimizations(model(x), mode="inference", fold_constants=False)
    return {"case": case, "graph": mf.Graph(root, optimize=True)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemm":
        return native.gemm(state["a"], state["b"], state["bias"], trans_a=case["layout"] == "TN",
                           trans_b=case["layout"] == "NT")
    if kind == "conv":
        window = {"stride": (case["stride"],) * 2, "padding": (case["size"] // 2,) * 2}
        y, cols = native.conv2d_forward(state["x"], state["w"], state["b"], **window)
        dx, dw, db = native.conv2d_backward(state["x"], state["w"], state["dy"], cols, need_bias_grad=case["bias"], **window)
        return {"y": y, "dx": dx, "dw": dw, "db": db}
    if kind == "pool":
        y, context = native.maxpool2d_forward(state["x"], kernel_size=(case["size"],) * 2, stride=(case["stride"],) * 2)
        return {"y": y, "dx": native.maxpool2d_backward(state["dy"], context)}
    if kind == "infer":
        state["graph"].forward()
        return state["graph"].target_node.value
    if kind == "train":
        state["step"].one_step()
        state["step"].update()
    else:
        state["graph"].forward()
        state["graph"].backward()
    return {"out": state["out"].value, "grads": [node.grad for node in state["grads"]]}


def _resnet_layers(h, w):
    """(ci, co, size, stride, output pixels) of ResNet18's convolutions."""
    h, w = (h - 1) // 2 + 1, (w - 1) // 2 + 1
    layers = [(3, 64, 7, 2, h * w)]
    h, w = (h - 3) // 2 + 1, (w - 3) // 2 + 1
    ci = 64
    for co, stride in ((64, 1), (128, 2), (256, 2), (512, 2)):
        h, w = (h - 1) // stride + 1, (w - 1) // stride + 1
        layers.append((ci, co, 3, stride, h * w))
        if stride != 1:
            layers.append((ci, co, 1, stride, h * w))
        layers += [(co, co, 3, 1, h * w)] * 3
        ci = co
    return layers


def work(case):
    """Operations of the matrix products; bytes of the inputs, weights, targets, outputs and gradients,
    each once (for a training step the activations that the backward needs, written and read once, and
    Adam's reads and writes of its four tensors)."""
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "dense":
        m, k, n = case["batch"], case["n_in"], case["n_out"]
        return {"bytes": 4 * (2 * m * k + 2 * k * n + 2 * m * n + 2 * n), "flops": 6 * m * n * k}
    if kind == "pool":
        big = case["batch"] * case["c"] * case["h"] * case["w"]
        small = case["batch"] * case["c"] * ((case["h"] - case["size"]) // case["stride"] + 1) * (
            (case["w"] - case["size"]) // case["stride"] + 1)
        return {"bytes": 4 * (2 * big + 2 * small), "flops": 0}
    n = case["batch"]
    if kind == "conv":
        pad = case["size"] // 2
        oh, ow = ((case[d] + 2 * pad - case["size"]) // case["stride"] + 1 for d in ("h", "w"))
        weights = case["ci"] * case["co"] * case["size"] ** 2
        return {"bytes": 4 * (2 * n * case["ci"] * case["h"] * case["w"] + 2 * weights + 2 * n * case["co"] * oh * ow),
                "flops": 6 * n * oh * ow * weights}
    if kind == "block":
        s = case["stride"]
        pixels = ((case["h"] - 1) // s + 1) * ((case["w"] - 1) // s + 1)
        weights = case["co"] * (case["ci"] + case["co"]) * 9 + (case["co"] * case["ci"] if s != 1 else 0)
        return {"bytes": 4 * (2 * n * case["ci"] * case["h"] * case["w"] + 2 * weights + 8 * n * case["co"] * pixels),
                "flops": 6 * n * pixels * weights}
    if kind == "stem":
        pixels = ((case["h"] - 1) // 2 + 1) * ((case["w"] - 1) // 2 + 1)
        oh, ow = (((case[d] - 1) // 2 + 1 - 3) // 2 + 1 for d in ("h", "w"))
        return {"bytes": 4 * (2 * n * 3 * case["h"] * case["w"] + 2 * n * case["co"] * pixels + 2 * n * case["co"] * oh * ow),
                "flops": 4 * n * pixels * case["co"] * 147}
    layers = _resnet_layers(case["h"], case["w"])
    macs = sum(ci * co * f * f * px for ci, co, f, _, px in layers)
    weights = sum(ci * co * f * f for ci, co, f, _, _ in layers) + 1024
    image = 3 * case["h"] * case["w"]
    if kind == "infer":
        return {"bytes": 4 * (n * image + weights), "flops": 2 * n * macs}
    stem = layers[0]
    activations = sum(co * px for _, co, _, _, px in layers)
    return {"bytes": 4 * (2 * n * image + 2 * n * activations + 9 * weights),
            "flops": n * (6 * macs - 2 * stem[4] * 64 * 147)}


def tolerance(case):
    """About four times the distance to the same pass in 64 bits, measured over the ranges of draw()."""
    kind = case["kind"]
    if kind in ("gemm", "dense"):
        return {"rel": 4e-6, "max": 4e-5}
    if kind == "conv":
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "pool":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "infer":
        return {"rel": 1e-5, "max": 1e-4}
    # A rounding that takes a ReLU or a max-pool to its other side changes single gradients wholly.
    if kind in ("block", "stem"):
        return {"rel": 5e-3, "max": 0.99}
    return {"rel": 2e-2, "max": 0.99}


def _leaf(t):
    return t.double().requires_grad_(True)


def _norm(x):
    """A training batch norm with gamma 1 and beta 0 as leaves of their own."""
    gamma, beta = _leaf(torch.ones(x.shape[1], device=x.device)), _leaf(torch.zeros(x.shape[1], device=x.device))
    return F.batch_norm(x, None, None, gamma, beta, training=True, eps=1e-5), [gamma, beta]


def exact(case, seed):
    """The pass in 64 bits by plain torch, with torch's own gradients."""
    kind, data = case["kind"], _inputs(case, seed)
    if kind == "gemm":
        a, b = data["a"].double(), data["b"].double()
        out = (a.t() if case["layout"] == "TN" else a) @ (b.t() if case["layout"] == "NT" else b)
        return out if data["bias"] is None else out + data["bias"].double()
    if kind == "infer":
        return _exact_resnet(data, seed, training=False)[0]
    if kind == "conv":
        leaves = [_leaf(data["x"]), _leaf(data["w"])] + ([_leaf(data["b"])] if case["bias"] else [])
        y = F.conv2d(*leaves, stride=case["stride"], padding=case["size"] // 2)
        dx, dw, *db = torch.autograd.grad(y, leaves, data["dy"].double())
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db[0] if db else None}
    if kind == "pool":
        x = _leaf(data["x"])
        y = F.max_pool2d(x, case["size"], case["stride"])
        return {"y": y.detach(), "dx": torch.autograd.grad(y, x, data["dy"].double())[0]}
    if kind == "train":
        out, leaves = _exact_resnet(data, seed, training=True)
    elif kind == "dense":
        leaves = [_leaf(data["x"]), _leaf(data["w"]), _leaf(data["b"])]
        out = leaves[0] @ leaves[1] + leaves[2]
    else:
        if kind == "block":
            x, weights = _leaf(data["x"]), [_leaf(w) for w in data["weights"]]
            features, leaves = _exact_block(x, weights, case["stride"])
            leaves = [x, *leaves]
        else:
            w = _leaf(data["w"])
            features, bn = _norm(F.conv2d(data["x"].double(), w, stride=2, padding=3))
            features, leaves = F.max_pool2d(features.relu(), 3, 2), [w, *bn]
        head = [_leaf(data["head"]), _leaf(torch.zeros(1, 10, device=DEVICE))]
        out, leaves = features.mean(dim=(2, 3)) @ head[0] + head[1], leaves + head
    loss = (out - data["t"].double()).square().mean()
    return {"out": out.detach(), "grads": list(torch.autograd.grad(loss, leaves))}


def _exact_block(x, weights, stride):
    y, bn1 = _norm(F.conv2d(x, weights[0], stride=stride, padding=1))
    y, bn2 = _norm(F.conv2d(y.relu(), weights[1], padding=1))
    leaves = [weights[0], *bn1, weights[1], *bn2]
    if len(weights) > 2:
        x, bn3 = _norm(F.conv2d(x, weights[2], stride=stride))
        leaves += [weights[2], *bn3]
    return (y + x).relu(), leaves


def _exact_resnet(data, seed, training):
    """ResNet18 over the parameters and running statistics of _resnet(seed): (logits, its leaves in the
    order of the model's params)."""
    draw_weight, rng = _weights(seed), np.random.default_rng(seed)
    leaves = []

    def leaf(value):
        leaves.append(_leaf(torch.as_tensor(np.asarray(value), device=DEVICE).float()))
        return leaves[-1]

    plan = [(64, 3, 7)]  # the kernels in the order they are drawn
    for width, ci, strided in ((64, 64, False), (128, 64, True), (256, 128, True), (512, 256, True)):
        plan += [(width, ci, 3), (width, width, 3)] + ([(width, ci, 1)] if strided else []) + [(width, width, 3)] * 2

    kernels = []
    for co, ci, f in plan:
        w = leaf(draw_weight((co, ci, f, f)))
        stats = tuple(torch.as_tensor(v, device=DEVICE).float().double()
                      for v in (rng.normal(0, 0.1, co), rng.uniform(0.5, 1.5, co)))
        kernels.append((w, leaf(np.ones(co)), leaf(np.zeros(co)), stats))
    head = leaf(draw_weight((512, 2))), leaf(np.zeros(2))
    following = iter(kernels)

    def unit(x, stride, pad):
        w, gamma, beta, (mean, var) = next(following)
        x = F.conv2d(x, w, stride=stride, padding=pad)
        if training:
            return F.batch_norm(x, None, None, gamma, beta, training=True, eps=1e-5)
        return F.batch_norm(x, mean, var, gamma, beta, eps=1e-5)

    def block(x, stride):
        y = unit(unit(x, stride, 1).relu(), 1, 1)
        return (y + (x if stride == 1 else unit(x, stride, 0))).relu()

    def network(x):
        x = F.max_pool2d(unit(x, 2, 3).relu(), 3, 2)
        for stride in (1, 2, 2, 2):
            x = block(block(x, stride), 1)
        return x.mean(dim=(2, 3)) @ head[0] + head[1]

    x = data["x"].double()
    if training:
        return network(x), leaves
    with torch.no_grad():
        logits = []
        for part in x.split(16):
            following = iter(kernels)
            logits.append(network(part))
    return torch.cat(logits), leaves
