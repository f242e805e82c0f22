"""What a user of this framework has it do, as cases that can be timed: training steps and inference of the networks in
``models.py`` / ``resnet20.py``, single adder layers as these and other networks contain them, and the column-matrix
operator.

    listed()          the named cases            draw(rng)         one more case of the same ranges
    prepare(case, s)  network / layer and inputs of seed ``s`` on the GPU
    run(state)        one pass through the public entry points, with its outputs
    work(case)        bytes and operations one pass cannot do without        tolerance(case)
"""
import math

import torch

DEV = "cuda"

# Input sizes of the networks: 32x32 images and ten classes (CIFAR), 224x224 and a thousand for ResNet-50.
ARCHS = {"resnet20": (32, 10), "vgg_small": (32, 10), "densenet_cifar": (32, 10), "resnet50": (224, 1000)}


def listed():
    return [
        # the training step the framework's headline number is quoted on: ResNet-20 on 32x32 images at batch 256, run as
        # the training script runs it (one captured HIP graph, fresh data copied into its input buffers)
        {"name": "train_resnet20_b256", "kind": "train", "arch": "resnet20", "batch": 256},
        # two other networks of the training script, eager steps (its --no-graph; also its tail batches)
        {"name": "train_vgg_small_b128", "kind": "train", "arch": "vgg_small", "batch": 128},
        {"name": "train_densenet_b64", "kind": "train", "arch": "densenet_cifar", "batch": 64},
        # a layer of ResNet-50's longest stage, whose maps are 14x14 (the gradients of that whole network, untrained, amplify
        # a last-bit difference to tens of per cent: no training step of it here)
        {"name": "layer_1x1_f32_14x14", "kind": "layer", "dtype": "float32", "batch": 64, "ci": 1024, "co": 256, "h": 14, "w": 14,
         "k": 1, "stride": 1, "pad": 0},
        # serving: one image at a time (latency), and a small batch of a large network
        {"name": "infer_resnet20_b1", "kind": "infer", "arch": "resnet20", "batch": 1},
        {"name": "infer_resnet50_b32", "kind": "infer", "arch": "resnet50", "batch": 32},
        # a layer of a user's own network: 5x5 taps (adder2d takes any kernel size)
        {"name": "layer_5x5_f32", "kind": "layer", "dtype": "float32", "batch": 64, "ci": 32, "co": 64, "h": 16, "w": 16,
         "k": 5, "stride": 1, "pad": 2},
        # channel counts, a map and a batch that are multiples of nothing: a small layer, launch-bound
        {"name": "layer_ragged_f32", "kind": "layer", "dtype": "float32", "batch": 7, "ci": 37, "co": 51, "h": 27, "w": 19,
         "k": 3, "stride": 1, "pad": 1},
        # the bfloat16-storage mode on the two kinds of layer a bottleneck block has
        {"name": "layer_3x3_bf16", "kind": "layer", "dtype": "bfloat16", "batch": 32, "ci": 64, "co": 64, "h": 56, "w": 56,
         "k": 3, "stride": 1, "pad": 1},
        {"name": "layer_1x1_bf16", "kind": "layer", "dtype": "bfloat16", "batch": 32, "ci": 128, "co": 512, "h": 28, "w": 28,
         "k": 1, "stride": 1, "pad": 0},
        # the literal operator of the reference's extension on an unfolded input: its own comparison shape, and the second
        # stage of ResNet-20 at batch 256
        {"name": "col_small", "kind": "col", "co": 32, "k": 288, "nl": 1024},
        {"name": "col_resnet20_b256", "kind": "col", "co": 32, "k": 288, "nl": 65536},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "infer", "layer", "layer", "layer", "col"])
    if kind == "train":
        arch = rng.choice(["resnet20", "vgg_small", "densenet_cifar"])
        most = {"resnet20": 512, "vgg_small": 160, "densenet_cifar": 64}[arch]
        return {"kind": kind, "arch": arch, "batch": _log_int(rng, 8, most)}
    if kind == "infer":
        arch = rng.choice(list(ARCHS))
        most = {"resnet20": 1024, "vgg_small": 256, "densenet_cifar": 256, "resnet50": 32}[arch]
        return {"kind": kind, "arch": arch, "batch": _log_int(rng, 1, most)}
    if kind == "layer":
        k = rng.choice([1, 1, 3, 3, 3, 5])
        h = _log_int(rng, 7, 64)
        case = {"kind": kind, "dtype": rng.choice(["float32", "float32", "bfloat16"]), "batch": 1,
                "ci": _log_int(rng, 3, 1024), "co": _log_int(rng, 8, 1024), "h": h, "w": max(7, h + rng.choice([0, 0, 0, -1, 3, 8])),
                "k": k, "stride": rng.choice([1, 1, 1, 2]), "pad": k // 2}
        # as many images as keep the pass below 4e9 terms and the tensors below 2^25 elements
        ho, wo = _out_hw(case)
        terms = case["co"] * case["ci"] * k * k * ho * wo
        elems = max(case["ci"] * case["h"] * case["w"], case["co"] * ho * wo)
        most = max(1, min(256, int(4e9) // terms, (1 << 25) // elems))
        case["batch"] = _log_int(rng, 1, most) if most > 1 else 1
        return case
    while True:
        case = {"kind": "col", "co": _log_int(rng, 8, 256), "k": _log_int(rng, 27, 2304), "nl": _log_int(rng, 64, 262144)}
        if case["k"] * case["nl"] <= 4e7 and case["co"] * case["k"] * case["nl"] <= 2e9:
            return case


def _out_hw(case):
    k, s, p = case["k"], case["stride"], case["pad"]
    return (case["h"] - k + 2 * p) // s + 1, (case["w"] - k + 2 * p) // s + 1


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen)


def _network(arch, seed):
    from addernetcuda_amd.train import build_network
    torch.manual_seed(seed)
    with torch.device(DEV):
        return build_network(arch, eta=0.1, num_classes=ARCHS[arch][1])


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(1000 + int(seed))
    kind = case["kind"]
    if kind in ("train", "infer"):
        size, classes = ARCHS[case["arch"]]
        net = _network(case["arch"], int(seed))
        images = _randn(gen, case["batch"], 3, size, size)          # normalised images
        if kind == "infer":
            # BatchNorm statistics as a trained network has them: those of its own activations
            norms = [m for m in net.modules() if isinstance(m, torch.nn.BatchNorm2d)]
            for m in norms:
                m.momentum = 1.0
            with torch.no_grad():
                net.train()(_randn(gen, 16, 3, size, size))
            for m in norms:
                m.momentum = 0.1
            return {"kind": kind, "net": net.eval(), "images": images}
        from addernetcuda_amd.optim import SGD
        from addernetcuda_amd.train import GraphedStep, train_step
        labels = torch.randint(0, classes, (case["batch"],), device=DEV, generator=gen)
        # the step size the cosine schedule ends on, so that every pass starts from the same weights
        opt = SGD(net.train().parameters(), lr=torch.zeros((), device=DEV), momentum=0.9, weight_decay=5e-4)
        state = {"kind": kind, "net": net, "opt": opt, "images": images, "labels": labels, "stream": None}
        if case["arch"] == "resnet20":
            state["step"], state["stream"] = GraphedStep(net, opt), torch.cuda.Stream()
            for _ in range(4):    # three eager steps and the capture: what the training script spends on its first batches
                _train_pass(state)
        else:
            state["step"] = lambda x, y: train_step(net, opt, x, y)
        return state
    if kind == "layer":
        from addernetcuda_amd.adder import adder2d
        torch.manual_seed(int(seed))
        with torch.device(DEV):
            layer = adder2d(case["ci"], case["co"], case["k"], stride=case["stride"], padding=case["pad"])
        dtype = getattr(torch, case["dtype"])
        # activations behind a BatchNorm and a ReLU; a gradient that a BatchNorm behind the layer has scaled down
        x = torch.relu(_randn(gen, case["batch"], case["ci"], case["h"], case["w"])).to(dtype).requires_grad_(True)
        gy = (_randn(gen, case["batch"], case["co"], *_out_hw(case)) * 0.1).to(dtype)
        return {"kind": kind, "layer": layer, "x": x, "gy": gy}
    w = _randn(gen, case["co"], case["k"]).requires_grad_(True)
    x = torch.relu(_randn(gen, case["k"], case["nl"])).requires_grad_(True)
    return {"kind": kind, "x": x, "w": w, "gy": _randn(gen, case["co"], case["nl"]) * 0.1}


def _train_pass(state):
    if state["stream"] is None:
        return state["step"](state["images"], state["labels"])
    here = torch.cuda.current_stream()
    state["stream"].wait_stream(here)
    with torch.cuda.stream(state["stream"]):
        loss = state["step"](state["images"], state["labels"])
    here.wait_stream(state["stream"])
    return loss


def _flat(grads):
    return torch.cat([g.reshape(-1) for g in grads])


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            return state["net"](state["images"])
    if kind == "train":
        loss = _train_pass(state)
        # every gradient of the step, as one vector of the adder weights' and one of all the others (a network has
        # several hundred parameters)
        named = [(n, p.grad) for n, p in state["net"].named_parameters()]
        return {"loss": loss, "adder_grads": _flat([g for n, g in named if n.endswith(".adder")]),
                "other_grads": _flat([g for n, g in named if not n.endswith(".adder")])}
    if kind == "layer":
        x, layer = state["x"], state["layer"]
        x.grad = layer.adder.grad = None
        y = layer(x)
        y.backward(state["gy"])
        return {"y": y.detach(), "gx": x.grad, "gw": layer.adder.grad}
    from addernetcuda_amd.adder import adder
    x, w = state["x"], state["w"]
    x.grad = w.grad = None
    y = adder.apply(w, x)
    y.backward(state["gy"])
    return {"y": y.detach(), "gx": x.grad, "gw": w.grad}


# Layers of a network on its usual input, as (count, Ci, H, Co, k, stride): adder layers, then ordinary ones.
def _layers(arch):
    if arch == "resnet20":
        return ([(6, 16, 32, 16, 3, 1), (1, 16, 32, 32, 1, 2), (1, 16, 32, 32, 3, 2), (5, 32, 16, 32, 3, 1),
                 (1, 32, 16, 64, 1, 2), (1, 32, 16, 64, 3, 2), (5, 64, 8, 64, 3, 1)], [(1, 3, 32, 16, 3, 1), (1, 64, 1, 10, 1, 1)])
    if arch == "vgg_small":
        return ([(1, 128, 32, 128, 3, 1), (1, 128, 16, 256, 3, 1), (1, 256, 16, 256, 3, 1), (1, 256, 8, 512, 3, 1),
                 (1, 512, 8, 512, 3, 1)], [(1, 3, 32, 128, 3, 1), (1, 8192, 1, 10, 1, 1)])
    if arch == "resnet50":
        adders, cin, h = [], 64, 56
        for planes, blocks, stride in ((64, 3, 1), (128, 4, 2), (256, 6, 2), (512, 3, 2)):
            for b in range(blocks):
                s = stride if b == 0 else 1
                adders += [(1, cin, h, planes, 1, 1), (1, planes, h, planes, 3, s)]
                if b == 0:
                    adders.append((1, cin, h, 4 * planes, 1, s))
                h, cin = h // s, 4 * planes
                adders.append((1, planes, h, 4 * planes, 1, 1))
        return adders, [(1, 3, 224, 64, 7, 2), (1, 2048, 1, 1000, 1, 1)]
    adders, planes, h, growth = [], 24, 32, 12
    for stage, blocks in enumerate((6, 12, 24, 16)):
        for _ in range(blocks):
            adders += [(1, planes, h, 4 * growth, 1, 1), (1, 4 * growth, h, growth, 3, 1)]
            planes += growth
        if stage < 3:
            adders.append((1, planes, h, planes // 2, 1, 1))
            planes, h = planes // 2, h // 2
    return adders, [(1, 3, 32, 24, 3, 1), (1, planes, 1, 10, 1, 1)]


def _terms(layers):
    return sum(n * ci * co * k * k * (h // s) ** 2 for n, ci, h, co, k, s in layers)


def _weights(layers):
    return sum(n * ci * co * k * k for n, ci, h, co, k, s in layers)


def work(case):
    """A term of an adder layer is 2 operations forward (subtract, add), 4 for the input's gradient (subtract, clamp,
    multiply, add) and 2 for the weight's (multiply, add).  Bytes: inputs and weights in, results and gradients out."""
    kind = case["kind"]
    if kind in ("train", "infer"):
        size, classes = ARCHS[case["arch"]]
        adders, others = _layers(case["arch"])
        n, params = case["batch"], _weights(adders) + _weights(others)
        train = kind == "train"
        return {"bytes": 4 * (n * (3 * size * size + classes) + (2 if train else 1) * params),
                "flops": n * ((8 if train else 2) * _terms(adders) + (6 if train else 2) * _terms(others))}
    if kind == "layer":
        ho, wo = _out_hw(case)
        nx, ny = case["batch"] * case["ci"] * case["h"] * case["w"], case["batch"] * case["co"] * ho * wo
        nw = case["co"] * case["ci"] * case["k"] ** 2
        return {"bytes": (2 if case["dtype"] == "bfloat16" else 4) * (2 * nx + 2 * ny) + 4 * 2 * nw,
                "flops": 8 * (nw * case["batch"] * ho * wo)}
    nx, ny, nw = case["k"] * case["nl"], case["co"] * case["nl"], case["co"] * case["k"]
    return {"bytes": 4 * (2 * nx + 2 * ny + 2 * nw), "flops": 8 * nw * case["nl"]}


def tolerance(case):
    """About four times what the path differs by from itself in float64."""
    kind = case["kind"]
    if kind == "train":
        # up to 5.3e-3 (adder weights) over batches 8..256: a last-bit difference flips a few ReLUs, and the gradients
        # of the weights behind them change by their own size
        return {"rel": 2e-2, "max": 0.99}
    if kind == "infer":
        # 4.1e-4 for ResNet-50's logits, below 3e-5 for the networks of 32x32 images
        return {"rel": 2e-3, "max": 2e-2} if case["arch"] == "resnet50" else {"rel": 1e-4, "max": 1e-3}
    if kind == "layer" and case["dtype"] == "bfloat16":
        return {"rel": 8e-3, "max": 1.6e-2}      # 2.1e-3 and 3.9e-3: the rounding of the stored results
    return {"rel": 3e-6, "max": 3e-5}            # 3.4e-7 and 3.0e-6, a little more where there are more terms
