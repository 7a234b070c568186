"""The workloads whose speed matters to a user of this framework, with their sizes.

Five kinds of work, each through the public entry points:

* ``layer``    one dilated convolution + ReLU as an autograd function, forward and backward
               with all three gradients: a layer inside somebody's own network;
* ``learn``    ``model.learn(input, target)``: one optimisation step whose loss is read back,
               what an interactive loop over small images does (launches and latency count);
* ``graph``    the same step recorded once with ``GraphedStep`` and replayed;
* ``train``    ``model.train(batches, 1)``: an epoch over a few batches that are on the GPU;
* ``predict``  ``model.net(input)`` without gradients: applying a trained network.

Images are standardised noise on a smooth background, the regression target is a smoothed
version of the input, labels are drawn uniformly; networks start from their usual
initialisation, with a final layer and an optimiser as after some training (the initial final
layer is zero, which would make every gradient of the block vanish, and the first steps of a
fresh Adam are the signs of the gradients, which amplify rounding without end)."""
import math

import torch

import msd_pytorch_amd as mp
from msd_pytorch_amd import conv2d, conv3d

DILATIONS = {"1-10": [1, 2, 3, 4, 5, 6, 7, 8, 9, 10], "1-8": [1, 2, 4, 8]}


def _net(name, kind, task, size, *, batch=1, c_in=1, c_out=1, depth=100, width=1, dilations="1-10",
         batches=1):
    """A case of a whole network; ``size`` is "HxW" or "DxHxW"."""
    case = {"kind": kind, "task": task, "size": size, "batch": batch, "c_in": c_in, "c_out": c_out,
            "depth": depth, "width": width, "dilations": dilations, "batches": batches}
    return {"name": name, **case} if name else case


def _layer(name, size, *, batch=1, c_in=1, c_out=1, dilation=1):
    case = {"kind": "layer", "size": size, "batch": batch, "c_in": c_in, "c_out": c_out, "dilation": dilation}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one small layer of a user's own network, differentiated: launches and host work only
        _layer("layer 2d 96x96", "96x96", c_in=12, dilation=3),
        # a layer of a volume with ragged rows: the operators outside the dense block
        _layer("layer 3d 40x61x75", "40x61x75", c_in=16, dilation=2),
        # the smallest network of the benchmark: a step of a few dozen launches, loss read back
        _net("learn 2d 256x256", "learn", "L2", "256x256", depth=10),
        # the same network as a recorded step: what the launches themselves cost
        _net("graph 2d 256x256", "graph", "L2", "256x256", depth=10),
        # slices with neighbours as channels, ragged, three labels, powers of two as dilations
        _net("train 2d 3x333x477", "train", "labels", "333x477", batch=3, c_in=5, c_out=3, depth=30, dilations="1-8",
             batches=2),
        # the usual depth on a batch of ordinary slices
        _net("train 2d 4x512x512", "train", "L2", "512x512", batch=4, batches=2),
        # the headline network: segmentation of one large slice into four labels
        _net("train 2d 1024x1024", "train", "labels", "1024x1024", c_out=4, batches=2),
        # the largest: two channels per layer, depth 200, a very large slice
        _net("train 2d 2048x2048 w2", "train", "L2", "2048x2048", c_in=2, depth=200, width=2),
        # a volume whose extents are all odd, absolute loss
        _net("train 3d 61x93x75", "train", "L1", "61x93x75", depth=20, batches=2),
        # the headline network for volumes
        _net("train 3d 128^3", "train", "L2", "128x128x128", depth=50, batches=2),
        # a trained network applied to one detector-sized slice with an odd number of columns
        _net("predict 2d 1500x1021", "predict", "labels", "1500x1021", c_out=4),
        # and to a whole volume
        _net("predict 3d 256^3", "predict", "L2", "256x256x256", depth=30),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edges(rng, ndim, lo, hi):
    """Extents around one common size, a third of them rounded to a multiple of 32."""
    base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    out = []
    for _ in range(ndim):
        n = int(min(hi, max(lo, base * rng.uniform(0.7, 1.4))))
        if rng.random() < 0.35:
            n = max(32, (n + 16) // 32 * 32)
        out.append(n)
    return "x".join(str(n) for n in out)


def draw(rng):
    """A case of the listed kinds anywhere in their ranges, at most as expensive as a step of
    the headline networks."""
    kind = rng.choice(["layer", "layer", "learn", "graph", "train", "train", "train", "predict", "predict"])
    ndim = rng.choice([2, 2, 3])
    while True:
        if kind == "layer":
            lo, hi = (32, 1024) if ndim == 2 else (16, 128)
            case = _layer(None, _edges(rng, ndim, lo, hi), batch=rng.choice([1, 1, 2, 4]), c_in=_log_int(rng, 1, 64),
                          c_out=rng.choice([1, 1, 1, 2, 3]), dilation=rng.randint(1, 10))
        else:
            small = kind in ("learn", "graph")
            if ndim == 2:
                lo, hi = (64, 384) if small else (128, 1536)
                depth = _log_int(rng, 6, 28) if small else rng.randint(20, 100)
            else:
                lo, hi = (16, 48) if small else (32, 192)
                depth = _log_int(rng, 6, 28) if small else rng.randint(10, 50)
            task = rng.choice(["L2", "L1", "labels"])
            case = _net(None, kind, task, _edges(rng, ndim, lo, hi), batch=rng.choice([1, 1, 2, 4]),
                        c_in=rng.choice([1, 1, 1, 2, 5]),
                        c_out=rng.randint(2, 6) if task == "labels" else rng.choice([1, 1, 2]),
                        depth=depth, width=rng.choice([1, 1, 1, 2]), dilations=rng.choice(["1-10", "1-10", "1-8"]),
                        batches=2 if kind == "train" else 1)
        if work(case)["flops"] <= 6e11:
            return case


def _size(case):
    return tuple(int(n) for n in case["size"].split("x"))


def _image(gen, batch, channels, size):
    """Unit-variance noise on a smooth wave."""
    x = torch.randn(batch, channels, *size, device="cuda", generator=gen)
    ramp = torch.linspace(0, 9, size[-1], device="cuda")
    return 0.8 * x + 0.8 * torch.sin(ramp)


def _smooth(x):
    """The regression target: a moving average along the rows."""
    return (x + x.roll(1, -1) + x.roll(-1, -1)) / 3


def _resume(optimizer, params):
    """The optimiser as a checkpoint restores it after a thousand steps."""
    saved = optimizer.state_dict()
    saved["state"] = {i: {"step": torch.tensor(1000.0), "exp_avg": torch.zeros_like(p),
                          "exp_avg_sq": torch.full_like(p, 1e-6)} for i, p in enumerate(params)}
    optimizer.load_state_dict(saved)


def prepare(case, seed):
    size = _size(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "layer":
        taps = 3 ** len(size)
        x = _image(gen, case["batch"], case["c_in"], size).requires_grad_()
        shape = (case["c_out"], case["c_in"], *([3] * len(size)))
        weight = torch.randn(shape, device="cuda", generator=gen) * math.sqrt(2 / (taps * case["c_in"]))
        bias = torch.randn(case["c_out"], device="cuda", generator=gen) * 0.1
        out = torch.empty(case["batch"], case["c_out"], *size, device="cuda")
        grad = torch.randn(out.shape, device="cuda", generator=gen)
        fn = conv2d.conv2d_relu if len(size) == 2 else conv3d.conv3d_relu
        return {"case": case, "fn": fn, "leaves": (x, weight.requires_grad_(), bias.requires_grad_()), "out": out,
                "grad": grad}

    torch.manual_seed(seed)
    dilations = DILATIONS[case["dilations"]]
    if case["task"] == "labels":
        model = mp.MSDSegmentationModel(case["c_in"], case["c_out"], case["depth"], case["width"],
                                        dilations=dilations, ndim=len(size))
    else:
        model = mp.MSDRegressionModel(case["c_in"], case["c_out"], case["depth"], case["width"],
                                      dilations=dilations, loss=case["task"], ndim=len(size))
    with torch.no_grad():
        for p in model.msd.final_layer.parameters():
            p.normal_(0, 0.1, generator=gen)
    state = {"case": case, "model": model, "params": list(model.msd.parameters())}
    if case["kind"] == "predict":
        state["x"] = _image(gen, case["batch"], case["c_in"], size)
        return state
    if case["kind"] == "graph":
        model.optimizer = torch.optim.Adam(state["params"], capturable=True)
    _resume(model.optimizer, state["params"])
    batches = []
    for _ in range(case["batches"]):
        x = _image(gen, case["batch"], case["c_in"], size)
        if case["task"] == "labels":
            y = torch.randint(0, case["c_out"], (case["batch"], 1, *size), device="cuda", generator=gen)
        else:
            y = _smooth(x[:, :1]).expand(-1, case["c_out"], *size).contiguous()
        batches.append((x, y))
    if case["kind"] == "graph":
        model.set_input(batches[0][0])
        model.set_target(batches[0][1])
        state["step"] = mp.GraphedStep(model, update=True)
    state["batches"] = batches
    return state


def _joined(tensors):
    return torch.cat([t.reshape(-1) for t in tensors])


def run(state):
    case = state["case"]
    if case["kind"] == "layer":
        x, weight, bias = state["leaves"]
        out = state["fn"](x, weight, bias, state["out"], 1, case["dilation"])
        return out.detach(), torch.autograd.grad(out, state["leaves"], state["grad"])
    model = state["model"]
    if case["kind"] == "predict":
        with torch.no_grad():
            return model.net(state["x"])
    params = state["params"]
    if case["kind"] == "train":
        model.train(state["batches"], 1)
        # one tensor each: a network of this depth has about a hundred parameters
        return {"loss": model.loss.detach(), "output": model.output, "grads": _joined(p.grad for p in params),
                "params": _joined(p.detach() for p in params)}
    x, y = state["batches"][0]
    if case["kind"] == "graph":
        state["step"](x, y)
        loss = model.loss
    else:
        loss = model.learn(x, y)
    return {"loss": loss, "output": model.output, "grads": [p.grad for p in params],
            "params": [p.detach() for p in params]}


def work(case):
    """Bytes: inputs, targets, outputs, parameters and (in training) gradients and the two
    moments of Adam once each, and the activations of every layer written once in the forward
    pass and read once in the backward pass.  Operations: two per multiply-add of the
    convolutions and the final layer, in each of the three products of a training step (the
    first layer of a network needs no gradient of its input)."""
    size = _size(case)
    voxels, taps = math.prod(size) * case["batch"], 3 ** len(size)
    if case["kind"] == "layer":
        weights = case["c_in"] * case["c_out"] * taps
        planes = case["c_in"] + case["c_out"]
        return {"bytes": 4 * (voxels * (2 * planes + case["c_out"]) + 3 * weights), "flops": 6 * voxels * weights}
    depth, width, c_in, c_out = case["depth"], case["width"], case["c_in"], case["c_out"]
    hidden = depth * width
    convs = taps * width * sum(c_in + i * width for i in range(depth))
    final = (c_in + hidden) * c_out
    params = convs + hidden + final + c_out
    if case["kind"] == "predict":
        return {"bytes": 4 * (voxels * (c_in + c_out) + params), "flops": 2 * voxels * (convs + final)}
    labels = case["task"] == "labels"
    target = 2 if labels else c_out                      # labels are 64-bit integers
    first = taps * width * c_in
    steps = case["batches"]
    return {"bytes": 4 * steps * (voxels * (c_in + target + c_out + 2 * hidden) + 8 * params),
            "flops": 2 * steps * voxels * (3 * (convs + final) - first)}


def tolerance(case):
    """A layer or a forward pass is 32-bit sums in another order.  In training an activation
    within rounding of zero may get the other sign, which moves a whole voxel in and out of the
    gradients of everything below it, and a bias gradient is a sum of both signs over all voxels
    that nearly cancels: the same network on kernels with other orders of summation differs by
    up to 2e-4 of a gradient's norm, mostly by 1e-6."""
    return {"rel": 1e-5} if case["kind"] in ("layer", "predict") else {"rel": 1e-3}
