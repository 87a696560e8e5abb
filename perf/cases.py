"""What this framework is used for, as measurable cases: training steps and inference passes of ``ConvBlock`` and of the
stand-alone depthwise convolution, called the way a PyTorch program calls them (eagerly, or replayed as the HIP graphs
of ``pyramidconvblock_amd.graphs``).

    listed()            the standing cases
    draw(rng)           one more case from the ranges that these stand for
    prepare(case, seed) inputs on the GPU, the module and, for graph cases, its captured graph
    run(state)          one pass, and everything it computes: outputs, input gradient, parameter gradients
    work(case)          bytes and operations that a pass cannot do without
    tolerance(case)     how far another correct implementation of the same precision may be off

A case is a dict of plain values:

    op      "block" (ConvBlock(dim, kernel_size) with its default scales 1 and 1/2) or "conv" (OptimizedDepthwiseConv2d
            with 'same' padding)
    mode    "train": forward and backward, "infer": forward under no_grad
    launch  "eager": one call of the module per pass, "graph": one replay of a captured pass
    dtype   "bf16", "fp16" or "fp32"
    B, H, W, C, k   batch, image extents, channels (the block's dim) and filter size

Ranges: batches of 1 to 128 images of 7 to 112 pixels a side, odd and even; 32 to 1152 channels, multiples of 8; odd
filters from 3 to 17; up to the work of the largest listed case.  Graphs are drawn up to 256 channels (wider blocks run
library products, which programs rather launch than capture).
"""
import math

import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, op, mode, launch, dtype, shape, k):
    B, H, W, C = shape
    return {"name": name, "op": op, "mode": mode, "launch": launch, "dtype": dtype, "B": B, "H": H, "W": W, "C": C, "k": k}


def listed():
    return [
        # a small block in full precision: unit tests, debugging, small models; nothing but latency and launches
        _case("block_train_small_fp32", "block", "train", "eager", "fp32", (2, 32, 32, 64), 7),
        # one image through a trained model: serving latency
        _case("block_infer_one_bf16", "block", "infer", "eager", "bf16", (1, 56, 56, 128), 13),
        # an inference batch with the largest filter, as a captured model replays it
        _case("block_infer_graph_bf16", "block", "infer", "graph", "bf16", (32, 56, 56, 128), 17),
        # the training step that the benchmark reports, as a captured model replays it
        _case("block_train_graph_bf16", "block", "train", "graph", "bf16", (32, 56, 56, 128), 13),
        # the same step in full precision, launched eagerly
        _case("block_train_fp32", "block", "train", "eager", "fp32", (32, 56, 56, 128), 13),
        # a high-resolution stage: fewer channels, more pixels, the largest filter
        _case("block_train_highres_fp16", "block", "train", "eager", "fp16", (8, 112, 112, 96), 17),
        # odd extents and a channel count off the powers of two: no tile, vector or pooled size comes out even
        _case("block_train_ragged_bf16", "block", "train", "eager", "bf16", (3, 57, 61, 200), 9),
        _case("block_train_ragged_graph_fp32", "block", "train", "graph", "fp32", (3, 57, 61, 200), 15),
        # a wide block on small maps: the deep stage of a large model
        _case("block_train_wide_fp16", "block", "train", "eager", "fp16", (4, 64, 64, 1152), 13),
        # the depthwise convolution by itself, as a layer of somebody else's block: inference, and training when wide
        _case("conv_infer_bf16", "conv", "infer", "eager", "bf16", (32, 56, 56, 128), 13),
        _case("conv_train_wide_fp16", "conv", "train", "eager", "fp16", (8, 64, 64, 1152), 9),
        # a large training batch: throughput
        _case("block_train_large_bf16", "block", "train", "eager", "bf16", (128, 56, 56, 128), 13),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = "conv" if rng.random() < 0.2 else "block"
    mode = "infer" if rng.random() < 0.3 else "train"
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    k = rng.choice([3, 5, 7, 9, 11, 13, 15, 17])
    C = 8 * _log_int(rng, 4, 144)
    H = _log_int(rng, 7, 112)
    W = min(112, max(7, H + rng.choice([0, 0, 0, 1, -1, 4, -3, H // 3])))
    B = _log_int(rng, 1, 128)
    launch = "graph" if C <= 256 and rng.random() < 0.4 else "eager"
    most = _cost(listed()[-1]) / (4 if dtype == "fp32" else 2)
    while B > 1 and _cost(dict(op=op, mode=mode, dtype=dtype, B=B, H=H, W=W, C=C, k=k)) > most:
        B //= 2
    case = _case("", op, mode, launch, dtype, (B, H, W, C), k)
    del case["name"]
    return case


def _cost(case):
    w = work(case)
    return w["bytes"] + w["flops"] / 50


def prepare(case, seed):
    import pyramidconvblock_amd as pcb
    from pyramidconvblock_amd.graphs import GraphedForward, GraphedStep

    dtype = DTYPES[case["dtype"]]
    shape = (case["B"], case["H"], case["W"], case["C"])
    torch.manual_seed(seed)   # the module's own default initialisation
    if case["op"] == "block":
        module = pcb.ConvBlock(dim=case["C"], kernel_size=case["k"])
    else:
        module = pcb.OptimizedDepthwiseConv2d(case["C"], case["k"], padding=case["k"] // 2)
    module = module.to(dtype).cuda()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    train, graph = case["mode"] == "train", None
    x = torch.randn(shape, generator=gen, device="cuda").to(dtype)
    g = torch.randn(shape, generator=gen, device="cuda").to(dtype) if train else None
    if case["launch"] == "graph":
        graph = GraphedStep(module, x, g) if train else GraphedForward(module, x)
    elif train:
        x.requires_grad_()
    params = list(module.parameters())
    return {"module": module, "params": params, "x": x, "g": g, "train": train, "graph": graph}


def run(state):
    graph = state["graph"]
    if graph is not None:
        y = graph.replay()
        return [y, graph.x.grad, *graph.param_grads] if state["train"] else [y]
    if not state["train"]:
        with torch.no_grad():
            return [state["module"](state["x"])]
    x, params = state["x"], state["params"]
    x.grad = None
    for p in params:
        p.grad = None
    y = state["module"](x)
    torch.autograd.backward(y, state["g"])
    return [y, x.grad, *[p.grad for p in params]]


def work(case):
    B, H, W, C, k = (case[n] for n in ("B", "H", "W", "C", "k"))
    es = 4 if case["dtype"] == "fp32" else 2
    N = B * H * W
    if case["op"] == "conv":
        params, flops = k * k * C, 2.0 * k * k * N * C
    else:
        I = C // 2
        n = B * (H // 2) * (W // 2)
        params = 2 * C * I + 2 * k * k * I + C * C + 2 * C
        # the two dense layers, both convolutions, and the mean branch's layer (one row per image)
        flops = 2.0 * 2 * N * C * I + 2.0 * k * k * (N + n) * I + 2.0 * B * C * C
    if case["mode"] == "infer":
        return {"bytes": es * (2.0 * N * C + params), "flops": flops}
    # x, the output, both their gradients; parameters and their gradients.  The backward is two products per product
    return {"bytes": es * (4.0 * N * C + 2 * params), "flops": 3 * flops}


def tolerance(case):
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}[case["dtype"]]}
