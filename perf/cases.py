"""What the speed of this framework is measured on: its public operators on voxelised surfaces.

A case is one pass of a user's program: a stack of submanifold convolutions trained or evaluated with its neighbor cache
built on the way (new coordinates) or kept from an earlier pass, a generic strided convolution (the downsampling step of a
sparse U-Net) with its output coordinates, or coordinates coded along a space-filling curve and back.

Fields of a case
  op       "subm" | "conv" | "serialize"
  res      side of the voxel grid; the active voxels are a spherical surface in it
  thick    False: |distance to the centre - 0.45 res| <= 0.5, the surface of the benchmark configurations
           True: the outer 1.25 voxels of the inscribed ball, the surface of the stacked-layer benchmark
  batch    samples per call;  shuffle: rows in random order instead of scan order
  ci, co   channels in and out (further layers of a stack are co -> co);  layers: their number
  dtype    "f16" | "bf16" | "f32"
  train    forward and all gradients, or forward alone under no_grad;  input_grad: whether the first layer's input wants one
  relu     the operator with the ReLU epilogue;  bias: whether the layers have one;  dilation: of a submanifold layer
  cache    "fresh": the pass builds the neighbor cache from the coordinates;  "kept": the program holds it
  kernel, stride, padding  of a generic convolution (the same on all axes)
  mode     "z_order" | "hilbert"
"""
import math

import torch

import flex_gemm
from flex_gemm.ops.serialize import decode_seq, encode_seq

spconv = flex_gemm.ops.spconv
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ELEMENT_BYTES = {"f16": 2, "bf16": 2, "f32": 4}

SUBM = {"op": "subm", "res": 64, "thick": True, "batch": 1, "shuffle": False, "ci": 64, "co": 64, "layers": 1, "dtype": "f16", "train": True,
        "input_grad": True, "relu": False, "bias": True, "dilation": 1, "cache": "fresh"}
CONV = {"op": "conv", "res": 64, "thick": True, "batch": 1, "shuffle": False, "ci": 64, "co": 64, "dtype": "f16", "train": True,
        "input_grad": True, "relu": False, "bias": True, "kernel": 2, "stride": 2, "padding": 0, "cache": "fresh"}
SERIALIZE = {"op": "serialize", "res": 256, "thick": False, "batch": 1, "shuffle": True, "mode": "hilbert"}


def listed():
    return [
        # one layer of a small network answering a single request: launches and host time are all there is
        dict(SUBM, name="subm_infer_tiny", res=16, ci=32, co=32, train=False, cache="kept"),
        # a training step of the coarse, cheap levels of a network, new coordinates every step
        dict(SUBM, name="subm_train_small", res=32, ci=64, co=64, layers=2, relu=True),
        # the stacked-layer benchmark's coarse end: few voxels under wide layers, the weights are the traffic
        dict(SUBM, name="subm_train_deep", res=16, ci=1024, co=1024, layers=8, dtype="bf16"),
        # the first layer of a network: a handful of input features, no gradient for them, an odd number of voxels' samples
        dict(SUBM, name="subm_train_stem", res=192, batch=3, ci=6, co=48, dtype="bf16", input_grad=False),
        # full-precision training of a medium layer
        dict(SUBM, name="subm_train_fp32", res=100, ci=96, co=96, dtype="f32", bias=False),
        # one forward pass at the middle of the range, coordinates seen for the first time (benchmark configuration 2)
        dict(SUBM, name="subm_infer_256", res=256, thick=False, ci=256, co=256, train=False),
        # the headline training step: 512^3 surface, 128 channels, cache reused (benchmark configuration 3)
        dict(SUBM, name="subm_train_512", res=512, thick=False, ci=128, co=128, cache="kept"),
        # very many voxels, narrow layers, rows in random order, cache built in the step (benchmark configuration 4)
        dict(SUBM, name="subm_train_1024", res=1024, thick=False, ci=32, co=32, layers=2, dtype="bf16", shuffle=True),
        # the widest layers: matrix products (benchmark configuration 5)
        dict(SUBM, name="subm_train_wide", res=128, thick=False, ci=1024, co=1024, cache="kept"),
        # the downsampling step of a U-Net in training: output coordinates, both maps, three passes
        dict(CONV, name="conv_down_train", res=256, ci=64, co=128, dtype="bf16"),
        # an overlapping downsampling convolution at inference
        dict(CONV, name="conv_down_infer", res=301, thick=False, ci=40, co=72, train=False, kernel=3, padding=1, relu=True),
        # ordering codes for the tokens of two large samples, and the coordinates back
        dict(SERIALIZE, name="serialize_1024", res=1024, batch=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng):
    kind = rng.random()
    if kind < 0.6:
        return 16 * _log_int(rng, 1, 64)
    return 8 * _log_int(rng, 1, 96) if kind < 0.8 else _log_int(rng, 8, 300)


def _fits(case):
    w, most = work(case), work(next(c for c in listed() if c["name"] == "subm_train_wide"))
    n = voxels(case)
    rate = 16 if case.get("dtype") == "f32" else 1           # the matrix units take 32-bit operands at a sixteenth of the rate
    return 100 <= n <= 2_700_000 * (2 if case["op"] == "serialize" else 1) and w["flops"] * rate <= most["flops"] and w["bytes"] <= 3e9


def draw(rng):
    while True:
        op = rng.choices(("subm", "conv", "serialize"), (70, 20, 10))[0]
        case = {"op": op, "res": _log_int(rng, 8, 1024), "thick": rng.random() < 0.5, "batch": rng.choice((1, 1, 1, 2, 3, 4)),
                "shuffle": rng.random() < 0.2}
        if op == "serialize":
            case = dict(SERIALIZE, **case, mode=rng.choice(("z_order", "hilbert")))
        else:
            case.update(ci=_channels(rng), dtype=rng.choices(("f16", "bf16", "f32"), (40, 40, 20))[0], train=rng.random() < 0.6,
                        bias=rng.random() < 0.8, cache=rng.choices(("fresh", "kept"), (65, 35))[0])
            case["co"] = case["ci"] if rng.random() < 0.6 else _channels(rng)
            case["relu"] = rng.random() < 0.4 and not (case["train"] and case["dtype"] == "f32")
            if op == "subm":
                if rng.random() < 0.15:
                    case.update(ci=rng.randint(3, 8), input_grad=False)
                case = dict(SUBM, **case) if "input_grad" in case else dict(SUBM, **case, input_grad=True)
                case["layers"] = rng.choice((1, 1, 2, 3, 4))
                case["dilation"] = 2 if rng.random() < 0.1 else 1
            else:
                k = rng.choice((2, 2, 3))
                case = dict(CONV, **case, kernel=k, padding=k // 2 if k == 3 else 0)
        if _fits(case):
            return case


def voxels(case):
    """Rows of the input, to within a percent or two."""
    res = case["res"]
    return int(case["batch"] * (3.93 * (res - 1.25) ** 2 if case["thick"] else 2.545 * res ** 2))


def _pairs_and_rows(case):
    """(valid (output, kernel position) pairs, output rows), from the densities of the two surfaces."""
    n = voxels(case)
    if case["op"] == "subm":
        per_row = 12.7 if case["thick"] else 10.6
        return int(n * (per_row if case["dilation"] == 1 else 0.6 * per_row)), n
    if case["kernel"] == 2:
        return n, int(n * (0.27 if case["thick"] else 0.31))
    return int(3.37 * n), int(n * (0.42 if case["thick"] else 0.5))


def work(case):
    n = voxels(case)
    if case["op"] == "serialize":
        code = 4 if (case["batch"] - 1).bit_length() + 3 * (case["res"] - 1).bit_length() <= 32 else 8
        return {"bytes": 2 * n * (16 + code), "flops": 0}
    pairs, rows = _pairs_and_rows(case)
    s = ELEMENT_BYTES[case["dtype"]]
    volume = 27 if case["op"] == "subm" else case["kernel"] ** 3
    bytes_, flops = 0, 0
    # the neighbor cache: coordinates in; map, codes, order and (training) pair lists out; a kept one is read
    if case["cache"] == "fresh":
        bytes_ += 16 * n + (4 * volume + 12) * rows
        if case["op"] == "conv":
            bytes_ += 16 * rows + (4 * volume * n if case["train"] else 0)
        if case["train"]:
            bytes_ += 8 * pairs
    else:
        bytes_ += 4 * volume * rows
    for layer in range(case.get("layers", 1)):
        ci, co = case["ci"] if layer == 0 else case["co"], case["co"]
        rows_in = n if layer == 0 else rows
        weight, x, y = s * volume * ci * co, s * rows_in * ci, s * rows * co
        bytes_ += weight + x + y                               # forward
        flops += 2 * pairs * ci * co
        if case["train"]:
            if layer > 0 or case["input_grad"]:
                bytes_ += weight + x + y
                flops += 2 * pairs * ci * co
            bytes_ += weight + x + y                           # weight gradient
            flops += 2 * pairs * ci * co
    return {"bytes": int(bytes_), "flops": int(flops)}


def tolerance(case):
    if case["op"] == "serialize":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    # one rounding to 16 bits per layer and pass; with a ReLU, an output whose sum is nearly zero may change sides
    rel = 2e-3 if case["dtype"] == "f16" else 1e-2
    return {"rel": 2 * rel if case["relu"] and case["train"] else rel}


def _surface(case, gen):
    """int32 [N, 4] rows (b, x, y, z) of the active voxels, in scan order unless the case shuffles them.  The centre lies off
    the grid's own, and every sample's surface is turned and mirrored by the seed: other coordinates, as many of them."""
    res, dev = case["res"], gen.device
    outer = res / 2 if case["thick"] else 0.45 * res + 0.5
    inner = res / 2 - 1.25 if case["thick"] else 0.45 * res - 0.5
    lo2, hi2 = math.ceil(256 * inner * inner), math.floor(256 * outer * outer)     # in sixteenths of a voxel: whole numbers
    axis = 16 * torch.arange(res, device=dev, dtype=torch.int32)
    sq = [(axis - (8 * res - 8 + off)) ** 2 for off in (1, 2, 3)]
    rows = []
    for b in range(case["batch"]):
        turn = torch.randperm(3, generator=gen, device=dev).tolist()
        flip = torch.randint(0, 2, (3,), generator=gen, device=dev).tolist()
        if case["op"] == "conv":
            flip = (0, 0, 0)                    # a strided grid is not its own mirror image: the number of outputs would change
        sx, sy, sz = [sq[t].flip(0) if f else sq[t] for t, f in zip(turn, flip)]
        step = max(1, min(res, (1 << 27) // (res * res)))
        for x0 in range(0, res, step):
            d2 = sx[x0:x0 + step, None, None] + (sy[None, :, None] + sz[None, None, :])
            at = ((d2 >= lo2) & (d2 <= hi2)).nonzero()
            at[:, 0] += x0
            rows.append(torch.cat([at.new_full((at.shape[0], 1), b), at], dim=1).to(torch.int32))
    coords = torch.cat(rows)
    if case["shuffle"]:
        coords = coords[torch.randperm(coords.shape[0], generator=gen, device=dev)]
    return coords.contiguous()


def _convolve(state, feats, weight, bias, cache):
    """One layer through its public operator: (output, cache)."""
    case = state["case"]
    if case["op"] == "subm":
        op = spconv.sparse_submanifold_conv3d_relu if case["relu"] else spconv.sparse_submanifold_conv3d
        return op(feats, state["coords"], state["shape"], weight, bias, cache, (case["dilation"],) * 3)
    op = spconv.sparse_conv3d_relu if case["relu"] else spconv.sparse_conv3d
    out, _, cache = op(feats, state["coords"], state["shape"], weight, bias, cache, state["out_coords"], (case["stride"],) * 3,
                       (case["padding"],) * 3)
    return out, cache


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    coords = _surface(case, gen)
    n, res = coords.shape[0], case["res"]
    state = {"case": case, "coords": coords, "shape": torch.Size([case["batch"], case.get("ci", 1), res, res, res])}
    if case["op"] == "serialize":
        return state
    dt = DTYPES[case["dtype"]]

    def normal(*size, scale=1.0):
        return (torch.randn(*size, generator=gen, device=dev) * scale).to(dt)

    k = 3 if case["op"] == "subm" else case["kernel"]
    state["feats"] = normal(n, case["ci"]).requires_grad_(case["train"] and case["input_grad"])
    state["layers"] = []
    for layer in range(case.get("layers", 1)):
        ci, co = case["ci"] if layer == 0 else case["co"], case["co"]
        weight = normal(co, k, k, k, ci, scale=1 / math.sqrt(k ** 3 * ci)).requires_grad_(case["train"])
        bias = normal(co).requires_grad_(case["train"]) if case["bias"] else None
        state["layers"].append((weight, bias))
    state["cache"], state["out_coords"] = None, None
    rows = n
    if case["op"] == "conv":
        fn = spconv.SparseConv3dFunction
        out_coords = fn._get_output_coords(coords, state["shape"], (k,) * 3, (case["stride"],) * 3, (case["padding"],) * 3, (1, 1, 1))
        rows = out_coords.shape[0]
        if case["cache"] == "kept":
            state["out_coords"] = out_coords
    if case["cache"] == "kept":
        with torch.set_grad_enabled(case["train"]):
            _, state["cache"] = _convolve(state, state["feats"], *state["layers"][0], None)
    if case["train"]:
        state["upstream"] = normal(rows, case["co"])
        state["leaves"] = [t for t in [state["feats"]] + [p for layer in state["layers"] for p in layer] if t is not None and t.requires_grad]
    return state


def run(state):
    case = state["case"]
    if case["op"] == "serialize":
        codes = encode_seq(state["coords"], state["shape"], case["mode"])
        return codes, decode_seq(codes, state["shape"], case["mode"])
    with torch.set_grad_enabled(case["train"]):
        h, cache = state["feats"], state["cache"]
        for weight, bias in state["layers"]:
            h, cache = _convolve(state, h, weight, bias, cache)
    if not case["train"]:
        return h
    return [h, *torch.autograd.grad(h, state["leaves"], state["upstream"])]
