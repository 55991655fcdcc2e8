"""What this package is used for, as cases that can be timed: SS2D's core, its three operators, whole blocks and models,
forward and backward, over the map sizes, batches, state counts and data types they meet.

A case is a plain dict; ``prepare`` makes what a program holds before the call (seeded inputs on the GPU, the module with
its weights), ``run`` is one pass through the public entry points, ``work`` what that pass cannot do without, ``tolerance``
how far another correct implementation at the same precision may be off.
"""
import math

import torch

from vmamba_amd.csm import cross_merge_fn, cross_scan_fn
from vmamba_amd.csms6s import selective_scan_fn
from vmamba_amd.ss2d import SS2D
from vmamba_amd.vssm import VSSBlock, vmamba_tiny_s1l8

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# VMamba-T's four stages: channels and map side of a 224 x 224 image
_STAGES = ((96, 56), (192, 28), (384, 14), (768, 7))
_TINY_DEPTHS = (2, 2, 8, 2)

# the largest listed case of each kind, in elements of the map (B * D * H * W) or pixels of the image batch
_CORE_MAX = 128 * 96 * 56 * 56
_OPS_MAX = 128 * 96 * 56 * 56
_TRAIN_OPS_MAX = 64 * 96 * 56 * 56
_TRAIN_OPS_N16_MAX = 16 * 192 * 28 * 28
_TRAIN_BLOCK_MAX = 64 * 384 * 14 * 14
_MODEL_MAX = 128 * 224 * 224


def _core(name, dtype, batch, dim, height, width, d_state=1):
    return dict(name=name, kind="core", dtype=dtype, batch=batch, dim=dim, height=height, width=width, d_state=d_state)


def _ops(name, dtype, batch, dim, height, width, d_state=1, train=False):
    return dict(name=name, kind="ops", dtype=dtype, batch=batch, dim=dim, height=height, width=width, d_state=d_state,
                train=train)


def listed():
    return [
        # SS2D.forward_core: the inference hot path of every block, behind the call the reference's users make.
        # One image at VMamba-T's last stage: an online request, the smallest call there is.
        _core("core_7x7_b1_bf16", "bf16", 1, 768, 7, 7),
        # Stage 2 in single precision, the precision of the reference's own throughput harness, an ordinary batch.
        _core("core_28x28_b32_fp32", "fp32", 32, 192, 28, 28),
        # Stage 1 of VMamba-T at batch 128: the headline shape.
        _core("core_56x56_b128_bf16", "bf16", 128, 96, 56, 56),
        # A map with odd sides, as images that are no multiple of 32 give, in half precision.
        _core("core_57x58_b48_fp16", "fp16", 48, 96, 57, 58),
        # Stage 1 of four 1024 x 1024 images, the dense-prediction size.
        _core("core_256x256_b4_bf16", "bf16", 4, 96, 256, 256),
        # The heavier block with 16 states per channel and twice the channels.
        _core("core_n16_56x56_b64_bf16", "bf16", 64, 192, 56, 56, d_state=16),
        # The three operators behind the reference's own call surfaces, inference, headline shape.
        _ops("ops_56x56_b128_bf16", "bf16", 128, 96, 56, 56),
        # The same operators in training: forward and backward, 16-bit activations, one state and sixteen.
        _ops("train_ops_56x56_b64_bf16", "bf16", 64, 96, 56, 56, train=True),
        _ops("train_ops_n16_28x28_b16_bf16", "bf16", 16, 192, 28, 28, d_state=16, train=True),
        # A whole block in training, single precision: stage 3, which has most of the blocks.
        dict(name="train_block_14x14_b64_fp32", kind="train_block", dtype="fp32", batch=64, dim=384, height=14, width=14),
        # The whole VMamba-T backbone at inference: one image (latency), and the benchmark's batch (throughput).
        dict(name="model_224_b1_bf16", kind="model", dtype="bf16", batch=1, side=224),
        dict(name="model_224_b128_bf16", kind="model", dtype="bf16", batch=128, side=224),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _map(rng, most, side_lo, side_hi, dim_hi=768, batch_hi=128):
    """dim, height, width, batch with dim * height * width * batch <= most: sides over the logarithm of their range, near
    squares and oblong ones, even and odd; channels a multiple of 16; the batch fills a random share of what is left."""
    while True:
        height = _log_int(rng, side_lo, side_hi)
        width = height if rng.random() < 0.5 else min(side_hi, max(side_lo, int(height * rng.uniform(0.6, 1.6))))
        dim = 16 * _log_int(rng, 3, dim_hi // 16)
        room = min(batch_hi, most // (dim * height * width))
        if room >= 1:
            return dim, height, width, _log_int(rng, 1, room)


def draw(rng):
    kind = rng.choice(["core"] * 6 + ["ops"] + ["train_ops"] * 2 + ["train_block"] + ["model"] * 2)
    if kind == "core":
        d_state = 16 if rng.random() < 1 / 6 else 1
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        most = _CORE_MAX // (2 if dtype == "fp32" else 1)
        dim, height, width, batch = _map(rng, most, 7, 256 if d_state == 1 else 64)
        case = _core("", dtype, batch, dim, height, width, d_state)
    elif kind == "ops":
        dtype = rng.choice(["bf16", "fp16", "fp32"])
        dim, height, width, batch = _map(rng, _OPS_MAX // (2 if dtype == "fp32" else 1), 7, 128)
        case = _ops("", dtype, batch, dim, height, width)
    elif kind == "train_ops":
        d_state = rng.choice([1, 16])
        dtype = rng.choice(["bf16", "fp16", "fp32"])
        most = (_TRAIN_OPS_MAX if d_state == 1 else _TRAIN_OPS_N16_MAX) // (2 if dtype == "fp32" else 1)
        dim, height, width, batch = _map(rng, most, 7, 64)
        case = _ops("", dtype, batch, dim, height, width, d_state, train=True)
    elif kind == "train_block":
        dim, height, width, batch = _map(rng, _TRAIN_BLOCK_MAX, 7, 56)
        case = dict(kind="train_block", dtype="fp32", batch=batch, dim=dim, height=height, width=width)
    else:
        side = 32 * rng.randint(4, 13)
        case = dict(kind="model", dtype=rng.choice(["bf16", "fp16"]),
                    batch=_log_int(rng, 1, min(128, _MODEL_MAX // (side * side))), side=side)
    case.pop("name", None)                        # drawn cases carry none
    return case


def _generator(seed):
    torch.manual_seed(seed)                       # the modules' own initialisers draw from the global generators
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def prepare(case, seed):
    g = _generator(seed)
    dtype = _DTYPES[case["dtype"]]
    kind, batch = case["kind"], case["batch"]
    if kind == "core":
        with torch.device("cuda"):
            op = SS2D(d_model=case["dim"], d_state=case["d_state"], dt_rank=_dt_rank(case), channel_first=False)
        op = op.to(dtype).eval()
        # forward_core's input comes from the depthwise convolution's SiLU
        x = torch.nn.functional.silu(_normal(g, batch, case["dim"], case["height"], case["width"])).to(dtype)
        return dict(kind=kind, op=op, x=x)
    if kind == "ops":
        D, H, W, N = case["dim"], case["height"], case["width"], case["d_state"]
        L, K = H * W, 4
        dt = torch.exp(torch.rand(K * D, generator=g, device="cuda") * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
        args = dict(
            x=_normal(g, batch, D, H, W, dtype=dtype),
            delta=_normal(g, batch, K * D, L, dtype=dtype),
            A=-torch.arange(1, N + 1, device="cuda", dtype=torch.float32).repeat(K * D, 1),
            B=_normal(g, batch, K, N, L, dtype=dtype),
            C=_normal(g, batch, K, N, L, dtype=dtype),
            D=torch.ones(K * D, device="cuda"),
            bias=dt + torch.log(-torch.expm1(-dt)))               # softplus of it is dt
        if case["train"]:
            for t in args.values():
                t.requires_grad_(True)
            args["grad"] = _normal(g, batch, D, L)
        return dict(kind=kind, train=case["train"], dims=(batch, K, D, H, W), **args)
    with torch.device("cuda"):
        if kind == "train_block":
            model = VSSBlock(case["dim"], channel_first=False)
        else:
            model = vmamba_tiny_s1l8(channel_first=False)
    model = model.to(dtype)
    if kind == "train_block":
        x = _normal(g, batch, case["height"], case["width"], case["dim"], dtype=dtype).requires_grad_(True)
        return dict(kind=kind, model=model.train(), x=x, grad=_normal(g, *x.shape, dtype=dtype))
    return dict(kind=kind, model=model.eval(), x=_normal(g, batch, 3, case["side"], case["side"], dtype=dtype))


def _three_operators(s):
    batch, K, D, H, W = s["dims"]
    xs = cross_scan_fn(s["x"])
    ys = selective_scan_fn(xs.view(batch, K * D, H * W), s["delta"], s["A"], s["B"], s["C"], s["D"], s["bias"], True, True)
    return cross_merge_fn(ys.view(batch, K, D, H, W))


def run(state):
    kind = state["kind"]
    if kind == "core":
        with torch.no_grad():
            return state["op"].forward_core(state["x"])
    if kind == "model":
        with torch.no_grad():
            return state["model"](state["x"])
    if kind == "ops":
        if not state["train"]:
            with torch.no_grad():
                return _three_operators(state)
        y = _three_operators(state)
        wanted = [state[k] for k in ("x", "delta", "A", "B", "C", "D", "bias")]
    else:
        y = state["model"](state["x"])
        wanted = [state["x"]] + list(state["model"].parameters())
    return [y.detach()] + list(torch.autograd.grad(y, wanted, state["grad"]))


def _dt_rank(case):
    # the heavier 16-state block widens d_model = dim / 2 by two: its step rank is that of d_model
    return math.ceil(case["dim"] / (32 if case["d_state"] > 1 else 16))


def _core_work(batch, dim, L, d_state, rank, size):
    """forward_core: the map in, the normalised map out, the weights; x_proj and dt_proj as products, the recurrence (a
    product and two multiply-adds with the output's, per position, direction and state), merge and norm."""
    C = rank + 2 * d_state
    E = batch * dim * L
    weights = 4 * dim * (C + rank + d_state + 2) * size + 2 * dim * size
    flops = 2 * 4 * E * (C + rank) + 4 * E * (6 * d_state + 6) + 12 * E
    return 2 * E * size + weights, flops


def _block_work(batch, dim, L, size):
    """Inference of one block: its input and output once, its weights once."""
    E = batch * dim * L
    _, core = _core_work(batch, dim, L, 1, math.ceil(dim / 16), size)
    return 2 * E * size + 10 * dim * dim * size, 2 * E * dim * 10 + 18 * E + core


def work(case):
    size = _DTYPES[case["dtype"]].itemsize
    batch = case["batch"]
    if case["kind"] == "model":
        cells = (case["side"] // 32) ** 2
        flops, weights = 0, 0
        for i, ((dim, _), depth) in enumerate(zip(_STAGES, _TINY_DEPTHS)):
            L = cells * 4 ** (3 - i)
            byte, flop = _block_work(batch, dim, L, size)
            flops += depth * flop
            weights += depth * (byte - 2 * batch * dim * L * size)
            if i:                                 # 3 x 3 convolution, stride 2
                flops += 2 * batch * L * dim * (dim // 2) * 9
                weights += dim * (dim // 2) * 9 * size
        flops += 2 * batch * cells * 1024 // 4 * 48 * 27 + 2 * batch * cells * 64 * 96 * 48 * 9 + 2 * batch * 768 * 1000
        weights += (48 * 27 + 96 * 48 * 9 + 768 * 1000) * size
        return {"bytes": batch * (3 * case["side"] ** 2 + 1000) * size + weights, "flops": flops}
    dim, L = case["dim"], case["height"] * case["width"]
    E = batch * dim * L
    if case["kind"] == "core":
        byte, flop = _core_work(batch, dim, L, case["d_state"], _dt_rank(case), size)
        return {"bytes": byte, "flops": flop}
    if case["kind"] == "train_block":
        _, flop = _block_work(batch, dim, L, size)
        return {"bytes": 5 * E * size + 20 * dim * dim * size, "flops": 3 * flop}      # x, y, dy, dx and one saved map
    N = case["d_state"]
    scan = 4 * E * (6 * N + 6)
    bc = 2 * batch * 4 * N * L
    # each of the three calls reads its tensors once and writes its result once (the scan's and the merge's are fp32)
    byte = 5 * E * size + (4 * E * (2 * size + 4) + bc * size) + 5 * E * 4
    if case["train"]:
        # the merge's adjoint, the scan's (u, delta, B, C and the fp32 gradient in; theirs out), the CrossScan's
        byte += 5 * E * 4 + (4 * E * (4 * size + 4) + 2 * bc * size) + 5 * E * size
    return {"bytes": byte, "flops": scan * (4 if case["train"] else 1)}


# About four times what the paths differ from the same computation in 64 bits (relative, and the largest difference over
# the root mean square); the 16-bit figures are the rounding of the results themselves, a model's that of its activations.
_TOLERANCES = {
    ("core", "bf16"): (6.5e-3, 1.6e-2), ("core", "fp16"): (8e-4, 2e-3), ("core", "fp32"): (1e-6, 1e-5),
    ("ops", "bf16"): (1e-6, 1e-5), ("ops", "fp16"): (1e-6, 1e-5), ("ops", "fp32"): (1e-6, 1e-5),      # fp32 results
    ("train_ops", "bf16"): (1e-2, 4e-2), ("train_ops", "fp16"): (1.2e-3, 5e-3), ("train_ops", "fp32"): (4e-6, 4e-5),
    ("train_block", "fp32"): (1e-5, 1e-4),
    ("model", "bf16"): (2e-2, 7e-2), ("model", "fp16"): (2.5e-3, 1e-2),
}


def tolerance(case):
    kind = "train_ops" if case.get("train") else case["kind"]
    rel, most = _TOLERANCES[kind, case["dtype"]]
    return {"rel": rel, "max": most}
