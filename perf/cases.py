"""Performance cases of viola_amd: what a training or serving program has the framework do, over the sizes it meets.

Six kinds of work, each through the package's public classes:

  linear   nn.Linear, inference or forward + backward, under the four scaling recipes
  mlp      nn.MLP (gated), inference or forward + backward
  experts  nn.GroupedExperts-style variable-group linear (mixture of experts), one call for all groups
  bound    one whole training step of a Linear under bind_optimizer: forward, backward, FP8Muon, FP8 write-back
  muon     FP8Muon.step on the matrices and vectors of a stack of transformer blocks
  wire     FP8Communication.roundtrip on gradient buckets

`listed()` names the cases, `draw(rng)` gives another one of the same ranges, `prepare(case, seed)` makes what a program
holds before the call, `run(state)` is one pass, `work(case)` the bytes and operations it cannot do without and
`tolerance(case)` how far two correct implementations may be apart.
"""

import math

import torch

import viola_amd
from viola_amd import nn, optim
from viola_amd.distributed import FP8Communication

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


# ---------------------------------------------------------------------------------------------------------- the cases
def _linear(tokens, n_in, n_out, scaling, train, *, weights="fp8", mode="memory", backward="e4m3", dtype="bf16"):
    return dict(kind="linear", tokens=tokens, n_in=n_in, n_out=n_out, scaling=scaling, train=train, weights=weights, mode=mode,
                backward=backward, dtype=dtype)


def _mlp(tokens, n_in, hidden, scaling, train, *, activation="silu", backward="e4m3", dtype="bf16"):
    return dict(kind="mlp", tokens=tokens, n_in=n_in, hidden=hidden, scaling=scaling, train=train, activation=activation,
                backward=backward, dtype=dtype)


def _experts(groups, tokens, n_in, n_out, train, *, backward="e4m3", dtype="bf16"):
    return dict(kind="experts", groups=groups, tokens=tokens, n_in=n_in, n_out=n_out, train=train, backward=backward, dtype=dtype)


def _bound(tokens, n_in, n_out, scaling, *, method="standard"):
    return dict(kind="bound", tokens=tokens, n_in=n_in, n_out=n_out, scaling=scaling, method=method)


def _muon(blocks, width, method, *, grads="fp32", rounding="nearest"):
    return dict(kind="muon", blocks=blocks, width=width, method=method, grads=grads, rounding=rounding)


def _wire(buckets, elements, *, fmt="e4m3", tile=256):
    return dict(kind="wire", buckets=buckets, elements=elements, format=fmt, tile=tile)


def listed():
    cases = {
        # a handful of sequences decoding one token each: the smallest call, all latency and launches
        "linear_decode": _linear(8, 1024, 4096, "grouped", False),
        # a long prompt through a projection of a 4096-wide model, weights frozen, the module's default recipe
        "linear_prefill": _linear(4096, 4096, 4096, "current", False),
        # fine-tuning with a tiny batch on a small layer: forward + backward where each launch is a few microseconds
        "linear_train_small": _linear(256, 512, 2048, "current", True, backward="e5m2"),
        # the benchmark's layer and batch
        "linear_train": _linear(8192, 1024, 4096, "grouped", True),
        # 50 images of 196 patches and a class token: a row count that is a multiple of nothing, FP16 activations
        "linear_train_ragged": _linear(50 * 197, 768, 3072, "grouped", True, dtype="fp16"),
        # attention output projection of a 4096-wide model over a full batch, block-scaled recipe
        "linear_train_wide": _linear(16384, 4096, 4096, "mxfp8", True),
        # the feed-forward of a diffusion-transformer block (width 1152), the recipe that hands h over as codes
        "mlp_train_block": _mlp(4096, 1152, 4608, "mxfp8", True, activation="gelu"),
        # the benchmark's MLP: the largest call
        "mlp_train_large": _mlp(16384, 4096, 11008, "grouped", True),
        # the benchmark's mixture-of-experts layer
        "experts_train": _experts(16, 32768, 4096, 1024, True),
        # a layer trained under a master weight, the whole step of a small model
        "bound_step": _bound(1024, 1024, 1024, "grouped"),
        # the optimizer step of the benchmark's parameter set (28 blocks of width 1152)
        "muon_blocks": _muon(28, 1152, "standard"),
        # one 25 MB gradient bucket encoded for the wire and decoded
        "wire_bucket": _wire(1, 6553600),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _spread(rng, low, high):
    """An integer from low to high, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _tokens(rng, low, high):
    """Row counts: half of them whole multiples of 64 (fixed batches), half of them anything (packed or cut sequences)."""
    n = _spread(rng, low, high)
    return max(64, n // 64 * 64) if n >= 64 and rng.random() < .5 else n


def _features(rng, low, high):
    """Layer widths: mostly multiples of 128, some of 32 or 8, a few (class counts, vocabularies) of nothing."""
    unit = rng.choices((128, 32, 8, 1), (60, 20, 12, 8))[0]
    return max(unit, _spread(rng, low, high) // unit * unit)


def draw(rng):
    kind = rng.choices(("linear", "mlp", "experts", "bound", "muon", "wire"), (40, 18, 12, 8, 12, 10))[0]
    backward, dtype = rng.choice(("e4m3", "e5m2")), rng.choices(("bf16", "fp16"), (75, 25))[0]
    scaling = rng.choices(("grouped", "current", "delayed", "mxfp8"), (35, 25, 10, 30))[0]
    while True:
        if kind == "linear":
            train = rng.random() < .65
            case = _linear(_tokens(rng, 32 if train else 1, 16384), _features(rng, 256, 8192), _features(rng, 256, 8192), scaling, train,
                           weights=rng.choices(("fp8", "bf16"), (80, 20))[0], mode=rng.choices(("memory", "fast"), (70, 30))[0],
                           backward=backward, dtype=dtype)
            if work(case)["flops"] <= 8e11:
                return case
        elif kind == "mlp":
            train = rng.random() < .65
            case = _mlp(_tokens(rng, 32 if train else 1, 16384), _features(rng, 256, 4096), _features(rng, 512, 11008), scaling, train,
                        activation=rng.choices(("silu", "gelu", "relu"), (60, 30, 10))[0], backward=backward, dtype=dtype)
            if work(case)["flops"] <= 8e11:
                return case
        elif kind == "experts":
            case = _experts(_spread(rng, 2, 64), _tokens(rng, 128, 32768), _features(rng, 256, 4096), _features(rng, 256, 4096),
                            rng.random() < .7, backward=backward, dtype=dtype)
            if work(case)["flops"] <= 8e11:
                return case
        elif kind == "bound":
            case = _bound(_tokens(rng, 64, 8192), _features(rng, 256, 2048), _features(rng, 256, 4096), scaling,
                          method=rng.choice(("standard", "gram")))
            if work(case)["flops"] <= 8e11:
                return case
        elif kind == "muon":
            case = _muon(_spread(rng, 1, 28), max(64, _spread(rng, 192, 1280) // 32 * 32), rng.choice(("standard", "gram")),
                         grads=rng.choice(("fp32", "bf16")), rounding=rng.choices(("nearest", "stochastic"), (75, 25))[0])
            if work(case)["flops"] <= 1.2e13:
                return case
        else:
            case = _wire(_spread(rng, 1, 8), _spread(rng, 1 << 14, 1 << 25), fmt=backward, tile=rng.choices((256, 128, 512), (70, 15, 15))[0])
            if case["buckets"] * case["elements"] <= 1 << 27:
                return case


# ------------------------------------------------------------------------------------------------ inputs and modules
def _normal(shape, scale, dtype, generator):
    return (torch.randn(shape, device="cuda", generator=generator) * scale).to(dtype)


def _generator(seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    return generator


def _layer_state(case, seed, module, n_out):
    """A module with the activations and, for training, the output gradient of one batch."""
    generator = _generator(seed)
    dtype = _DTYPES[case.get("dtype", "bf16")]
    x = _normal((case["tokens"], case["n_in"]), 1.0, dtype, generator)
    state = dict(kind=case["kind"], train=case.get("train", True), module=module, x=x)
    if state["train"]:
        x.requires_grad_()
        state["dy"] = _normal((case["tokens"], n_out), 1e-2, dtype, generator)
    return state


def _group_sizes(case, seed):
    """Rows per expert as a router deals them: uneven, and now and then an expert that gets nothing."""
    generator = torch.Generator().manual_seed(seed)
    share = torch.rand(case["groups"], generator=generator) + .2
    rows = torch.multinomial(share, case["tokens"], replacement=True, generator=generator)
    return torch.bincount(rows, minlength=case["groups"]).tolist()


def _muon_shapes(case):
    d = case["width"]
    return [(3 * d, d), (d, d), (4 * d, d), (d, 4 * d), (3 * d,), (d,), (4 * d,), (d,), (d,), (d,)] * case["blocks"]


def _muon_state(case, seed):
    """Parameters, gradients and optimizer state in flat buffers (as a bucketed data-parallel program keeps them), in the
    middle of a run: the momentum and the second moments are not zero."""
    generator = _generator(seed)
    shapes = _muon_shapes(case)
    tile = 256
    sizes = [-(-math.prod(shape) // tile) * tile for shape in shapes]          # every tensor starts on a tile
    begins = [sum(sizes[:i]) for i in range(len(sizes))]
    total = sum(sizes)
    values = _normal(total, .02, torch.float32, generator)
    gradients = _normal(total, 1e-3, _DTYPES[case["grads"]], generator)
    momentum = _normal(total, 112.0, torch.float32, generator).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    scales = torch.full((total // tile,), 3e-6, device="cuda")
    first, second = _normal(total, 1e-4, torch.float32, generator), torch.full((total,), 1e-7, device="cuda")
    viola_amd.set_gradient_dtype(case["grads"])
    parameters, entries = [], {}
    for index, (shape, size, begin) in enumerate(zip(shapes, sizes, begins)):
        count = math.prod(shape)
        parameter = torch.nn.Parameter(values[begin:begin + count].view(shape))
        parameter.grad_dtype = _DTYPES[case["grads"]]
        parameter.grad = gradients[begin:begin + count].view(shape)
        parameters.append(parameter)
        if len(shape) == 2:
            entries[index] = {"step": 10, "momentum_q": momentum[begin:begin + size],
                              "momentum_scale": scales[begin // tile:(begin + size) // tile]}
        else:
            entries[index] = {"step": 10, "exp_avg": first[begin:begin + count], "exp_avg_sq": second[begin:begin + count]}
    optimizer = optim.FP8Muon(parameters, lr=1e-3, weight_decay=.01, ns_method=case["method"], rounding=case["rounding"], rounding_seed=42)
    optimizer.load_state_dict({"state": entries, "param_groups": optimizer.state_dict()["param_groups"]})
    return dict(kind="muon", optimizer=optimizer, outputs=dict(parameters=values, momentum=momentum, scales=scales, first=first, second=second))


def prepare(case, seed):
    torch.manual_seed(seed)                                                    # the modules' own initialisation
    kind = case["kind"]
    if kind == "muon":
        return _muon_state(case, seed)
    if kind == "wire":
        generator = _generator(seed)
        codec = FP8Communication(case["elements"], device="cuda", fp8_format=case["format"], tile_size=case["tile"])
        # gradients: normal inside a tensor, their size different from one part of the bucket to the next
        buckets = [_normal(case["elements"], 10.0 ** -(2 + i % 3), torch.float32, generator) for i in range(case["buckets"])]
        return dict(kind="wire", codec=codec, buckets=buckets)
    viola_amd.set_gradient_dtype("bf16")
    viola_amd.set_master_weight_dtype("fp32")
    dtype = _DTYPES[case.get("dtype", "bf16")]
    if kind == "linear":
        module = nn.Linear(case["n_in"], case["n_out"], device="cuda", dtype=dtype, scaling=case["scaling"], mode=case["mode"],
                           weight_dtype=case["weights"], forward_dtype="e4m3", backward_dtype=case["backward"])
        return _layer_state(case, seed, module, case["n_out"])
    if kind == "mlp":
        module = nn.MLP(case["n_in"], case["hidden"], activation=case["activation"], device="cuda", dtype=dtype,
                        scaling=case["scaling"], forward_dtype="e4m3", backward_dtype=case["backward"])
        return _layer_state(case, seed, module, case["n_in"])
    if kind == "experts":
        module = nn.GroupedExperts(case["groups"], case["n_in"], case["n_out"], backward_dtype=case["backward"], device="cuda")
        return dict(_layer_state(case, seed, module, case["n_out"]), counts=_group_sizes(case, seed))
    assert kind == "bound", kind
    module = nn.Linear(case["n_in"], case["n_out"], device="cuda", dtype=torch.bfloat16, scaling=case["scaling"], backward_dtype="e4m3")
    optimizer = optim.bind_optimizer(module, optim.FP8Muon(module.parameters(), lr=1e-3, weight_decay=.01, ns_method=case["method"]))
    masters = [p for group in optimizer.param_groups for p in group["params"]]
    return dict(_layer_state(case, seed, module, case["n_out"]), optimizer=optimizer, masters=masters)


# ------------------------------------------------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "muon":
        state["optimizer"].step()
        return state["outputs"]
    if kind == "wire":
        return [state["codec"].roundtrip(bucket) for bucket in state["buckets"]]
    module, x = state["module"], state["x"]
    extra = (state["counts"],) if kind == "experts" else ()
    if not state["train"]:
        with torch.no_grad():
            return module(x, *extra)
    x.grad = None
    if kind == "bound":
        optimizer = state["optimizer"]
        optimizer.zero_grad()
        y = module(x)
        y.backward(state["dy"])
        optimizer.step()
        return dict(y=y.detach(), dx=x.grad, weight=module.weight.detach(), weight_scale=module.weight_scale, bias=module.bias.detach(),
                    masters=[m.detach() for m in state["masters"]],
                    momentum=[optimizer.state[m]["momentum_q"] for m in state["masters"] if m.dim() == 2])
    parameters = dict(module.named_parameters())
    for parameter in parameters.values():
        parameter.grad = None
    y = module(x, *extra)
    y.backward(state["dy"])
    return dict(y=y.detach(), dx=x.grad, gradients={name: parameter.grad for name, parameter in parameters.items()})


# ---------------------------------------------------------------------------------------------- what a pass has to do
def _gemm_work(tokens, n_in, n_out, train, value, weight):
    """One linear layer: x, W (and dy) in, y (and dx, dW in bf16) out; one product forward, two backward."""
    flops = 2 * tokens * n_in * n_out
    bytes_ = value * tokens * (n_in + n_out) + weight * n_in * n_out
    if train:
        bytes_ += value * tokens * (n_in + n_out) + 2 * n_in * n_out
    return dict(bytes=bytes_, flops=3 * flops if train else flops)


def _orthogonal_flops(rows, cols, method, steps=5):
    """Products of one Newton-Schulz chain, a symmetric product at half its size."""
    m, n = min(rows, cols), max(rows, cols)
    if method == "standard" or m == n:
        return steps * (m * m * n + m ** 3 + 2 * m * m * n)
    return 2 * m * m * n + 2 * 2 * m * m * n + 26 * m ** 3


def work(case):
    kind = case["kind"]
    value = _BYTES[case.get("dtype", "bf16")]
    if kind == "linear":
        return _gemm_work(case["tokens"], case["n_in"], case["n_out"], case["train"], value, 1 if case["weights"] == "fp8" else 2)
    if kind == "mlp":
        # x and y (dx and dy), the three weight matrices; the hidden activation itself need not leave the chip
        t, d, h = case["tokens"], case["n_in"], case["hidden"]
        flops, weights = 2 * t * d * 3 * h, 3 * d * h
        if not case["train"]:
            return dict(bytes=2 * value * t * d + weights, flops=flops)
        return dict(bytes=4 * value * t * d + weights + 2 * weights, flops=3 * flops)
    if kind == "experts":
        t, k, n, g = case["tokens"], case["n_in"], case["n_out"], case["groups"]
        flops, weights = 2 * t * k * n, g * k * n
        bytes_ = value * t * (k + n) + weights
        return dict(bytes=2 * value * t * (k + n) + 3 * weights, flops=3 * flops) if case["train"] else dict(bytes=bytes_, flops=flops)
    if kind == "bound":
        layer = _gemm_work(case["tokens"], case["n_in"], case["n_out"], True, 2, 1)
        size = case["n_in"] * case["n_out"]
        # master read and written, momentum codes read and written, new FP8 weight written
        return dict(bytes=layer["bytes"] + (8 + 2 + 1) * size,
                    flops=layer["flops"] + _orthogonal_flops(case["n_out"], case["n_in"], case["method"]))
    if kind == "muon":
        bytes_ = flops = 0
        for shape in _muon_shapes(case):
            size = math.prod(shape)
            gradient = _BYTES[case["grads"]] * size
            if len(shape) == 2:
                bytes_ += gradient + (8 + 2) * size
                flops += _orthogonal_flops(*shape, case["method"])
            else:
                bytes_ += gradient + 24 * size
        return dict(bytes=bytes_, flops=flops)
    # value in, packet out, packet in, value out
    return dict(bytes=case["buckets"] * case["elements"] * 2 * (4 + 1 + 4 / case["tile"]), flops=0)


def tolerance(case):
    """16-bit results of FP32 sums in another order: half an ulp either way (bf16 about 2e-3 in the 2-norm). An MLP's
    backward pass sees three such roundings on the way. An optimizer step changes a weight by about a hundredth, computed
    through fifteen or more bf16 products; its FP8 state is the same to the bit. The wire codec is exact."""
    kind = case["kind"]
    if kind == "wire":
        return "exact"
    if kind == "muon":
        return {"rel": 3e-4}
    if kind == "mlp":
        return {"rel": 1e-2}
    return {"rel": 5e-3}
