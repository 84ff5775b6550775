"""The calls whose time on the GPU is tracked, through the package's public entry points.

A case is one of three calls of a program that uses the package:

* ``layer``: ``HFFNRuntime.forward`` (or ``PreparedRuntime.forward``) of one layer on N tokens, inference;
* ``step``: one decode step's feed-forward calls of a whole model, one per layer, each output copied to where the model
  keeps it (``PreparedRuntime``);
* ``train``: ``HFFNTrainRuntime.step`` of one layer (forward with z, backward, AdamW).

Layers have the widths, densities, value types and supports that the package's workloads, tests and benchmarks use:
every neuron the same number of slots (``even``), a number of slots drawn from 0 to twice the mean with empty rows among
them (``ragged``), or clipped-normal numbers with indices biased towards a few inputs (``zipf``). Everything is drawn
on the GPU from the seed.
"""
from __future__ import annotations

import math

import torch

from hffn_amd.prepared_runtime import PreparedRuntime
from hffn_amd.runtime import HFFNLayer, HFFNRuntime
from hffn_amd.train_runtime import HFFNTrainRuntime

HYPER = dict(lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=1e-2)
WEIGHT_STD, BIAS_STD, GRAD_STD = 0.02, 0.01, 0.1
MOST_SLOT_TOKENS = 1.3e10  # a drawn call multiplies at most this many slots by tokens (a fifth of it when training)

# (d_model, d_ff): the widths of the test layers and of the 70M, 160M, 410M, 1.4B and 2.8B shapes; then widths that are
# no multiples of 256, as an odd-sized model has them.
WIDTHS = ((256, 1024), (512, 2048), (768, 3072), (1024, 4096), (2048, 8192), (2560, 10240), (400, 1608), (1104, 4424))
TRAIN_WIDTHS = WIDTHS[:4]


def _case(name, kind, widths, density, tokens, support="even", values="float32", prepared=False, layers=1):
    case = {"kind": kind, "d_model": widths[0], "d_ff": widths[1], "density": density, "tokens": tokens,
            "support": support, "values": values, "prepared": prepared, "layers": layers}
    return {"name": name, **case} if name else case


def listed():
    return [
        # Greedy decoding of one sequence, the lowest latency a serving program asks for.
        _case("decode_410m_d50_n1", "layer", WIDTHS[3], 0.5, 1, prepared=True),
        # Decoding a batch of 16 sequences on a sparse bfloat16 layer.
        _case("decode_1p4b_d20_bf16_n16", "layer", WIDTHS[4], 0.2, 16, values="bf16"),
        # All 24 feed-forward calls of one decode step of eight sequences.
        _case("decode_step_410m_d50_n8", "step", WIDTHS[3], 0.5, 8, prepared=True, layers=24),
        # A ragged batch (continuous batching, a short prompt) on the irregular test layer, empty rows included.
        _case("batch_512_d10_ragged_n37", "layer", WIDTHS[1], 0.1, 37, support="ragged"),
        # One 128-token prompt on the smallest model of the request benchmark.
        _case("prompt_70m_d20_n128", "layer", WIDTHS[1], 0.2, 128),
        # Four 128-token prompts in one call, low density.
        _case("prompt_160m_d10_n512", "layer", WIDTHS[2], 0.1, 512),
        # The headline: a 2048-token prefill of the 410M shape at half density.
        _case("prompt_410m_d50_n2048", "layer", WIDTHS[3], 0.5, 2048),
        # A prefill of an odd length on the sparse bfloat16 layer.
        _case("prompt_1p4b_d20_bf16_n1999", "layer", WIDTHS[4], 0.2, 1999, values="bf16"),
        # The largest: a 4096-token prefill of the 2.8B shape, uneven fan-in.
        _case("prompt_2p8b_d80_zipf_bf16_n4096", "layer", WIDTHS[5], 0.8, 4096, support="zipf", values="bf16"),
        # Training: a small step (few tokens), the training benchmark's largest cell, a large batch of a sparse layer.
        _case("train_512_2048_d20_n8", "train", WIDTHS[1], 0.2, 8),
        _case("train_1024_4096_d50_n512", "train", WIDTHS[3], 0.5, 512),
        _case("train_1024_4096_d10_n2048", "train", WIDTHS[3], 0.1, 2048),
    ]


def draw(rng):
    log = lambda low, high: math.exp(rng.uniform(math.log(low), math.log(high)))  # noqa: E731
    train = rng.random() < 0.25
    d_model, d_ff = rng.choice(TRAIN_WIDTHS if train else WIDTHS)
    support = rng.choice(("even", "even", "ragged", "zipf"))
    density = round(log(0.05, 0.5 if train or support == "ragged" else 0.8), 3)
    most = MOST_SLOT_TOKENS / (5 if train else 1) / (2 * d_model * d_ff * density)
    tokens = max(1, min(round(log(1, 2048 if train else 4096)), int(most)))
    if train:
        return _case("", "train", (d_model, d_ff), density, tokens, support=support)
    values = rng.choice(("float32", "bf16"))
    return _case("", "layer", (d_model, d_ff), density, tokens, support=support, values=values, prepared=rng.random() < 0.4)


# ------------------------------------------------------------------------------------------------------------- inputs

def _normal(generator, shape, std=1.0):
    return torch.randn(shape, generator=generator, device="cuda") * std


def _degrees(generator, case):
    """Slots of every neuron on one side. Uneven ones are one drawn set of numbers in an order of the seed's, so that the
    total, and with it the length of the stores, is the case's."""
    d, h, mean = case["d_model"], case["d_ff"], max(1, round(case["density"] * case["d_model"]))
    if case["support"] == "even":
        return torch.full((h,), mean, device="cuda", dtype=torch.int64)
    fixed = torch.Generator("cuda").manual_seed(h)
    if case["support"] == "ragged":
        degrees = torch.randint(0, min(2 * mean, d) + 1, (h,), generator=fixed, device="cuda")
    else:
        drawn = torch.round(mean + 0.15 * mean * torch.randn(h, generator=fixed, device="cuda"))
        degrees = drawn.clamp(max(1, mean // 8), d).long()
    return degrees[torch.randperm(h, generator=generator, device="cuda")]


def _side(generator, case):
    """(offsets, indices, values) of one side, hidden-major: every neuron's slots at distinct, sorted indices."""
    d, h = case["d_model"], case["d_ff"]
    degrees = _degrees(generator, case)
    keys = torch.rand((h, d), generator=generator, device="cuda").clamp_(min=1e-30)
    if case["support"] == "zipf":  # weighted sampling without replacement: the largest log-weight plus Gumbel keys
        rank = torch.randperm(d, generator=generator, device="cuda").float()
        keys = -1.1 * torch.log(rank + 1.0)[None, :] - torch.log(-torch.log(keys.clamp_(max=1 - 1e-7)))
    order = keys.argsort(dim=1, descending=True)
    taken = torch.zeros((h, d), dtype=torch.bool, device="cuda")
    taken.scatter_(1, order, torch.arange(d, device="cuda")[None, :] < degrees[:, None])
    offsets = torch.zeros(h + 1, dtype=torch.int32, device="cuda")
    offsets[1:] = torch.cumsum(degrees, 0).int()
    index = taken.nonzero()[:, 1].to(torch.int16)
    values = _normal(generator, index.numel(), WEIGHT_STD)
    return offsets, index, values.bfloat16() if case["values"] == "bf16" else values


def _layer(generator, case):
    """The arguments of ``HFFNLayer.from_hidden_major``."""
    d, h = case["d_model"], case["d_ff"]
    up, down = _side(generator, case), _side(generator, case)
    return d, h, _normal(generator, h, BIAS_STD), *up, _normal(generator, d, BIAS_STD), *down


def _inputs(case, seed):
    """The layers' arguments, their inputs and (training) the gradients of their outputs."""
    generator = torch.Generator("cuda").manual_seed(seed)
    shape = (case["tokens"], case["d_model"])
    layers = [_layer(generator, case) for _ in range(case["layers"])]
    xs = [_normal(generator, shape) for _ in range(case["layers"])]
    return layers, xs, _normal(generator, shape, GRAD_STD) if case["kind"] == "train" else None


def prepare(case, seed):
    layers, xs, gy = _inputs(case, seed)
    layers = [HFFNLayer.from_hidden_major(*layer) for layer in layers]
    runtime = (PreparedRuntime if case["prepared"] else HFFNRuntime)(layers, "cuda")
    state = {"kind": case["kind"], "runtime": runtime, "xs": xs}
    if case["kind"] == "step":
        state["outs"] = [torch.empty_like(x) for x in xs]
    if case["kind"] == "train":
        state["train"] = HFFNTrainRuntime(runtime, **HYPER, max_tokens=case["tokens"])
        state["train"].reserve(case["tokens"])
        state["gy"] = gy
    return state


# --------------------------------------------------------------------------------------------------------------- run

def run(state):
    if state["kind"] == "layer":
        return state["runtime"].forward(0, state["xs"][0])
    if state["kind"] == "step":
        for index, (x, out) in enumerate(zip(state["xs"], state["outs"])):
            out.copy_(state["runtime"].forward(index, x))
        return state["outs"]
    train = state["train"]
    gx = train.step(0, state["xs"][0], state["gy"])
    return {"gx": gx, "gradients": train.gradients(0), "parameters": train.parameters(0)}


def work(case):
    """The slots of both sides (2-byte indices and the values), offsets and biases, inputs and outputs once; two
    operations per slot and token. Training also reads and writes values, both moments, writes the gradients, and
    multiplies every slot by every token three times."""
    d, h, n, layers = case["d_model"], case["d_ff"], case["tokens"], case["layers"]
    slots = 2 * h * max(1, round(case["density"] * d))
    value = 2 if case["values"] == "bf16" else 4
    bytes_ = slots * (2 + value) + 8 * (h + d) + 8 * n * d
    flops = 2.0 * slots * n
    if case["kind"] == "train":
        bytes_ += slots * (4 + 4 + 8 + 8) + 4 * n * d  # written values, gradients, moments read and written; gy
        flops = 3 * flops + 12 * slots
    return {"bytes": float(layers * bytes_), "flops": float(layers * flops)}


def tolerance(case):
    """Float32 sums of hundreds to thousands of products, in any order or as splits into 16-bit parts: up to 1e-6 of the
    result against 64 bits (1.5e-7 to 1e-6 measured over the cases). A training step adds AdamW, whose first updates
    divide a gradient by its own size: where it is next to zero the sign of an update, up to 2 lr or a fifth of a
    bias, follows the rounding (5e-6 of a drawn layer's biases)."""
    return {"rel": 2e-5, "max": 0.2} if case["kind"] == "train" else {"rel": 4e-6, "max": 1e-4}


# ------------------------------------------------------------------------------------------------------------- exact

def _dense(case, offsets, index, values):
    """The neurons' rows [d_ff, d_model] of one side in float64."""
    owner = torch.repeat_interleave(torch.arange(case["d_ff"], device="cuda"), offsets.diff().long())
    dense = torch.zeros((case["d_ff"], case["d_model"]), dtype=torch.float64, device="cuda")
    dense[owner, index.long()] = values.double()
    return dense, owner


def _adamw(value, gradient):
    """The first AdamW update in float64."""
    value = value.double()
    return value * (1.0 - HYPER["lr"] * HYPER["weight_decay"]) - HYPER["lr"] * gradient / (gradient.abs() + HYPER["eps"])


def exact(case, seed):
    layers, xs, gy = _inputs(case, seed)
    outs = []
    for (_, _, b_up, up_offsets, up_idx, up_val, b_down, down_offsets, down_idx, down_val), x in zip(layers, xs):
        w_up, up_owner = _dense(case, up_offsets, up_idx, up_val)
        w_down, down_owner = _dense(case, down_offsets, down_idx, down_val)
        x = x.double()
        z = x @ w_up.T + b_up.double()
        phi = 0.5 * (1.0 + torch.special.erf(z / math.sqrt(2.0)))
        act = z * phi
        if gy is None:
            outs.append(act @ w_down + b_down.double())
            continue
        gy = gy.double()
        gz = (gy @ w_down.T) * (phi + z * torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi))
        order = torch.argsort(down_idx.long(), stable=True)  # the gradient and the values of the down side are output-major
        gradients = {"up_val": (gz.T @ x)[up_owner, up_idx.long()], "b_up": gz.sum(0),
                     "out_val": (act.T @ gy)[down_owner, down_idx.long()][order], "b_down": gy.sum(0)}
        values = {"up_val": up_val, "b_up": b_up, "out_val": down_val[order], "b_down": b_down}
        return {"gx": gz @ w_up, "gradients": gradients,
                "parameters": {name: _adamw(values[name], gradients[name]) for name in values}}
    return outs if case["kind"] == "step" else outs[0]
