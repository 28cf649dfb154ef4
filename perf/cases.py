"""What the performance of this library is measured on.

Each case is a use of a public entry point as a training or a serving program makes it: a
training step (forward, and the backward through autograd), a prefill of a prompt that hands its
state on, or some steps of a decode loop.  `listed` holds one case for each use and size class;
`draw` makes further ones of the same ranges: batches of 1 to 64 (256 when decoding), widths of
64 to 4096 channels, 16 to 65536 timesteps (1 to 16 in a decode step), up to 2^27 elements a tensor.
"""
from __future__ import annotations

import math

import torch

from fast_sequential_scan_amd import (scan_cm, scan_cu, scan_cu_fp16, scan_cu_single, scan_gated,
                                      scan_gated_with_state, scan_with_state)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# op -> (tensors of bs*seq*d elements a pass reads and writes, flops per element)
#   train     scan_cu / scan_cu_single / scan_cu_fp16: forward reads alpha, beta, writes h; backward
#             reads alpha, h, dout, writes two gradients
#   train_cm  the same on (bs, d, seq) tensors, scan_cm
#   train_state    scan_with_state with gradients: a segment of a longer sequence
#   train_gated    scan_gated: forward as above; backward reads gate, x, h, dout, writes two gradients
#   prefill, prefill_gated   scan_with_state / scan_gated_with_state without gradients
#   decode, decode_gated     the same for the few tokens of a decode step, DECODE_STEPS times, each
#             step from the state that the one before left
OPS = {
    "train": (8, 5), "train_cm": (8, 5), "train_state": (8, 5), "train_gated": (9, 24),
    "prefill": (3, 2), "prefill_gated": (3, 9), "decode": (3, 2), "decode_gated": (3, 9),
}
DECODE_STEPS = 4


def _case(name, op, dtype, bs, seq, d, recipe):
    return {"name": name, "op": op, "dtype": dtype, "bs": bs, "seq": seq, "d": d, "recipe": recipe}


def listed():
    return [
        # tokens of a small batch, one by one, through a Hawk block that computes alpha and beta itself: all launch and host time
        _case("decode", "decode", "bf16", 8, 1, 1024, "hawk"),
        # tokens of a server's batch, one by one, through the gated block
        _case("decode_gated", "decode_gated", "bf16", 64, 1, 2048, "sigmoid"),
        # one segment of a chunked prefill, its state coming in and going out
        _case("prefill_gated", "prefill_gated", "bf16", 4, 2048, 2048, "sigmoid"),
        # the README's example shape: a training step bound by launches
        _case("train_small", "train", "bf16", 2, 1024, 768, "normal"),
        # Hawk training from the gates' pre-activations
        _case("train_gated", "train_gated", "bf16", 16, 2048, 512, "sigmoid"),
        # a sequence length that is no power of two
        _case("train_ragged", "train", "bf16", 8, 3000, 1024, "sigmoid"),
        # the benchmark's headline shape
        _case("train_headline", "train", "bf16", 8, 4096, 1024, "sigmoid"),
        # the long end of the benchmark's sweep over sequence lengths, long memory
        _case("train_longest", "train", "bf16", 8, 32768, 1024, "sigmoid_plus2"),
        # one document of prime length, few channels: all parallelism has to come from the sequence
        _case("train_one_sequence", "train", "bf16", 1, 65521, 256, "sigmoid"),
        # single precision
        _case("train_fp32", "train", "fp32", 8, 2048, 1536, "hawk"),
        # channel-major tensors, one token shorter than a power of two as next-token training leaves them
        _case("train_cm", "train_cm", "bf16", 8, 2047, 1024, "sigmoid"),
        # truncated back-propagation: a ragged segment between two states, half precision, width no multiple of 64
        _case("train_segment", "train_state", "fp16", 2, 777, 328, "near_one"),
    ]


def _log_int(rng, low, high):
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    op = rng.choice(("train",) * 6 + ("train_cm", "train_cm", "train_state", "train_gated", "train_gated", "prefill",
                                      "prefill_gated", "decode", "decode_gated"))
    dtype = rng.choice(("bf16",) * 6 + ("fp16", "fp32"))
    gated = op.endswith("gated")
    # (a gate near saturation rounds alpha to 1 in 16 bits: the gated recipes stop at +2)
    recipe = rng.choice(("sigmoid", "sigmoid_plus2") if gated else ("normal", "hawk", "sigmoid", "sigmoid_plus2", "near_one"))
    while True:
        d = _log_int(rng, 64, 4096)
        if rng.random() < 0.75:
            d = max(64, d // 64 * 64)
        if op.startswith("decode"):
            bs, seq = _log_int(rng, 1, 256), _log_int(rng, 1, 16)
            break
        bs, seq = _log_int(rng, 1, 64), _log_int(rng, 16, 65536)
        if 1 << 17 <= bs * seq * d <= 1 << 27:
            break
    return {"op": op, "dtype": dtype, "bs": bs, "seq": seq, "d": d, "recipe": recipe}


def _pair(recipe, shape, gen):
    """alpha and beta of a recurrence, in fp32."""
    x = torch.randn(shape, generator=gen, device="cuda")
    beta = torch.randn(shape, generator=gen, device="cuda")
    shift = {"normal": None, "hawk": 0.0, "sigmoid": 0.0, "sigmoid_plus2": 2.0, "near_one": 6.0}[recipe]
    alpha = x if shift is None else torch.sigmoid(x + shift)
    if recipe in ("hawk", "near_one"):
        beta = beta * torch.sqrt(1.0 - alpha * alpha)
    return alpha, beta


def _inputs(case, shape, gen):
    """(alpha, beta), or (gate, x) of a gated case, in the case's type."""
    if case["op"].endswith("gated"):
        first = torch.randn(shape, generator=gen, device="cuda") + (2.0 if case["recipe"] == "sigmoid_plus2" else 0.0)
        second = torch.randn(shape, generator=gen, device="cuda")
    else:
        first, second = _pair(case["recipe"], shape, gen)
    return first.to(DTYPES[case["dtype"]]), second.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op, bs, seq, d = case["op"], case["bs"], case["seq"], case["d"]
    shape = (bs, d, seq) if op == "train_cm" else (bs, seq, d)
    state = {"op": op, "dtype": case["dtype"]}
    if op.startswith("decode"):
        state["tokens"] = [_inputs(case, shape, gen) for _ in range(DECODE_STEPS)]
    else:
        state["first"], state["second"] = _inputs(case, shape, gen)
    if op.startswith("train"):
        state["first"].requires_grad_(True)
        state["second"].requires_grad_(True)
        state["grad"] = torch.randn(shape, generator=gen, device="cuda").to(DTYPES[case["dtype"]])
    if not op.startswith("train") or op == "train_state":
        state["h_before"] = torch.randn((bs, d), generator=gen, device="cuda")
    if op == "train_state":
        state["h_before"].requires_grad_(True)
        state["grad_last"] = torch.randn((bs, d), generator=gen, device="cuda")
    return state


_PLAIN = {"bf16": scan_cu, "fp16": scan_cu_fp16, "fp32": scan_cu_single}


def run(state):
    op = state["op"]
    if op.startswith("decode"):
        step = scan_gated_with_state if op == "decode_gated" else scan_with_state
        outs, last = [], state["h_before"]
        for first, second in state["tokens"]:
            h, last = step(first, second, last)
            outs.append(h)
        return outs, last
    first, second = state["first"], state["second"]
    if op == "prefill":
        return scan_with_state(first, second, state["h_before"])
    if op == "prefill_gated":
        return scan_gated_with_state(first, second, state["h_before"])
    if op == "train_state":
        h, last = scan_with_state(first, second, state["h_before"])
        return (h, last) + torch.autograd.grad((h, last), (first, second, state["h_before"]), (state["grad"], state["grad_last"]))
    scan = _PLAIN[state["dtype"]] if op == "train" else scan_cm if op == "train_cm" else scan_gated
    h = scan(first, second)
    return (h,) + torch.autograd.grad(h, (first, second), state["grad"])


def work(case):
    tensors, flops = OPS[case["op"]]
    steps = DECODE_STEPS if case["op"].startswith("decode") else 1
    n = case["bs"] * case["seq"] * case["d"]
    states = {"train": 0, "train_cm": 0, "train_gated": 0, "train_state": 5}.get(case["op"], 2)
    size = 4 if case["dtype"] == "fp32" else 2
    return {"bytes": steps * (tensors * n * size + states * case["bs"] * case["d"] * 4), "flops": steps * flops * n}


def tolerance(case):
    # Four times the largest distance (over the norm; of one value) from the same recurrence in 64 bits seen
    # over sixty cases, gated ones from the alpha and beta that the storage type holds: bf16 2.5e-3
    # and 2.4e-2, fp16 2.9e-4 and 2.3e-3, fp32 3.2e-7 and 9.4e-6.
    return {"bf16": {"rel": 1e-2, "max": 9.5e-2}, "fp16": {"rel": 1.2e-3, "max": 9.2e-3},
            "fp32": {"rel": 1.3e-6, "max": 3.8e-5}}[case["dtype"]]
