"""The work a program has this framework do, as measurable cases: calls of mhc.MHCLayer, forward alone
and forward + backward, over the batch sizes, widths, stream counts and data types that it is used with.

A case is a dict of plain values:

    mode     "train": forward + backward with gradients of x and of every parameter
             "infer": the layer in eval mode under torch.no_grad()
    dynamic  per-sample coefficients projected from x, or shared parameters
    dtype    "bf16":  bfloat16 activations in and out
             "mixed": float32 activations in and out, bfloat16 arithmetic (compute_dtype=torch.bfloat16)
             "fp32":  float32 throughout (the constructor's default)
    B, n, C  samples (tokens), residual streams, hidden size
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("mhc.cu_amd"))

from mhc import MHCLayer  # noqa: E402


def _case(mode, dynamic, dtype, B, n, C):
    return {"mode": mode, "dynamic": dynamic, "dtype": dtype, "B": B, "n": n, "C": C}


def listed():
    return [
        # a serving step: a handful of sequences advance by one token; latency and launches count
        dict(_case("infer", True, "bf16", 7, 4, 1280), name="decode"),
        # the static layer's forward at the shape of the first benchmark configuration
        dict(_case("infer", False, "fp32", 320, 4, 1280), name="static_forward"),
        # a prompt's tokens pass through the layer once; their number is whatever the prompt has
        dict(_case("infer", True, "bf16", 3001, 4, 2560), name="prefill"),
        # training at the benchmark's four configurations with dynamic coefficients
        dict(_case("train", True, "bf16", 320, 4, 1280), name="train_small"),
        dict(_case("train", True, "bf16", 1280, 4, 2560), name="train_large"),
        dict(_case("train", True, "bf16", 256, 8, 1280), name="train_n8"),
        dict(_case("train", True, "bf16", 128, 32, 1280), name="train_n32"),
        # float32 tensors around bfloat16 arithmetic: what the benchmark tables run
        dict(_case("train", True, "mixed", 512, 4, 1920), name="train_mixed"),
        # the layer as its constructor makes it, float32 throughout
        dict(_case("train", True, "fp32", 2560, 4, 1280), name="train_fp32"),
        # shared coefficients, the other half of the benchmark tables
        dict(_case("train", False, "bf16", 1280, 4, 2560), name="train_static"),
        # a small model whose sizes are no multiples of anything
        dict(_case("train", True, "bf16", 333, 3, 1230), name="train_ragged"),
        # one micro-batch of a large training run
        dict(_case("train", True, "bf16", 8192, 4, 2560), name="train_tokens"),
    ]


#: the most activation elements B * n * C of a drawn case: those of the largest listed case, fewer where an
#: element costs more (32-bit storage and arithmetic, more streams)
_MOST = 8192 * 4 * 2560


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "static_forward", "prefill", "train", "train", "train_wide", "mixed", "fp32", "static"])
    n = rng.choice([4, 4, 4, 2, 3, 8, 8, 5, 6])
    C = _spread(rng, 256, 4096)
    if rng.random() < 0.75:  # most models' hidden sizes are multiples of 64
        C = max(256, C // 64 * 64)
    if kind == "decode":
        return _case("infer", True, "bf16", _spread(rng, 1, 64), n, C)
    if kind == "train_wide":
        return _case("train", True, "bf16", _spread(rng, 16, 192), rng.choice([12, 16, 24, 32, 32]), max(256, min(C // 64 * 64, 1600)))
    most = _MOST * min(4, n) // n // {"mixed": 3, "fp32": 16, "static_forward": 2}.get(kind, 1)
    if C % 8:  # sizes that are no multiple of a 16-byte access are met in small models
        most = min(most, 8_000_000, 100_000_000 // (n * n + 2 * n))
    B = min(_spread(rng, 64, 8192), most // (n * C))
    if kind == "static_forward":
        return _case("infer", False, rng.choice(["fp32", "bf16"]), B, n, C)
    if kind == "prefill":
        return _case("infer", True, "bf16", B, n, C)
    if kind == "static":
        return _case("train", False, rng.choice(["bf16", "bf16", "mixed"]), B, n, C)
    return _case("train", True, {"train": "bf16"}.get(kind, kind), B, n, C)


def prepare(case, seed):
    """A layer whose parameters have moved away from their initial values, activations and, for
    training, the gradient that arrives from above."""
    torch.manual_seed(seed)
    B, n, C, dtype = case["B"], case["n"], case["C"], case["dtype"]
    act = torch.bfloat16 if dtype == "bf16" else torch.float32
    with torch.device("cuda"):
        layer = MHCLayer(C, n, use_dynamic_h=case["dynamic"], output_dtype=torch.bfloat16 if dtype == "bf16" else None,
                         compute_dtype=torch.bfloat16 if dtype == "mixed" else None)
        with torch.no_grad():
            layer.rmsnorm_weight.normal_(1.0, 0.1)
            if case["dynamic"]:
                for b in (layer.b_pre, layer.b_post, layer.b_res):
                    b.normal_(0.0, 0.5)
                for a in (layer.alpha_pre, layer.alpha_post, layer.alpha_res):
                    a.fill_(0.1)
            else:
                for h in (layer.H_pre, layer.H_post, layer.H_res):
                    h.normal_(0.0, 1.0)
        state = {"layer": layer, "x": torch.randn(B, n, C, dtype=act), "params": list(layer.parameters())}
        if case["mode"] == "train":
            layer.train()
            state["dy"] = torch.randn(B, n, C, dtype=act)
            state["x"].requires_grad_(True)
        else:
            layer.eval()
    return state


def run(state):
    layer, x = state["layer"], state["x"]
    if "dy" not in state:
        with torch.no_grad():
            return layer(x)
    x.grad = None
    for p in state["params"]:
        p.grad = None
    y = layer(x)
    y.backward(state["dy"])
    return [y.detach(), x.grad] + [p.grad for p in state["params"]]


def work(case):
    """Activations, parameters and gradients once each; the multiplications of the projection, of the
    aggregate and of the mix, and in the backward those of their gradients."""
    B, n, C = case["B"], case["n"], case["C"]
    size = 2 if case["dtype"] == "bf16" else 4
    D = n * n + 2 * n if case["dynamic"] else 0
    act, train = B * n * C, case["mode"] == "train"
    nbytes = 2 * size * act + 4 * D * n * C + 2 * C
    flops = 2 * act * D + 2 * act * (n + 2)
    if train:
        nbytes += 2 * size * act + 4 * D * n * C + 2 * C
        flops += 4 * act * D + 2 * act * (2 * n + 4)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["dtype"] != "fp32":
        return {"rel": 1e-2}  # bfloat16 operands and results
    # float32 sums; the gradients of the three alphas are sums over all samples of terms of both signs
    return {"rel": 2e-5}
