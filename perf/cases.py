"""What the speed of this backend is measured on: calls of its nine public functions
(dslperfgap_amd/viperbench/*/hip_impl.py) over the shapes, element types and options they
are used with.

A case is a dict of plain values: ``op`` (the function, ``ce_step`` being the forward, the
mean loss and the backward of one training step), ``shape`` ("rows x cols", or the whole
shape where ``dim`` names the axis), ``dtype`` and the op's own options.  ``listed()`` are
the cases of record, ``draw()`` gives further ones of the same ranges: 1 to 65536 rows, 64
to 131072 columns, up to 2^27 elements, whole multiples of a model width's 64 and ragged
lengths alike, fp32 / fp16 / bf16, reduced axes in last, first and middle place.

Inputs are drawn on the GPU from the seed.  Outputs are returned whole; of the three
cross-entropy buffers, which are as large as the logits, only the first
n_rows * (column blocks) values are ever written, and these are what a caller reads.
"""
import math

import torch

from dslperfgap_amd.viperbench.argmax.hip_impl import argmax
from dslperfgap_amd.viperbench.cross_entropy.hip_impl import (cross_entropy_bwd,
                                                              cross_entropy_fwd, loss_mean)
from dslperfgap_amd.viperbench.layer_norm.hip_impl import layer_norm
from dslperfgap_amd.viperbench.log_softmax.hip_impl import log_softmax
from dslperfgap_amd.viperbench.logsumexp.hip_impl import logsumexp
from dslperfgap_amd.viperbench.max_reduction.hip_impl import max_reduction
from dslperfgap_amd.viperbench.mean_reduction.hip_impl import mean_reduction
from dslperfgap_amd.viperbench.rms_norm.hip_impl import rms_norm
from dslperfgap_amd.viperbench.softmax.hip_impl import softmax

DEVICE = "cuda"
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZES = {"fp32": 4, "fp16": 2, "bf16": 2}
IGNORED = -100


def listed():
    return [
        # the norm of one decode step of 64 sequences: latency
        {"name": "layer_norm_decode", "op": "layer_norm", "shape": "64x1024", "dtype": "bf16",
         "weight": "bf16", "bias": True},
        # the norm ahead of a wide MLP (this repository's C5)
        {"name": "layer_norm_wide", "op": "layer_norm", "shape": "2048x20480", "dtype": "bf16",
         "weight": "bf16", "bias": True},
        # the norm of a prefill of 8192 tokens (C2)
        {"name": "rms_norm_prefill", "op": "rms_norm", "shape": "8192x4096", "dtype": "bf16",
         "weight": "bf16"},
        # attention scores, 1% of them large (C3)
        {"name": "softmax_scores", "op": "softmax", "shape": "16384x4096", "dtype": "fp32",
         "mask": False},
        # token log-probabilities over a vocabulary that is no multiple of a vector, 16-bit
        # logits widened to fp32 as a scoring program asks for them
        {"name": "log_softmax_vocab", "op": "log_softmax", "shape": "1024x50257",
         "dtype": "bf16", "out": "fp32", "dim": 1},
        # class log-probabilities over the channel axis of an image batch
        {"name": "log_softmax_channels", "op": "log_softmax", "shape": "16x64x128x128",
         "dtype": "fp32", "out": "fp32", "dim": 1},
        # the partition function over the rows of C3
        {"name": "logsumexp_rows", "op": "logsumexp", "shape": "16384x4096", "dtype": "fp32"},
        # one step's loss and gradient in fp32 (C4, forward and backward)
        {"name": "ce_step_fp32", "op": "ce_step", "shape": "8192x32000", "dtype": "fp32",
         "smoothing": 0.0, "scale": 1.0, "z": 0.0, "labels": "i64"},
        # the same from 16-bit logits over a ragged vocabulary, with label smoothing, the
        # z-loss and ignored (padding) tokens
        {"name": "ce_step_bf16", "op": "ce_step", "shape": "4096x50257", "dtype": "bf16",
         "smoothing": 0.1, "scale": 1.0, "z": 1e-4, "labels": "i64"},
        # the reference benchmark's large row mean
        {"name": "mean_rows", "op": "mean_reduction", "shape": "8192x32768", "dtype": "fp32",
         "dim": 1},
        # max over time of a batch of token features (a middle axis)
        {"name": "max_over_time", "op": "max_reduction", "shape": "64x512x768",
         "dtype": "fp16", "dim": 1},
        # greedy choice of the next token for a batch of sequences: few, long rows
        {"name": "argmax_tokens", "op": "argmax", "shape": "64x50304", "dtype": "fp16",
         "dim": 1},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _length(rng, lo, hi):
    """A length: half of the time a multiple of 64, as model widths are, else any."""
    n = int(_log_uniform(rng, lo, hi))
    if rng.random() < 0.5 and n >= 64:
        n -= n % 64
    return max(lo, min(hi, n))


def draw(rng):
    op = rng.choice(["layer_norm", "rms_norm", "softmax", "log_softmax", "logsumexp", "ce_step",
                     "ce_blocks", "mean_reduction", "max_reduction", "argmax"])
    case = {"op": op, "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    elements = _log_uniform(rng, 1 << 14, 1 << 27)
    cols = _length(rng, 1000 if op.startswith("ce") else 64, 131072)
    rows = max(1, min(65536, int(elements / cols)))
    case["shape"] = f"{rows}x{cols}"
    if op in ("layer_norm", "rms_norm"):
        case["weight"] = rng.choice([case["dtype"], "fp32"])
        if op == "layer_norm":
            case["bias"] = rng.random() < 0.8
    elif op == "softmax":
        case["mask"] = rng.random() < 0.3
    elif op == "ce_step":
        case.update(smoothing=rng.choice([0.0, 0.1]), scale=rng.choice([1.0, 1.0, 0.5]),
                    z=rng.choice([0.0, 1e-4]), labels=rng.choice(["i64", "i32"]))
    elif op == "ce_blocks":
        case.update(smoothing=rng.choice([0.0, 0.1]), scale=1.0, z=0.0, labels="i64",
                    block=rng.choice([1024, 2048, 8192]))
    elif op != "logsumexp":
        if op == "log_softmax":
            case["out"] = rng.choice([case["dtype"], "fp32"])
        case["dim"] = 1
        if rng.random() < 0.5:  # a first or middle axis
            n = _length(rng, 2, 8192)
            inner = _length(rng, 2, 8192)
            outer = max(1, min(4096, int(elements / (n * inner))))
            outer = 1 if rng.random() < 0.3 else outer
            case["shape"] = f"{n}x{inner}" if outer == 1 else f"{outer}x{n}x{inner}"
            case["dim"] = 0 if outer == 1 else 1
    return case


def _shape(case):
    return tuple(int(s) for s in case["shape"].split("x"))


def _blocks(case):
    """(block size, column blocks) of a cross-entropy case."""
    cols = _shape(case)[1]
    size = case.get("block", 1 << 18)
    return size, -(-cols // size)


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    op, shape, dtype = case["op"], _shape(case), DTYPES[case["dtype"]]

    def randn(*size):
        return torch.randn(*size, device=DEVICE, generator=g)

    x = randn(*shape)
    state = {"case": case}
    if op in ("layer_norm", "rms_norm"):
        wdt = DTYPES[case["weight"]]
        x = 0.5 + 2.0 * x
        state["w"] = (1.0 + 0.1 * randn(shape[1])).to(wdt)
        if case.get("bias"):
            state["b"] = (0.1 * randn(shape[1])).to(wdt)
    elif op in ("softmax", "log_softmax", "logsumexp"):
        x = 3.0 * x
        if op == "softmax" and case["mask"]:  # padded keys: each row's tail at the lowest value
            keep = torch.randint(1, shape[1] + 1, (shape[0], 1), device=DEVICE, generator=g)
            x = torch.where(torch.arange(shape[1], device=DEVICE) < keep, x,
                            torch.finfo(dtype).min)
        else:
            x[torch.rand(*shape, device=DEVICE, generator=g) < 0.01] = 20.0
    elif op in ("ce_step", "ce_blocks"):
        rows, cols = shape
        x = 2.0 * x
        labels = torch.randint(0, cols, (rows,), device=DEVICE, generator=g)
        labels[torch.rand(rows, device=DEVICE, generator=g) < 0.05] = IGNORED
        state["labels"] = labels.to(torch.int32) if case["labels"] == "i32" else labels
        state["dloss"] = torch.full((rows,), 1.0 / rows, device=DEVICE)
    state["x"] = x.to(dtype)
    return state


def _ce_args(case):
    size, blocks = _blocks(case)
    smooth = case["smoothing"]
    return (smooth, case["scale"], case["z"], IGNORED, _shape(case)[1], 0, size, smooth > 0.0)


def run(state):
    case, x = state["case"], state["x"]
    op = case["op"]
    if op == "layer_norm":
        return layer_norm(x, state["w"], state.get("b"))
    if op == "rms_norm":
        return rms_norm(x, (x.shape[1],), state["w"])
    if op == "softmax":
        return softmax(x)
    if op == "log_softmax":
        if case["out"] == case["dtype"]:
            return log_softmax(x, dim=case["dim"])
        return log_softmax(x, dim=case["dim"], dtype=DTYPES[case["out"]])
    if op == "logsumexp":
        return logsumexp(x)
    if op == "mean_reduction":
        return mean_reduction(x, case["dim"])
    if op == "max_reduction":
        return max_reduction(x, case["dim"])
    if op == "argmax":
        return argmax(x, case["dim"])
    args = _ce_args(case)
    rows = x.shape[0]
    loss, lse, z = cross_entropy_fwd(x, state["labels"], *args, op == "ce_blocks")
    n = rows * _blocks(case)[1]
    out = [loss.view(-1)[:n], lse.view(-1)[:n], z.view(-1)[:n]]
    if op == "ce_step":
        out.append(loss_mean(loss, rows))
        out.append(cross_entropy_bwd(state["dloss"], x, lse, state["labels"], *args))
    return out


def work(case):
    op, shape, e = case["op"], _shape(case), SIZES[case["dtype"]]
    n = math.prod(shape)
    if op in ("layer_norm", "rms_norm"):
        vectors = 1 + bool(case.get("bias"))
        return {"bytes": 2 * n * e + vectors * shape[1] * SIZES[case["weight"]], "flops": 8 * n}
    if op == "softmax":
        return {"bytes": 2 * n * e, "flops": 5 * n}
    if op == "log_softmax":
        return {"bytes": n * (e + SIZES[case["out"]]), "flops": 5 * n}
    if op == "logsumexp":
        return {"bytes": n * e + shape[0] * e, "flops": 4 * n}
    if op in ("ce_step", "ce_blocks"):
        rows = shape[0]
        lab = 4 if case["labels"] == "i32" else 8
        fwd = n * e + rows * lab + 12 * rows * _blocks(case)[1]
        if op == "ce_blocks":
            return {"bytes": fwd, "flops": 4 * n}
        # the mean reads the losses; the backward reads the logits again, the labels, lse
        # and dloss, and writes dlogits
        return {"bytes": fwd + 4 * rows + 2 * n * e + rows * (lab + 8), "flops": 8 * n}
    out = {"mean_reduction": e, "max_reduction": e + 8, "argmax": 8}[op]
    return {"bytes": n * e + n // shape[case["dim"]] * out, "flops": n}


# Relative error (2-norm) and largest difference of another correct implementation: four
# times the largest distance between this backend and exact() over the listed and 150 drawn
# cases.  fp32 results carry the rounding of their 32-bit sums and of the hardware's 1-ulp
# exponential and logarithm (9.4e-8 and 1.2e-6 at most; 5.5e-7 and 2e-6 for the mean, which
# cancels), 16-bit results half an ulp of their type (fp16 2.4e-4 and 4.9e-4, and 4.6e-4 and
# 6.9e-4 for gradients among the subnormals; bf16 2.2e-3 and 3.9e-3).
TOLERANCE = {
    "fp32": {"rel": 4e-7, "max": 5e-6},
    "fp16": {"rel": 1e-3, "max": 2e-3},
    "bf16": {"rel": 8e-3, "max": 1.6e-2},
}
MEAN_FP32 = {"rel": 2e-6, "max": 8e-6}


def tolerance(case):
    op = case["op"]
    if op in ("max_reduction", "argmax"):
        return "exact"  # a value and the first place of the input
    if op == "ce_blocks":
        return TOLERANCE["fp32"]
    if op == "mean_reduction" and case["dtype"] == "fp32":
        return MEAN_FP32
    return TOLERANCE[case.get("out", case["dtype"])]


def exact(case, seed):
    op = case["op"]
    if op == "argmax":
        return None
    state = prepare(case, seed)
    x = state.pop("x").double()
    if op in ("layer_norm", "rms_norm"):
        w = state["w"].double()
        if op == "rms_norm":
            return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * w
        d = x - x.mean(1, keepdim=True)
        y = d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-5) * w
        return y + state["b"].double() if "b" in state else y
    if op == "softmax":
        return torch.softmax(x, 1)
    if op == "log_softmax":
        return torch.log_softmax(x, case["dim"])
    if op == "logsumexp":
        return torch.logsumexp(x, 1)
    if op == "mean_reduction":
        return x.mean(case["dim"])
    if op == "max_reduction":
        return x.amax(case["dim"]), None
    return _exact_ce(case, state, x)


def _exact_ce(case, state, x):
    rows, cols = x.shape
    smooth, zs = case["smoothing"], case["z"]
    split = case["op"] == "ce_blocks"
    size, blocks = _blocks(case)
    labels = state["labels"].long()
    live = labels != IGNORED
    at = labels.clamp(min=0)
    x *= case["scale"]
    losses, lses, zlosses = [], [], []
    for cb in range(blocks):
        part = x[:, cb * size:(cb + 1) * size]
        lse = torch.logsumexp(part, 1)
        here = live & (at >= cb * size) & (at < cb * size + part.shape[1])
        logit = x.gather(1, at[:, None])[:, 0]
        mean = part.sum(1) / cols
        base = torch.zeros_like(lse) if split else lse
        loss = torch.where(here, base - (1.0 - smooth) * logit, smooth * base)
        loss = loss - smooth * mean
        z = torch.zeros_like(lse) if split else zs * lse * lse
        losses.append(torch.where(live, loss + z, 0.0))
        zlosses.append(torch.where(live, z, 0.0))
        lses.append(lse)
    out = [torch.cat(losses), torch.cat(lses), torch.cat(zlosses)]
    if split:
        return out
    lse = lses[0]
    out.append(out[0].mean())
    grad = torch.exp(x.sub_(lse[:, None])).mul_((1.0 + 2.0 * zs * lse)[:, None])
    grad -= smooth / cols
    grad[torch.arange(rows, device=x.device), at] -= 1.0 - smooth
    grad *= (torch.where(live, state["dloss"].double(), 0.0) * case["scale"])[:, None]
    return out + [grad]
