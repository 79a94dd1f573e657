"""The work that users of streaming attention have it do, as measurable cases.

Every case is one call of a public entry point (`streaming_attention` or `self_attention`), for
training followed by its backward pass.  Sizes are those of bench.py's workloads, of the reference's
benchmark grid and of the test suite, or generic ones of the same ranges.

A case holds
  what    "train" (forward + backward), "infer" (forward only), "dense" (`self_attention`)
  dtype, B, H, T, D   the [B, H, T, D] problem
  C, R    chunk length and number of earlier chunks a query sees (unused by "dense")
  lens    "full" (lens=None), "half" (uniform in [T/2, T]), "any" (uniform in [1, T]) or
          "log" (log-uniform in [min(64, T), T])
  packed  q, k, v are views of one [B, T, 3, H, D] projection output instead of tensors of their own
  lse     the log-sum-exp is asked for as well ("infer" only)
"""
import math
import os
import random
import sys

import torch

import kernels_amd

sys.path.insert(0, os.path.dirname(os.path.abspath(kernels_amd.__file__)))

from self_attention import self_attention  # noqa: E402
from streaming_attention import streaming_attention  # noqa: E402


def _case(what, dtype, B, H, T, D, C=0, R=0, lens="full", packed=False, lse=False, name=None):
    c = dict(what=what, dtype=dtype, B=B, H=H, T=T, D=D, C=C, R=R, lens=lens, packed=packed, lse=lse)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # one short utterance through a streaming encoder layer: latency, no backward pass
        _case("infer", "float16", 1, 8, 200, 64, 10, 9, name="infer_one_utterance_fp16"),
        # a debugging-size float32 training step, the one the CPU can check
        _case("train", "float32", 2, 4, 512, 64, 64, 2, "half", name="train_small_fp32"),
        # dense variable-length encoder layer
        _case("dense", "float16", 8, 12, 1500, 64, lens="half", name="dense_encoder_fp16"),
        # batch transcription with short chunks: the reference's benchmark grid, forward
        _case("infer", "float16", 128, 12, 1354, 64, 10, 9, name="infer_batch_fp16_chunk10"),
        # training on the same grid, its largest length and other chunk size
        _case("train", "float16", 128, 12, 3000, 64, 32, 2, name="train_batch_fp16_chunk32"),
        # small heads, short chunks, a large batch of sequences of every length
        _case("train", "float16", 225, 4, 993, 32, 16, 2, "any", name="train_heads32_fp16"),
        # strongly padded batch of short windows
        _case("train", "float16", 16, 8, 2048, 128, 64, 1, "log", name="train_ragged_fp16"),
        # medium context, head dimension 64
        _case("train", "bfloat16", 8, 16, 4096, 64, 128, 4, name="train_4k_heads64_bf16"),
        # wide heads, q, k and v read in place from the projection's output
        _case("train", "bfloat16", 4, 16, 4096, 256, 128, 4, packed=True, name="train_4k_heads256_bf16"),
        # float32 training at full precision
        _case("train", "float32", 4, 16, 4096, 128, 128, 4, name="train_4k_fp32"),
        # the headline workload
        _case("train", "bfloat16", 4, 16, 16384, 128, 256, 8, "half", name="train_16k_bf16"),
        # the longest context
        _case("train", "bfloat16", 1, 32, 65536, 128, 512, 16, name="train_64k_bf16"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _fits(c):
    """Whether a drawn case costs no more than the largest listed one and its tensors are of a usual size."""
    w, most = work(c), work(listed()[-1])
    rate = 20 if c["dtype"] == "float32" else 3 if c["D"] < 128 or c["C"] < 128 else 1
    return w["flops"] * rate <= most["flops"] and w["bytes"] <= 6e9


def draw(rng):
    while True:
        kind = rng.choice(["small", "grid", "narrow", "ragged", "medium", "wide", "fp32", "long", "dense"])
        half = rng.choice(["float16", "bfloat16"])
        what = rng.choice(["train", "infer"])
        lse = what == "infer" and rng.random() < 0.25
        packed = rng.random() < 0.25
        if kind == "small":       # a few short sequences of any type
            c = _case(what, rng.choice(["float32", half]), rng.randint(1, 4), rng.randint(1, 8), _log(rng, 50, 640),
                      rng.choice([32, 64, 128]), _log(rng, 8, 128), rng.randint(0, 9), rng.choice(["full", "half", "any"]),
                      packed, lse)
        elif kind == "grid":      # large batches, windows of about a hundred keys
            C = _log(rng, 8, 64)
            c = _case(what, half, _log(rng, 16, 128), rng.choice([8, 12, 16]), _log(rng, 257, 3000), 64, C,
                      max(1, 128 // C - rng.randint(1, 3)), rng.choice(["full", "half"]), packed, lse)
        elif kind == "narrow":    # small heads
            c = _case(what, half, _log(rng, 16, 256), rng.choice([4, 6, 8]), _log(rng, 257, 1024), rng.choice([16, 32]),
                      _log(rng, 10, 64), rng.randint(1, 5), rng.choice(["full", "any"]), packed, lse)
        elif kind == "ragged":
            c = _case(what, half, _log(rng, 8, 48), rng.choice([8, 12, 16]), _log(rng, 1024, 4096), rng.choice([64, 128]),
                      _log(rng, 32, 128), rng.randint(0, 3), "log", packed, lse)
        elif kind == "medium":
            c = _case(what, half, rng.randint(1, 8), rng.choice([8, 12, 16]), _log(rng, 1024, 16384), rng.choice([64, 128]),
                      _log(rng, 64, 512), rng.randint(1, 8), rng.choice(["full", "half"]), packed, lse)
        elif kind == "wide":
            c = _case(what, half, rng.randint(1, 4), rng.choice([8, 16]), _log(rng, 512, 4096), 256, _log(rng, 32, 256),
                      rng.randint(1, 6), rng.choice(["full", "half"]), packed, lse)
        elif kind == "fp32":
            c = _case(what, "float32", rng.randint(1, 8), rng.choice([4, 8, 16]), _log(rng, 512, 4096),
                      rng.choice([32, 64, 128]), _log(rng, 16, 256), rng.randint(1, 6), rng.choice(["full", "half"]),
                      packed, lse)
        elif kind == "long":
            c = _case(what, half, 1, rng.choice([8, 16, 32]), _log(rng, 16384, 65536), 128, _log(rng, 256, 512),
                      rng.randint(8, 16), "full", packed, lse)
        else:
            c = _case("dense", rng.choice(["float32", half, half]), rng.randint(1, 16), rng.choice([4, 8, 12]),
                      _log(rng, 64, 2048), rng.choice([32, 64, 128]), lens=rng.choice(["full", "half"]), packed=packed)
        if _fits(c):
            return c


def _lengths(case):
    """The batch's lengths in some order; prepare() shuffles them, so that the work does not depend on the seed."""
    B, T, mode = case["B"], case["T"], case["lens"]
    rng = random.Random(20)
    if mode == "full":
        return [T] * B
    if mode == "half":
        return [rng.randint((T + 1) // 2, T) for _ in range(B)]
    if mode == "any":
        return [rng.randint(1, T) for _ in range(B)]
    lo = math.log(min(64, T))
    return [int(round(math.exp(lo + rng.random() * (math.log(T) - lo)))) for _ in range(B)]


def prepare(case, seed):
    B, H, T, D = (case[n] for n in "BHTD")
    dtype = getattr(torch, case["dtype"])
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(seed)
    grad = case["what"] == "train"

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32).to(dtype)

    if case["packed"]:
        qkv = normal(B, T, 3, H, D)
        q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    else:
        q, k, v = (normal(B, H, T, D) for _ in range(3))
    lens = None
    if case["lens"] != "full":
        lengths = _lengths(case)
        random.Random(seed).shuffle(lengths)
        lens = torch.tensor(lengths, dtype=torch.int32).to(dev)
    return {"what": case["what"], "C": case["C"], "R": case["R"], "lse": case["lse"], "lens": lens,
            "q": q.requires_grad_(grad), "k": k.requires_grad_(grad), "v": v.requires_grad_(grad),
            "d_o": normal(B, H, T, D) if grad else None}


def run(state):
    q, k, v, lens = state["q"], state["k"], state["v"], state["lens"]
    if state["what"] == "train":
        out = streaming_attention(q, k, v, lens, state["C"], state["R"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["d_o"])
        return {"o": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    with torch.inference_mode():
        if state["what"] == "dense":
            return self_attention(q, k, v, lens)
        return streaming_attention(q, k, v, lens, state["C"], state["R"], return_lse=state["lse"])


def work(case):
    """Inputs at valid positions read once, outputs written once (zeros at padded positions included); two products
    of 2*D flop per allowed (query, key) pair forward, five backward."""
    B, H, T, D = (case[n] for n in "BHTD")
    lengths = _lengths(case)
    es = 4 if case["dtype"] == "float32" else 2
    pairs = 0
    for L in lengths:
        if case["what"] == "dense":
            pairs += L * L
            continue
        C, R = case["C"], case["R"]
        for c in range(-(-L // C)):
            pairs += (min((c + 1) * C, L) - c * C) * (min((c + 1) * C, L) - max(0, c - R) * C)
    valid, rows = sum(lengths) * H, B * H * T
    if case["what"] == "train":
        return {"bytes": float(4 * valid + 4 * rows) * D * es, "flops": 14.0 * D * H * pairs}
    return {"bytes": float(3 * valid + rows) * D * es + (4.0 * rows if case["lse"] else 0.0), "flops": 4.0 * D * H * pairs}


def tolerance(case):
    """Four times the largest error seen against a float64 evaluation of the same problems: relative 8.2e-7 / 4.2e-4 /
    3.4e-3 and largest 1.5e-5 / 7.8e-3 / 5.9e-2 for float32 / float16 / bfloat16 (dK and dV, which sum rounded
    probabilities over a window, are the worst)."""
    return {"float32": {"rel": 3.3e-6, "max": 6e-5}, "float16": {"rel": 1.7e-3, "max": 0.032},
            "bfloat16": {"rel": 1.4e-2, "max": 0.24}}[case["dtype"]]
