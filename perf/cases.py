"""Workloads of bucketed approximate top-k as its users call it, for timing on one GPU.

``listed()`` names the workloads, ``draw(rng)`` makes another one of the same ranges,
``prepare(case, seed)`` builds what a program holds before the call (inputs in GPU
memory), ``run(state)`` is one call through the package's public entry points,
``work(case)`` the bytes and operations the call cannot do without, and
``tolerance(case)`` how far a correct result may be from another.

A case is a plain dict:

    entry        "topk": approx_topk.topk; "indices": compact_indices.topk_indices (int32);
                 "argmax": bucketed_argmax.topk_triton; "train": differentiable.topk and
                 the gradient of its values with respect to the input
    rows, n      the input is [rows, n], the top-k dim last
    dtype        "float32", "float16" or "bfloat16"
    k, j, k_mult, interleaved   as the operator's arguments
    data         "normal": N(0, 1); "scores": N(0, 1) / sqrt(128), attention scores before the
                 softmax; "logits": N(0, 1) with Zipf boosts on a hundredth of the columns;
                 "trend": a slow trend under noise, neighbouring elements correlated
"""
from __future__ import annotations

import math
import os
import sys

import torch

# the package of the working folder, the repository's root
sys.path.insert(0, os.path.abspath("pytorch-approx-topk_amd"))

import approx_topk  # noqa: E402
from approx_topk.experimental import bucketed_argmax, compact_indices, differentiable  # noqa: E402

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}

# Most input bytes of a drawn case: a quarter of the largest listed input.
_DRAWN_BYTES = 128 << 20


def _case(entry, rows, n, dtype, k, j=1, k_mult=1, interleaved=True, data="normal"):
    return {"entry": entry, "rows": rows, "n": n, "dtype": dtype, "k": k, "j": j, "k_mult": k_mult,
            "interleaved": interleaved, "data": data}


def listed():
    cases = {
        # the smallest call: a handful of rows between the other steps of a model, bound by
        # launches and by the host
        "small_batch": _case("topk", 4, 65536, "float32", 1024),
        # one token of a decoding loop: 32 heads pick the keys and values to gather, and only the
        # positions are used
        "decode_positions": _case("indices", 32, 20480, "float16", 512, j=2, k_mult=2, data="scores"),
        # the operator's headline: many candidates of long rows, one stage
        "headline": _case("topk", 128, 1 << 20, "float32", 65536, j=2),
        # the same in a 16-bit type with four elements a bucket, the largest listed
        "headline_bf16": _case("topk", 256, 1 << 20, "bfloat16", 65536, j=4),
        # prefill of sparse attention: 32 sequences x 32 heads, two stages
        "attention_scores": _case("topk", 1024, 32768, "float16", 2048, j=4, k_mult=4, data="scores"),
        # sampling from a vocabulary: few of many logits, two stages
        "vocabulary_logits": _case("topk", 256, 131072, "float32", 64, j=1, k_mult=8, data="logits"),
        # the same with a vocabulary of no round size, as most are, so that rows start anywhere
        "ragged_logits": _case("topk", 256, 100003, "bfloat16", 64, j=1, k_mult=8, data="logits"),
        # one long correlated row over the whole GPU, two stages
        "long_row": _case("topk", 1, 1 << 26, "float32", 16384, j=4, k_mult=2, data="trend"),
        # ranking all entities of a knowledge graph for a few queries: very few of very many
        "entity_ranking": _case("topk", 16, 2653751, "float32", 10, j=2, k_mult=4),
        # contiguous buckets of uneven lengths
        "contiguous_ragged": _case("topk", 512, 40001, "float32", 1000, j=2, interleaved=False),
        # bucketed arg-max over a padded row
        "argmax_ragged": _case("argmax", 256, 50001, "float16", 1000),
        # a training step through sparse activations: forward and backward
        "train_activations": _case("train", 2048, 16384, "float32", 1024, j=2, k_mult=2),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: every entry point, sizes spread over their logarithm, half of them round."""
    entry = rng.choice(("topk", "topk", "topk", "topk", "indices", "argmax", "train"))
    dtype = rng.choice(tuple(_DTYPES))
    es = _BYTES[dtype]
    n = _log_uniform(rng, 1 << 12, 1 << 24)
    if rng.random() < 0.5:
        n = 1 << (n.bit_length() - 1)
    # a training step reads its input, writes a gradient as large and keeps both
    room = max(1, _DRAWN_BYTES // (4 if entry == "train" else 1) // (n * es))
    rows = _log_uniform(rng, 1, min(room, 4096))
    if entry == "argmax":
        j, k_mult = 1, 1
    else:
        j = rng.choice((1, 2, 4))
        k_mult = rng.choice((1, 1, 2, 4, 8))
    # sixteen elements or more for every candidate; k a multiple of 4, so that every j divides it
    k = _log_uniform(rng, 16, max(16, min(n // 16, 65536) // k_mult))
    k = 1 << (k.bit_length() - 1) if n & (n - 1) == 0 else k // 4 * 4
    interleaved = entry != "topk" or rng.random() < 0.75
    data = rng.choice(("normal", "scores", "logits", "trend"))
    return _case(entry, rows, n, dtype, k, j, k_mult, interleaved, data)


def _input(case, generator):
    rows, n = case["rows"], case["n"]
    x = torch.randn(rows, n, generator=generator, device="cuda")
    if case["data"] == "scores":
        x *= 128 ** -0.5
    elif case["data"] == "logits":
        # 12 * rank ^ -1.1, as of a Zipf law, on distinct columns of every row, its own ones
        boosted = max(1, n // 100)
        rank = torch.arange(boosted, device="cuda")
        first = torch.randint(n, (rows, 1), generator=generator, device="cuda")
        columns = (first + 97 * rank) % n
        x.scatter_add_(1, columns, (12.0 * (rank + 1.0) ** -1.1).expand(rows, boosted))
    elif case["data"] == "trend":
        x += torch.linspace(-0.5, 0.5, n, device="cuda")
    return x.to(_DTYPES[case["dtype"]])


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "x": _input(case, generator)}
    if case["entry"] == "train":
        state["x"].requires_grad_()
        state["grad"] = torch.randn(case["rows"], case["k"], generator=generator, device="cuda").to(
            _DTYPES[case["dtype"]])
    return state


def run(state):
    case, x = state["case"], state["x"]
    if case["entry"] == "topk":
        return approx_topk.topk(x, case["k"], -1, j=case["j"], k_mult=case["k_mult"],
                                interleaved=case["interleaved"])
    if case["entry"] == "indices":
        return compact_indices.topk_indices(x, case["k"], -1, j=case["j"], k_mult=case["k_mult"])
    if case["entry"] == "argmax":
        return bucketed_argmax.topk_triton(x, case["k"], -1, case["interleaved"])
    values, indices = differentiable.topk(x, case["k"], -1, j=case["j"], k_mult=case["k_mult"])
    (grad_x,) = torch.autograd.grad(values, x, state["grad"])
    return values.detach(), indices, grad_x


def work(case):
    es = _BYTES[case["dtype"]]
    read = case["rows"] * case["n"] * es
    results = case["rows"] * case["k"]
    total = read + results * (4 if case["entry"] == "indices" else es + 8)
    if case["entry"] == "train":  # the gradient of the values and the indices read, that of the input written
        total += results * (es + 8) + read
    return {"bytes": total, "flops": case["rows"] * case["n"]}  # one comparison an element


def tolerance(case):
    """The selection is a total order (value, then lower index) and copies bits: nothing may differ.
    The gradient moves bits as well, to distinct positions."""
    return "exact"
