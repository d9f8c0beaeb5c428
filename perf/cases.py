"""Performance cases of the Sparse-Linear Attention operators on one GPU.

``listed()`` are the workloads the framework is meant for, ``draw(rng)`` gives more of the same ranges; ``prepare``
makes what a user's program holds before the call, ``run`` is one pass through the public entry points.

Kinds of case:
  forward     ``SparseLinearAttention`` under ``no_grad`` (serving a diffusion step)
  train       ``SparseLinearAttention`` forward and backward, gradients of q, k, v and of ``proj_l``
  packed      ``forward_packed`` forward and backward on a packed ``(B, L, 3, H, D)`` projection (a DiT block in training)
  sage        ``SageSparseLinearAttention``, the quantised forward (serving)
  attention   ``_attention.apply`` forward and backward over a map built beforehand (the kernel benchmark's convention)
  complement  ``SparseLinearAttention(..., linear_mode="complement")`` forward and backward
"""
from __future__ import annotations

import math

import torch

from sla_amd import SageSparseLinearAttention, SparseLinearAttention
from sla_amd.inputs import make_proj
from sparse_linear_attention.kernel import _attention
from sparse_linear_attention.utils import get_block_map

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
FRAMES = 21                     # latent frames of the video grids the sequence lengths stand for
TRAINING = ("train", "packed", "attention", "complement")


def listed():
    return [
        # One head pair of a short sequence, 32-bit inputs and the constructor's defaults: a call whose time is latency.
        {"name": "forward_small", "kind": "forward", "B": 1, "H": 2, "L": 1024, "D": 64, "BLKQ": 64, "topk": 0.2,
         "fmap": "softmax", "dtype": "fp32", "structured": False},
        # Self-attention of a small video DiT at inference; the headline configuration.
        {"name": "forward_video", "kind": "forward", "B": 1, "H": 12, "L": 32760, "D": 128, "BLKQ": 64, "topk": 0.05,
         "fmap": "elu", "dtype": "bf16", "structured": True},
        # Two images or short clips at head dimension 64, a length that fills no block.
        {"name": "forward_d64", "kind": "forward", "B": 2, "H": 16, "L": 7813, "D": 64, "BLKQ": 128, "topk": 0.1,
         "fmap": "relu", "dtype": "bf16", "structured": True},
        # The usage example's shape, fine-tuned.
        {"name": "train_example", "kind": "train", "B": 2, "H": 4, "L": 4096, "D": 128, "BLKQ": 64, "topk": 0.2,
         "fmap": "softmax", "dtype": "bf16", "structured": False},
        # Fine-tuning the small video DiT.
        {"name": "train_video", "kind": "train", "B": 1, "H": 12, "L": 32760, "D": 128, "BLKQ": 64, "topk": 0.05,
         "fmap": "elu", "dtype": "bf16", "structured": True},
        # Fine-tuning the large video DiT: the largest call.
        {"name": "train_large", "kind": "train", "B": 1, "H": 40, "L": 75600, "D": 128, "BLKQ": 64, "topk": 0.05,
         "fmap": "relu", "dtype": "bf16", "structured": True},
        # Training at head dimension 64 in half precision, odd length.
        {"name": "train_d64", "kind": "train", "B": 2, "H": 8, "L": 6001, "D": 64, "BLKQ": 64, "topk": 0.1,
         "fmap": "softmax", "dtype": "fp16", "structured": True},
        # A transformer block in training: packed projection in, token-major activations out, 128-row query blocks.
        {"name": "packed_block", "kind": "packed", "B": 1, "H": 12, "L": 9360, "D": 128, "BLKQ": 128, "topk": 0.1,
         "fmap": "softmax", "dtype": "bf16", "structured": True},
        # The quantised operator serving the large model.
        {"name": "sage_large", "kind": "sage", "B": 1, "H": 40, "L": 32760, "D": 128, "BLKQ": 128, "topk": 0.1,
         "fmap": "softmax", "dtype": "bf16", "structured": True},
        # The quantised operator on short, odd sequences at head dimension 64.
        {"name": "sage_d64", "kind": "sage", "B": 2, "H": 8, "L": 5003, "D": 64, "BLKQ": 128, "topk": 0.2,
         "fmap": "elu", "dtype": "bf16", "structured": True},
        # evaluate/bench_kernel.py's shape: the attention operator alone, iid inputs, map built outside.
        {"name": "attention_kernel", "kind": "attention", "B": 2, "H": 16, "L": 32760, "D": 128, "BLKQ": 128,
         "topk": 0.05, "fmap": "", "dtype": "bf16", "structured": False},
        # The variant whose linear branch leaves the selected blocks out, in training.
        {"name": "complement_train", "kind": "complement", "B": 1, "H": 12, "L": 16380, "D": 128, "BLKQ": 64,
         "topk": 0.05, "fmap": "elu", "dtype": "bf16", "structured": True},
    ]


def draw(rng):
    most = work(next(c for c in listed() if c["name"] == "train_large"))["flops"]
    while True:
        kind = rng.choice(("forward", "forward", "train", "train", "packed", "sage", "attention", "complement"))
        D = rng.choice((64, 128, 128))
        L = int(round(math.exp(rng.uniform(math.log(1024), math.log(75600)))))
        BLKQ = 128 if kind == "sage" else rng.choice((64, 64, 128))
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
        if kind in ("forward", "train") and rng.random() < 0.2:
            dtype = "fp32"
        # in half precision the divisors of the elu and relu maps leave the format's range on long sequences
        fmaps = ("softmax",) if dtype == "fp16" else ("elu", "relu", "softmax")
        case = {"kind": kind, "B": rng.choice((1, 1, 2)), "H": rng.choice((2, 4, 8, 12, 16, 24, 40)), "L": L, "D": D,
                "BLKQ": BLKQ, "topk": rng.choice((0.05, 0.1, 0.2) if L >= 4096 else (0.1, 0.2)),
                "fmap": "" if kind == "attention" else rng.choice(fmaps), "dtype": dtype,
                "structured": rng.random() < 0.7}
        if work(case)["flops"] <= 0.25 * most and case["B"] * case["H"] * L * D <= 40 * 75600 * 64:
            return case


def _field(heads, L, D, gen):
    """(heads, L, D) smooth unit-variance field over a FRAMES x rows x columns latent grid of 16:9 frames, flattened and
    cut to L tokens: low-frequency sinusoids with a phase per head and channel, as neighbouring tokens of a video share
    their content."""
    frame = -(-L // FRAMES)
    cols = max(1, math.ceil(math.sqrt(frame * 16 / 9)))
    rows = -(-frame // cols)
    t = torch.arange(L, device="cuda")
    f = (t // (rows * cols)).float() / FRAMES
    y = (t // cols % rows).float() / rows
    x = (t % cols).float() / cols
    modes = ((1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (0, 1, 1), (2, 0, 1))
    field = torch.zeros(heads, L, D, device="cuda")
    for af, ay, ax in modes:
        arg = 2 * math.pi * (af * f + ay * y + ax * x)
        phase = 2 * math.pi * torch.rand(heads, 1, D, device="cuda", generator=gen)
        field += torch.sin(arg.view(1, L, 1) + phase)
    return field / math.sqrt(len(modes) / 2)


def _qkv(case, seed):
    """q, k, v and the gradient of the output, each (B, H, L, D) on the GPU.  Structured inputs: q and k are a shared
    smooth field plus noise (the quantised operator's k also carries a bias per channel, which its smoothing removes);
    v and the gradient are iid normal."""
    B, H, L, D = (case[n] for n in ("B", "H", "L", "D"))
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, device="cuda", generator=gen)

    q = torch.empty(B, H, L, D, device="cuda", dtype=dt)
    k, v, do = torch.empty_like(q), torch.empty_like(q), torch.empty_like(q)
    step = max(1, (1 << 25) // (L * D))                        # heads at a time, so that the 32-bit values stay small
    for b in range(B):
        for h in range(0, H, step):
            n = min(step, H - h)
            if case["structured"]:
                field = _field(n, L, D, gen)
                q[b, h:h + n] = 0.5 * randn(n, L, D) + field
                field += 0.5 * randn(n, L, D)
                if case["kind"] == "sage":
                    field += 2.0 * randn(n, 1, D)
                k[b, h:h + n] = field
            else:
                q[b, h:h + n] = randn(n, L, D)
                k[b, h:h + n] = randn(n, L, D)
            v[b, h:h + n] = randn(n, L, D)
            do[b, h:h + n] = randn(n, L, D)
    return q, k, v, do


def _module(case, seed):
    half = case["dtype"] == "fp16"
    if case["kind"] == "sage":
        mod = SageSparseLinearAttention(case["D"], case["topk"], case["fmap"], use_bf16=not half)
    else:
        mod = SparseLinearAttention(case["D"], case["topk"], case["fmap"], case["BLKQ"], 64, use_bf16=not half,
                                    linear_mode="complement" if case["kind"] == "complement" else "global")
    weight, bias = make_proj(case["D"], seed + 1)
    with torch.no_grad():
        mod.proj_l.weight.copy_(weight)
        mod.proj_l.bias.copy_(bias)
    return mod.cuda()


def prepare(case, seed):
    kind = case["kind"]
    q, k, v, do = _qkv(case, seed)
    state = {"kind": kind, "do": do}
    if kind == "packed":
        # what nn.Linear(dim, 3 * dim) leaves behind; the output's gradient arrives in the same token-major order
        state["qkv"] = torch.stack([t.permute(0, 2, 1, 3) for t in (q, k, v)], dim=2).requires_grad_(True)
        state["do"] = do.permute(0, 2, 1, 3).contiguous()
    else:
        state["q"], state["k"], state["v"] = (t.requires_grad_(kind in TRAINING) for t in (q, k, v))
    if kind == "attention":
        with torch.no_grad():
            state["map"], state["lut"], state["T"] = get_block_map(q, k, topk_ratio=case["topk"], BLKQ=case["BLKQ"])
        state["BLKQ"] = case["BLKQ"]
    else:
        state["mod"] = _module(case, seed)
    if kind not in TRAINING:
        del state["do"]
    return state


def run(state):
    kind = state["kind"]
    if kind in ("forward", "sage"):
        with torch.no_grad():
            return state["mod"](state["q"], state["k"], state["v"])
    if kind == "packed":
        inputs = [state["qkv"]]
        out = state["mod"].forward_packed(state["qkv"])
    elif kind == "attention":
        inputs = [state["q"], state["k"], state["v"]]
        out = _attention.apply(*inputs, state["map"], state["lut"], state["T"], state["BLKQ"], 64)
    else:
        inputs = [state["q"], state["k"], state["v"]]
        out = state["mod"](*inputs)
    if kind != "attention":
        inputs += [state["mod"].proj_l.weight, state["mod"].proj_l.bias]
    grads = torch.autograd.grad(out, inputs, state["do"])
    return {"out": out.detach(), "grads": list(grads)}


def work(case):
    """Floating-point operations of the matrix products (the selected tiles, and the linear branch through its D x D
    states) and bytes of the tensors that go in and come out."""
    B, H, L, D = (case[n] for n in ("B", "H", "L", "D"))
    blocks = -(-L // 64)
    selected = min(blocks, int(case["topk"] * blocks))
    tensor = B * H * L * D
    training = case["kind"] in TRAINING
    tile = 2.0 * B * H * L * min(L, selected * 64) * D          # one product over the selected tiles
    state = 2.0 * tensor * D                                    # one product with a D x D state
    flops = tile * (7 if training else 2)                       # backward: S again, dP, dV, dQ, dK
    if case["kind"] != "attention":
        flops += state * (6 if training else 2)                 # backward: d(phi q), d(state), d(phi k), dV
    size = 4 if case["dtype"] == "fp32" else 2
    return {"bytes": float(tensor * size * (8 if training else 4)), "flops": flops}


def tolerance(case):
    # Four times the relative error measured against 64-bit arithmetic over the same selected blocks (lengths up to 2000):
    # bf16 at most 5.7e-3 (dq of structured inputs, a difference of sums), fp16 at most 6.5e-4; the quantised operator
    # against exact attention over the same quantised q, k, v at most 1.8e-2 (probabilities rounded to e4m3).
    if case["kind"] == "sage":
        return {"rel": 0.07}
    return {"rel": 0.0025 if case["dtype"] == "fp16" else 0.02}
