"""The work this framework is measured on: ACSR sparse attention through its public entry points.

A case is one pass of a user's program: a forward of ``RegularAttention`` (one fused kernel), the same module as the
reference's three operators (``fused=False``), a training step (``attention_with_grad`` and its gradients), or the ACSR of a
mask that came as a tensor (``create_acsr``).  Sizes are those of the benchmark configurations and of the reference's own
end-to-end script, plus generic small, ragged and odd ones.  Inputs are drawn on the GPU from the seed; the module, with the
metadata of its mask, is what a program keeps between calls.
"""
from __future__ import annotations

import math
import os
import sys

import torch

for _p in (os.getcwd(), os.path.join(os.getcwd(), "triton-fun_amd", "SPLAT")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import acsr_helpers as A  # noqa: E402
from r_attention import RegularAttention, attention_with_grad  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BLOCK = 16  # BLOCK_SIZE_Y / BLOCK_SIZE_X / BLOCK_HEIGHT, as everywhere in the reference


def listed():
    return [
        # One short sequence, one head: a call that is all latency (benchmark configuration 1).
        dict(name="fwd_f32_smallest", op="forward", dtype="f32", pattern="causal", width=64, step=1, B=1, H=1, L=512, d=64,
             layout="rows"),
        # The reference's end-to-end script: batch 32, 12 heads of 64, window 128 to both sides, float32.
        dict(name="fwd_f32_reference", op="forward", dtype="f32", pattern="windowed", width=257, step=1, B=32, H=12, L=1024,
             d=64, layout="rows"),
        # Inference of a mid-sized model in half precision (configuration 2).
        dict(name="fwd_f16_causal", op="forward", dtype="f16", pattern="causal", width=256, step=1, B=4, H=16, L=4096, d=64,
             layout="rows"),
        # Sparse-Transformer rows: a local window and every 128th key before it, two segments (configuration 3).
        dict(name="fwd_bf16_strided", op="forward", dtype="bf16", pattern="strided", width=128, step=128, B=2, H=16, L=8192,
             d=64, layout="rows"),
        # A prompt of a length that no tile divides, K stored as the reference stores it ([B, H, d, L] contiguous).
        dict(name="fwd_bf16_ragged_keys", op="forward", dtype="bf16", pattern="windowed", width=201, step=1, B=2, H=6, L=1037,
             d=128, layout="keys"),
        # The headline: long sequences, heads of 128, causal window 512 (configuration 5).
        dict(name="fwd_bf16_causal_long", op="forward", dtype="bf16", pattern="causal", width=512, step=1, B=4, H=16, L=16384,
             d=128, layout="rows"),
        # The reference's three operators with the compressed matrices in memory (configuration 4's shape).
        dict(name="ops_bf16_dilated", op="operators", dtype="bf16", pattern="dilated", width=512, step=2, B=2, H=32, L=8192,
             d=128, layout="rows"),
        # The operators at a head dimension that the fused kernel has no variant for, and rows of an odd number of slots.
        dict(name="ops_f16_d80_ragged", op="operators", dtype="f16", pattern="windowed", width=129, step=1, B=2, H=8, L=2000,
             d=80, layout="rows"),
        # A training step with heads of 128 (configuration 4's shape): forward, then the gradients of q, k and v.
        dict(name="train_bf16_dilated", op="train", dtype="bf16", pattern="dilated", width=512, step=2, B=2, H=32, L=8192,
             d=128, layout="rows"),
        # A small training step on token-major activations ([B, L, H, d] seen as [B, H, L, d]), ragged length.
        dict(name="train_f16_ragged_tokens", op="train", dtype="f16", pattern="causal", width=200, step=1, B=2, H=4, L=777,
             d=64, layout="tokens"),
        # A training step in full precision.
        dict(name="train_f32_causal", op="train", dtype="f32", pattern="causal", width=128, step=1, B=2, H=8, L=2048, d=64,
             layout="rows"),
        # The mask of a batch of packed documents (every row sees a causal window of its own document), given as a tensor.
        dict(name="build_documents", op="build", width=512, L=8192),
    ]


# ------------------------------------------------------------------------------------------------ what a mask holds

def _patterns(case):
    L, w, s = case["L"], case["width"], case["step"]
    kind = case["pattern"]
    if kind == "causal":
        return A.causal_windowed_pattern(L, w - 1)
    if kind == "windowed":
        return A.windowed_pattern(L, w // 2)
    if kind == "dilated":
        return A.dilated_pattern(L, w, s)
    if kind == "blocked":
        return A.blocked_pattern(L, w // 2)
    return A.strided_patterns(L, w, s)


def _nnz(case):
    """Live entries of the mask, from the patterns' definitions."""
    L, w, s = case["L"], case["width"], case["step"]
    i = torch.arange(L, dtype=torch.int64)
    kind = case["pattern"]
    if kind == "causal":
        n = torch.clamp(i + 1, max=w)
    elif kind == "windowed":
        n = torch.clamp(i + w // 2, max=L - 1) - torch.clamp(i - w // 2, min=0) + 1
    elif kind == "dilated":  # columns i - w*s//2 + s*t, t < w, inside [0, L)
        c0 = i - w * s // 2
        lo = torch.clamp(torch.div(-c0 + s - 1, s, rounding_mode="floor"), min=0)
        hi = torch.clamp(torch.div(L - 1 - c0, s, rounding_mode="floor"), max=w - 1)
        n = torch.clamp(hi - lo + 1, min=0)
    elif kind == "blocked":
        p = w // 2
        b = torch.div(i, p, rounding_mode="floor")
        n = torch.where(b == 0, torch.full_like(i, min(p, L)), torch.clamp((b + 1) * p, max=L) - (b - 1) * p)
    else:  # the local window and the far columns j <= i - w with j % s == s - 1
        n = torch.clamp(i + 1, max=w) + torch.div(torch.clamp(i - w + 1, min=0), s, rounding_mode="floor")
    return int(n.sum())


# ------------------------------------------------------------------------------------------------ drawn cases

def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["forward"] * 4 + ["operators"] * 2 + ["train"] * 3 + ["build"])
    if op == "build":
        return dict(op=op, width=_spread(rng, 32, 1024), L=_spread(rng, 512, 8192))
    case = dict(op=op, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                pattern=rng.choice(["causal", "causal", "windowed", "dilated", "blocked", "strided"]))
    L = _spread(rng, 128, 16384)
    if rng.random() < 0.5:
        L = L // 64 * 64
    width, step = _spread(rng, 16, min(512, L // 2)), 1
    if case["pattern"] == "windowed":
        width |= 1
    elif case["pattern"] == "blocked":
        width = max(32, width // 16 * 16)
    elif case["pattern"] == "dilated":
        step = rng.choice([2, 2, 3, 4])
        width = max(8, min(width, L // (2 * step)))
    elif case["pattern"] == "strided":
        width = min(width, 256)
        step = max(rng.choice([16, 32, 64, 128]), L // 128)
    d = rng.choice([64, 128] if op != "operators" else [32, 64, 64, 80, 96, 128])
    layout = rng.choice(["rows", "rows", "tokens"] + (["keys"] if op != "train" else []))
    case.update(width=width, step=step, B=1, H=1, L=L, d=d, layout=layout)
    # heads: up to the arithmetic of the headline (a step of training and of float32 weighs more) and 1 GB of operands
    weight = {"forward": 1.0, "operators": 2.0, "train": 4.0}[op] * (10.0 if case["dtype"] == "f32" else 1.0)
    most = min(2.0e11 / (weight * 4.0 * d * _nnz(case)), 1.0e9 / (weight * 4.0 * L * d * 2.0), 384.0)
    heads = _spread(rng, 1, max(1.0, most))
    case["H"] = min(heads, rng.choice([4, 8, 12, 16, 32]))
    case["B"] = max(1, heads // case["H"])
    return case


# ------------------------------------------------------------------------------------------------ a pass

def _documents(case, g, dev):
    """Boolean [L, L]: row i sees the last ``width`` positions up to i of its own document; document lengths vary."""
    L = case["L"]
    starts = torch.rand(L, generator=g, device=dev) < 4.0 / max(L, 64) + 1.0 / 1024.0
    starts[0] = True
    pos = torch.arange(L, device=dev)
    first = torch.where(starts, pos, torch.zeros_like(pos)).cummax(0).values
    lo = torch.maximum(first, pos - (case["width"] - 1))
    return (pos[None, :] >= lo[:, None]) & (pos[None, :] <= pos[:, None])


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(int(seed))
    if case["op"] == "build":
        return dict(op="build", mask=_documents(case, g, dev), dev=dev)
    B, H, L, d, dt = case["B"], case["H"], case["L"], case["d"], DTYPES[case["dtype"]]

    def activations(layout):
        if layout == "tokens":  # a projection's output, heads after tokens
            return torch.randn(B, L, H, d, generator=g, device=dev).to(dt).transpose(1, 2)
        return torch.randn(B, H, L, d, generator=g, device=dev).to(dt)
    layout = case["layout"]
    q, k, v = (activations(layout) for _ in range(3))
    attn = RegularAttention(B, L, H, d, _patterns(case), BLOCK, BLOCK, dev, dt, scale=d ** -0.5,
                            fused=case["op"] != "operators")
    if case["op"] == "train":
        grad = activations(layout)
        for t in (q, k, v):
            t.requires_grad_(True)
        return dict(op="train", attn=attn, q=q, k=k, v=v, grad=grad)
    kT = k.transpose(2, 3)
    if layout == "keys":
        kT = kT.contiguous()
    return dict(op=case["op"], attn=attn, x=[q, kT, v])


def run(state):
    if state["op"] == "build":
        # (a program holds the mask as booleans and hands their bytes over)
        return A.create_acsr(state["mask"].view(torch.uint8), BLOCK, state["dev"])
    if state["op"] == "train":
        q, k, v = state["q"], state["k"], state["v"]
        out = attention_with_grad(q, k, v, state["attn"])
        return (out.detach(), *torch.autograd.grad(out, (q, k, v), state["grad"]))
    return state["attn"](state["x"])


def work(case):
    L = case["L"]
    if case["op"] == "build":  # the mask's bytes, five arrays of L and two of L / BLOCK
        return {"bytes": float(L) * L + 20.0 * L + 8.0 * math.ceil(L / BLOCK), "flops": 0.0}
    es = 4 if case["dtype"] == "f32" else 2
    heads, d = case["B"] * case["H"], case["d"]
    dense = float(heads) * L * d * es
    live = float(heads) * _nnz(case)
    if case["op"] == "forward":  # q, k, v read, the output written; two products
        return {"bytes": 4 * dense, "flops": 4.0 * d * live}
    if case["op"] == "operators":  # the same, and the scores and the probabilities written and read
        return {"bytes": 4 * dense + 4 * live * es, "flops": 4.0 * d * live}
    # training: q, k, v and the upstream gradient read, the output and three gradients written; seven products
    return {"bytes": 8 * dense, "flops": 14.0 * d * live}


def tolerance(case):
    if case["op"] == "build":
        return "exact"
    # probabilities (and, in training, score gradients) are rounded to the type between the products; float32 throughout for f32
    return {"rel": {"bf16": 1e-2, "f16": 2e-3, "f32": 1e-5}[case["dtype"]]}
