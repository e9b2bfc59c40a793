"""The workloads whose speed and results are measured: calls of `tattn.attention` as training and
inference programs make them, over the sizes, layouts, element types and masks that the tests
and the benchmark of this repository use.

A case: batch `z`, heads `h`, sequence length `n`, head dim `d`, `dtype`, `causal`, `layout`
("heads": [z, h, n, d] tensors; "tokens": views of [z, n, h, d] activations, as a projection
leaves them) and `train` (forward and backward, returning O and the three gradients; otherwise
the forward alone without autograd).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "triton-attn_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from tattn import attention  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

# Counted operations of the largest listed case: no drawn case costs more.
MOST_FLOPS = 14 * 16 * 16384 * 16384 * 64
# One fp32 product takes the matrix cores about as long as sixteen 16-bit ones.
FP32_WEIGHT = 16


def _case(name, z, h, n, d, dtype, causal, train, layout="heads"):
    return {"name": name, "z": z, "h": h, "n": n, "d": d, "dtype": dtype, "causal": causal, "train": train,
            "layout": layout}


def listed():
    return [
        # A single small call: two sequences of 128 tokens in float32. Latency of one launch.
        _case("fp32_small_forward", 2, 4, 128, 64, "fp32", False, False),
        # The smallest training call: 70 tokens, 3 heads, activations as the projection leaves them.
        _case("fp16_small_train", 2, 3, 70, 32, "fp16", True, True, "tokens"),
        # Attention over very many short rows: 65,536 (batch, head) pairs of 24 tokens.
        _case("fp16_many_short_rows_train", 1024, 64, 24, 16, "fp16", False, True),
        # The benchmark's shortest rows, trained with a causal mask.
        _case("fp16_512_causal_train", 32, 16, 512, 64, "fp16", True, True),
        # The benchmark's middle length, trained without a mask.
        _case("fp16_4096_train", 4, 16, 4096, 64, "fp16", False, True),
        # The benchmark's longest rows: the costliest training call.
        _case("fp16_16384_train", 1, 16, 16384, 64, "fp16", False, True),
        # Causal prefill of one 2,048-token prompt: few rows, one sequence, no gradients.
        _case("bf16_prompt_forward", 1, 16, 2048, 64, "bf16", True, False, "tokens"),
        # The benchmark's middle length as a causal forward.
        _case("fp16_4096_causal_forward", 4, 16, 4096, 64, "fp16", True, False),
        # Odd sizes: 11 sequences of 1,500 tokens, 12 heads, trained with a causal mask.
        _case("fp16_ragged_causal_train", 11, 12, 1500, 64, "fp16", True, True, "tokens"),
        # Head dim 128 in bfloat16, as large language models train it.
        _case("bf16_d128_causal_train", 2, 16, 4096, 128, "bf16", True, True, "tokens"),
        # Full-precision training.
        _case("fp32_1024_train", 4, 16, 1024, 64, "fp32", False, True),
        # Small heads in bfloat16, without a mask.
        _case("bf16_d32_train", 16, 16, 1000, 32, "bf16", False, True),
    ]


def _flops(case):
    f = 4.0 * case["z"] * case["h"] * case["n"] ** 2 * case["d"] * (0.5 if case["causal"] else 1.0)
    return f * (3.5 if case["train"] else 1.0)


def draw(rng):
    dtype = rng.choice(["fp16", "fp16", "fp16", "bf16", "bf16", "bf16", "fp32"])
    d = rng.choice([16, 32, 64, 64, 64, 64, 128, 128])
    longest = 4096 if dtype == "fp32" else 16384
    n = round(math.exp(rng.uniform(math.log(16), math.log(longest))))
    if rng.random() < 0.5 and n > 128:  # half of the longer rows in whole blocks, half as they come
        n = max(128, round(n / 128) * 128)
    h = rng.choice([1, 3, 4, 8, 12, 16, 16, 32])
    tokens = math.exp(rng.uniform(math.log(max(n, 1024)), math.log(max(2 * n, 32768))))
    z = max(1, round(tokens / n))
    case = {"z": z, "h": h, "n": n, "d": d, "dtype": dtype, "causal": rng.random() < 0.5,
            "train": rng.random() < 0.6, "layout": rng.choice(["heads", "heads", "tokens"])}
    weight = FP32_WEIGHT if dtype == "fp32" else max(1, 64 // d)  # narrow heads: the exponentials bound them
    while _flops(case) * weight > MOST_FLOPS * 0.9 and (case["z"] > 1 or case["h"] > 1):
        if case["z"] > 1:
            case["z"] -= max(1, case["z"] // 8)
        else:
            case["h"] -= 1
    return case


def _inputs(case, seed):
    """q, k, v and dO as [z, h, n, d] values drawn N(0, 1), in the case's layout."""
    z, h, n, d = case["z"], case["h"], case["n"], case["d"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (z, n, h, d) if case["layout"] == "tokens" else (z, h, n, d)
    return [torch.randn(shape, device="cuda", dtype=DTYPES[case["dtype"]], generator=g) for _ in range(4)]


def prepare(case, seed):
    q, k, v, do = _inputs(case, seed)
    if case["train"]:
        for t in (q, k, v):
            t.requires_grad_()
    return {"q": q, "k": k, "v": v, "do": do, "causal": case["causal"], "train": case["train"],
            "tokens": case["layout"] == "tokens"}


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    if state["tokens"]:
        o = attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), causal=state["causal"]).transpose(1, 2)
    else:
        o = attention(q, k, v, causal=state["causal"])
    if not state["train"]:
        return {"o": o}
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    elements = case["z"] * case["h"] * case["n"] * case["d"]
    # Forward: q, k, v in and O out. Training: dO in and the three gradients out as well (O and
    # the row statistics stay a matter of the implementation).
    return {"bytes": float(elements * size * (8 if case["train"] else 4)), "flops": _flops(case)}


def tolerance(case):
    # Measured against `exact` over the listed and drawn cases and stated at about four times:
    # fp16 3.4e-4, bf16 2.7e-3, fp32 7.6e-7 at most.
    return {"rel": {"fp16": 1.4e-3, "bf16": 1.1e-2, "fp32": 3e-6}[case["dtype"]]}


def exact(case, seed):
    """Attention and its gradients in float64 from the materialised probabilities, head by head."""
    scale = 1.0 / math.sqrt(case["d"])
    q, k, v, do = _inputs(case, seed)
    if case["layout"] == "tokens":
        q, k, v, do = (t.transpose(1, 2) for t in (q, k, v, do))
    n = case["n"]
    flat = [t.reshape(-1, n, case["d"]) for t in (q, k, v, do)]
    outs = [torch.empty(flat[0].shape, dtype=torch.float64, device="cuda") for _ in range(4 if case["train"] else 1)]
    heads = max(1, (1 << 27) // (n * n))  # slices at a time: about 1 GB per n x n matrix
    hidden = torch.ones(n, n, dtype=torch.bool, device="cuda").triu_(1) if case["causal"] else None
    for s in range(0, flat[0].shape[0], heads):
        a, b, c, g = (t[s:s + heads].double() for t in flat)
        p = torch.matmul(a, b.transpose(1, 2).contiguous()).mul_(scale)
        if hidden is not None:
            p.masked_fill_(hidden, -math.inf)
        p = torch.softmax(p, dim=-1)
        o = torch.matmul(p, c)
        outs[0][s:s + heads] = o
        if not case["train"]:
            continue
        outs[3][s:s + heads] = torch.matmul(p.transpose(1, 2).contiguous(), g)
        ds = torch.matmul(g, c.transpose(1, 2).contiguous()).sub_((g * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
        del p
        outs[1][s:s + heads] = torch.matmul(ds, b)
        outs[2][s:s + heads] = torch.matmul(ds.transpose(1, 2).contiguous(), a)
        del ds
    outs = [t.reshape(q.shape) for t in outs]
    if case["layout"] == "tokens":
        outs = [t.transpose(1, 2).contiguous() for t in outs]
    return dict(zip(("o", "dq", "dk", "dv"), outs))
