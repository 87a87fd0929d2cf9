"""What is timed: the work that a user of this package has it do, through its public entry points.

Three entry points carry it: the sparse MoE block (router, expert sort, three expert projections, combine) in
inference with bf16 or 4-bit expert weights and in training; the same block with LoRA adapters through the fast-LoRA
forward; and ``moe_fused_linear`` by itself, forward and backward.  Unless a case says otherwise the sizes are those
of this repository's benchmark: 128 experts, 8 per token, hidden 2048, intermediate 768, bf16.

A case is a dict of plain values:

* ``kind``   "block" (forward under ``no_grad``), "train" (block, forward and backward), "lora" (the block with
             adapters through the fast-LoRA forward, forward and backward), "linear" (``moe_fused_linear``, forward and
             backward);
* ``tokens`` (block, train, lora) or ``rows`` (linear), ``experts``, ``top_k``, ``hidden``, ``inter``; for "linear" the
             operand is (rows, hidden) and the weight (experts, inter, hidden);
* ``weights`` "bf16", "fp32", "nf4" (blocks of 64, fp32 scales) or "nf4dq" (the scales quantised once more to 8 bits,
             the 4-bit layer's default); activations are fp32 with "fp32" and bf16 otherwise;
* ``zipf``   exponent of the experts' popularity (0: near-uniform);
* ``rank``   rank of the adapters ("lora").
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "transformers-qwen3-moe-fused_amd"))

from qwen3_moe_fused.fast_lora import fast_Qwen3MoeFusedSparseMoeBlock_forward  # noqa: E402
from qwen3_moe_fused.functional import moe_fused_linear  # noqa: E402
from qwen3_moe_fused.lora import LoraMoeFusedLinear  # noqa: E402
from qwen3_moe_fused.modular_qwen3_moe_fused import MoeFusedLinear, Qwen3MoeFusedSparseMoeBlock  # noqa: E402
from qwen3_moe_fused.quantize.layer import MoeFusedLinear4bit  # noqa: E402

DEV = "cuda"
PROJECTIONS = ("gate_proj", "up_proj", "down_proj")
WEIGHT_STD = 0.02
# the hidden states' first channel is a constant of this size (real hidden states have a few such channels): with
# the router's first column the experts' log-popularity over it, the routing is skewed
MASSIVE = 8.0


def _case(name, kind, tokens, weights, experts=128, top_k=8, hidden=2048, inter=768, zipf=0.0, rank=0):
    return {"name": name, "kind": kind, "tokens": tokens, "weights": weights, "experts": experts, "top_k": top_k,
            "hidden": hidden, "inter": inter, "zipf": zipf, "rank": rank}


def listed():
    return [
        # one user, one token at a time, on the 4-bit layer's default format
        _case("decode_1_nf4dq", "block", 1, "nf4dq"),
        # a small decode batch on packed weights (benchmark configuration 5)
        _case("decode_16_nf4", "block", 16, "nf4"),
        # a decode batch on unquantised weights
        _case("decode_32_bf16", "block", 32, "bf16"),
        # a large decode batch, or a short prompt, on the 4-bit layer's default format
        _case("serve_256_nf4dq", "block", 256, "nf4dq"),
        # a long prompt on packed weights (benchmark configuration 5)
        _case("prefill_16384_nf4", "block", 16384, "nf4"),
        # a prompt of no round length on unquantised weights
        _case("prefill_3001_bf16", "block", 3001, "bf16"),
        # full fine-tuning: one training step of the block (benchmark configurations 2 and 3)
        _case("train_4096_bf16", "train", 4096, "bf16"),
        # LoRA fine-tuning with skewed routing (benchmark configuration 4)
        _case("lora_8192_zipf", "lora", 8192, "bf16", zipf=1.2, rank=16),
        # QLoRA fine-tuning on the 4-bit layer's default format
        _case("qlora_2048_nf4dq", "lora", 2048, "nf4dq", rank=16),
        # the library's own operator, forward and backward, in bf16 (the down projection of configuration 3)
        _case("linear_32768_bf16", "linear", 32768, "bf16", hidden=768, inter=2048),
        # the same in float32, at the size of the tests and benchmarks that check the kernels
        _case("linear_1024_fp32", "linear", 1024, "fp32"),
        # the smallest call: one training step of a toy block in float32 (benchmark configuration 1)
        _case("toy_256_fp32", "train", 256, "fp32", experts=8, top_k=2, hidden=64, inter=128),
    ]


def draw(rng):
    """The ranges: 1 to 16384 tokens in inference, 64 to 8192 in training (4096 for all weights), 64 to 32768 rows of
    the operator (4096 in float32); half of the drawn cases at the benchmark's sizes, the others with 8 to 160 experts,
    hidden 512 to 4096 and intermediate 256 to 1536 in steps of 32, as expert models have them, and in float32 also
    sizes that are a multiple of nothing."""

    def log_between(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    most = max(_cost(c) for c in listed())
    while True:
        kind, weights = rng.choice((("block", "nf4"), ("block", "nf4dq"), ("block", "bf16"), ("block", "bf16"),
                                    ("train", "bf16"), ("train", "fp32"), ("lora", "bf16"), ("lora", "nf4"),
                                    ("lora", "nf4dq"), ("linear", "bf16"), ("linear", "bf16"), ("linear", "fp32")))
        c = {"kind": kind, "tokens": 0, "weights": weights, "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768,
             "zipf": 0.0, "rank": rng.choice((8, 16, 32)) if kind == "lora" else 0}
        if rng.random() < 0.5 or (kind, weights) == ("train", "fp32"):
            c["experts"] = rng.choice((8, 16, 60, 64, 96, 128, 160))
            c["top_k"] = rng.choice((1, 2, 4, 6, 8))
            c["hidden"], c["inter"] = 32 * log_between(16, 128), 32 * log_between(8, 48)
        if (kind, weights) == ("linear", "bf16") and rng.random() < 0.5:
            c["hidden"], c["inter"] = c["inter"], c["hidden"]
        if kind == "block":
            c["tokens"] = log_between(1, 16384)
        elif weights == "fp32":
            c["tokens"] = log_between(64, 4096 if kind == "linear" else 512)
            c["hidden"] += rng.choice((0, 0, 1, 4, 7))
            if kind == "train":
                c["hidden"], c["inter"] = max(16, c["hidden"] // 8), max(16, c["inter"] // 8)
        elif kind == "linear":
            c["tokens"] = log_between(64, 32768)
        else:
            c["tokens"] = log_between(64, 4096 if kind == "train" else 8192)
        if kind != "linear" and rng.random() < 0.3:
            c["zipf"] = round(rng.uniform(0.5, 1.3), 2)
        if _cost(c) <= most:
            return c


def _cost(c):
    """Rough time of a pass: the bytes and operations of ``work``, float32 operations at the rate of its units."""
    w = work(c)
    return w["bytes"] / 5e12 + w["flops"] / (1e14 if c["weights"] == "fp32" else 8e14)


def _routed_experts(c):
    """Experts that are expected to get rows."""
    e, rows = c["experts"], c["tokens"] * (1 if c["kind"] == "linear" else c["top_k"])
    if c["zipf"]:
        p = [(i + 1.0) ** -c["zipf"] for i in range(e)]
        p = [v / sum(p) for v in p]
    else:
        p = [1.0 / e] * e
    return sum(1.0 - (1.0 - v) ** rows for v in p)


def work(case):
    c = case
    size = 4 if c["weights"] == "fp32" else 2
    h, i, e, r = c["hidden"], c["inter"], c["experts"], c["rank"]
    hit = _routed_experts(c)
    per_weight = {"bf16": 2.0, "fp32": 4.0, "nf4": 0.5 + 4.0 / 64, "nf4dq": 0.5 + 1.0 / 64}[c["weights"]]
    if c["kind"] == "linear":
        # x, dy in; y, dx out; the weights once, their gradient once
        io = size * c["tokens"] * 2 * (h + i)
        return {"bytes": io + hit * h * i * per_weight + e * h * i * size, "flops": 6.0 * c["tokens"] * h * i}
    rows = c["tokens"] * c["top_k"]
    router = 2.0 * c["tokens"] * h * e
    flops = 6.0 * rows * h * i + router
    nbytes = size * (2 * c["tokens"] * h + e * h + c["tokens"] * e) + 3 * hit * h * i * per_weight
    if c["kind"] == "train":
        flops *= 3
        nbytes += size * (2 * c["tokens"] * h + e * h) + 3 * e * h * i * size
    elif c["kind"] == "lora":
        # frozen base weights: the input gradients of the three projections and of the router; adapters both ways
        adapters = 3 * r * (h + i)
        flops += 6.0 * rows * h * i + 2 * router + 6.0 * rows * adapters
        nbytes += size * (2 * c["tokens"] * h + e * h) + size * e * 2 * adapters
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance of the path's results from the same path in float64 (given its routing): the
    operator rounds once, 0.0017 of the norm and 0.004 of a value; the block's chain of roundings comes to 0.0047 to
    0.0068 of the norm and up to 0.16 of a value (gradients of experts with few rows); float32 sums to 8e-7 and 5e-6.
    Two implementations that both round differ by as much as sqrt(2) times that."""
    if case["weights"] == "fp32":
        return {"rel": 4e-6, "max": 4e-5}
    if case["kind"] == "linear":
        return {"rel": 6e-3, "max": 0.02}
    return {"rel": 2e-2, "max": 0.5 if case["kind"] == "lora" else 0.3}


def _normal(g, shape, dtype, std=1.0):
    return torch.empty(shape, device=DEV, dtype=dtype).normal_(0.0, std, generator=g)


def _expert_weight(g, c, out_features, in_features):
    """A projection with weights from N(0, 0.02)."""
    dtype = torch.float32 if c["weights"] == "fp32" else torch.bfloat16
    w = torch.nn.Parameter(_normal(g, (c["experts"], out_features, in_features), dtype, WEIGHT_STD))
    if c["weights"] in ("nf4", "nf4dq"):
        return MoeFusedLinear4bit(in_features, out_features, c["experts"], weight=w, quant_type="nf4",
                                  compute_dtype=torch.bfloat16, compress_statistics=c["weights"] == "nf4dq",
                                  device="meta").to(DEV)
    proj = MoeFusedLinear(in_features, out_features, c["experts"], device="meta")
    proj.weight = w
    return proj


def _routing(g, c):
    """(hidden, router weight): logits of about unit variance, plus the experts' log-popularity."""
    dtype = torch.float32 if c["weights"] == "fp32" else torch.bfloat16
    x = _normal(g, (1, c["tokens"], c["hidden"]), dtype)
    w = _normal(g, (c["experts"], c["hidden"]), torch.float32, c["hidden"] ** -0.5)
    if c["zipf"]:
        order = torch.randperm(c["experts"], device=DEV, generator=g)
        x[..., 0] = MASSIVE
        w[:, 0] = -c["zipf"] * torch.log(order.float() + 1.0) / MASSIVE
    return x, w.to(dtype)


def prepare(case, seed):
    c = case
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype = torch.float32 if c["weights"] == "fp32" else torch.bfloat16
    if c["kind"] == "linear":
        # every row's expert drawn uniformly, rows sorted by expert
        sel = torch.randint(0, c["experts"], (c["tokens"],), device=DEV, generator=g)
        return {"kind": "linear", "m_sizes": torch.bincount(sel, minlength=c["experts"]).to(torch.int32),
                "x": _normal(g, (c["tokens"], c["hidden"]), dtype).requires_grad_(),
                "w": _normal(g, (c["experts"], c["inter"], c["hidden"]), dtype, WEIGHT_STD).requires_grad_(),
                "dy": _normal(g, (c["tokens"], c["inter"]), dtype)}
    with torch.device("meta"):
        block = Qwen3MoeFusedSparseMoeBlock(SimpleNamespace(
            num_experts=c["experts"], num_experts_per_tok=c["top_k"], norm_topk_prob=True, hidden_size=c["hidden"],
            moe_intermediate_size=c["inter"], hidden_act="silu"))
    hidden, router = _routing(g, c)
    block.gate.weight = torch.nn.Parameter(router)
    for name in PROJECTIONS:
        out_f, in_f = (c["hidden"], c["inter"]) if name == "down_proj" else (c["inter"], c["hidden"])
        proj = _expert_weight(g, c, out_f, in_f)
        if c["kind"] == "lora":
            proj.weight.requires_grad_(False)
            with torch.device(DEV):  # where the adapter's parameters are made
                proj = LoraMoeFusedLinear(proj, "default", r=c["rank"], lora_alpha=2 * c["rank"])
            with torch.no_grad():
                for p in list(proj.lora_A.values()) + list(proj.lora_B.values()):
                    p.weight = torch.nn.Parameter(_normal(g, p.weight.shape, dtype, 0.01))
        setattr(block, name, proj)
    state = {"kind": c["kind"], "block": block, "hidden": hidden}
    if c["kind"] != "block":
        hidden.requires_grad_()
        state["dout"] = _normal(g, hidden.shape, dtype)
    return state


def run(state):
    if state["kind"] == "block":
        with torch.no_grad():
            return state["block"](state["hidden"])
    if state["kind"] == "linear":
        x, w = state["x"], state["w"]
        x.grad = w.grad = None
        y = moe_fused_linear(x, w, state["m_sizes"])
        y.backward(state["dy"])
        return y.detach(), x.grad, w.grad
    block, hidden = state["block"], state["hidden"]
    block.zero_grad(set_to_none=True)
    hidden.grad = None
    if state["kind"] == "lora":
        out, logits = fast_Qwen3MoeFusedSparseMoeBlock_forward(block, hidden)
    else:
        out, logits = block(hidden)
    out.backward(state["dout"])
    return {"out": out.detach(), "logits": logits.detach(), "hidden.grad": hidden.grad,
            **{name: p.grad for name, p in block.named_parameters() if p.grad is not None}}
