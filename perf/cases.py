"""What the performance of this framework is measured on: the calls that a serving or training program makes.

A case is a dict of plain values.  ``kind`` names the program:

``ffn``      the quantized expert FFN on activations that arrive int8 per token (``MoeFfnW8A8.forward``): what an inference
             engine with a W8A8 checkpoint runs in every layer.
``layer``    the whole MoE layer operator by operator, from 16-bit hidden states and fp32 router logits: gating top-k,
             routing with dynamic quantisation, the two grouped GEMMs and the combine with the shared expert's rows added.
``permute``  token permutation and combine around experts of the caller's own (16-bit rows, capacity per expert with
             dropped and padded rows): what a program with unquantized experts, a training step among them, uses.

Shapes: those of ``synth.CONFIGS`` (DeepSeek-V3-, Mixtral- and Qwen3-MoE-shaped, and the small one) and generic ones whose
inner sizes are no multiples of 128, as tensor-parallel shards of an expert have.  Values are those of the measurement
plan: N(0, 1) hidden states quantized per token, uniform int8 weights, N(0, 1) router logits (``skew``: Zipf popularity).
"""
import math

import torch

from __graft_entry__ import load_package

pkg = load_package()
aclnn = pkg.aclnn


def _ffn(name, tokens, hidden, inter, experts, top_k, skew=0.0, routing="v2", weights="k_major", out="bf16"):
    return {"name": name, "kind": "ffn", "tokens": tokens, "hidden": hidden, "inter": inter, "experts": experts,
            "top_k": top_k, "skew": skew, "routing": routing, "weights": weights, "out": out}


def _layer(name, tokens, hidden, inter, experts, top_k, skew=0.0, dtype="bf16", quant="v3", shared=True):
    return {"name": name, "kind": "layer", "tokens": tokens, "hidden": hidden, "inter": inter, "experts": experts,
            "top_k": top_k, "skew": skew, "dtype": dtype, "quant": quant, "shared": shared}


def _permute(name, tokens, hidden, experts, top_k, skew=0.0, dtype="bf16", capacity_factor=1.25):
    return {"name": name, "kind": "permute", "tokens": tokens, "hidden": hidden, "experts": experts, "top_k": top_k,
            "skew": skew, "dtype": dtype, "capacity_factor": capacity_factor}


def listed():
    return [
        # one user's next token: every launch and every host microsecond shows
        _ffn("decode_1_token", 1, 4096, 1536, 128, 8),
        # a small model, or a short prompt through one expert-parallel rank: latency
        _ffn("small_256_tokens", 256, 1024, 1024, 8, 2),
        # a decode step of a serving batch: the touched experts' weights are streamed once for a handful of rows each
        _ffn("decode_64_tokens", 64, 4096, 1536, 128, 8),
        # the same step from hidden states and router logits, fp16, with a ragged batch
        _layer("layer_decode_23_tokens", 23, 4096, 1536, 128, 8, dtype="fp16", quant="quant_v2"),
        # decode on an expert-parallel rank that holds 64 experts in the blocked weight layout
        _ffn("decode_blocked_weights", 100, 7168, 2048, 64, 8, routing="v3", weights="nz"),
        # inner sizes off the 128 grid, a ragged batch
        _ffn("ragged_sizes", 301, 2880, 1440, 32, 4),
        # a prompt chunk on plain row-major weights, fp16 out
        _ffn("chunk_row_major_weights", 1000, 4096, 14336, 8, 2, routing="v3", weights="row_major", out="fp16"),
        # a whole layer over a prompt
        _layer("layer_prefill", 2047, 4096, 1536, 128, 8),
        # prefill with many experts: each sees about 128 rows, bound by memory
        _ffn("prefill_many_experts", 4096, 7168, 2048, 256, 8),
        # prefill with few experts of thousands of rows: bound by the matrix cores; the largest case
        _ffn("prefill_few_experts", 16384, 4096, 14336, 8, 2),
        # the load imbalance of real routers: one expert with thirty times the mean, a third of them idle
        _ffn("prefill_skewed", 8192, 7168, 2048, 256, 8, skew=1.2),
        # permutation and combine around unquantized experts with a capacity
        _permute("permute_with_capacity", 4096, 7168, 64, 8, skew=0.6),
    ]


# The largest listed case costs this much; drawn ones stay below it.
_MAX_OPS = 6 * 16384 * 2 * 4096 * 14336
_MAX_WEIGHT_BYTES = 3 * 256 * 7168 * 2048
_MAX_ROW_BYTES = 4096 * 8 * 7168 * 2


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng):
    """(hidden, inter, experts, top_k): one of the repository's, or a generic one on a grid of 64 or of 32."""
    if rng.random() < 0.5:
        return rng.choice([(1024, 1024, 8, 2), (7168, 2048, 256, 8), (7168, 2048, 64, 8), (4096, 14336, 8, 2), (4096, 1536, 128, 8)])
    while True:
        grid = rng.choice([32, 64, 128, 256])
        hidden = max(1024, _log_uniform(rng, 1024, 7168) // grid * grid)
        inter = max(512, _log_uniform(rng, 512, 14336) // grid * grid)
        experts = rng.choice([8, 16, 32, 60, 64, 128, 160, 256])
        top_k = rng.choice([2, 4, 6, 8])
        if 3 * experts * hidden * inter <= _MAX_WEIGHT_BYTES:
            return hidden, inter, experts, top_k


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "ffn", "layer", "layer", "permute"])
    while True:
        hidden, inter, experts, top_k = _shape(rng)
        tokens = _log_uniform(rng, 1, 16384)
        rows = tokens * top_k
        if kind == "permute":
            tokens = max(tokens, 16)
            if rows * hidden * 2 <= _MAX_ROW_BYTES:
                break
        elif 6 * rows * hidden * inter <= _MAX_OPS and rows * hidden <= 65536 * 7168:
            break
    skew = rng.choice([0.0, 0.0, 0.6, 1.2]) if experts >= 32 else 0.0
    if kind == "permute":
        case = _permute("", tokens, hidden, experts, top_k, skew, rng.choice(["bf16", "bf16", "fp16"]), rng.choice([1.0, 1.25, 2.0]))
    elif kind == "layer":
        case = _layer("", tokens, hidden, inter, experts, top_k, skew, rng.choice(["bf16", "bf16", "fp16"]),
                      rng.choice(["v3", "v3", "quant_v2"]), rng.random() < 0.5)
    else:
        weights = rng.choice(["k_major", "k_major", "k_major", "nz", "row_major"])
        case = _ffn("", tokens, hidden, inter, experts, top_k, skew, rng.choice(["v2", "v2", "v3"]), weights,
                    rng.choice(["bf16", "bf16", "fp16"]))
    del case["name"]
    return case


_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _logits(case, device, generator):
    """Router logits fp32 [tokens, experts]."""
    experts = case["experts"]
    logits = torch.randn((case["tokens"], experts), device=device, generator=generator)
    if case["skew"] > 0:
        rank = torch.randperm(experts, device=device, generator=generator).float() + 1
        logits -= case["skew"] * torch.log(rank)
    return logits


def _top_k(case, logits):
    weight, idx = torch.topk(torch.softmax(logits, dim=1), case["top_k"], dim=1)
    return idx.int().contiguous(), (weight / weight.sum(dim=1, keepdim=True)).contiguous()


def _capacity(case):
    mean = case["tokens"] * case["top_k"] / case["experts"]
    return min(case["tokens"], max(1, math.ceil(case["capacity_factor"] * mean)))


def prepare(case, seed):
    device = torch.device("cuda")
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    tokens, hidden, experts = case["tokens"], case["hidden"], case["experts"]
    state = {"case": case}
    logits = _logits(case, device, g)
    if case["kind"] == "permute":
        state["x"] = torch.randn((tokens, hidden), device=device, generator=g).to(_DTYPES[case["dtype"]])
        state["residual"] = torch.randn((tokens, hidden), device=device, generator=g).to(_DTYPES[case["dtype"]])
        idx, weight = _top_k(case, logits)
        state["idx"], state["weight"], state["capacity"] = idx, weight.to(_DTYPES[case["dtype"]]), _capacity(case)
        return state
    inter = case["inter"]
    w13 = torch.empty((experts, 2 * inter, hidden), dtype=torch.int8, device=device).random_(-127, 128, generator=g)
    w2 = torch.empty((experts, hidden, inter), dtype=torch.int8, device=device).random_(-127, 128, generator=g)
    w13_scale = torch.empty((experts, 2 * inter), device=device).uniform_(1e-3, 1e-2, generator=g)
    w2_scale = torch.empty((experts, hidden), device=device).uniform_(1e-3, 1e-2, generator=g)
    if case["kind"] == "layer":
        dtype = _DTYPES[case["dtype"]]
        state["x"] = torch.randn((tokens, hidden), device=device, generator=g).to(dtype)
        state["logits"] = logits
        state["shared"] = torch.randn((tokens, hidden), device=device, generator=g).to(dtype) if case["shared"] else None
        # channel scales that keep the experts' rows at the magnitude of the hidden states, well inside fp16's range
        state["weights"] = (w13.transpose(1, 2), w13_scale * 0.05, w2.transpose(1, 2), w2_scale * 0.05)
        return state
    x = torch.randn((tokens, hidden), device=device, generator=g).bfloat16().float()
    x_scale = x.abs().amax(dim=1) / 127.0
    state["xq"] = torch.clamp(torch.round(x / x_scale[:, None]), -127, 127).to(torch.int8)
    state["x_scale"] = x_scale
    state["idx"], state["weight"] = _top_k(case, logits)
    if case["out"] == "fp16":
        w13_scale *= 0.05
        w2_scale *= 0.05
        state["weight"] = state["weight"].half()
    state["ffn"] = pkg.MoeFfnW8A8(w13, w13_scale, w2, w2_scale, out_dtype=_DTYPES[case["out"]], routing=case["routing"],
                                  weight_nz=case["weights"] == "nz", weight_row_major=case["weights"] == "row_major")
    return state


def _run_layer(case, s):
    experts, top_k = case["experts"], case["top_k"]
    w13, w13_scale, w2, w2_scale = s["weights"]
    weight, idx, _ = aclnn.moe_gating_top_k_softmax_v2(s["logits"], top_k, renorm=1)
    if case["quant"] == "v3":
        rows, row_idx, counts, row_scale = aclnn.moe_init_routing_v3(s["x"], idx, expert_num=experts, expert_tokens_num_type=0,
                                                                     quant_mode=1)
    else:
        rows, row_idx, counts, _, row_scale = aclnn.moe_init_routing_quant_v2(
            s["x"], idx, 1, expert_num=experts, expert_tokens_count_or_cumsum_flag=1)
    h, h_scale = aclnn.grouped_matmul_swiglu_quant(rows, w13, counts, w13_scale, row_scale)
    y = torch.empty((rows.shape[0], case["hidden"]), dtype=_DTYPES[case["dtype"]], device=rows.device)
    aclnn.grouped_matmul_v4([h], [w2], scale=[w2_scale], per_token_scale=[h_scale], group_list=counts, split_item=3,
                            group_type=0, group_list_type=0, act_type=0, out=[y])
    out = aclnn.moe_finalize_routing_v2(y, row_idx, x1=s["shared"], scales=weight.half() if y.dtype == torch.float16 else weight,
                                        drop_pad_mode=2)
    return {"out": out, "weight": weight, "idx": idx}


def _run_permute(case, s):
    experts = case["experts"]
    rows, row_idx, _, counts = aclnn.moe_init_routing_v2(s["x"], s["idx"], 0, s["capacity"], experts, 1, 0, True)
    out = aclnn.moe_finalize_routing_v2(rows, row_idx, x1=s["residual"], scales=s["weight"], drop_pad_mode=3)
    return {"rows": rows, "row_idx": row_idx, "counts": counts, "out": out}


def run(state):
    case = state["case"]
    if case["kind"] == "layer":
        return _run_layer(case, state)
    if case["kind"] == "permute":
        return _run_permute(case, state)
    return state["ffn"].forward(state["xq"], state["x_scale"], state["idx"], state["weight"])


def _experts_touched(case):
    """Experts with at least one row, on one sample of the case's routing."""
    g = torch.Generator()
    g.manual_seed(1)
    idx, _ = _top_k(case, _logits(case, torch.device("cpu"), g))
    return torch.unique(idx).numel()


def work(case):
    tokens, hidden, experts, top_k = case["tokens"], case["hidden"], case["experts"], case["top_k"]
    rows = tokens * top_k
    if case["kind"] == "permute":
        slots = experts * _capacity(case)
        # rows in and out of the permutation, the residual and the result, ids, weights, indices and counts
        return {"bytes": 2 * hidden * (tokens + slots + tokens + tokens) + rows * (4 + 2 + 4) + 4 * experts,
                "flops": 2 * rows * hidden}
    inter = case["inter"]
    weights = _experts_touched(case) * (3 * hidden * inter + 4 * (2 * inter + hidden))
    if case["kind"] == "layer":
        # hidden states, the shared expert's rows and the result; logits in, weights and ids out
        other = 2 * tokens * hidden * (3 if case["shared"] else 2) + 4 * tokens * experts + 8 * rows
    else:
        other = tokens * (hidden + 4) + 8 * rows + 2 * tokens * hidden
    return {"bytes": weights + other, "flops": 6 * rows * hidden * inter}


def tolerance(case):
    """About four times what these paths differ by from float64 restatements on the same inputs (2-norm / largest):
    permutation and combine 1.8e-3 / 3.9e-3 (one bf16 rounding); whole layer 2.8e-3 / 6.6e-2; expert FFN 4.6e-3 / 3.1e-2
    (the int8 requantisation between the two GEMMs moves an activation across a rounding boundary now and then)."""
    if case["kind"] == "permute":
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["kind"] == "layer":
        return {"rel": 1.1e-2, "max": 2.5e-1, "differ": 1e-4}
    return {"rel": 1.6e-2, "max": 1.2e-1}
