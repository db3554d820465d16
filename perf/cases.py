"""The routed MoE layer's work, as a serving program has it done: one pass per call of a case.

A case is one layer of a model at one batch size, through `ops.MoeLayer` (the whole layer in one
call) or through the separate operators (`entry` "operators"). The layers are the two Qwen3-MoE
shapes of the benchmark, whole, as a tensor-parallel rank's half of the intermediate width (`split`
2) or as an expert-parallel rank's window of the experts; the batches run from one decoded token
through continuous batches of decodes and chunked prefill to whole prompts. Weights are bf16,
block-scaled e4m3 or MXFP4, ~N(0, 0.02) before quantisation; hidden rows are ~N(0, 1) bf16. Decode
batches route near-uniformly, prompts mostly by a Zipf(1.1) router bias.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "uniserve-v1_amd"))

from uniserve_moe import ops  # noqa: E402
from uniserve_moe.checkpoint import quantize_blocks_e4m3, quantize_blocks_mxfp4  # noqa: E402

#: hidden, experts, top, intermediate
SHAPES = {"30b": (2048, 128, 8, 768), "235b": (4096, 128, 8, 1536)}


def _case(model, weights, tokens, zipf=False, split=1, first=0, held=128, entry="layer", name=None):
    case = {"model": model, "weights": weights, "tokens": tokens, "zipf": zipf, "split": split, "first": first,
            "held": held, "entry": entry}
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # One user's decode step on the larger model.
        _case("235b", "fp8", 1, name="one-235b-fp8"),
        # A handful of concurrent decodes.
        _case("30b", "bf16", 5, name="few-30b-bf16"),
        # A small continuous batch, four-bit experts.
        _case("235b", "mx", 23, name="decode-235b-mx"),
        # The benchmark's decode batch.
        _case("30b", "bf16", 64, name="decode-30b-bf16"),
        # A busy server's decode batch, whatever number of sequences is live.
        _case("30b", "fp8", 200, name="decode-30b-fp8"),
        # A very large one, or decodes with a short prompt's chunk among them.
        _case("30b", "bf16", 301, name="batch-30b-bf16"),
        # A chunk of a prompt's prefill.
        _case("30b", "fp8", 777, zipf=True, name="chunk-30b-fp8"),
        # The same layer issued operator by operator, with the shared expert's join at its end.
        _case("30b", "bf16", 512, entry="operators", name="operators-30b-bf16"),
        # One of eight expert-parallel ranks: sixteen of the experts, every rank's tokens.
        _case("235b", "fp8", 2048, first=48, held=16, name="ep-235b-fp8"),
        # Whole prompts: the benchmark's prefill batches, and a ragged one.
        _case("30b", "bf16", 8192, zipf=True, name="prefill-30b-bf16"),
        _case("30b", "mx", 6007, zipf=True, name="prefill-30b-mx"),
        _case("235b", "fp8", 4096, zipf=True, name="prefill-235b-fp8"),
    ]


def draw(rng):
    model = rng.choice(["30b", "30b", "235b"])
    weights = rng.choice(["bf16", "fp8", "mx"])
    entry, split, first, held = "layer", 1, 0, 128
    kind = rng.random()
    if kind < 0.15:
        weights, entry = "bf16", "operators"
    elif kind < 0.3:
        held = rng.choice([16, 32])
        first = held * rng.randrange(128 // held)
    elif kind < 0.45 and not (model == "30b" and weights == "mx"):
        split = 2  # (MXFP4 stacks hold whole 256-channel chunks: 384 are not)
    most = 8192 if model == "30b" else (2048 if weights == "bf16" else 4096)
    tokens = min(most, int(round(math.exp(rng.uniform(0.0, math.log(most))))))
    zipf = entry == "layer" and rng.random() < (0.75 if tokens > 512 else 0.25)
    return _case(model, weights, tokens, zipf, split, first, held, entry)


def _sizes(case):
    hidden, experts, top, intermediate = SHAPES[case["model"]]
    return case["tokens"], hidden, experts, top, intermediate // case["split"]


def _bias(case, device):
    if not case["zipf"]:
        return None
    experts = SHAPES[case["model"]][1]
    return -1.1 * torch.log(torch.arange(experts, device=device, dtype=torch.float32) + 1.0)


def _normal(shape, std, generator):
    return (torch.randn(shape, generator=generator, device="cuda") * std).to(torch.bfloat16)


def _tokens(case, generator):
    """Everything of the case but the expert stacks."""
    tokens, hidden, experts, _, _ = _sizes(case)
    made = {"x": _normal((tokens, hidden), 1.0, generator), "router": _normal((experts, hidden), 0.02, generator),
            "bias": _bias(case, "cuda")}
    if case["entry"] == "operators":
        made["shared"] = _normal((tokens, hidden), 0.2, generator)
        made["shared_gate"] = _normal((tokens, 1), 1.0, generator)
    return made


def _stacks(case, generator):
    """The held experts' two stacks and their scales, in the form the weights' kind takes."""
    _, hidden, _, _, intermediate = _sizes(case)
    made = []
    for rows, width in ((2 * intermediate, hidden), (hidden, intermediate)):
        parts, scales = [], []
        for at in range(0, case["held"], 16):
            part = _normal((min(16, case["held"] - at), rows, width), 0.02, generator)
            scale = None
            if case["weights"] == "fp8":
                part, scale = quantize_blocks_e4m3(part)
            elif case["weights"] == "mx":
                part, scale = quantize_blocks_mxfp4(part)
            parts.append(part)
            scales.append(scale)
        made.append((torch.cat(parts), None if scales[0] is None else torch.cat(scales)))
    return made


def prepare(case, seed):
    tokens, hidden, experts, top, intermediate = _sizes(case)
    generator = torch.Generator(device="cuda").manual_seed(seed)
    state = _tokens(case, generator)
    (state["up_gate"], s1), (state["down"], s2) = _stacks(case, generator)
    if case["entry"] == "operators":
        state["experts"], state["top"] = experts, top
        return state
    kind = {"bf16": "bf16", "fp8": "f8e4m3", "mx": "f4e2m1"}[case["weights"]]
    state["layer"] = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=kind)
    state["options"] = {"router_bias": state["bias"]}
    if case["weights"] == "fp8":
        state["options"].update(up_gate_scales=s1, down_scales=s2)
    elif case["weights"] == "mx":
        # Converted once, at load, to the layout the prefill kernels fetch in runs.
        state["options"].update(up_gate_scales=ops.mx_stage_major_scales(s1),
                                down_scales=ops.mx_stage_major_scales(s2), scale_layout="stage")
    if case["held"] != experts:
        state["options"]["window"] = (case["first"], case["held"])
    return state


def run(state):
    x, router = state["x"], state["router"]
    if "layer" in state:
        return state["layer"](x, router, state["up_gate"], state["down"], **state["options"])
    tokens, experts, top = x.shape[0], state["experts"], state["top"]
    ids, weights = ops.topk_softmax(ops.router_gemm(x, router), top)
    maps = ops.moe_sort(ids, weights, experts)
    gated = ops.gather_gemm(x, state["up_gate"], top, maps, ops.permuted_rows(tokens, top, experts))
    products = ops.route_gemm(gated, state["down"], maps)
    out = ops.moe_unpermute(products, maps[ops.EXPANDED_TO_PERMUTED], weights)
    return ops.sigmoid_gated_add_(out, state["shared"], state["shared_gate"]), ids, weights


def work(case):
    """Weights of the experts some route names, the rows in and out, the router; the routes'
    products. (The routing is drawn as the inputs' distributions give it.)"""
    tokens, hidden, experts, top, intermediate = _sizes(case)
    rng = np.random.default_rng(0)
    scores = rng.standard_normal((tokens, experts), dtype=np.float32) * (0.02 * math.sqrt(hidden))
    if case["zipf"]:
        scores += _bias(case, "cpu").numpy()
    ids = np.argpartition(-scores, top - 1, axis=1)[:, :top]
    ids = ids[(ids >= case["first"]) & (ids < case["first"] + case["held"])]
    touched = len(np.unique(ids))
    element = {"bf16": 2.0, "fp8": 1.0 + 4.0 / 128 / 128, "mx": 0.5 + 1.0 / 32}[case["weights"]]
    moved = touched * 3 * hidden * intermediate * element + tokens * hidden * 4 + hidden * experts * 2
    if case["entry"] == "operators":
        moved += tokens * hidden * 2 + tokens * top * 8
    return {"bytes": int(moved), "flops": int(ids.size * 6 * hidden * intermediate + 2 * tokens * hidden * experts)}


def tolerance(case):
    # About four times the layer's measured distance from `exact` (2-norm): bf16 0.0029, where the
    # gated rows, the products and the output each round once; e4m3 0.011 and MXFP4 0.015, where
    # the gated rows round into e4m3 as well and a neighbour of a tie goes the other way. A token
    # whose last two picks tie may take the other expert.
    return {"rel": {"bf16": 1.2e-2, "fp8": 4e-2, "mx": 6e-2}[case["weights"]], "differ": 1e-2}


def _e4m3_rows(rows):
    """Rows through e4m3 with a scale of amax / 448 per 128 channels, decoded again."""
    groups = rows.reshape(rows.shape[0], -1, 128)
    amax = groups.abs().amax(dim=2, keepdim=True)
    scale = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    codes = (groups / scale).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn)
    return (codes.double() * scale).reshape(rows.shape)


def _mxfp8_rows(rows):
    """Rows through MXFP8: e4m3 with the smallest power of two that saturates nothing per 32."""
    groups = rows.reshape(rows.shape[0], -1, 32)
    amax = groups.abs().amax(dim=2, keepdim=True)
    mantissa, exponent = torch.frexp(torch.where(amax > 0, amax, torch.ones_like(amax)))
    exponent = exponent - 9 + (mantissa > 0.875).int()  # 448 = 0.875 * 2^9
    scale = torch.ldexp(torch.ones_like(amax), exponent)
    codes = (groups / scale).float().to(torch.float8_e4m3fn)
    return (codes.double() * scale).reshape(rows.shape)


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _decoded(codes, scales, kind):
    """One expert's matrix in 64 bits."""
    if kind == "bf16":
        return codes.double()
    if kind == "fp8":
        blocks = scales.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
        return codes.view(torch.float8_e4m3fn).double() * blocks
    table = torch.tensor(_E2M1, dtype=torch.float64, device=codes.device)
    pairs = torch.stack([table[(codes & 15).long()], table[(codes >> 4).long()]], dim=2).reshape(codes.shape[0], -1)
    return pairs * torch.exp2(scales.double() - 127.0).repeat_interleave(32, 1)


def exact(case, seed):
    tokens, hidden, experts, top, intermediate = _sizes(case)
    generator = torch.Generator(device="cuda").manual_seed(seed)
    made = _tokens(case, generator)
    (up_gate, s1), (down, s2) = _stacks(case, generator)
    rounded = {"bf16": lambda rows: rows, "fp8": _e4m3_rows, "mx": _mxfp8_rows}[case["weights"]]

    # The router Linear's output is bf16 by definition; equal scores take the lower expert first.
    scores = made["x"].double() @ made["router"].double().t()
    if made["bias"] is not None:
        scores = scores + made["bias"].double()
    chances = torch.softmax(scores.to(torch.bfloat16).double(), dim=1)
    ordered, order = torch.sort(chances, dim=1, descending=True, stable=True)
    ids, weights = order[:, :top], ordered[:, :top]
    weights = weights / weights.sum(dim=1, keepdim=True)

    rows = rounded(made["x"].double())
    out = torch.zeros((tokens, hidden), dtype=torch.float64, device="cuda")
    for held in range(case["held"]):
        token, pick = torch.nonzero(ids == case["first"] + held, as_tuple=True)
        if token.numel() == 0:
            continue
        both = rows[token] @ _decoded(up_gate[held], None if s1 is None else s1[held], case["weights"]).t()
        up, gate = both[:, :intermediate], both[:, intermediate:]
        gated = rounded(up * gate * torch.sigmoid(gate))
        product = gated @ _decoded(down[held], None if s2 is None else s2[held], case["weights"]).t()
        out.index_add_(0, token, product * weights[token, pick].unsqueeze(1))
    if case["entry"] != "operators":
        return out
    out = out + torch.sigmoid(made["shared_gate"].double()) * made["shared"].double()
    return out, ids, weights
