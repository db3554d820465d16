"""The prefill front end where several workgroups share 32 tokens - eight, four or two, with expert
counts that fill, half fill and miss their shares - and in layers without a sort: given the layer's own
scores, the ids, weights and expert load are the topk_softmax entry's bit for bit, the hidden codes and
scales the quantisers', and (without a sort) each visible route is named at its own expanded index. The
scores are the oracle's router within one bf16 step of FP32 sums in another order."""

import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_helpers import announce, bf16_bits, bf16_values, kernels_of, normal_bf16
from test_gpu_layer_routing import quantised
from uniserve_moe import ops

pytestmark = pytest.mark.gpu

CASES = {
    # name: tokens, hidden, experts, top, weights, window, live
    "9 tokens, eight shares, no sort": (9, 4096, 128, 8, "f4e2m1", None, None),
    "31 tokens, eight shares, no sort": (31, 512, 100, 8, "bf16", None, None),
    "300 tokens, eight shares, no sort, window + live": (300, 1024, 128, 8, "f8e4m3", (40, 64), 290),
    "700 tokens, eight shares of 60 experts + live": (700, 512, 60, 8, "bf16", None, 699),
    "1025 tokens, four shares": (1025, 512, 128, 8, "f8e4m3", None, None),
    "1536 tokens, four shares of 33 experts": (1536, 256, 33, 6, "f8e4m3", None, 1500),
    "2048 tokens, four shares": (2048, 512, 128, 8, "f4e2m1", (8, 112), None),
    "2049 tokens, two shares": (2049, 512, 128, 8, "f4e2m1", (8, 112), None),
}


@pytest.mark.parametrize("case", list(CASES))
def test_split_front_is_the_separate_operators(device, case):
    tokens, hidden, experts, top, wdtype, window, live = CASES[case]
    announce("split front", case)
    intermediate = 256
    x = normal_bf16((tokens, hidden), 101, device=device)
    router = normal_bf16((experts, hidden), 102, 0.02, device)
    offset, local = (0, experts) if window is None else window
    up_gate = normal_bf16((local, 2 * intermediate, hidden), 103, 0.02, device)
    down = normal_bf16((local, hidden, intermediate), 104, 0.02, device)
    *_, up_dev, down_dev, args = quantised(wdtype, up_gate, down, device)
    mapping = torch.from_numpy(np.random.default_rng(105).permutation(experts).astype(np.int32)).to(device)
    load = torch.zeros(experts, dtype=torch.int64, device=device)
    live_t = None if live is None else torch.tensor([live], dtype=torch.int32, device=device)
    layer = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=wdtype)
    layer(x, router, up_dev, down_dev, live_tokens=live_t, mapping=mapping, load=load, window=window, **args)
    torch.cuda.synchronize()
    scores = layer.view("scores", torch.bfloat16, (tokens, experts)).clone()
    want = O.bf16_decode(O.router_gemm(bf16_bits(x), bf16_bits(router), None)).astype(np.float64)
    magnitude = np.abs(bf16_values(x)) @ np.abs(bf16_values(router)).T
    assert (np.abs(bf16_values(scores) - want) <= 2.0**-7 * np.abs(want) + 2.0 * hidden * 2.0**-24 * magnitude).all()

    want_load = torch.zeros_like(load)
    want_ids, want_weights = ops.topk_softmax(scores, top, True, None, mapping, live_t, want_load)
    ids = layer.view("ids", torch.int32, (tokens, top))
    assert torch.equal(ids, want_ids) and torch.equal(load, want_load)
    weights = layer.view("weights", torch.float32, (tokens, top))
    assert torch.equal(weights.view(torch.int32), want_weights.view(torch.int32))
    if wdtype != "bf16":
        want_q, want_s = (ops.quantize_fp8 if wdtype == "f8e4m3" else ops.quantize_mxfp8)(x)
        assert torch.equal(layer.view("hidden_q", torch.uint8, (tokens, hidden)), want_q)
        if wdtype == "f8e4m3":  # (MXFP4 layers with a sort park their scales by route)
            got_s = layer.view("hidden_s", torch.float32, (tokens, hidden // 128))
            assert torch.equal(got_s.view(torch.int32), want_s.view(torch.int32))
    if case.count("no sort"):
        route = torch.arange(tokens * top, device=device, dtype=torch.int32).reshape(tokens, top)
        seen = (ids >= offset) & (ids < offset + local) & (route < (tokens if live is None else live) * top)
        want_e2p = torch.where(seen, route, torch.full_like(route, -1))
        assert torch.equal(layer.view("expanded_to_permuted", torch.int32, (tokens, top)), want_e2p)
    else:
        maps = ops.moe_sort(ids.contiguous(), weights.contiguous(), experts, local=(offset, offset + local), live_tokens=live_t)
        got = layer.view("expanded_to_permuted", torch.int32, (tokens * top,))
        assert torch.equal(got, maps[ops.EXPANDED_TO_PERMUTED][: tokens * top])


@pytest.mark.parametrize("tokens", [31, 300, 900, 1100, 2000, 2100])
def test_scores_do_not_depend_on_the_share(device, tokens):
    """Eight, four or two workgroups share a token's experts, and all walk K from the same stage: equal
    router rows in different shares give equal scores (so the lower expert comes first), and every score
    is bit for bit the single-launch front end's, which serves past 4096 tokens."""
    announce("split front, equal router rows", tokens)
    hidden, experts, top, intermediate, most = 4096, 128, 8, 128, 4128
    x = normal_bf16((most, hidden), 111, device=device)
    half = normal_bf16((experts // 2, hidden), 112, 0.02, device)
    router = torch.cat([half, half])
    up_gate = normal_bf16((experts, 2 * intermediate, hidden), 113, 0.02, device)
    down = normal_bf16((experts, hidden, intermediate), 114, 0.02, device)
    scores = {}
    for count in (tokens, most):
        layer = ops.MoeLayer(hidden, experts, top, intermediate, count)
        layer(x[:count], router, up_gate, down)
        torch.cuda.synchronize()
        scores[count] = layer.view("scores", torch.int16, (count, experts))[:tokens].clone()
        if count == tokens:
            ids = layer.view("ids", torch.int32, (tokens, top)).clone()
    assert torch.equal(scores[tokens][:, : experts // 2], scores[tokens][:, experts // 2 :])
    assert torch.equal(scores[tokens], scores[most])
    values = scores[tokens].view(torch.bfloat16).float()
    want = torch.sort(values, dim=1, descending=True, stable=True).indices[:, :top]  # ties: the lower expert
    assert torch.equal(ids.long(), want)


@pytest.mark.parametrize("wdtype", ["bf16", "f8e4m3", "f4e2m1"])
@pytest.mark.parametrize("tokens, shares", [(1024, 8), (1025, 4), (2048, 4), (2049, 2), (4096, 2), (4097, 1)])
def test_shares_fill_the_chip_once(device, tokens, shares, wdtype):
    """Eight, four or two workgroups per 32 tokens, at most 256 in all, whatever the weights; one where
    the tokens alone make more than 128."""
    announce("split front, shares", tokens, wdtype)
    hidden, experts, top, intermediate = 512, 32, 8, 256
    x = normal_bf16((tokens, hidden), 121, device=device)
    router = normal_bf16((experts, hidden), 122, 0.02, device)
    up_gate = normal_bf16((experts, 2 * intermediate, hidden), 123, 0.02, device)
    down = normal_bf16((experts, hidden, intermediate), 124, 0.02, device)
    *_, up_dev, down_dev, args = quantised(wdtype, up_gate, down, device)
    layer = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=wdtype)
    out = torch.empty((tokens, hidden), dtype=torch.bfloat16, device=device)
    names = kernels_of(lambda: layer(x, router, up_dev, down_dev, out=out, **args))
    quant = {"bf16": 0, "f8e4m3": 1, "f4e2m1": 2}[wdtype]
    want = f"split_scores_kernelILi{quant}ELi{shares}EE" if shares > 1 else f"prefill_front_kernelILi{quant}EE"
    assert want in names[0], names
