"""The expert-major decode products where an expert has as many rows as a pass takes, one fewer, one
more, several passes' worth, or more runs than there are workgroup columns for - and uneven K
quarters - against the oracle's layer. (Small e4m3 and MXFP4 layers take the split stream kernels; the
wide ones are named in test_wide_kernels_of_many_rows.) A router bias sends every token to the same experts, so their
row counts are the token count exactly."""

import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_helpers import announce, assert_bf16_bar, bf16_bits, bf16_values, kernels_of, normal_bf16
from test_gpu_layer_routing import quantised
from uniserve_moe import ops

pytestmark = pytest.mark.gpu

CASES = {
    # name: tokens, hidden, experts, top, intermediate, window, live
    "a pass less one": (31, 512, 64, 4, 256, None, None),
    "a pass": (32, 1024, 64, 4, 256, None, None),
    "a pass and one": (33, 512, 64, 4, 256, None, None),
    "two passes and one, 20 and 6 lines of K": (65, 1280, 64, 4, 384, None, None),
    "some rows not live": (100, 512, 64, 4, 256, None, 70),
    "a window of three experts": (300, 512, 128, 8, 256, (2, 3), None),
    "a window of four experts, a run ends on a pass": (288, 512, 128, 8, 256, (0, 4), None),
    "fewer routes than experts": (40, 512, 128, 2, 256, None, None),
}


@pytest.mark.parametrize("wdtype", ["bf16", "f8e4m3", "f4e2m1"])
@pytest.mark.parametrize("case", list(CASES))
def test_experts_of_many_rows(device, case, wdtype):
    tokens, hidden, experts, top, intermediate, window, live = CASES[case]
    if wdtype == "f4e2m1":
        intermediate = 512 if intermediate == 384 else intermediate  # whole 256-element chunks
    announce("row runs", case, wdtype)
    offset, local = (0, experts) if window is None else window
    x = normal_bf16((tokens, hidden), 81, device=device)
    router = normal_bf16((experts, hidden), 82, 0.02, device)
    up_gate = normal_bf16((local, 2 * intermediate, hidden), 83, 0.02, device)
    down = normal_bf16((local, hidden, intermediate), 84, 0.02, device)
    bias = np.where(np.arange(experts) < top, 40.0, 0.0).astype(np.float32)
    w1, w2, s1, s2, up_dev, down_dev, args = quantised(wdtype, up_gate, down, device)
    layer = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=wdtype)
    live_t = None if live is None else torch.tensor([live], dtype=torch.int32, device=device)
    out = layer(x, router, up_dev, down_dev, router_bias=torch.from_numpy(bias).to(device), live_tokens=live_t,
                window=window, **args)
    torch.cuda.synchronize()
    got = bf16_values(out)
    want_bits, want_ids, _, _ = O.moe_layer(
        bf16_bits(x), bf16_bits(router), w1, w2, top, up_gate_scales=s1, down_scales=s2, router_bias=bias, live=live,
        window=None if window is None else (offset, local))
    ids = layer.view("ids", torch.int32, (tokens, top)).cpu().numpy()
    served = tokens if live is None else live
    np.testing.assert_array_equal(ids[:served], want_ids[:served])
    assert (np.sort(ids[:served], axis=1) == np.arange(top)).all()  # every token names the same experts
    assert (got[served:] == 0).all()
    assert_bf16_bar(got[:served], O.bf16_decode(want_bits).astype(np.float64)[:served], case,
                    max_rel=2e-2 if wdtype == "bf16" else 4e-2)


@pytest.mark.parametrize("wdtype", ["bf16", "f8e4m3"])
def test_spread_walks_of_the_two_workgroup_kernel(device, wdtype):
    """Between one and four rounds of resident workgroups its items start their K walks at different
    stages and wrap around: bf16 FC1 over 20 stages of K and FC2 over 8; e4m3, whose rows are spread
    at whole 4 KB, FC1 over 32."""
    tokens, hidden, experts, top, intermediate = (
        (1024, 1280, 128, 8, 512) if wdtype == "bf16" else (4096, 4096, 16, 2, 1024))
    announce("spread walks", wdtype)
    x = normal_bf16((tokens, hidden), 91, device=device)
    router = normal_bf16((experts, hidden), 92, 0.02, device)
    up_gate = normal_bf16((experts, 2 * intermediate, hidden), 93, 0.02, device)
    down = normal_bf16((experts, hidden, intermediate), 94, 0.02, device)
    w1, w2, s1, s2, up_dev, down_dev, args = quantised(wdtype, up_gate, down, device)
    layer = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=wdtype)
    out = layer(x, router, up_dev, down_dev, **args)
    torch.cuda.synchronize()
    tiles = int(layer.view("num_non_exiting_tiles", torch.int32, (1,)).item())
    assert 512 <= tiles * (intermediate // 128) <= 2048
    want_bits, want_ids, _, _ = O.moe_layer(bf16_bits(x), bf16_bits(router), w1, w2, top, up_gate_scales=s1,
                                            down_scales=s2)
    np.testing.assert_array_equal(layer.view("ids", torch.int32, (tokens, top)).cpu().numpy(), want_ids)
    assert_bf16_bar(bf16_values(out), O.bf16_decode(want_bits).astype(np.float64), wdtype,
                    max_rel=2e-2 if wdtype == "bf16" else 4e-2)


PLAIN_WALKS = {
    # name: weights, tokens, hidden, experts, top, intermediate, FC1 spread, FC2 spread
    "bf16 rows of 4 KB and 2 KB": ("bf16", 768, 2048, 16, 2, 1024, True, True),
    "bf16 rows of more than 4 KB": ("bf16", 768, 2560, 16, 2, 512, False, True),
    "bf16, four rounds of possible FC2 items": ("bf16", 2100, 2048, 128, 8, 512, True, False),
    "e4m3 rows of 4 KB and 1 KB": ("f8e4m3", 768, 4096, 16, 2, 1024, True, False),
}


@pytest.mark.parametrize("case", list(PLAIN_WALKS))
def test_which_walks_may_be_spread(device, case):
    wdtype, tokens, hidden, experts, top, intermediate, fc1, fc2 = PLAIN_WALKS[case]
    announce("plain walks", case)
    x = normal_bf16((tokens, hidden), 95, device=device)
    router = normal_bf16((experts, hidden), 96, 0.02, device)
    up_gate = normal_bf16((experts, 2 * intermediate, hidden), 97, 0.02, device)
    down = normal_bf16((experts, hidden, intermediate), 98, 0.02, device)
    *_, up_dev, down_dev, args = quantised(wdtype, up_gate, down, device)
    layer = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=wdtype)
    out = torch.empty((tokens, hidden), dtype=torch.bfloat16, device=device)
    names = kernels_of(lambda: layer(x, router, up_dev, down_dev, out=out, **args))
    pairs = [name for name in names if "pair_kernel" in name]
    assert ["Lb1ELb%dEE" % fc1 in pairs[0], "Lb0ELb%dEE" % fc2 in pairs[1]] == [True, True], names


_FP8, _MX = "wide_fp8_kernelILb", "wide_mx_kernelILb"
WIDE = {
    # name: weights, tokens, hidden, experts, top, intermediate, window, live, FC1's and FC2's kernels. (At
    # most 48 runs past the first passes are shared out to columns of their own, or as many as experts:
    # eight experts of 300 rows have 72 and take them 64 rows at a time, of 288 rows 64.)
    "e4m3, a pass and one": ("f8e4m3", 33, 1024, 64, 8, 1024, None, None, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi4ELi1ELb0EE"),
    "e4m3, two passes and one, some rows not live": (
        "f8e4m3", 90, 2048, 64, 8, 768, None, 65, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi2ELi2ELb0EE"),
    "e4m3, compact grid": (
        "f8e4m3", 15, 4096, 128, 8, 512, None, None, _FP8 + "1ELi2ELi2ELb1EE", "stream_fp8_kernelILb0ELb0ELi1ELb1E"),
    "e4m3, window, FC2 of 4 lines": (
        "f8e4m3", 300, 1024, 128, 8, 512, (0, 16), None, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi2ELi2ELb0EE"),
    "e4m3, window, FC2 of 4 lines, a width of an odd number of 128 columns": (
        "f8e4m3", 100, 640, 128, 8, 512, (0, 16), None, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi4ELi1ELb0EE"),
    "e4m3, window, FC2 of 8 lines": (
        "f8e4m3", 288, 512, 128, 8, 1024, (0, 16), None, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi4ELi1ELb0EE"),
    "e4m3, window, FC2 of 6 lines": (
        "f8e4m3", 288, 2048, 128, 8, 768, (0, 16), None, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi2ELi2ELb0EE"),
    "e4m3, window, some rows not live": (
        "f8e4m3", 200, 1024, 128, 8, 1024, (4, 20), 150, _FP8 + "1ELi2ELi2ELb1EE", _FP8 + "0ELi4ELi1ELb0EE"),
    "mx, a pass and one": ("f4e2m1", 33, 1024, 64, 8, 512, None, None, _MX + "1ELi2ELi2ELb1EE", _MX + "0ELi2ELi2ELb0EE"),
    "mx, two passes and one, some rows not live": (
        "f4e2m1", 90, 2048, 64, 8, 768, None, 65, _MX + "1ELi2ELi2ELb1EE", _MX + "0ELi1ELi4ELb0EE"),
    "mx, compact grid": (
        "f4e2m1", 12, 1024, 128, 8, 512, None, None, "stream_mx_kernelILb1ELb0ELb1ELi1ELb1EE", _MX + "0ELi2ELi2ELb0EE"),
    "mx, window, FC2 of 2 lines": (
        "f4e2m1", 300, 1024, 128, 8, 512, (0, 16), None, _MX + "1ELi2ELi2ELb1EE", _MX + "0ELi2ELi2ELb0EE"),
    "mx, window, FC2 of 3 lines": (
        "f4e2m1", 288, 2048, 128, 8, 768, (0, 16), None, _MX + "1ELi2ELi2ELb1EE", _MX + "0ELi1ELi4ELb0EE"),
    "mx, window, some rows not live": (
        "f4e2m1", 200, 1024, 128, 8, 768, (4, 20), 150, _MX + "1ELi2ELi2ELb1EE", _MX + "0ELi1ELi4ELb0EE"),
    "bf16, window": ("bf16", 300, 512, 128, 8, 256, (0, 16), None, "wide_kernelILb1ELb1ELi2EE", "wide_kernelILb0ELb1ELi2EE"),
}


@pytest.mark.parametrize("case", list(WIDE))
def test_wide_kernels_of_many_rows(device, case):
    """The wide kernels by name - also of a window that holds the much-named experts - where further
    columns share out the rows past an expert's first pass."""
    wdtype, tokens, hidden, experts, top, intermediate, window, live, fc1, fc2 = WIDE[case]
    announce("wide kernels", case)
    local = experts if window is None else window[1]
    x = normal_bf16((tokens, hidden), 101, device=device)
    router = normal_bf16((experts, hidden), 102, 0.02, device)
    up_gate = normal_bf16((local, 2 * intermediate, hidden), 103, 0.02, device)
    down = normal_bf16((local, hidden, intermediate), 104, 0.02, device)
    bias = np.where(np.arange(experts) < top, 40.0, 0.0).astype(np.float32)
    bias_dev = torch.from_numpy(bias).to(device)
    live_t = None if live is None else torch.tensor([live], dtype=torch.int32, device=device)
    w1, w2, s1, s2, up_dev, down_dev, args = quantised(wdtype, up_gate, down, device)
    layer = ops.MoeLayer(hidden, experts, top, intermediate, tokens, weight_dtype=wdtype)
    out = torch.empty((tokens, hidden), dtype=torch.bfloat16, device=device)

    def call():
        layer(x, router, up_dev, down_dev, out=out, router_bias=bias_dev, live_tokens=live_t, window=window, **args)

    names = kernels_of(call)
    assert any(fc1 in name for name in names) and any(fc2 in name for name in names), names
    call()
    torch.cuda.synchronize()
    want_bits, want_ids, _, _ = O.moe_layer(bf16_bits(x), bf16_bits(router), w1, w2, top, up_gate_scales=s1,
                                            down_scales=s2, router_bias=bias, live=live, window=window)
    served = tokens if live is None else live
    np.testing.assert_array_equal(layer.view("ids", torch.int32, (tokens, top)).cpu().numpy()[:served], want_ids[:served])
    assert_bf16_bar(bf16_values(out)[:served], O.bf16_decode(want_bits).astype(np.float64)[:served], case,
                    max_rel=2e-2 if wdtype == "bf16" else 4e-2)
