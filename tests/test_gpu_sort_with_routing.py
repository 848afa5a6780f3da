"""Batches whose pairs are sorted by the launches that route and quantise them: what the sort leaves - row ranges, counts, places and their
inverse - and the quantised rows, on both sides of the sizes where a wave routes one token, two and four, of the rule's ends, and for an
expert-parallel share, against the stand-alone sort of the ids the routing left and the oracle's quantiser."""
import numpy as np
import pytest
import torch

from conftest import bits

pytestmark = pytest.mark.gpu

from oracle import c_oracle as co  # noqa: E402


@pytest.mark.parametrize("M,E,K,quant,H,scoring,n_group", [
    (1536, 128, 8, "int8", 256, "softmax", 1), (1537, 128, 8, "int8", 256, "softmax", 1),      # 12288 pairs, and the first beyond
    (2048, 128, 8, "none", 128, "softmax", 1), (2049, 128, 8, "int8", 128, "softmax", 1),      # one token a wave, two
    (4097, 100, 8, "int8", 128, "softmax", 1), (8192, 128, 8, "int8", 128, "softmax", 1),      # three, four
    (8193, 64, 4, "int8", 128, "softmax", 1),                                                  # five: a sort of its own
    (1025, 17, 17, "none", 128, "softmax", 1), (600, 128, 64, "none", 128, "softmax", 1),      # a chunk of 1024 pairs
    (2047, 128, 8, "int8", 128, "sigmoid", 8), (1999, 130, 8, "fp8", 256, "sigmoid", 5),        # up to 128 experts; more
    (1600, 64, 8, "fp8", 128, "sigmoid", 1), (1999, 120, 8, "fp8", 256, "sigmoid", 5),          # groups of 24: scores in LDS
    (1600, 96, 8, "int8", 2048, "softmax", 1), (1600, 96, 8, "int8", 2064, "softmax", 1),        # rows of a wave, of four
    (1600, 96, 8, "int8", 8192, "softmax", 1), (3000, 128, 8, "w4", 128, "softmax", 1),
    (8193, 130, 8, "fp8", 1024, "sigmoid", 5)])                                                # two groups of 128 a lane
@pytest.mark.parametrize("share", [False, True])
def test_sort_of_a_routed_batch(M, E, K, quant, H, scoring, n_group, share):
    from vllm_kunlun_amd import _lib as L, _plan, synth
    base = "dsv3-decode" if scoring == "sigmoid" else "qwen3-decode"
    shape = synth.scaled(synth.SHAPES[base], M=M, H=H, E=E, K=K, I=128, I_shared=0, quant=quant, n_group=n_group,
                         topk_group=max(1, n_group // 2), group_size=128)
    sl = synth.make_layer(shape, "cuda", seed=M)
    logits = sl.logits
    if share:  # the layer's experts are the last ones of half as many again: their routing needs logits (and a bias) for all
        if scoring == "sigmoid":
            pytest.skip("the group arithmetic of a share is the softmax cases'")
        logits = torch.cat([torch.randn(M, E // 2, device="cuda"), sl.logits], 1).contiguous()
    if quant == "int8":
        sl.x[M // 2, 5], sl.x[M - 1, 1] = float("nan"), float("inf")
    P = M * K
    lay = sl.layer
    fmt = {"int8": L.KMOE_FMT_INT8, "fp8": L.KMOE_FMT_FP8_BLOCK, "none": L.KMOE_FMT_BF16, "w4": L.KMOE_FMT_W4A16}[quant]
    weights = [getattr(lay, n + ("_weight_packed" if quant == "w4" else "_weight")) for n in ("w13", "w2")]
    aux = [getattr(lay, n + "_weight_scale", None) for n in ("w13", "w2")]
    aux = [None if a is None or quant == "none" else a.data for a in aux]
    if quant == "int8":
        aux = [a.reshape(E, -1) for a in aux]
    out = torch.empty_like(sl.x)
    plan = _plan.make_moe_plan(fmt, sl.x, logits, out, K, weights[0].data, weights[1].data, aux[0], aux[1], scoring, True, n_group,
                               shape.topk_group, shape.routed_scale, sl.bias if not share else None,
                               group_size=128 if quant == "w4" else None, first_expert=E // 2 if share else 0)
    plan()
    first = E // 2 if share else 0
    ids = plan.view("topk_ids", P, torch.int32).clone()
    want = [torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (P, P, E, E + 1)]
    nbytes = L.lib.kmoe_align_workspace_bytes(P, E)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    L.check(L.lib.kmoe_align_local(L.ptr(ids), P, E, first, *(L.ptr(t) for t in want), L.ptr(ws), nbytes, L.stream()))
    live = int(want[3][-1])
    got = [plan.view(n, c, torch.int32) for n, c in (("moe_index", P), ("sorted_src", P), ("expert_m", E), ("lod", E + 1))]
    assert torch.equal(got[0], want[0]) and torch.equal(got[1][:live], want[1][:live])
    assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3])
    if quant in ("int8", "fp8") and not plan.layout.codes_chunked:
        ref = co.quant_i8_rows(bits(sl.x)) if quant == "int8" else co.quant_fp8_group128(bits(sl.x))
        codes = plan.view("xq", M * H, torch.uint8).cpu().numpy().reshape(M, H)
        scales = plan.view("xmax", ref[1].size, torch.float32).cpu().numpy()
        assert np.array_equal(codes, ref[0].view(np.uint8)) and np.array_equal(scales.view(np.uint32), ref[1].reshape(-1).view(np.uint32))
