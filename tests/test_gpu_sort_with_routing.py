"""What a batch's launches before the first GEMM leave: experts and weights against the oracle's routing, the sort - row ranges, counts,
places and their inverse - against a stable sort of those experts, and the quantised rows against the oracle's quantiser. On both sides of
the sizes where the sort goes from one launch to two and the fp8 quantiser to two groups a lane, for an expert-parallel share, and for
groups whose scores lie in LDS."""
import numpy as np
import pytest
import torch

from conftest import bits

pytestmark = pytest.mark.gpu

from oracle import c_oracle as co  # noqa: E402


@pytest.mark.parametrize("M,E,K,quant,H,scoring,n_group", [
    (1536, 128, 8, "int8", 256, "softmax", 1), (1537, 128, 8, "int8", 256, "softmax", 1),
    (2048, 128, 8, "none", 128, "softmax", 1), (2049, 128, 8, "int8", 128, "softmax", 1),
    (4097, 100, 8, "int8", 128, "softmax", 1), (8192, 128, 8, "int8", 128, "softmax", 1),      # 32776 pairs: two launches
    (8193, 64, 4, "int8", 128, "softmax", 1),                                                  # 32772
    (1025, 17, 17, "none", 128, "softmax", 1), (600, 128, 64, "none", 128, "softmax", 1),      # every expert; the most a token may have
    (2047, 128, 8, "int8", 128, "sigmoid", 8), (1999, 130, 8, "fp8", 256, "sigmoid", 5),        # groups of 16; of 26: scores in LDS
    (1600, 64, 8, "fp8", 128, "sigmoid", 1), (1999, 120, 8, "fp8", 256, "sigmoid", 5),          # no groups; of 24
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
    w_ref, ids_ref = co._route(logits.cpu().numpy(), K, scoring, True, n_group, shape.topk_group, shape.routed_scale,
                               sl.bias.cpu().numpy() if sl.bias is not None and not share else None)
    assert np.array_equal(plan.view("topk_ids", P, torch.int32).cpu().numpy(), ids_ref.ravel())
    assert np.array_equal(plan.view("topk_w", P, torch.float32).cpu().numpy().view(np.uint32), w_ref.ravel().view(np.uint32))
    key = ids_ref.ravel() - first
    here = np.flatnonzero((key >= 0) & (key < E))
    src = here[np.argsort(key[here], kind="stable")]
    place = np.full(P, -1, np.int32)
    place[src] = np.arange(src.size)
    counts = np.bincount(key[here], minlength=E)
    for name, want in (("moe_index", place), ("sorted_src", src), ("expert_m", counts), ("lod", np.concatenate([[0], counts.cumsum()]))):
        assert np.array_equal(plan.view(name, want.size, torch.int32).cpu().numpy(), want), name
    if quant in ("int8", "fp8") and not plan.layout.codes_chunked:
        ref = co.quant_i8_rows(bits(sl.x)) if quant == "int8" else co.quant_fp8_group128(bits(sl.x))
        codes = plan.view("xq", M * H, torch.uint8).cpu().numpy().reshape(M, H)
        scales = plan.view("xmax", ref[1].size, torch.float32).cpu().numpy()
        assert np.array_equal(codes, ref[0].view(np.uint8)) and np.array_equal(scales.view(np.uint32), ref[1].reshape(-1).view(np.uint32))
