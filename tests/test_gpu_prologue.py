"""The launch in front of a layer's first GEMM (routing, with the quantisation of the activations where the format has
one): router logits in the activations' own 16-bit type must give the bits of the same logits widened to float32, for
every format and slot count of the routing kernel; a layer call whose argument block is kept from an earlier call must
follow what changed in between."""
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), ".."))
from conftest import bits  # noqa: E402
from oracle import c_oracle as co  # noqa: E402

pytestmark = pytest.mark.gpu


# experts on both sides of a routing kernel's slot counts (128, 256, 512), groups that are a power of two and not
@pytest.mark.parametrize("E,n_group", [(8, 2), (96, 3), (128, 8), (129, 1), (192, 4), (256, 8), (320, 5), (520, 4)])
@pytest.mark.parametrize("quant", ["int8", "fp8", "none"])
@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sixteen_bit_logits_route_like_their_float32_values(E, n_group, quant, scoring, dtype):
    from vllm_kunlun_amd import synth
    base = "dsv3-decode" if scoring == "sigmoid" else "qwen3-decode"
    topk_group = max(1, n_group // 2)
    shape = synth.scaled(synth.SHAPES[base], M=37, H=256, E=E, K=4, I=128, I_shared=0, quant=quant,
                         n_group=n_group if scoring == "sigmoid" else 1, topk_group=topk_group)
    sl = synth.make_layer(shape, "cuda", seed=E, dtype=dtype)
    logits = (sl.logits * 2).to(dtype)  # (16-bit values repeat: ties go to the lower expert either way)
    a = sl.layer(sl.x, logits)
    b = sl.layer(sl.x, logits.float())
    assert torch.equal(a, b) and float(a.float().abs().max()) > 0


def test_kept_argument_block_follows_the_call():
    """The second call of a layer reuses the first one's argument block: another batch size, other inputs, other
    options, another layer at the same sizes and weights that were swapped must all be seen."""
    from vllm_kunlun_amd import synth
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=48, H=256, E=16, K=4, I=128)
    sl, other = synth.make_layer(shape, "cuda", seed=1), synth.make_layer(shape, "cuda", seed=2)
    m = sl.layer.quant_method
    full = m.apply_monolithic(sl.layer, sl.x, sl.logits)
    assert torch.equal(m.apply_monolithic(sl.layer, sl.x, sl.logits), full)
    for n in (1, 17, 48):
        assert torch.equal(m.apply_monolithic(sl.layer, sl.x[:n], sl.logits[:n]), full[:n])
    doubled = m.apply_monolithic(sl.layer, sl.x, sl.logits, out_scale=2.0)
    assert torch.equal(doubled.float(), 2 * full.float())
    want = other.layer.quant_method.apply_monolithic(other.layer, sl.x, sl.logits)
    assert not torch.equal(want, full)
    for name in ("w13_weight", "w2_weight", "w13_weight_scale", "w2_weight_scale"):
        getattr(sl.layer, name).data = getattr(other.layer, name).data
    assert torch.equal(m.apply_monolithic(sl.layer, sl.x, sl.logits), want)
    with pytest.raises(ValueError):
        m.apply_monolithic(sl.layer, sl.x, sl.logits[:5])
    with pytest.raises(ValueError):
        m.apply_monolithic(sl.layer, sl.x[:, :128].contiguous(), sl.logits)
    with pytest.raises(RuntimeError):
        m.apply_monolithic(sl.layer, sl.x.cpu(), sl.logits.cpu())
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        on_side = m.apply_monolithic(sl.layer, sl.x, sl.logits)
    torch.cuda.synchronize()
    assert torch.equal(on_side, want)


# pairs and experts on both sides of every choice of launches, the last chunk full and not, ids of other ranks' experts
@pytest.mark.parametrize("P", [0, 255, 256, 257, 1024, 1025, 8192, 8193, 24576, 24577, 131073, 300000])
@pytest.mark.parametrize("E,first", [(1, 0), (256, 0), (257, 3), (1000, 0)])
def test_stable_sort_by_expert(P, E, first):
    from vllm_kunlun_amd import _lib as L
    ids = torch.randint(first - 2, first + E + 2, (P,), generator=torch.Generator().manual_seed(P + E)).clamp(min=0)
    ids[: P // 3] = first + E // 2
    local = torch.where((ids >= first) & (ids < first + E), ids - first, torch.full_like(ids, E))
    order = torch.argsort(local, stable=True)
    counts = torch.bincount(local, minlength=E + 1)[:E]
    kept = int(counts.sum())
    index = torch.full((P,), -1)
    index[order[:kept]] = torch.arange(kept)
    nbytes = L.lib.kmoe_align_workspace_bytes(P, E)
    dev = ids.int().cuda()
    out = [torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (max(P, 1), max(P, 1), E, E + 1)]
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    L.check(L.lib.kmoe_align_local(L.ptr(dev), P, E, first, *(L.ptr(t) for t in out), L.ptr(ws), nbytes, L.stream()))
    moe_index, sorted_src, expert_m, lod = (t.cpu().long() for t in out)
    assert torch.equal(moe_index[:P], index) and torch.equal(sorted_src[:kept], order[:kept])
    assert torch.equal(expert_m, counts) and torch.equal(lod, torch.cat([torch.zeros(1), counts.cumsum(0)]).long())


# the one launch's batches of ids (two and eight a thread) and its end, none of the pairs here and all of them
@pytest.mark.parametrize("P", [0, 2048, 2049, 4097, 16384, 16385, 32767, 32768, 32769])
@pytest.mark.parametrize("E,first", [(40, 0), (384, 1000), (1000, 0)])
def test_stable_sort_in_one_launch(P, E, first):
    test_stable_sort_by_expert(P, E, first)


# the ends of the rule that goes by the number of experts
@pytest.mark.parametrize("P", [24576, 24577, 32768, 32769])
@pytest.mark.parametrize("E,first", [(1, 0), (63, 0), (64, 7)])
def test_stable_sort_by_number_of_experts(P, E, first):
    test_stable_sort_by_expert(P, E, first)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fp8_group_quantiser_on_every_mantissa(dtype):
    """Groups whose maximum has every mantissa, over the exponents where the quotients come from the reciprocal and those
    where they are divided; zeros of both signs, subnormals, infinities and NaNs among the values."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(3)
    half = dtype == torch.float16
    mantissas = 1024 if half else 128
    exponents = [0, 1, 14, 15, 16, 30] if half else [0, 1, 60, 70, 76, 77, 127, 195, 196, 250, 254]
    top = torch.tensor([(e << (10 if half else 7)) | m for e in exponents for m in range(mantissas)], dtype=torch.int32)
    groups = len(top)
    x = torch.randint(0, 1 << 15, (groups, 128), generator=gen, dtype=torch.int32) % (top[:, None] + 1)
    near = torch.randint(0, (4 << 10) if half else (10 << 7), (groups, 128), generator=gen, dtype=torch.int32)
    x[:, :96] = (top[:, None] - near[:, :96]).clamp(min=0)  # most values within a few exponents of the maximum
    x[:, 5] = top
    x[:, 6] = 0
    x[::7, 9] = 0x7c00 if half else 0x7f80  # infinity: an infinite scale
    x[::5, 11] = 0x7e00 if half else 0x7fc0  # NaN: not part of the maximum
    x[3] = 0
    x |= torch.randint(0, 2, x.shape, generator=gen, dtype=torch.int32) << 15
    x = torch.from_numpy(x.numpy().astype(np.uint16).view(np.int16)).view(dtype).reshape(groups // 2, 256)
    R = x.shape[0]
    q_ref, s_ref = co.quant_fp8_group128(bits(x), f16=half)
    dx = x.cuda()
    q = torch.zeros(R, 256, dtype=torch.uint8, device="cuda")
    s = torch.zeros(R, 2, dtype=torch.float32, device="cuda")
    L.check(L.lib.kmoe_quant_fp8_group128_dt(L.ptr(dx), 256, R, 256, L.ptr(q), 256, L.ptr(s), L.act_dtype(dx, "test"), L.stream()))
    assert np.array_equal(s.cpu().numpy().view(np.uint32), s_ref.view(np.uint32))
    assert np.array_equal(q.cpu().numpy(), q_ref)


@pytest.mark.parametrize("E,K,n_group", [(8, 4, 2), (64, 8, 1), (129, 8, 1), (256, 8, 8), (520, 8, 4)])
@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
def test_nan_scores_still_give_every_pair_an_expert(E, K, n_group, scoring):
    """Rows whose scores are NaN with every bit set (memory filled with -1), all of them or all but two: K different
    experts of the layer, numbers before NaNs."""
    from vllm_kunlun_amd import _lib as L
    logits = torch.randn(6, E, generator=torch.Generator().manual_seed(E))
    nan = torch.full((1,), -1, dtype=torch.int32).view(torch.float32)
    bias = torch.zeros(E)
    if scoring == "softmax":
        logits[1], logits[3, 2:] = nan, nan
        logits[5, : E - 2] = nan
    else:  # (the sigmoid of a NaN is a number; a NaN in the correction bias reaches the comparison)
        bias[2:] = nan
    logits, bias = logits.cuda(), bias.cuda()
    w = torch.empty(6, K, device="cuda")
    ids = torch.full((6, K), -7, dtype=torch.int32, device="cuda")
    if scoring == "softmax":
        L.check(L.lib.kmoe_softmax_topk(L.ptr(logits), 6, E, K, 1, L.ptr(w), L.ptr(ids), L.stream()))
    else:
        L.check(L.lib.kmoe_sigmoid_group_topk_norm(L.ptr(logits), L.ptr(bias), 6, E, K, n_group, max(1, n_group // 2), 1.0,
                                                   L.ptr(w), L.ptr(ids), L.stream()))
    ids = ids.cpu().long()
    assert int(ids.min()) >= 0 and int(ids.max()) < E
    assert all(len(set(row.tolist())) == K for row in ids)
    if scoring == "softmax":
        assert set(ids[3, :2].tolist()) == {0, 1} and set(ids[5, :2].tolist()) == {E - 2, E - 1}


@pytest.mark.parametrize("M", [1, 40])  # a column of workgroups per pair, and one per expert
def test_nan_logits_of_a_token_leave_the_others_alone(M):
    from vllm_kunlun_amd import synth
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=M + 1, H=256, E=64, K=8, I=128)
    sl = synth.make_layer(shape, "cuda", seed=M)
    want = sl.layer(sl.x, sl.logits)
    logits = sl.logits.clone()
    logits[0] = torch.full((1,), -1, dtype=torch.int32).view(torch.float32).cuda()
    got = sl.layer(sl.x, logits)
    assert torch.equal(got[1:], want[1:])


# one group a lane and two, the last workgroup full and not, rows apart from each other
@pytest.mark.parametrize("R,C", [(511, 16384), (512, 16384), (513, 16384), (21846, 384), (1, 128)])
def test_fp8_groups_of_large_batches(R, C):
    from vllm_kunlun_amd import _lib as L
    x = torch.randn(R, C, generator=torch.Generator().manual_seed(R)).bfloat16()
    q_ref, s_ref = co.quant_fp8_group128(bits(x))
    apart = torch.full((R, C + 8), float("inf"), dtype=torch.bfloat16, device="cuda")
    apart[:, :C] = x.cuda()
    q = torch.full((R * C + 64,), 99, dtype=torch.uint8, device="cuda")
    s = torch.full((R * C // 128 + 16,), -7.0, device="cuda")
    L.check(L.lib.kmoe_quant_fp8_group128_dt(L.ptr(apart), C + 8, R, C, L.ptr(q), C, L.ptr(s), L.act_dtype(apart, "test"), L.stream()))
    assert np.array_equal(q[:R * C].cpu().numpy().reshape(R, C), q_ref) and bool((q[R * C:] == 99).all())
    got = s[:R * C // 128].cpu().numpy()
    assert np.array_equal(got.view(np.uint32), s_ref.reshape(-1).view(np.uint32)) and bool((s[R * C // 128:] == -7).all())
