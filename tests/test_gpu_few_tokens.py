"""Batches of a few tokens, whose second quantisation, down projection and combine are one launch: the launch's limits (row
lengths on both sides of its two forms, waves, remainders of the steps in flight), and the calls that stay apart."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), ".."))
from conftest import bits, from_bits, rel_l2  # noqa: E402
from oracle import c_oracle as co  # noqa: E402

pytestmark = pytest.mark.gpu

FUSED = "down projection and combine"


def _named(call):
    from vllm_kunlun_amd import _lib as L
    L.lib.kmoe_trace_kernels(1)
    out = call()
    named = L.lib.kmoe_traced_kernels().decode()
    L.lib.kmoe_trace_kernels(0)
    return out, named


@pytest.mark.parametrize("fmt,I", [("int8", 64), ("int8", 1024), ("int8", 1088), ("int8", 2048), ("int8", 2112), ("fp8", 128),
                                   ("fp8", 1152), ("fp8", 2048), ("fp8", 2176), ("none", 96), ("none", 1056), ("none", 2048),
                                   ("none", 2080), ("w4", 128), ("w4", 1152), ("w4", 2048), ("w4", 2176)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_of_every_length(fmt, I, dtype):
    """Against the same tokens in a batch with a column per expert: the same bits in int8; elsewhere sums split otherwise
    move a 16-bit result by its rounding (2^-9 of it, and the same again behind the second GEMM: 4e-3)."""
    from vllm_kunlun_amd import synth
    M, E, K = 3, 48, 6
    big = E // K + 2
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=big, H=256, E=E, K=K, I=I, quant=fmt)
    sl = synth.make_layer(shape, "cuda", seed=I, dtype=dtype)
    whole = sl.layer(sl.x, sl.logits)
    part, named = _named(lambda: sl.layer(sl.x[:M], sl.logits[:M]))
    padded = -(-I // 64) * 64 if fmt == "int8" else I
    assert (FUSED in named) == (padded <= 2048), named
    if fmt == "int8":
        assert torch.equal(part, whole[:M])
    else:
        assert rel_l2(part, whole[:M]) <= 4e-3


@pytest.mark.parametrize("M,K,H,I,steps", [(1, 2, 4096, 2048, 8), (4, 2, 4096, 2048, 8), (1, 4, 2048, 512, 8), (2, 4, 2048, 896, 3), (3, 3, 512, 1152, 8),
                                           (1, 8, 4096, 1920, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_packed_steps_in_flight(M, K, H, I, steps, dtype):
    """4-bit weights: deep rings where the launch has no more waves than a row values."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], M=M, E=40, K=K, H=H, I=I, quant="w4"), "cuda", seed=I, dtype=dtype)
    out, named = _named(lambda: _call(sl))
    assert f"{steps} steps in flight>" in named[named.index("few_down_kernel"):], named
    _check(sl, out)


@pytest.mark.parametrize("M,fused", [(6, True), (7, False), (8, False)])
def test_packed_layers_whose_tokens_may_share_experts_end_apart(M, fused):
    """Qwen3 dims, 4-bit: one launch at the end up to six tokens; with more, samples of one prompt would read shared weights too often."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], M=M, quant="w4"), "cuda", seed=M)
    _, named = _named(lambda: _call(sl))
    assert (FUSED in named) == fused, named


@pytest.mark.parametrize("fmt", ["int8", "fp8"])
@pytest.mark.parametrize("K,fused", [(1, True), (15, True), (16, False)])
@pytest.mark.parametrize("scales", [(1.0, 1.0), (0.5, 0.75)])
def test_shared_expert_rides_along(fmt, K, fused, scales):
    """A wave for the shared expert beside one per routed expert, up to 16; with the caller's epilogue (scale of the routed
    sum, scale of the shared expert's rows)."""
    from vllm_kunlun_amd import synth
    M, E = 3, 64
    big = E // K + 2
    shape = synth.scaled(synth.SHAPES["dsv3-fp8-decode" if fmt == "fp8" else "dsv3-decode"], M=big, H=384, E=E, K=K, I=256, I_shared=256, n_group=1,
                         topk_group=1)
    sl = synth.make_layer(shape, "cuda", seed=K)
    kw = dict(sl.apply_kwargs(), out_scale=scales[0], shared_scale=scales[1])
    m = sl.layer.quant_method
    whole = m.apply_monolithic(sl.layer, sl.x, sl.logits, **kw)
    part, named = _named(lambda: m.apply_monolithic(sl.layer, sl.x[:M].contiguous(), sl.logits[:M].contiguous(), **kw))
    assert (FUSED in named) == fused, named
    if fmt == "int8":
        assert torch.equal(part, whole[:M])
    else:
        assert rel_l2(part, whole[:M]) <= 4e-3


def test_batches_that_read_too_much_twice_stay_apart():
    from vllm_kunlun_amd import synth
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=14, H=2048, E=128, K=8, I=768)
    sl = synth.make_layer(shape, "cuda", seed=1)
    for M, fused in ((1, True), (10, True), (14, False)):
        out, named = _named(lambda: sl.layer(sl.x[:M], sl.logits[:M]))
        assert (FUSED in named) == fused, (M, named)
        assert torch.equal(out, sl.layer(sl.x, sl.logits)[:M])


@pytest.mark.parametrize("fmt,dims,most", [("int8", dict(H=7168, E=48, K=4, I=2048), 2),   # 59 MB a token
                                           ("fp8", dict(H=4096, E=176, K=4, I=1536), 4),   # 25 MB
                                           ("w4", dict(H=7168, E=128, K=4, I=2048), 2)])    # 29 MB
def test_batches_that_could_read_too_much_twice_stay_apart(fmt, dims, most):
    """Up to `most` tokens end in one launch: with one more, tokens that all chose the same experts would lose more there than
    tokens of uniform routing gain. The bits (int8) are the same on both sides, with such tokens."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], M=most + 1, quant=fmt, **dims), "cuda", seed=2)
    sl.logits[:, :dims["K"]] += 12.0
    part, named = _named(lambda: sl.layer(sl.x[:most], sl.logits[:most]))
    assert FUSED in named, named
    whole, named = _named(lambda: sl.layer(sl.x, sl.logits))
    assert FUSED not in named, named
    if fmt == "int8":
        assert torch.equal(part, whole[:most])
    else:
        assert rel_l2(part, whole[:most]) <= 4e-3


ROUTED = "routing, quantisation, sort and gate_up"


@pytest.mark.parametrize("fmt", ["int8", "fp8", "none", "w4"])
@pytest.mark.parametrize("M,K,E", [(1, 1, 2), (1, 16, 17), (2, 8, 128), (3, 6, 129), (4, 16, 65), (4, 8, 256), (4, 3, 257), (3, 8, 512),
                                   (4, 4, 513), (5, 4, 128)])
@pytest.mark.parametrize("H", [128, 640])
def test_routing_in_the_gate_up_launch(fmt, M, K, E, H):
    """Up to four tokens are routed, quantised and sorted by the gate_up launch: experts on both sides of a wave's 64 slots,
    tokens that share experts, parts of K that are empty for some waves. Against the same tokens in a batch with a
    column per expert."""
    from vllm_kunlun_amd import synth
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=max(M + 1, E // K + 2), H=H, E=E, K=K, I=128, quant=fmt)
    sl = synth.make_layer(shape, "cuda", seed=M * E + K)
    sl.logits[:M, :K // 2] += 4.0  # shared experts
    whole = sl.layer(sl.x, sl.logits)
    part, named = _named(lambda: sl.layer(sl.x[:M], sl.logits[:M]))
    assert (ROUTED in named) == (M <= 4 and M * K < E and E <= 512), named
    if fmt == "int8":
        assert torch.equal(part, whole[:M])
    else:
        assert rel_l2(part, whole[:M]) <= 4e-3


@pytest.mark.parametrize("fmt,M,fused", [("int8", 3, True), ("int8", 4, False), ("fp8", 3, True), ("fp8", 4, False), ("none", 1, True),
                                         ("none", 2, False), ("w4", 1, True), ("w4", 2, False)])
def test_long_rows_stay_apart(fmt, M, fused):
    """The gate_up launch holds all its rows in LDS: where they are too long for five workgroups a CU, routing is a launch of
    its own again; a shared expert's column has a row per token."""
    from vllm_kunlun_amd import synth
    E, K = 32, 4
    shared = fmt in ("int8", "fp8")
    base = "qwen3-decode" if not shared else ("dsv3-fp8-decode" if fmt == "fp8" else "dsv3-decode")
    over = dict(I_shared=128, n_group=4, topk_group=2) if shared else {}
    shape = synth.scaled(synth.SHAPES[base], M=E // K + 2, H=7168, E=E, K=K, I=128, quant=fmt, **over)
    sl = synth.make_layer(shape, "cuda", seed=3)
    sl.logits[:M, :K] += 6.0  # every token on the same experts
    kw = sl.apply_kwargs()
    m = sl.layer.quant_method
    run = (lambda x, l: m.apply_monolithic(sl.layer, x, l, **kw)) if shared else (lambda x, l: sl.layer(x, l))  # noqa: E731
    whole = run(sl.x, sl.logits)
    part, named = _named(lambda: run(sl.x[:M].contiguous(), sl.logits[:M].contiguous()))
    assert (ROUTED in named) == fused, named
    if fmt == "int8":
        assert torch.equal(part, whole[:M])
    else:
        assert rel_l2(part, whole[:M]) <= 4e-3


@pytest.mark.parametrize("kind", ["nan", "inf", "zero", "tiny"])
def test_rows_that_are_not_all_numbers(kind):
    """int8: a token whose row has a NaN, an infinity or nothing to scale by gets the codes the quantiser gives it, and the
    other tokens keep their results."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], M=10, H=640, E=64, K=8, I=128), "cuda", seed=9)
    value = {"nan": float("nan"), "inf": float("inf"), "zero": 0.0, "tiny": 1e-40}[kind]
    if kind in ("zero", "tiny"):
        sl.x[1] = 0
    sl.x[1, 639] = value
    whole = sl.layer(sl.x, sl.logits)
    part, named = _named(lambda: sl.layer(sl.x[:3], sl.logits[:3]))
    assert ROUTED in named
    assert torch.equal(part.view(torch.int16)[[0, 2]], whole[:3].view(torch.int16)[[0, 2]])
    assert torch.equal(torch.isnan(part[1]), torch.isnan(whole[1])) and torch.equal(part[1].nan_to_num(), whole[1].nan_to_num())


def _oracle(sl, M):
    """The C oracle's output of a layer's first M tokens."""
    s, f16 = sl.shape, sl.x.dtype == torch.float16
    w13, a13, w2, a2, shared = sl.host_weights()
    kw = dict(K=s.K, scoring=s.scoring, n_group=s.n_group, topk_group=s.topk_group, routed_scale=s.routed_scale, f16=f16,
              bias=None if sl.bias is None else sl.bias.cpu().numpy())
    x, logits = bits(sl.x[:M]), sl.logits[:M].float().cpu().numpy()
    if s.quant == "int8":
        shared = None if shared is None else tuple(t.numpy() for t in shared)
        return co.forward_w8a8(x, logits, w13.numpy(), a13.numpy(), w2.numpy(), a2.numpy(), shared=shared, **kw)
    if s.quant == "fp8":
        w13, w2 = w13.view(torch.uint8), w2.view(torch.uint8)
        shared = None if shared is None else tuple((t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t).numpy() for t in shared)
        return co.forward_fp8(x, logits, w13.numpy(), a13.numpy(), w2.numpy(), a2.numpy(), shared=shared, **kw)
    if s.quant == "w4":
        return co.forward_bf16(x, logits, co.dequant_w4_bf16(w13.numpy(), bits(a13), s.group_size, f16=f16),
                               co.dequant_w4_bf16(w2.numpy(), bits(a2), s.group_size, f16=f16), **kw)
    return co.forward_bf16(x, logits, bits(w13), bits(w2), **kw)


def _call(sl):
    if sl.shared is None:
        return sl.layer(sl.x, sl.logits)
    return sl.layer.quant_method.apply_monolithic(sl.layer, sl.x, sl.logits, **sl.apply_kwargs())


def _check(sl, out):
    """int8: the oracle's bits. Elsewhere the oracle's sums run in another order, which moves a 16-bit result by its rounding
    (2^-9 of it, and the same again behind the second GEMM): 4e-3."""
    ref = _oracle(sl, sl.shape.M)
    if sl.shape.quant == "int8":
        assert (bits(out) == ref).all()
    else:
        assert rel_l2(out, from_bits(ref).view(out.dtype)) <= 4e-3


@pytest.mark.parametrize("fmt,dims,dtype", [
    ("int8", dict(M=6, H=2048, E=64, K=8, I=768), torch.bfloat16),     # 75 MB of down projections
    ("int8", dict(M=9, H=1024, E=256, K=16, I=512), torch.float16),    # 75 MB, 144 pairs
    ("int8", dict(M=3, H=4096, E=96, K=6, I=1024, I_shared=1024, n_group=1, topk_group=1), torch.bfloat16),  # ... a shared expert
    ("fp8", dict(M=4, H=4096, E=96, K=4, I=1152), torch.bfloat16),
    ("none", dict(M=6, H=2048, E=64, K=6, I=512), torch.bfloat16),
    ("none", dict(M=6, H=2048, E=64, K=6, I=512), torch.float16),
    ("w4", dict(M=2, H=4096, E=128, K=16, I=1152), torch.bfloat16)], ids=str)
@pytest.mark.parametrize("common", [0, 1, 2])
def test_down_projections_of_more_than_64_mb(fmt, dims, dtype, common):
    """Launches of few tokens' down projection beyond 64 MB: experts of one token, of some and (`common` of them) of every
    token, against the oracle."""
    from vllm_kunlun_amd import synth
    base = "dsv3-decode" if "I_shared" in dims else "qwen3-decode"
    sl = synth.make_layer(synth.scaled(synth.SHAPES[base], quant=fmt, **dims), "cuda", seed=common, dtype=dtype)
    M, E = dims["M"], dims["E"]
    if common == 0:  # no expert twice (as far as they go)
        for m in range(M):
            sl.logits[m, [(m * dims["K"] + k) % E for k in range(dims["K"])]] += 9.0
    sl.logits[:, :common] += 12.0
    out, named = _named(lambda: _call(sl))
    assert FUSED in named, named
    _check(sl, out)


@pytest.mark.parametrize("fmt,dims", [
    ("int8", dict(M=4, H=4096, E=40, K=4, I=768)),                   # 101 MB of gate_up projections
    ("int8", dict(M=3, H=4096, E=48, K=8, I=768, I_shared=768, n_group=4, topk_group=2)),   # ... sigmoid routing, a shared expert
    ("fp8", dict(M=4, H=4096, E=40, K=4, I=640)),
    ("fp8", dict(M=4, H=4096, E=40, K=4, I=640, I_shared=640, n_group=4, topk_group=2)),
    ("none", dict(M=3, H=2048, E=40, K=8, I=768)),
    ("w4", dict(M=2, H=4096, E=80, K=16, I=640))], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("common", [0, 2])
def test_gate_up_projections_of_more_than_64_mb(fmt, dims, dtype, common):
    """Layers whose first launch routes and streams more than 64 MB, so that it reads its weights past the caches, with experts of one
    token and (`common` of them) of every token, against the oracle."""
    from vllm_kunlun_amd import synth
    base = ("dsv3-fp8-decode" if fmt == "fp8" else "dsv3-decode") if "I_shared" in dims else "qwen3-decode"
    sl = synth.make_layer(synth.scaled(synth.SHAPES[base], quant=fmt, **dims), "cuda", seed=7 + common, dtype=dtype)
    sl.logits[:, :common] += 12.0
    out, named = _named(lambda: _call(sl))
    assert ROUTED in named, named
    _check(sl, out)


@pytest.mark.parametrize("fmt", ["int8", "fp8", "none", "w4"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,H,I", [(1, 8, 640, 384), (4, 6, 256, 1152), (7, 3, 1152, 128), (9, 8, 256, 1024)])
def test_few_tokens_match_the_oracle(fmt, dtype, M, K, H, I):
    """Batches on both sides of the launch that routes (4 tokens), experts shared and not."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], M=M, H=H, E=96, K=K, I=I, quant=fmt), "cuda", seed=M, dtype=dtype)
    sl.logits[:, :K // 3] += 9.0
    out, named = _named(lambda: _call(sl))
    assert FUSED in named and (ROUTED in named) == (M <= 4), named
    _check(sl, out)


@pytest.mark.parametrize("dims,shape", [
    (dict(M=5, E=48, K=4, H=3072, I=2176), "4 channel fragments"),   # 20 columns, whose down launch splits 17 steps
    (dict(M=5, E=40, K=6, H=3072, I=384), "2 channel fragments"),    # few workgroups
    (dict(M=9, E=96, K=8, H=3200, I=640), "4 channel fragments"),    # 25 steps; a column per pair
    (dict(M=20, E=64, K=4, H=3072, I=512), "4 channel fragments"),   # ... per expert
    (dict(M=6, E=96, K=4, H=2944, I=640), None)], ids=str)            # shorter rows
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_packed_launches_on_long_rows_match_the_oracle(dims, shape, dtype):
    """4-bit layers of a few tokens whose gate_up launch splits its long rows over four waves, with as many channels a wave as leave
    enough workgroups."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], quant="w4", **dims), "cuda", seed=dims["M"], dtype=dtype)
    out, named = _named(lambda: _call(sl))
    gate_up = [k for k in named.replace(">", ">\n").splitlines() if "SiLU-mul" in k]
    assert len(gate_up) == 1 and "sorts the pairs itself" in gate_up[0], named
    assert ("K split 4" in gate_up[0]) == (shape is not None) and (shape is None or shape in gate_up[0]), named
    if dims["I"] > 2048:
        assert "plain" in named and named.count("K split 4") == 2, named
    _check(sl, out)


@pytest.mark.parametrize("fmt,dims,launches", [
    ("int8", dict(M=7, E=256, K=4, H=1600, I=512), ["SiLU-mul, 4 steps in flight, K split 2"]),   # 25 steps
    ("fp8", dict(M=7, E=256, K=4, H=3200, I=512), ["SiLU-mul, 2 steps in flight, K split 2"]),    # 25 steps
    ("none", dict(M=9, E=64, K=7, H=4096, I=2048), ["SiLU-mul, 4 steps in flight, K split 4", "plain, 4 steps in flight, K split 4"]),
    ("none", dict(M=9, E=96, K=7, H=3040, I=2016), ["SiLU-mul, 4 steps in flight, K split 2", "plain, 4 steps in flight, K split 2"]),
    ("none", dict(M=16, E=96, K=4, H=3072, I=2048), ["SiLU-mul, 4 steps in flight, K split 2", "plain, 4 steps in flight, K split 2"]),
    ("none", dict(M=9, E=64, K=4, H=1024, I=512), ["SiLU-mul, 2 steps in flight, K split 4"]),
    ("none", dict(M=16, E=48, K=4, H=2048, I=512), ["SiLU-mul, 4 steps in flight, K split 4"]),   # a column per expert
    ("none", dict(M=16, E=48, K=4, H=2016, I=512), ["SiLU-mul, 2 steps in flight, K split 4"]),
    ("none", dict(M=16, E=31, K=4, H=2048, I=512), ["SiLU-mul, 2 steps in flight, K split 4"])], ids=str)   # fewer workgroups than CUs
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_columns_of_pairs_of_large_layers_match_the_oracle(fmt, dims, launches, dtype):
    """Layers of a few tokens, whose column-per-pair launches split K over four waves where they are large, have 16-bit weights, long rows and
    few columns; steps in flight of smaller ones."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], quant=fmt, **dims), "cuda", seed=dims["M"], dtype=dtype)
    out, named = _named(lambda: _call(sl))
    assert all(k in named for k in launches) and ("a column per pair" in named) == (dims["M"] * dims["K"] < dims["E"]), named
    _check(sl, out)


@pytest.mark.parametrize("fmt,H,M,dtype,fragments", [
    ("int8", 4160, 32, torch.float16, 4), ("int8", 4160, 31, torch.bfloat16, 2), ("int8", 4096, 32, torch.bfloat16, 2),
    ("fp8", 6272, 32, torch.bfloat16, 4), ("fp8", 6144, 32, torch.float16, 2), ("fp8", 8064, 32, torch.bfloat16, 4), ("fp8", 8192, 32, torch.bfloat16, 2)])
def test_four_rows_per_expert_of_large_layers_match_the_oracle(fmt, H, M, dtype, fragments):
    """gate_up launches of large layers with long rows from four rows per expert on, whose waves take four channel fragments; some experts have
    more rows than a pass, some none."""
    from vllm_kunlun_amd import synth
    sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], quant=fmt, M=M, E=32, K=4, H=H, I=4096), "cuda", seed=H, dtype=dtype)
    sl.logits[:20, :2] += 9.0
    sl.logits[:, 30:] -= 9.0
    out, named = _named(lambda: _call(sl))
    assert f"{fragments} channel fragments per wave, SiLU-mul, {2 if fmt == 'fp8' else 4} steps in flight, K split {fragments}" in named, named
    _check(sl, out)


@pytest.mark.parametrize("fmt,I_shared", [("int8", 0), ("int8", 2048), ("fp8", 0), ("fp8", 2048), ("none", 0), ("w4", 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_most_rows_of_the_greatest_length(fmt, I_shared, dtype):
    """Sixteen waves with rows of 2048 values, the most LDS the launch asks for (16-bit rows: more than 64 KB), against the oracle."""
    from vllm_kunlun_amd import synth
    base, K = ("dsv3-fp8-decode" if fmt == "fp8" else "dsv3-decode", 15) if I_shared else ("qwen3-decode", 16)
    over = dict(I_shared=I_shared, n_group=1, topk_group=1) if I_shared else {}
    sl = synth.make_layer(synth.scaled(synth.SHAPES[base], M=1, H=256, E=32, K=K, I=2048, quant=fmt, **over), "cuda", seed=K, dtype=dtype)
    out, named = _named(lambda: _call(sl))
    assert FUSED in named and "16 waves" in named, named
    _check(sl, out)


@pytest.mark.parametrize("variable", ["KMOE_QUANT_IN_GEMM", "KMOE_SORT_IN_GEMM"])
def test_switches_keep_the_launches_apart(variable):
    """Each of them set to 0 (read once per process, hence a child process) gives a few-token layer its launches back: the output
    bits stay (int8), and the first quantisation's codes and maxima stand in the workspace."""
    import subprocess
    code = r"""
import sys, zlib
sys.path.insert(0, sys.argv[1]); sys.path.insert(0, sys.argv[2])
import torch
from vllm_kunlun_amd import _lib as L, synth
sl = synth.make_layer(synth.scaled(synth.SHAPES["qwen3-decode"], M=3, H=512, E=64, K=6, I=768), "cuda", seed=4)
m = sl.layer.quant_method
L.lib.kmoe_trace_kernels(1)
out = sl.layer(sl.x, sl.logits)
L.lib.kmoe_trace_kernels(0)
named = L.lib.kmoe_traced_kernels().decode()
lay, ws = m.last_layout, m.last_workspace
x_max = ws[lay.xmax: lay.xmax + 12].view(torch.float32)
print(zlib.crc32(out.view(torch.int16).cpu().numpy().tobytes()), int("few_" in named), int(torch.equal(x_max, sl.x.float().abs().amax(1))))
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = []
    for flag in ("1", "0"):
        run = subprocess.run([sys.executable, "-c", code, root, os.path.join(root, "vllm-kunlun_amd")], env=dict(os.environ, **{variable: flag}),
                             capture_output=True, text=True, timeout=110)
        assert run.returncode == 0, run.stderr[-2000:]
        got.append(run.stdout.split())
    assert got[0][0] == got[1][0] and got[0][1] == "1" and got[1][1:] == ["0", "1"], got


@pytest.mark.parametrize("fmt,H", [("int8", 128), ("int8", 7680), ("int8", 7808), ("int8", 8448), ("int8", 8576), ("fp8", 256), ("fp8", 8192),
                                   ("none", 7680), ("none", 12672), ("w4", 256), ("w4", 7808)])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("infinite", [False, True])
def test_one_token_whose_row_the_other_waves_bring(fmt, H, grouped, infinite):
    """One token: waves 1 to 3 bring its row to LDS, in one round of loads up to 7680 values, beside the routing's scores (sigmoid),
    int8 up to 8448 values, whose copy in 16 bits shares the space; with an infinity in the row, which the usual way does not take."""
    from vllm_kunlun_amd import synth
    base = ("dsv3-fp8-decode" if fmt == "fp8" else "dsv3-decode") if grouped and fmt in ("int8", "fp8") else "qwen3-decode"
    over = dict(I_shared=128, n_group=4, topk_group=2) if base != "qwen3-decode" else {}
    sl = synth.make_layer(synth.scaled(synth.SHAPES[base], M=1, H=H, E=96, K=4, I=128, quant=fmt, **over), "cuda", seed=H)
    if infinite:
        sl.x[0, H - 3] = float("inf")
    out, named = _named(lambda: _call(sl))
    assert ROUTED in named, named
    if infinite:  # as the launches apart make it
        two = torch.cat([sl.x, sl.x[:0].new_zeros(40, H)])
        logits = torch.cat([sl.logits, sl.logits.new_zeros(40, sl.logits.shape[1])])
        sl.x, sl.logits = two, logits
        whole = _call(sl)[:1]
        for value in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(value(out), value(whole))
        assert rel_l2(out.nan_to_num(0, 0, 0), whole.nan_to_num(0, 0, 0)) <= 4e-3
    else:
        _check(sl, out)


@pytest.mark.parametrize("fmt,H", [("int8", 128), ("int8", 7680), ("int8", 7808), ("int8", 8448), ("fp8", 256), ("fp8", 8192)])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("kind", ["nan", "nans", "zero", "tiny", "huge"])
def test_one_token_whose_row_is_not_all_numbers(fmt, H, grouped, kind):
    """A row that the other waves bring and whose result is finite all the same: a NaN in each wave's part (no maximum, the lowest
    code), nothing but zeros, values so small that their scale has no reciprocal, the type's largest. int8: the oracle's bits."""
    from vllm_kunlun_amd import synth
    base = ("dsv3-fp8-decode" if fmt == "fp8" else "dsv3-decode") if grouped else "qwen3-decode"
    over = dict(I_shared=128, n_group=4, topk_group=2) if grouped else {}
    sl = synth.make_layer(synth.scaled(synth.SHAPES[base], M=1, H=H, E=96, K=4, I=128, quant=fmt, **over), "cuda", seed=H)
    at = [3, H // 3 + 1, H - 3]
    if kind == "nan":
        sl.x[0, H - 3] = float("nan")
    elif kind == "nans":
        sl.x[0, at] = float("nan")
    elif kind == "huge":
        sl.x[0, at] = 3e38
    else:
        sl.x[0] = 0
        sl.x[0, at] = 1e-40 if kind == "tiny" else 0.0
    out, named = _named(lambda: _call(sl))
    assert ROUTED in named, named
    ref = from_bits(_oracle(sl, 1)).to(out.device)
    if kind == "huge":  # (its products may overflow: then where and to what is the oracle's, too)
        for value in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(value(out), value(ref))
        out, ref = out.nan_to_num(0, 0, 0), ref.nan_to_num(0, 0, 0)
    assert bool(torch.isfinite(out).all())
    if fmt == "int8":
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    else:
        # the two roundings of _check, and the codes between them: an activation rounded the other way (2^-8 of it) moves its fp8 code (steps
        # of 2^-4) one time in sixteen, sqrt(s / 16) 2^-4 for a share s of them: 8e-3 for a quarter, with the roundings 9e-3
        assert rel_l2(out, ref) <= 9e-3
