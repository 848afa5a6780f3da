"""The work whose speed this repository is held to: one MoE layer call (and one dense W8A8 MLP) per pass, through the
entry points a serving engine calls, on the layer shapes of the benchmark (Qwen3-30B-A3B, DeepSeek-V3, Kimi-K2).

A state is what the engine has in hand at that moment: a layer whose weights went through
process_weights_after_loading, a batch of hidden states and the router logits (or the gate's weight where the gate
projection runs inside the call). A pass is the call itself, host code included.
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

_PACKAGE = os.path.join(os.getcwd(), "vllm-kunlun_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

# hidden, experts, experts per token, intermediate, routing, scale of the routed sum, shared expert's intermediate,
# largest batch. The token range goes from one request's decode step to the prefill chunk of the benchmark.
MODELS = {
    "qwen3": dict(H=2048, E=128, K=8, I=768, scoring="softmax", n_group=1, topk_group=1, scale=1.0, most=8192),
    "dsv3": dict(H=7168, E=256, K=8, I=2048, scoring="sigmoid", n_group=8, topk_group=4, scale=2.5, most=4096),
    "kimi": dict(H=7168, E=384, K=8, I=2048, scoring="sigmoid", n_group=1, topk_group=1, scale=2.5, most=2048),
}
# what is served on which shape: (model, format)
SERVED = [("qwen3", "int8"), ("dsv3", "int8"), ("dsv3", "fp8"), ("qwen3", "bf16"), ("qwen3", "w4"), ("kimi", "w4"),
          ("dsv3", "linear")]
BYTES = {"int8": 1.0, "fp8": 1.0, "bf16": 2.0, "w4": 0.5, "linear": 1.0}
GROUP = {"qwen3": 128, "kimi": 32}  # values per scale of the 4-bit checkpoints


def _case(model, fmt, tokens, act="bf16", hot=0, gate=False, name=None):
    """hot: that many experts get +2.0 on their logits (an uneven load); gate: the router's projection runs inside the
    call; act: the activations' type."""
    c = dict(model=model, format=fmt, tokens=tokens, act=act, hot=hot, gate=gate)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one request decoding alone: latency, launches and host code
        _case("qwen3", "int8", 1, name="qwen3-int8-1"),
        # the decode batch of the benchmark
        _case("qwen3", "int8", 64, name="qwen3-int8-64"),
        # a mixed step of decodes and one prefill chunk: an odd size, an uneven load, float16 as the recipes run it
        _case("qwen3", "int8", 777, act="f16", hot=8, name="qwen3-int8-777-skew"),
        # the prefill chunk of the benchmark
        _case("qwen3", "int8", 8192, name="qwen3-int8-8192"),
        # the headline: a decode batch of the large model, gate and shared expert in the call
        _case("dsv3", "int8", 128, gate=True, name="dsv3-int8-128-gate"),
        # its prefill chunk
        _case("dsv3", "int8", 4096, name="dsv3-int8-4096"),
        # the same model from an fp8 block-scaled checkpoint: a small decode batch and a ragged prefill chunk
        _case("dsv3", "fp8", 23, name="dsv3-fp8-23"),
        _case("dsv3", "fp8", 3001, name="dsv3-fp8-3001"),
        # unquantized weights: a prefill chunk
        _case("qwen3", "bf16", 4096, name="qwen3-bf16-4096"),
        # 4-bit weights: a decode batch (groups of 128) and a prefill chunk of the largest model (groups of 32)
        _case("qwen3", "w4", 64, name="qwen3-w4-64"),
        _case("kimi", "w4", 2048, name="kimi-w4-2048"),
        # the shared expert as an engine runs it on its own: two W8A8 Linears around SiLU-mul
        _case("dsv3", "linear", 100, name="dsv3-linear-100"),
    ]


def draw(rng):
    model, fmt = rng.choice(SERVED)
    most = MODELS[model]["most"]
    tokens = max(1, min(most, int(round(math.exp(rng.uniform(0.0, math.log(most)))))))
    act = "f16" if rng.random() < 0.25 else "bf16"
    gate = model == "dsv3" and fmt != "linear" and rng.random() < 0.33
    hot = 8 if fmt != "linear" and not gate and rng.random() < 0.25 else 0
    return _case(model, fmt, tokens, act, hot, gate)


def _normal(shape, g, sigma, most, dtype):
    """Codes of quantised N(0, sigma) values, clamped to +-most."""
    v = torch.randn(shape, generator=g, device="cuda").mul_(sigma).clamp_(-most, most)
    return v.to(dtype) if dtype.is_floating_point else v.round_().to(dtype)


def _fill_codes(w, g, sigma, most):
    """Fills the [..., n, k] codes of a weight with quantised normal values, a few matrices at a time."""
    flat = w.view(-1, w.shape[-2], w.shape[-1])
    step = max(1, (1 << 27) // flat[0].numel())
    for e in range(0, flat.shape[0], step):
        part = flat[e:e + step]
        part.copy_(_normal(part.shape, g, sigma, most, part.dtype))


def _fill_nibbles(w, g, sigma):
    step = max(1, (1 << 26) // w[0].numel())
    for e in range(0, w.shape[0], step):
        part = w[e:e + step]
        low, high = (_normal(part.shape, g, sigma, 7, torch.int8).add_(8).view(torch.uint8) for _ in range(2))
        part.copy_(low | (high << 4))


def _fill_scales(s, g, value):
    s.copy_(torch.randn(s.shape, generator=g, device="cuda").mul_(0.03).clamp_(-0.2, 0.2).add_(1.0).mul_(value))


def _make_linear(m, g):
    """The two Linears of a dense MLP after loading: gate_up [2I, H] and down [H, I]."""
    from vllm_kunlun_amd.quantization.kernels.scale_mm import KunlunScaledMMLinearKernel
    kernel, layers = KunlunScaledMMLinearKernel(), []
    for n, k in ((2 * m["I"], m["H"]), (m["H"], m["I"])):
        layer = torch.nn.Module()
        w, s = torch.empty((n, k), dtype=torch.int8, device="cuda"), torch.empty((n, 1), device="cuda")
        _fill_codes(w, g, 36.0, 127)
        _fill_scales(s, g, 0.02 / 36.0)
        layer.weight = torch.nn.Parameter(w, requires_grad=False)
        layer.weight_scale = torch.nn.Parameter(s, requires_grad=False)
        kernel.process_weights_after_loading(layer)
        layers.append(layer)
    return SimpleNamespace(kernel=kernel, up=layers[0], down=layers[1])


def _make_layer(m, model, fmt, act, g):
    """The FusedMoE layer of a checkpoint with weights ~ N(0, 0.02), after process_weights_after_loading."""
    from vllm_kunlun_amd.ops.fused_moe.layer import FusedMoE
    from vllm_kunlun_amd.quantization.compressed_tensors import compressed_tensors_moe as ct
    method = None
    if fmt == "int8":
        method = ct.KunlunCompressedTensorsW8A8Int8MoEMethod()
    elif fmt == "fp8":
        method = ct.KunlunCompressedTensorsW8A8Fp8MoEMethod()
    elif fmt == "w4":
        scheme = SimpleNamespace(num_bits=4, type="int", symmetric=True, dynamic=False, strategy="group",
                                 group_size=GROUP[model])
        method = ct.KunlunCompressedTensorsWNA16MoEMethod(scheme, None, None)
    bias = torch.randn(m["E"], generator=g, device="cuda") * 0.01 if m["scoring"] == "sigmoid" else None
    layer = FusedMoE(num_experts=m["E"], top_k=m["K"], hidden_size=m["H"], intermediate_size=m["I"], renormalize=True,
                     use_grouped_topk=m["n_group"] > 1, num_expert_group=m["n_group"], topk_group=m["topk_group"],
                     scoring_func=m["scoring"], routed_scaling_factor=m["scale"], e_score_correction_bias=bias,
                     quant_method=method, device="cuda", params_dtype=act)
    with torch.no_grad():
        for name in ("w13", "w2"):
            w = getattr(layer, name + ("_weight_packed" if fmt == "w4" else "_weight")).data
            if fmt == "bf16":
                _fill_codes(w, g, 0.02, 1.0)
                continue
            sigma = {"int8": 36.0, "fp8": 107.0, "w4": 2.5 if GROUP.get(model) == 128 else 3.3}[fmt]
            if fmt == "w4":
                _fill_nibbles(w, g, sigma)
            else:
                _fill_codes(w, g, sigma, 127 if fmt == "int8" else 448)
            _fill_scales(getattr(layer, name + "_weight_scale").data, g, 0.02 / sigma)
    layer.quant_method.process_weights_after_loading(layer)
    return layer


def _make_shared(m, fmt, g):
    """The dense shared expert in the layer's format, tiled as the routed weights are: what `shared_expert=` takes."""
    from vllm_kunlun_amd._plan import tile_pair_
    dtype = torch.int8 if fmt == "int8" else torch.float8_e4m3fn
    sigma, most = (36.0, 127) if fmt == "int8" else (107.0, 448)
    out = []
    for n, k in ((2 * m["I"], m["H"]), (m["H"], m["I"])):
        w = torch.empty((n, k), dtype=dtype, device="cuda")
        s = torch.empty((n,) if fmt == "int8" else (n // 128, k // 128), device="cuda")
        _fill_codes(w, g, sigma, most)
        _fill_scales(s, g, 0.02 / sigma * (127.0 if fmt == "int8" else 1.0))  # int8: the channel's largest magnitude
        out += [w, s]
    tile_pair_(out[0], out[2])
    return tuple(out)


def prepare(case, seed):
    m, fmt, M = MODELS[case["model"]], case["format"], case["tokens"]
    act = torch.float16 if case["act"] == "f16" else torch.bfloat16
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    state = SimpleNamespace(case=case)
    state.x = torch.randn((M, m["H"]), generator=g, device="cuda").to(act)
    if fmt == "linear":
        state.mlp = _make_linear(m, g)
        return state
    state.kwargs = {}
    if case["model"] == "dsv3":
        state.kwargs["shared_expert"] = _make_shared(m, fmt, g)
    logits = torch.randn((M, m["E"]), generator=g, device="cuda")
    if case["gate"]:
        gate = torch.randn((m["E"], m["H"]), generator=g, device="cuda") * (1.0 / math.sqrt(m["H"]))
        state.kwargs["router_weight"] = gate.to(act)
        state.logits = None
    else:
        if case["hot"]:
            logits[:, torch.arange(case["hot"], device="cuda") * (m["E"] // case["hot"])] += 2.0
        # Qwen3's gate is an ordinary 16-bit Linear; the sigmoid-routed models' gate gives float32
        state.logits = logits.to(act) if case["model"] == "qwen3" else logits
    state.layer = _make_layer(m, case["model"], fmt, act, g)
    return state


def run(state):
    if state.case["format"] == "linear":
        mlp = state.mlp
        y = mlp.kernel.apply_weights(mlp.up, state.x)
        h = torch.empty((y.shape[0], y.shape[1] // 2), dtype=y.dtype, device=y.device)
        torch.ops._C.silu_and_mul(h, y)
        return mlp.kernel.apply_weights(mlp.down, h)
    layer = state.layer
    if state.kwargs:
        return layer.quant_method.apply_monolithic(layer, state.x, state.logits, **state.kwargs)
    return layer(state.x, state.logits)


def work(case):
    """Every expert that is hit is read once (with its scales), the batch and the logits (or the gate) are read once,
    the result is written once; two operations per weight and row."""
    m, fmt, M = MODELS[case["model"]], case["format"], case["tokens"]
    H, I, E, K = m["H"], m["I"], m["E"], m["K"]
    weights = 3 * H * I

    def one_expert(n13, n2):
        scales = {"int8": 4 * (n13 + n2), "linear": 4 * (n13 + n2), "fp8": 4 * weights // (128 * 128), "bf16": 0,
                  "w4": 2 * weights // GROUP.get(case["model"], 128)}[fmt]
        return weights * BYTES[fmt] + scales

    if fmt == "linear":
        return {"bytes": one_expert(2 * I, H) + 2 * M * H * 2, "flops": 2.0 * M * weights}
    hit = E * (1.0 - (1.0 - K / E) ** M)  # experts that at least one of M tokens chooses
    data = hit * one_expert(2 * I, H) + 2 * M * H * 2
    flops = 2.0 * M * K * weights
    if case["gate"]:
        data, flops = data + E * H * 2, flops + 2.0 * M * E * H
    else:
        data += M * E * (2 if case["model"] == "qwen3" else 4)
    if case["model"] == "dsv3":
        data, flops = data + one_expert(2 * I, H), flops + 2.0 * M * weights
    return {"bytes": data, "flops": flops}


def tolerance(case):
    """16-bit results of products whose operands and intermediate rows are rounded to 8 or 16 bits: a correct
    implementation that rounds an intermediate the other way now and then stays within 1e-2."""
    return {"rel": 1e-2}
