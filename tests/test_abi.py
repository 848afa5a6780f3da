"""The C ABI without a GPU: libkmoe.so loads, exports every function that
include/kmoe.h declares, and rejects bad arguments with status codes before any
HIP call (so these run on a CPU-only host). No compute call is made here."""
import ctypes as C
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def L():
    from vllm_kunlun_amd import _lib
    return _lib


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "kmoe.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(kmoe_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_functions():
    names = _declared_functions()
    assert "kmoe_moe_forward" in names and "kmoe_grouped_gemm_i8" in names and len(names) >= 15


def test_library_exports_every_declared_symbol(L):
    for name in _declared_functions():
        assert hasattr(L.lib, name), f"{name} is declared in include/kmoe.h but not exported by libkmoe.so"
    assert set(_declared_functions()) == set(L.EXPORTS), "the ctypes binding must cover exactly the declared ABI"
    assert b"gfx950" in L.lib.kmoe_version()


def test_struct_layouts_match_the_header(L, tmp_path):
    """The ctypes mirrors against the C declarations themselves: a C program that includes include/kmoe.h
    prints sizeof and the offsets of a few late fields of every argument struct (gcc, host only)."""
    import subprocess
    structs = {"kmoe_gemm_i8_args": (L.GemmI8Args, ["lod", "acc_out", "w_tail", "tail_src0", "act_dtype"]),
               "kmoe_gemm_bf16_args": (L.GemmBf16Args, ["lod", "y", "bias", "act_limit"]),
               "kmoe_gemm_fp8_args": (L.GemmFp8Args, ["w_scale", "y", "w_tail", "tail_src0"]),
               "kmoe_gemm_w4_args": (L.GemmW4Args, ["w_scale", "lod", "y", "w_layout"]),
               "kmoe_moe_args": (L.MoEArgs, ["logits", "I_shared", "out", "w_gate", "ws_layout", "group_size",
                                             "act_dtype", "shared_scale", "tile_variant", "first_expert", "flags"]),
               "kmoe_moe_layout": (L.MoELayout, ["align_ws", "down", "sh_out", "n_logit_planes"])}
    lines = ["#include <stdio.h>", "#include <stddef.h>", '#include "kmoe.h"', "int main(void) {"]
    for name, (_, fields) in structs.items():
        lines.append(f'  printf("{name} %zu", sizeof({name}));')
        for f in fields:
            lines.append(f'  printf(" %zu", offsetof({name}, {f}));')
        lines.append('  printf("\\n");')
    lines += ["  return 0;", "}"]
    src = tmp_path / "layout.c"
    src.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    for line in filter(None, out):
        name, size, *offsets = line.split()
        cls, fields = structs[name]
        assert C.sizeof(cls) == int(size), name
        assert [getattr(cls, f).offset for f in fields] == [int(o) for o in offsets], name


def test_null_and_shape_errors_are_status_codes(L):
    lib = L.lib
    assert lib.kmoe_softmax_topk(None, 4, 8, 2, 1, None, None, None) == -1
    assert b"NULL" in lib.kmoe_last_error()
    one = C.c_void_p(0x1000)  # never dereferenced: validation fails first
    assert lib.kmoe_softmax_topk(one, 4, 0, 2, 1, one, one, None) == -2
    assert lib.kmoe_clock_probe(None, 1, 8, None) == -1
    assert lib.kmoe_clock_probe(one, 0, 8, None) == -2 and lib.kmoe_clock_probe(one, 1, 1, None) == -2
    assert lib.kmoe_softmax_topk(one, 4, 8, 9, 1, one, one, None) == -2          # K > E
    assert lib.kmoe_softmax_topk(one, 4, 2048, 8, 1, one, one, None) == -2       # E too large
    assert lib.kmoe_sigmoid_group_topk_norm(one, None, 4, 30, 4, 4, 2, 1.0, one, one, None) == -2  # E % n_group
    assert lib.kmoe_sigmoid_group_topk_norm(one, None, 4, 8, 4, 8, 2, 1.0, one, one, None) == -2   # groups of 1
    assert lib.kmoe_sigmoid_group_topk_norm(one, None, 4, 32, 8, 8, 1, 1.0, one, one, None) == -2  # K > kept experts
    assert lib.kmoe_align(one, 10, 4096, one, one, one, one, None, 0, None) == -2
    assert lib.kmoe_align(one, 100000, 64, one, one, one, one, None, 0, None) == -4  # needs a workspace
    assert b"workspace" in lib.kmoe_last_error()
    assert lib.kmoe_quant_i8_rows(one, 100, 4, 100, one, 100, one, None) == -2     # C % 8
    assert lib.kmoe_quant_fp8_group128(one, 200, 4, 200, one, 200, one, None) == -2
    assert lib.kmoe_silu_and_mul(one, 20, 4, 10, one, 10, None) == -2
    assert lib.kmoe_combine(one, 64, one, one, None, 4, 65, 64, 1.0, None, 0, one, 64, None) == -2  # K > 64
    assert lib.kmoe_grouped_gemm_i8(None, None) == -1


def test_gemm_argument_validation(L):
    g = L.GemmI8Args()
    assert L.lib.kmoe_grouped_gemm_i8(g, None) == -1
    for f in ("a", "a_max", "w", "w_max", "lod", "y"):
        setattr(g, f, 0x1000)
    g.E, g.n, g.k, g.rows, g.lda, g.ldy, g.src_div = 4, 64, 100, 10, 112, 64, 1
    assert L.lib.kmoe_grouped_gemm_i8(g, None) == -2 and b"k=100" in L.lib.kmoe_last_error()
    g.k, g.lda, g.act = 128, 128, 7
    assert L.lib.kmoe_grouped_gemm_i8(g, None) == -3
    g.act, g.n = 1, 48
    assert L.lib.kmoe_grouped_gemm_i8(g, None) == -2   # SwiGLU needs n % 32 == 0
    g.n, g.act, g.a = 64, 0, 0x1001
    assert L.lib.kmoe_grouped_gemm_i8(g, None) == -2 and b"misaligned" in L.lib.kmoe_last_error()
    # the tile kernel (variants 5-11) moves K in 128-byte chunks: a single 64-byte step is refused, not run
    g.a, g.k, g.lda, g.w_layout, g.variant = 0x1000, 64, 64, L.KMOE_W_TILED, 5
    assert L.lib.kmoe_grouped_gemm_i8(g, None) == -3 and b"k >= 128" in L.lib.kmoe_last_error()


def test_forward_validation_and_workspace_layout(L):
    a = L.MoEArgs()
    lay = L.MoELayout()
    a.M, a.H, a.E, a.K, a.I = 64, 2048, 128, 8, 768
    assert L.lib.kmoe_moe_workspace_layout(a, lay) == 0
    P = 64 * 8
    assert lay.total_bytes >= P * 2048 * 2 + P * 768 * 3 + 64 * 2048
    offs = [getattr(lay, n) for n, _ in L.MoELayout._fields_[1:-3]] + [lay.logit_planes]
    assert offs == sorted(offs) and all(o % 256 == 0 for o in offs)
    a.K = 200
    assert L.lib.kmoe_moe_workspace_layout(a, lay) == -2
    a.K = 8
    assert L.lib.kmoe_moe_forward(a, None, 0, None) == -1        # tensor pointers missing
    for f in ("logits", "x", "w13", "w13_max", "w2", "w2_max", "out"):
        setattr(a, f, 0x1000)
    assert L.lib.kmoe_moe_forward(a, None, 0, None) == -4        # no workspace
    assert L.lib.kmoe_moe_forward(a, C.c_void_p(0x10000), 16, None) == -4
    a.scoring = 9
    assert L.lib.kmoe_moe_forward(a, C.c_void_p(0x10000), 1 << 40, None) == -3


def test_python_errors_follow_the_reference_convention(L):
    with pytest.raises(ValueError):
        L.check(-2)
    with pytest.raises(NotImplementedError):
        L.check(-3)
    with pytest.raises(RuntimeError):
        L.check(-5)


def test_method_selection_mirrors_reference():
    """get_moe_method: same scheme for gate/up/down, None -> unquantized, dynamic-token
    W8A8 -> the int8 method, anything else -> RuntimeError (reference:
    compressed_tensors_moe.py:43-108)."""
    import torch
    from vllm_kunlun_amd.ops.fused_moe.layer import FusedMoEConfig, KunlunUnquantizedFusedMoEMethod
    from vllm_kunlun_amd.quantization.compressed_tensors.compressed_tensors_moe import (
        KunlunCompressedTensorsMoEMethod, KunlunCompressedTensorsW8A8Int8MoEMethod)

    class Cfg:
        def __init__(self, schemes):
            self.schemes = schemes

        def get_scheme_dict(self, layer, name):
            return self.schemes[name.rsplit(".", 1)[-1]]

    layer = torch.nn.Module()
    layer.moe_config = FusedMoEConfig(experts_per_token=2)
    w8 = {"weights": dict(num_bits=8, strategy="channel", symmetric=True, dynamic=False),
          "input_activations": dict(num_bits=8, strategy="token", symmetric=True, dynamic=True), "format": "int-quantized"}
    m = KunlunCompressedTensorsMoEMethod.get_moe_method(Cfg(dict(gate_proj=w8, up_proj=w8, down_proj=w8)), layer, "l.e")
    assert isinstance(m, KunlunCompressedTensorsW8A8Int8MoEMethod) and m.is_monolithic
    m = KunlunCompressedTensorsMoEMethod.get_moe_method(Cfg(dict(gate_proj=None, up_proj=None, down_proj=None)), layer,
                                                       "l.e")
    assert isinstance(m, KunlunUnquantizedFusedMoEMethod)
    with pytest.raises(ValueError):
        KunlunCompressedTensorsMoEMethod.get_moe_method(Cfg(dict(gate_proj=w8, up_proj=None, down_proj=w8)), layer, "l.e")
    static = dict(w8, input_activations=dict(num_bits=8, strategy="tensor", symmetric=True, dynamic=False))
    with pytest.raises(RuntimeError):
        KunlunCompressedTensorsMoEMethod.get_moe_method(Cfg(dict(gate_proj=static, up_proj=static, down_proj=static)),
                                                       layer, "l.e")


def test_process_weights_after_loading_turns_scales_into_maxes():
    import torch
    from vllm_kunlun_amd import synth
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=4, H=64, E=4, K=2, I=32)
    sl = synth.make_w8a8_layer(shape, "cpu", seed=0)
    w13 = sl.layer.w13_weight.float()
    mx = sl.layer.w13_weight_scale
    assert mx.shape == (4, 64, 1) and torch.all(mx > 0)
    assert torch.all(w13.abs().amax(-1, keepdim=True) == 127)      # per-channel quantisation reaches +-127
    before = mx.clone()
    sl.layer.quant_method.process_weights_after_loading(sl.layer)  # a second call multiplies again: it is in place
    assert torch.allclose(sl.layer.w13_weight_scale, before * 127.0)


def test_static_workspace_forward_refuses_what_does_not_fit(L):
    a = L.MoEArgs()
    a.M, a.H, a.E, a.K, a.I = 4096, 7168, 256, 8, 2048  # needs ~0.9 GB of intermediates
    a.format = L.KMOE_FMT_INT8
    assert L.lib.kmoe_moe_forward_static(C.byref(a), None) == -4
    assert b"built-in buffer" in L.lib.kmoe_last_error()


def test_kernel_trace_record_is_per_thread_and_empty_without_launches(L):
    lib = L.lib
    lib.kmoe_trace_kernels(1)
    assert lib.kmoe_traced_kernels() == b""
    lib.kmoe_trace_kernels(0)
    assert lib.kmoe_traced_kernels() == b""


@pytest.mark.skipif(torch.cuda.is_available(), reason="names the kernel a launch would take, on addresses that are not memory")
def test_packed_launches_on_rows_beyond_4_gib_do_not_take_32_bit_offsets(L):
    """Which kernel kmoe_grouped_gemm_w4a16 launches (the record is written before the launch, which fails without a
    GPU): 32-bit row offsets only where rows * lda * 2 bytes, and a row beyond, stay below 4 GiB and the rows are the
    launch's own."""
    def kernel(rows, lda, E=384, k=2048, act=0, variant=0, gather=False):
        g = L.GemmW4Args()
        for f in ("a", "w", "w_scale", "lod", "y"):
            setattr(g, f, 0x10000)
        g.row_src = 0x10000 if gather else None
        g.E, g.n, g.k, g.rows, g.lda, g.ldy, g.src_div = E, 7168, k, rows, lda, 7168, 1
        g.group_size, g.act, g.variant, g.w_layout = 32, act, variant, L.KMOE_W_TILED
        L.lib.kmoe_trace_kernels(1)
        assert L.lib.kmoe_grouped_gemm_w4a16(g, None) == -5
        L.lib.kmoe_trace_kernels(0)
        return L.lib.kmoe_traced_kernels().decode()

    most = (1 << 32) // (2 * 2048) - 2  # the most rows of 2048 values
    for rows in (384, most):
        assert "w4_tile_kernel" in kernel(rows, 2048)
    for rows in (most + 1, 131072 * 8):
        assert "stream_gemm_kernel" in kernel(rows, 2048) and "32-bit" not in kernel(rows, 2048)
    assert "32-bit" in kernel(384, 2048, act=1)                      # few rows per expert: the split launch
    assert "32-bit" not in kernel(384, 1 << 23, act=1)               # ... far apart
    assert "32-bit" not in kernel(2, 1 << 32, act=1)                 # (a stride whose product leaves 32 bits itself)
    assert "32-bit" not in kernel(384, 2048, act=1, gather=True)     # ... or gathered from who knows where
    for variant in (1, 2, 4):
        assert "32-bit" not in kernel(384, 2048, variant=variant) and "stream_gemm_kernel" in kernel(most + 1, 2048, variant=variant)
    g_tile = L.GemmW4Args()
    for f in ("a", "w", "w_scale", "lod", "y"):
        setattr(g_tile, f, 0x10000)
    g_tile.E, g_tile.n, g_tile.k, g_tile.rows, g_tile.lda, g_tile.ldy, g_tile.src_div = 4, 64, 128, 1 << 20, 4096, 64, 1
    g_tile.group_size, g_tile.variant, g_tile.w_layout = 32, 64, L.KMOE_W_TILED
    assert L.lib.kmoe_grouped_gemm_w4a16(g_tile, None) == -2 and b"32 bits" in L.lib.kmoe_last_error()


@pytest.mark.skipif(torch.cuda.is_available(), reason="names the kernel a launch would take, on addresses that are not memory")
@pytest.mark.parametrize("k,most", [(4096, 768), (4224, 96)])
def test_few_rows_per_expert_decide_the_packed_gate_up_kernel(L, k, most):
    """A packed gate_up launch on 384 experts: the streaming kernel up to two rows per expert, and with rows longer than 4096
    values up to a row for every fourth; tiles beyond, also where all but that many rows are other ranks'."""
    def kernel(rows, hint=0):
        g = L.GemmW4Args()
        for f in ("a", "w", "w_scale", "lod", "y"):
            setattr(g, f, 0x10000)
        g.E, g.n, g.k, g.rows, g.lda, g.ldy, g.src_div, g.rows_hint = 384, 4096, k, rows, k, 2048, 1, hint
        g.group_size, g.act, g.w_layout = 32, 1, L.KMOE_W_TILED
        L.lib.kmoe_trace_kernels(1)
        assert L.lib.kmoe_grouped_gemm_w4a16(g, None) == -5
        L.lib.kmoe_trace_kernels(0)
        return L.lib.kmoe_traced_kernels().decode()

    for rows, hint in ((1, 0), (most, 0), (8 * most, most)):
        assert "stream_gemm_kernel" in kernel(rows, hint)
    for rows, hint in ((most + 1, 0), (8 * most, 0), (8 * most, most + 1)):
        assert "w4_tile_kernel" in kernel(rows, hint)


@pytest.mark.skipif(torch.cuda.is_available(), reason="names the kernel a launch would take, on addresses that are not memory")
@pytest.mark.parametrize("E,n,k,top,most", [
    (384, 4096, 7168, 8, 16), (160, 3072, 5120, 6, 16),  # long rows: tokens that one pass holds, and at most a row per expert
    (64, 6144, 6144, 4, 16), (64, 4096, 7168, 8, 8),
    (128, 1536, 2048, 8, 48), (64, 5120, 3584, 6, 42),   # shorter: three passes, and at most four rows
    (32, 4096, 8192, 4, 8), (32, 2048, 2048, 4, 32)])    # few workgroups
def test_tokens_that_share_experts_decide_the_packed_gate_up_kernel(L, E, n, k, top, most):
    """A packed gate_up launch for a number of tokens, which the rows' sources say: where no expert can need more than a pass or a few, or tiles
    would leave the GPU idle, the streaming kernel, which splits the contraction, up to a row per expert (rows of at most 4096 values: four)."""
    def kernel(tokens):
        g = L.GemmW4Args()
        for f in ("a", "w", "w_scale", "lod", "y", "row_src"):
            setattr(g, f, 0x10000)
        g.E, g.n, g.k, g.rows, g.lda, g.ldy, g.src_div = E, n, k, tokens * top, k, n // 2, top
        g.group_size, g.act, g.w_layout = 32, 1, L.KMOE_W_TILED
        L.lib.kmoe_trace_kernels(1)
        assert L.lib.kmoe_grouped_gemm_w4a16(g, None) == -5
        L.lib.kmoe_trace_kernels(0)
        return L.lib.kmoe_traced_kernels().decode()

    for tokens in (1, 2, 5, 8, 13, most):
        assert ("stream_gemm_kernel" if tokens <= most else "w4_tile_kernel") in kernel(tokens)
    assert "w4_tile_kernel" in kernel(most + 1)


@pytest.mark.skipif(torch.cuda.is_available(), reason="names the kernel a launch would take, on addresses that are not memory")
@pytest.mark.parametrize("E,n,k,split", [(128, 2048, 3072, 4), (129, 2048, 3072, 2), (128, 8192, 3072, 2), (64, 8192, 3584, 4), (64, 8192, 4992, 4),
                                         (64, 16384, 3584, 2), (64, 16384, 4992, 2), (64, 16384, 5120, 4), (8, 8192, 2944, 2)])
def test_many_workgroups_of_short_work_split_packed_rows_two_ways(L, E, n, k, split):
    """A packed gate_up launch on the streaming kernel: rows from 3072 values on split four ways, shorter than 3584 and 5120 values only while
    that makes no more than 4096 and 8192 workgroups."""
    g = L.GemmW4Args()
    for f in ("a", "w", "w_scale", "lod", "y"):
        setattr(g, f, 0x10000)
    g.E, g.n, g.k, g.rows, g.lda, g.ldy, g.src_div = E, n, k, 4, k, n // 2, 1
    g.group_size, g.act, g.w_layout = 32, 1, L.KMOE_W_TILED
    L.lib.kmoe_trace_kernels(1)
    assert L.lib.kmoe_grouped_gemm_w4a16(g, None) == -5
    L.lib.kmoe_trace_kernels(0)
    assert f"K split {split}" in L.lib.kmoe_traced_kernels().decode()


@pytest.mark.skipif(torch.cuda.is_available(), reason="names the kernel a launch would take, on addresses that are not memory")
def test_dense_products_beyond_32_bit_offsets_stay_on_the_streaming_kernel(L):
    """kmoe_grouped_gemm_i8 with a tail matrix alone: the split-K kernel where its 32-bit offsets reach all activations (asked for
    the compute units first, which fails without a GPU), else the streaming kernel (noted before its launch fails)."""
    def call(a_rows, k):
        g = L.GemmI8Args()
        for f in ("a", "a_max", "w", "w_max", "lod", "y", "w_tail", "w_max_tail"):
            setattr(g, f, 0x10000)
        g.E, g.n, g.k, g.rows, g.ldy, g.a_rows, g.tail_rows = 1, 64, k, 0, 64, a_rows, 3
        g.w_layout, g.a_layout = L.KMOE_W_TILED, L.KMOE_A_CHUNKED
        L.lib.kmoe_trace_kernels(1)
        rc = L.lib.kmoe_grouped_gemm_i8(g, None)
        L.lib.kmoe_trace_kernels(0)
        return rc, L.lib.kmoe_traced_kernels().decode(), L.lib.kmoe_last_error()

    reach = 0xfff00000
    rc, kernel, error = call(reach // 4096 - 1, 4096)
    assert rc == -5 and kernel == "" and b"query the device" in error
    for a_rows in (reach // 4096, 1 << 20, (1 << 20) + 1):
        rc, kernel, error = call(a_rows, 4096)
        assert rc == -5 and "stream_gemm_kernel<i8" in kernel, (a_rows, error)
