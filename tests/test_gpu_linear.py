"""The dense W8A8 linear: the split-K kernel's tiles and channel fragments at their edges, and the
call kept on the layer following what changes in between."""
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), ".."))
from conftest import bits  # noqa: E402
from oracle import c_oracle as co  # noqa: E402

pytestmark = pytest.mark.gpu


def _linear(n, k, seed):
    from vllm_kunlun_amd.quantization.kernels.scale_mm import KunlunScaledMMLinearKernel
    g = torch.Generator().manual_seed(seed)
    layer = torch.nn.Module()
    codes = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    scale = torch.rand(n, generator=g) * 0.02 + 0.001
    layer.weight = torch.nn.Parameter(codes.cuda(), requires_grad=False)
    layer.weight_scale = torch.nn.Parameter(scale.cuda(), requires_grad=False)
    layer.input_scale = layer.input_zero_point = layer.azp_adj = None
    kern = KunlunScaledMMLinearKernel()
    kern.process_weights_after_loading(layer)
    return kern, layer, codes, layer.weight_scale.detach().cpu().reshape(-1)


# rows on both sides of the slices' sizes and of their choice, one channel fragment per wave and two, few K steps (an
# empty share for some of a workgroup's waves) and a remainder of the steps in flight
@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64, 65, 128, 129, 255, 257])
@pytest.mark.parametrize("n,k", [(16, 64), (64, 448), (4112, 192), (144, 1728), (48, 4160)])
def test_dense_slices(rows, n, k):
    kern, layer, codes, w_max = _linear(n, k, n + k)
    x = (torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)) * 1.5).bfloat16()
    out = kern.apply_weights(layer, x.cuda())
    xq, x_max = co.quant_i8_rows(bits(x))
    ref, _ = co.grouped_gemm_i8(xq, x_max, codes.numpy()[None], w_max.numpy()[None], np.array([0, rows], np.int32))
    assert np.array_equal(bits(out), ref)


# up to four rows are quantised by the GEMM's own launch, five are not, and of a matrix of more than two workgroups per CU only one; one channel fragment per workgroup and two, K up to
# the most it takes and beyond, rows of zeros and of one tiny value
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,k", [(16, 64), (4096, 576), (4112, 640), (80, 8192), (48, 8256), (16384, 64), (16400, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_quantised_in_the_launch(rows, n, k, dtype):
    from vllm_kunlun_amd import _lib as L
    kern, layer, codes, w_max = _linear(n, k, n + k)
    x = (torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)) * 1.5).to(dtype)
    if rows > 1:
        x[1] = 0
        x[rows - 1, k - 1] = 1e-7 if rows != 2 else 0
    f16 = dtype == torch.float16
    L.lib.kmoe_trace_kernels(1)
    out = kern.apply_weights(layer, x.cuda())
    named = L.lib.kmoe_traced_kernels().decode()
    L.lib.kmoe_trace_kernels(0)
    assert ("quantises its rows itself" in named) == (rows <= (4 if n <= 16384 else 1) and k <= 8192), named
    xq, x_max = co.quant_i8_rows(bits(x), f16=f16)
    ref, _ = co.grouped_gemm_i8(xq, x_max, codes.numpy()[None], w_max.numpy()[None], np.array([0, rows], np.int32), f16=f16)
    assert np.array_equal(bits(out), ref)


# every tile of the split-K kernel at its remainders (rows split evenly over the tiles, channels past the last fragment)
@pytest.mark.parametrize("rows,n", [(16, 4112), (23, 8176), (49, 4080), (65, 8176), (127, 8144), (250, 4080), (511, 1552), (512, 48)])
def test_tiles_of_the_split_kernel(rows, n):
    from vllm_kunlun_amd import _lib as L
    k = 1216
    kern, layer, codes, w_max = _linear(n, k, n)
    x = (torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)) * 1.5).bfloat16()
    L.lib.kmoe_trace_kernels(1)
    out = kern.apply_weights(layer, x.cuda())
    named = L.lib.kmoe_traced_kernels().decode()
    L.lib.kmoe_trace_kernels(0)
    assert "dense_i8_kernel" in named, named
    xq, x_max = co.quant_i8_rows(bits(x))
    ref, _ = co.grouped_gemm_i8(xq, x_max, codes.numpy()[None], w_max.numpy()[None], np.array([0, rows], np.int32))
    assert np.array_equal(bits(out), ref)


# k a multiple of 2048: every wave starts its part of K at a step of its own (the next k does not), on each tile and
# where the launch quantises the rows
@pytest.mark.parametrize("rows,n", [(3, 64), (16, 48), (24, 4112), (64, 4112), (100, 4080), (200, 4112)])
@pytest.mark.parametrize("k", [2048, 2112, 6144])
def test_k_steps_begun_apart(rows, n, k):
    kern, layer, codes, w_max = _linear(n, k, n + k)
    x = (torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)) * 1.5).bfloat16()
    out = kern.apply_weights(layer, x.cuda())
    xq, x_max = co.quant_i8_rows(bits(x))
    ref, _ = co.grouped_gemm_i8(xq, x_max, codes.numpy()[None], w_max.numpy()[None], np.array([0, rows], np.int32))
    assert np.array_equal(bits(out), ref)


# tiles of 32 x 128, 64 x 128 and beyond: rows and channels at their edges, an odd number of 64-byte steps, both types
@pytest.mark.parametrize("rows,n", [(289, 4096), (384, 4112), (513, 4000), (449, 7168), (1100, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_tiles(rows, n, dtype):
    k = 192
    kern, layer, codes, w_max = _linear(n, k, n)
    x = (torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)) * 1.5).to(dtype)
    out = kern.apply_weights(layer, x.cuda())
    f16 = dtype == torch.float16
    xq, x_max = co.quant_i8_rows(bits(x), f16=f16)
    ref, _ = co.grouped_gemm_i8(xq, x_max, codes.numpy()[None], w_max.numpy()[None], np.array([0, rows], np.int32), f16=f16)
    assert np.array_equal(bits(out), ref)


# several experts on the small tiles: 32 rows, 64 rows (more channel blocks than CUs for the former) and neither, uneven
# and empty experts, with and without a tail expert
@pytest.mark.parametrize("counts", [[70, 0, 33], [1, 64, 65, 0, 20, 31, 90, 17], [300, 40]])
@pytest.mark.parametrize("n", [272, 3088, 6160])
@pytest.mark.parametrize("tail", [0, 45])
def test_small_tiles_of_several_experts(counts, n, tail):
    from vllm_kunlun_amd import _lib as L
    from vllm_kunlun_amd import _plan
    k, rows, E = 192, sum(counts), len(counts)
    gen = torch.Generator().manual_seed(n + tail)
    a = torch.randint(-127, 128, (rows + tail, k), generator=gen, dtype=torch.int8)
    a_max, w_max = torch.rand(rows + tail, generator=gen) + 0.5, torch.rand(E + 1, n, generator=gen) + 0.5
    w = torch.randint(-127, 128, (E + 1, n, k), generator=gen, dtype=torch.int8)
    lod = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ref, _ = co.grouped_gemm_i8(a.numpy(), a_max.numpy(), w.numpy(), w_max.numpy(), np.append(lod, rows + tail).astype(np.int32))
    da, dmax, dw, dw_max, dlod = a.cuda(), a_max.cuda(), w.cuda(), w_max.cuda(), torch.from_numpy(lod).cuda()
    assert _plan.tile_int8_weights_(dw)
    y = torch.full((rows + tail, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    g = L.GemmI8Args()
    g.a, g.lda, g.a_max, g.src_div, g.w, g.w_max, g.lod = da.data_ptr(), k, dmax.data_ptr(), 1, dw.data_ptr(), dw_max.data_ptr(), dlod.data_ptr()
    g.E, g.n, g.k, g.rows, g.y, g.ldy, g.w_layout = E, n, k, rows, y.data_ptr(), n, L.KMOE_W_TILED
    if tail:
        g.w_tail, g.w_max_tail = dw[E].data_ptr(), dw_max[E].data_ptr()
        g.tail_row0, g.tail_rows, g.tail_src0 = rows, tail, rows
    L.check(L.lib.kmoe_grouped_gemm_i8(g, L.stream()))
    assert np.array_equal(bits(y), ref)


@pytest.mark.parametrize("kind", ["buffer", "attribute"])
def test_scale_that_is_no_parameter(kind):
    kern, layer, codes, w_max = _linear(64, 128, 5)
    x = torch.randn(9, 128, generator=torch.Generator().manual_seed(1)).bfloat16()
    want = kern.apply_weights(layer, x.cuda())
    scale = layer.weight_scale.data
    del layer.weight_scale
    if kind == "buffer":
        layer.register_buffer("weight_scale", scale)
    else:
        layer.weight_scale = scale
    for _ in range(2):
        assert torch.equal(kern.apply_weights(layer, x.cuda()), want)


def test_kept_call_follows_the_layer():
    kern, layer, *_ = _linear(256, 512, 1)
    _, other, *_ = _linear(256, 512, 2)
    x = torch.randn(48, 512, device="cuda").bfloat16()
    first = kern.apply_weights(layer, x)
    want = kern.apply_weights(other, x)
    assert torch.equal(kern.apply_weights(layer, x[:5]), first[:5])
    assert kern.apply_weights(layer, x.half()).dtype == torch.float16
    layer.weight, layer.weight_scale, layer._kmoe_w_1nk = other.weight, other.weight_scale, other._kmoe_w_1nk
    assert torch.equal(kern.apply_weights(layer, x), want)
