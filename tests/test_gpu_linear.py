"""The dense W8A8 linear on the weight-streaming kernel: the launch's slices and channel fragments at their edges, and the
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
