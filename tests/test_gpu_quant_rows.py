"""Row quantisation to int8 where the arithmetic for rows of ordinary numbers hands over to the general one: rows with NaNs
and infinities, rows so small that 127 / max overflows, and the largest numbers of both types."""
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), ".."))
from conftest import bits  # noqa: E402
from oracle import c_oracle as co  # noqa: E402

pytestmark = pytest.mark.gpu


def _rows(R, C, dtype):
    """Rows of every kind in turn, each with the special value at another place (one of the row's last values among them)."""
    g = torch.Generator().manual_seed(R + C)
    x = torch.randn(R, C, generator=g).to(dtype)
    top = torch.finfo(dtype).max
    smallest = torch.finfo(dtype).smallest_normal * 2.0 ** -(7 if dtype == torch.bfloat16 else 10)
    for r in range(R):
        at = (r * 37 + C - 1) % C
        kind = r % 8
        if kind == 1:
            x[r, at] = float("nan")
        elif kind == 2:
            x[r, at], x[r, 0] = float("-inf"), 0.0
        elif kind == 3:
            x[r] = float("nan")
        elif kind == 4:
            x[r] = 0
            x[r, at] = -smallest
        elif kind == 5:
            x[r, at] = top
        elif kind == 6:
            x[r] = 0
        elif kind == 7:
            x[r] = torch.arange(C).remainder(255).sub(127).to(dtype) * 0.5  # halves: ties of the rounding
            x[r, at] = 127.0
    return x


# widths on both sides of every kernel's limit: half a wave, a wave and a workgroup per row
@pytest.mark.parametrize("R,C", [(2056, 768), (2050, 64), (19, 1024), (18, 1088), (17, 2048), (16, 2112), (9, 8192), (9, 8256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chunked", [False, True])
def test_rows_of_every_kind(R, C, dtype, chunked):
    from vllm_kunlun_amd import _lib as L
    x = _rows(R, C, dtype)
    want, want_max = co.quant_i8_rows(bits(x), f16=dtype == torch.float16)
    dx = x.cuda()
    q = torch.empty(R * C, dtype=torch.int8, device="cuda")
    top = torch.empty(R, dtype=torch.float32, device="cuda")
    if chunked:
        L.check(L.lib.kmoe_quant_i8_rows_chunked_dt(L.ptr(dx), C, R, C, L.ptr(q), L.ptr(top), L.act_dtype(dx), L.stream()))
        got = q.view(C // 64, R, 64).transpose(0, 1).reshape(R, C)
    else:
        L.check(L.lib.kmoe_quant_i8_rows_dt(L.ptr(dx), C, R, C, L.ptr(q), C, L.ptr(top), L.act_dtype(dx), L.stream()))
        got = q.view(R, C)
    assert np.array_equal(top.cpu().numpy().view(np.uint32), want_max.view(np.uint32))
    assert np.array_equal(got.cpu().numpy(), want)


# the widths and numbers of rows at which the threads of a row, or their vectors, change; part of the last workgroup's rows
# are there, and rows apart from each other leave what lies between alone
@pytest.mark.parametrize("R,C", [(9, 256), (9, 320), (30, 512), (30, 576), (256, 1088), (257, 1088), (257, 1536), (257, 1600), (256, 2048),
                                 (257, 2048), (5, 4096), (5, 4160), (5, 16384), (5, 16448), (3, 32768), (3, 32832)])
@pytest.mark.parametrize("chunked", [False, True])
def test_threads_and_vectors_of_a_row(R, C, chunked):
    from vllm_kunlun_amd import _lib as L
    x = _rows(R, C, torch.bfloat16)
    want, want_max = co.quant_i8_rows(bits(x))
    apart = torch.full((R, C + 64), float("inf"), dtype=torch.bfloat16, device="cuda")
    apart[:, :C] = x.cuda()
    q = torch.full((R * C + 64,), 99, dtype=torch.int8, device="cuda")
    top = torch.empty(R, dtype=torch.float32, device="cuda")
    args = (L.ptr(apart), C + 64, R, C, L.ptr(q)) + (() if chunked else (C,)) + (L.ptr(top), L.act_dtype(apart), L.stream())
    L.check((L.lib.kmoe_quant_i8_rows_chunked_dt if chunked else L.lib.kmoe_quant_i8_rows_dt)(*args))
    codes = q[:R * C]
    got = codes.view(C // 64, R, 64).transpose(0, 1).reshape(R, C) if chunked else codes.view(R, C)
    assert np.array_equal(top.cpu().numpy().view(np.uint32), want_max.view(np.uint32))
    assert np.array_equal(got.cpu().numpy(), want) and bool((q[R * C:] == 99).all())
