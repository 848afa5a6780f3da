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


# short rows, four of them a wave: parts of a wave's rows there, both sides of the widths and of the number of rows
@pytest.mark.parametrize("R,C", [(1, 16), (15, 128), (17, 64), (2047, 192), (2048, 192), (2049, 256), (2051, 128), (2050, 144)])
def test_short_rows(R, C):
    from vllm_kunlun_amd import _lib as L
    x = _rows(R, C, torch.bfloat16)
    want, want_max = co.quant_i8_rows(bits(x))
    dx = x.cuda()
    q = torch.full((R * C + 64,), 99, dtype=torch.int8, device="cuda")
    top = torch.full((R + 16,), -7.0, device="cuda")
    L.check(L.lib.kmoe_quant_i8_rows_dt(L.ptr(dx), C, R, C, L.ptr(q), C, L.ptr(top), 0, L.stream()))
    assert np.array_equal(top[:R].cpu().numpy().view(np.uint32), want_max.view(np.uint32)) and bool((top[R:] == -7).all())
    assert np.array_equal(q[:R * C].view(R, C).cpu().numpy(), want) and bool((q[R * C:] == 99).all())


# rows of more bytes than the memory-side cache, whose vectors are asked for in turn, on both sides of its widths and size
@pytest.mark.parametrize("R,C", [(43690, 3072), (42368, 3136), (32767, 4096), (32768, 4096), (32264, 4160), (29128, 4608), (28728, 4672)])
def test_rows_beyond_the_memory_side_cache(R, C):
    from vllm_kunlun_amd import _lib as L
    few = 64
    x = _rows(few, C, torch.bfloat16)
    want, want_max = co.quant_i8_rows(bits(x))
    dx = x.cuda().repeat(-(-R // few), 1)[:R].contiguous()
    q = torch.empty(R, C, dtype=torch.int8, device="cuda")
    top = torch.empty(R, dtype=torch.float32, device="cuda")
    L.check(L.lib.kmoe_quant_i8_rows_dt(L.ptr(dx), C, R, C, L.ptr(q), C, L.ptr(top), 0, L.stream()))
    dw, dm = torch.from_numpy(want).cuda(), torch.from_numpy(want_max.copy()).view(torch.int32).cuda()
    assert torch.equal(q, dw.repeat(-(-R // few), 1)[:R]) and torch.equal(top.view(torch.int32), dm.repeat(-(-R // few))[:R])


def test_the_most_rows_there_can_be():
    """Rows up to the last that 31 bits count: the last workgroup's rows past them are none."""
    from vllm_kunlun_amd import _lib as L
    R, C, end = 2 ** 31 - 2, 8, 40
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("60 GB of rows")
    x = torch.zeros(R, C, dtype=torch.bfloat16, device="cuda")
    tail = _rows(end, C, torch.bfloat16)
    x[-end:] = tail.cuda()
    q = torch.empty(R * C + 64, dtype=torch.int8, device="cuda")
    q[R * C - end * C:] = 99
    top = torch.full((R + 16,), -7.0, device="cuda")
    L.check(L.lib.kmoe_quant_i8_rows_dt(L.ptr(x), C, R, C, L.ptr(q), C, L.ptr(top), 0, L.stream()))
    want, want_max = co.quant_i8_rows(bits(tail))
    assert np.array_equal(q[(R - end) * C:R * C].view(end, C).cpu().numpy(), want) and bool((q[R * C:] == 99).all())
    assert np.array_equal(top[R - end:R].cpu().numpy().view(np.uint32), want_max.view(np.uint32)) and bool((top[R:] == -7).all())
    assert not bool(q[:(R - end) * C].view(torch.int64).any()) and not bool(top[:R - end].any())
    del x, q, top
    torch.cuda.empty_cache()


# rows that the down projection's launch quantises itself (32 tokens: up to four rows a wave), their last vectors in one load
# of a lane and in two: rows of zeros, NaNs, infinities and the smallest numbers among ordinary ones
@pytest.mark.parametrize("I", [64, 576, 1024])
def test_rows_quantised_by_the_down_launch(I):
    from vllm_kunlun_amd import _lib as L
    from vllm_kunlun_amd import _plan
    from oracle import torch_moe as tm
    M, E, K, H = 32, 8, 2, 256
    g = torch.Generator().manual_seed(I)
    x = (torch.randn(M, H, generator=g) * 1.5).bfloat16()
    x[3], x[4, 7], x[5, 0], x[6], x[7] = 0, float("inf"), float("nan"), x[6] * 2.0 ** -126, x[7] * 1e38
    logits = torch.randn(M, E, generator=g)
    w, ids = co._route(logits.numpy(), K, "softmax", True, None, None, 1.0, None)
    w13q, s13 = tm.quantize_weight_per_channel(torch.randn(E * 2 * I, H, generator=g) * 0.05)
    w2q, s2 = tm.quantize_weight_per_channel(torch.randn(E * H, I, generator=g) * 0.05)
    w13q, w2q = w13q.view(E, 2 * I, H), w2q.view(E, H, I)
    w13_max, w2_max = (s13 * 127.0).view(E, 2 * I), (s2 * 127.0).view(E, H)
    d13, d2 = w13q.clone().cuda(), w2q.clone().cuda()
    assert _plan.tile_pair_(d13, d2)
    out = torch.empty(M, H, dtype=torch.bfloat16, device="cuda")
    plan = _plan.make_moe_plan(L.KMOE_FMT_INT8, x.cuda(), logits.cuda(), out, K, d13, d2, w13_max.cuda(), w2_max.cuda(),
                               scoring_func="softmax", renormalize=True)
    plan()
    moe_index, src, _, lod = co.align(ids, E)
    xq, x_max = co.quant_i8_rows(bits(x))
    act, _ = co.grouped_gemm_i8(xq, x_max, w13q.numpy(), w13_max.numpy(), lod, act=1, row_src=src, src_div=K)
    aq, a_max = co.quant_i8_rows(act)
    down, _ = co.grouped_gemm_i8(aq, a_max, w2q.numpy(), w2_max.numpy(), lod)
    ref = co.combine(down, moe_index, w)
    got, nan = bits(out), np.isnan((ref.astype(np.uint32) << 16).view(np.float32))
    assert nan.any() and not nan.all()
    assert np.array_equal(np.isnan((got.astype(np.uint32) << 16).view(np.float32)), nan)
    assert np.array_equal(got[~nan], ref[~nan])
