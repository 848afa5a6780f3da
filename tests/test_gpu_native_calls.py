"""Calls with a native body (csrc/torch_calls.cpp) against their Python bodies: the same results, refusals and counted writes."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _linear(n=64, k=256, device="cuda"):
    from vllm_kunlun_amd.quantization.kernels.scale_mm import KunlunScaledMMLinearKernel
    g = torch.Generator().manual_seed(n)
    layer, kernel = torch.nn.Module(), KunlunScaledMMLinearKernel()
    layer.weight = torch.nn.Parameter(torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8).to(device), requires_grad=False)
    layer.weight_scale = torch.nn.Parameter((torch.rand(n, 1, generator=g) * 0.02 + 0.001).to(device), requires_grad=False)
    kernel.process_weights_after_loading(layer)
    kernel.apply_weights(layer, torch.zeros(1, k, dtype=torch.bfloat16, device=device))
    return kernel, layer, layer.__dict__["_kmoe_dynamic"]


@pytest.mark.parametrize("rows", [1, 4, 5, 100, 512, 513])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear(rows, dtype):
    kernel, layer, call = _linear()
    x = torch.randn(rows, 256, device="cuda", dtype=dtype)
    got = kernel.apply_weights(layer, x)
    native, call.native = call.native, None
    want = kernel.apply_weights(layer, x)
    call.native = native
    assert native is not None and (native(x) is None) == (rows > call.split_max)
    assert torch.equal(got, want) and got.dtype == dtype and not got.requires_grad
    assert torch.equal(kernel.apply_weights(layer, x.view(1, rows, 256)), want.view(1, rows, 64))  # (the Python body's)
    wide = torch.randn(rows, 300, device="cuda", dtype=dtype)[:, :256]
    assert torch.equal(kernel.apply_weights(layer, wide), kernel.apply_weights(layer, wide.contiguous()))
    assert kernel.apply_weights(layer, x[:0]).shape == (0, 64)


def test_linear_refuses_what_it_refused():
    kernel, layer, _ = _linear()
    with pytest.raises(ValueError):
        kernel.apply_weights(layer, torch.zeros(3, 128, dtype=torch.bfloat16, device="cuda"))
    with pytest.raises(NotImplementedError):
        kernel.apply_weights(layer, torch.zeros(3, 256, device="cuda"))
    with pytest.raises(RuntimeError):
        kernel.apply_weights(layer, torch.zeros(3, 256, dtype=torch.bfloat16))


def test_linear_from_threads_on_their_own_streams():
    kernel, layer, _ = _linear()
    x = [torch.randn(r, 256, device="cuda", dtype=torch.bfloat16) for r in (1, 7, 60, 300)]
    want = [kernel.apply_weights(layer, t) for t in x]
    torch.cuda.synchronize()
    got = [None] * len(x)

    def run(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                got[i] = kernel.apply_weights(layer, x[i])
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(x))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("shape", [(1, 16), (7, 4096), (2, 3, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_and_mul(shape, dtype):
    from vllm_kunlun_amd.ops import _custom_ops as ops
    x = torch.randn(shape, device="cuda").to(dtype)
    out, want = (torch.zeros(*shape[:-1], shape[-1] // 2, device="cuda", dtype=dtype) for _ in range(2))
    torch.ops._C.silu_and_mul(out, x)
    ops.silu_and_mul(want, x)
    assert torch.equal(out, want) and out._version == 1
    torch.ops._C.silu_and_mul(out, x, -1, True)
    assert out._version == 2
    with torch.inference_mode():
        torch.ops._C.silu_and_mul(torch.zeros_like(out), x)


@pytest.mark.parametrize("case", ["type", "mixed", "odd", "shape", "strided", "device", "empty"])
def test_silu_and_mul_refuses_what_it_refused(case):
    from vllm_kunlun_amd.ops import _custom_ops as ops
    x, out = torch.zeros(4, 16, device="cuda", dtype=torch.bfloat16), torch.zeros(4, 8, device="cuda", dtype=torch.bfloat16)
    x, out = {"type": (x.float(), out.float()), "mixed": (x, out.half()), "odd": (x[:, :15].contiguous(), out), "shape": (x, out[:3]),
              "strided": (x[:, ::2], out[:, :4]), "device": (x, out.cpu()), "empty": (x[:0], out[:0])}[case]
    with pytest.raises(Exception) as python:
        ops.silu_and_mul(out, x)
    with pytest.raises(type(python.value)) as native:
        torch.ops._C.silu_and_mul(out, x)
    assert str(native.value) == str(python.value) and out._version == 0
