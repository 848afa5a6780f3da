"""The package without its extension of host code: never built, or built for another torch. A warning, and the calls in Python."""
import os
import subprocess
import sys

import pytest

PROJECT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-kunlun_amd")

CODE = """
import warnings
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import torch
    from vllm_kunlun_amd import _lib as L
    from vllm_kunlun_amd.ops import _custom_ops
    from vllm_kunlun_amd.quantization.kernels import scale_mm
assert L.torch_calls is None and L.lib.kmoe_version()
assert [w for w in seen if issubclass(w.category, RuntimeWarning) and "kmoe_torch.so" in str(w.message)], seen
try:
    torch.ops._C.silu_and_mul(torch.zeros(2, 4, dtype=torch.bfloat16), torch.zeros(2, 8, dtype=torch.bfloat16))
except RuntimeError as problem:
    assert "run on the GPU only" in str(problem), problem
else:
    raise AssertionError("a CPU tensor was taken")
if torch.cuda.is_available():
    x = torch.randn(3, 16, device="cuda", dtype=torch.bfloat16)
    out = torch.empty(3, 8, device="cuda", dtype=torch.bfloat16)
    torch.ops._C.silu_and_mul(out, x)
    want = (torch.nn.functional.silu(x[:, :8].float()) * x[:, 8:].float()).bfloat16()
    assert (out.float() - want.float()).abs().max() <= 2.0 ** -7 * want.float().abs().max()
    layer, kernel = torch.nn.Module(), scale_mm.KunlunScaledMMLinearKernel()
    layer.weight = torch.nn.Parameter(torch.ones(64, 256, dtype=torch.int8, device="cuda"), requires_grad=False)
    layer.weight_scale = torch.nn.Parameter(torch.ones(64, 1, device="cuda"), requires_grad=False)
    kernel.process_weights_after_loading(layer)
    assert torch.equal(kernel.apply_weights(layer, torch.ones(3, 256, device="cuda", dtype=torch.bfloat16)), torch.full((3, 64), 256.0, device="cuda").bfloat16())
print("ran")
"""


@pytest.mark.parametrize("content", [None, b"not a library"], ids=["missing", "foreign"])
@pytest.mark.parametrize("where", ["cpu", pytest.param("gpu", marks=pytest.mark.gpu)])
def test_import(tmp_path, content, where):
    (tmp_path / "lib").mkdir()
    os.symlink(os.path.join(PROJECT, "lib", "libkmoe.so"), tmp_path / "lib" / "libkmoe.so")
    os.symlink(os.path.join(PROJECT, "vllm_kunlun_amd"), tmp_path / "vllm_kunlun_amd")
    if content is not None:
        (tmp_path / "lib" / "kmoe_torch.so").write_bytes(content)
    env = dict(os.environ, PYTHONPATH=str(tmp_path))
    if where == "cpu":
        env.update(HIP_VISIBLE_DEVICES="", CUDA_VISIBLE_DEVICES="")
    done = subprocess.run([sys.executable, "-c", CODE], env=env, cwd=tmp_path, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.strip().endswith("ran"), done.stdout + done.stderr
