"""How the operators meet autograd (CPU, with operators of the same registration whose bodies need no GPU): a backward
pass through a result is refused, and an argument that a kernel wrote counts as written."""
import gc

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from vllm_kunlun_amd.ops import _custom_ops as ops


def _fill(t):
    t.detach().untyped_storage().copy_(torch.ones(t.untyped_storage().nbytes() // 4).untyped_storage())  # unseen by autograd


@ops.operator("kmoe_test::twice", mutates_args=())
def twice(x: torch.Tensor, bias: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor, bool]:
    return x.detach() * 2, torch.ones(x.shape, dtype=torch.int8), True


@ops.operator("kmoe_test::fill", mutates_args=("out", "more"))
def fill(x: torch.Tensor, out: torch.Tensor, more: torch.Tensor | None, n: int = 1) -> None:
    for t in (out, more):
        if t is not None:
            _fill(t)


OPS = torch.ops.kmoe_test


def test_backward_through_a_result_is_refused():
    x = torch.ones(3, requires_grad=True)
    y, codes, flag = OPS.twice(x)
    assert torch.equal(y.detach(), torch.full((3,), 2.0)) and flag is True and not codes.requires_grad
    with pytest.raises(RuntimeError, match="no autograd formula"):
        (y * x).sum().backward()
    w = torch.ones(3, requires_grad=True)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        OPS.twice(torch.ones(3), w)[0].sum().backward()
    with torch.no_grad():
        assert not OPS.twice(x)[0].requires_grad
    with torch.inference_mode():
        assert not OPS.twice(x)[0].requires_grad
    assert not OPS.twice(torch.ones(3))[0].requires_grad
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: OPS.twice(t)[0].sum())(torch.ones(3))


@pytest.mark.parametrize("mode", [torch.enable_grad, torch.no_grad, torch.inference_mode])
def test_a_written_argument_counts_as_written(mode):
    x = torch.ones(3, requires_grad=True)
    w, more = torch.zeros(3), torch.zeros(6)
    y = x * w  # saves w
    with mode():
        OPS.fill(torch.ones(3), w, more[:3])
    assert w._version == 1 and more._version == 1 and torch.equal(w, torch.ones(3))
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()
    before = x._version
    OPS.fill(x.detach(), w, None)
    assert w._version == 2 and x._version == before
    with torch.inference_mode():
        inner = torch.zeros(3)
        OPS.fill(inner, inner, None)
    OPS.fill(inner, inner, None)  # (an inference tensor has no version)


def test_traced_calls_count_writes_too():
    from torch.library import register_fake
    register_fake("kmoe_test::fill", ops._fake_writes(ops._WRITTEN["kmoe_test::fill"]))
    with FakeTensorMode():
        w = torch.zeros(3)
        OPS.fill(torch.ones(3), w, None)
        assert w._version == 1
    gc.collect()


def test_every_operator_is_registered_this_way():
    written = {"_C::moe_softmax_topk": (1, 2), "_C::moe_softmax_topk_norm": (1, 2), "_C::moe_sigmoid_group_topk_norm": (1, 2, 3),
               "_moe_C::topk_softmax": (0, 1, 2), "_C::gen_block_statistic": (1,), "_C::moe_pre_sorted": (3, 4, 5, 6),
               "_C::quant2d": (1, 2), "_C::moe_fc": (5,), "_C::silu_and_mul": (0,), "_C::moe_post": (4,)}
    assert {k: tuple(sorted(v)) for k, v in ops._WRITTEN.items() if not k.startswith("kmoe_test")} == written
    with FakeTensorMode():
        x, out = torch.zeros(4, 16, dtype=torch.bfloat16), torch.zeros(4, 8, dtype=torch.bfloat16)
        torch.ops._C.silu_and_mul(out, x)
        assert out._version == 1
        leaf = torch.zeros(4, 16, dtype=torch.bfloat16, requires_grad=True)
        y = torch.ops._C.swigluoai_and_mul(leaf)
        with pytest.raises(RuntimeError, match="no autograd formula"):
            y.sum().backward()
