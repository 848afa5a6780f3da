"""Host-side rules of the argument plumbing, without a GPU: which memory counts as re-tiled weights
(the mark follows the storage through views, `.data`, `.t()` and Parameter wrappers, and dies with
it), which views of such memory an operator refuses, one workspace per (device, stream), and a plan's
refusal to launch on another stream than the one it was built on."""
import gc

import pytest
import torch

from vllm_kunlun_amd import _lib as L
from vllm_kunlun_amd import _plan


def test_tiled_mark_follows_the_storage_not_the_tensor_object():
    w = torch.zeros(3, 32, 128, dtype=torch.int8)
    assert not _plan.is_tiled(w) and _plan.weight_layout(w) == L.KMOE_W_ROWMAJOR
    _plan._mark_tiled(w, 32, 128)          # what tile_int8_weights_ does after re-arranging the bytes
    p = torch.nn.Parameter(w, requires_grad=False)
    for view in (w, w.data, w.detach(), p, p.data, w[1], w.view(1, 3, 32, 128), w[1:], w[0].t().t()):
        assert _plan.is_tiled(view)
        assert _plan.weight_layout(view) == L.KMOE_W_TILED
    assert not _plan.is_tiled(w.clone())   # a copy is other memory (and would hold tiled bytes unmarked: do not copy)
    # views that would read scrambled values are refused, not served as row-major
    for bad in (w[0].t(), w[:, :16], w[:, :, :64], w.view(3, 64, 64), w.view(torch.bfloat16)[..., :32]):
        assert _plan.is_tiled(bad)
        with pytest.raises(ValueError):
            _plan.weight_layout(bad)
    # bf16 weights are tiled on their bytes: k counts bytes
    wb = torch.zeros(2, 16, 32, dtype=torch.bfloat16)
    _plan._mark_tiled(wb, 16, 64)
    assert _plan.weight_layout(wb) == L.KMOE_W_TILED


def test_tiled_mark_dies_with_the_storage():
    w = torch.zeros(16, 64, dtype=torch.int8)
    _plan._mark_tiled(w, 16, 64)
    key = w.untyped_storage()._cdata
    view = w.t()
    del w
    gc.collect()
    assert key in _plan._TILED             # the view keeps the memory, and the mark, alive
    del view
    gc.collect()
    assert key not in _plan._TILED         # a later tensor at the same address does not inherit it


def test_one_workspace_per_device_and_stream():
    ws = _plan._Workspace()
    cpu = torch.device("cpu")
    a = ws.get(100, cpu, stream_id=1)
    assert ws.get(50, cpu, stream_id=1) is a              # grows only
    b = ws.get(100, cpu, stream_id=2)
    assert b.data_ptr() != a.data_ptr()                    # another stream never shares scratch
    big = ws.get(1000, cpu, stream_id=1)
    assert big.numel() >= 1000 and ws.get(10, cpu, stream_id=1) is big


def test_plan_refuses_another_stream(monkeypatch):
    plan = _plan.MoEPlan(args=None, layout=None, workspace=torch.zeros(8, dtype=torch.uint8), keepalive=[],
                         stream_id=0x10)
    monkeypatch.setattr(_plan, "_current_stream_id", lambda device: 0x20)
    with pytest.raises(RuntimeError, match="built on stream 0x10"):
        plan()


def _kept_call(*tensors):
    plan = _plan.MoEPlan(L.MoEArgs(), None, None, [])
    return _plan._LayerCall(plan, tensors, experts=4)


@pytest.mark.parametrize("change", [lambda d: d.transpose(1, 2), lambda d: d.view(torch.float16), lambda d: d.view(2, 32, 16),
                                    lambda d: d.clone(), lambda d: d[:, :, :8]])
def test_kept_block_is_dropped_when_a_weight_becomes_another_view(change):
    """The same Parameter over the same memory with other strides, another type or another shape (which filling a block
    refuses) must not be served from the block kept for it."""
    w = torch.nn.Parameter(torch.zeros(4, 16, 16, dtype=torch.bfloat16), requires_grad=False)
    call = _kept_call(w, torch.zeros(4))
    assert not call.holds()  # (the second tensor is gone)
    scale = torch.zeros(4)
    call = _kept_call(w, scale)
    assert call.holds()
    w.data = w.data[:]
    assert call.holds()
    kept = w.data  # (the memory stays alive: another tensor cannot take its place)
    w.data = change(w.data)
    assert not call.holds()
    w.data = kept
    assert call.holds()


def test_kept_block_is_dropped_when_re_arranged_memory_is_freed():
    """Weights that were re-tiled, freed, and loaded again row-major: the allocator may hand out the same address, so
    the block that says "tiled" must not outlive the mark."""
    memory = torch.zeros(4096, dtype=torch.int8)  # two storages over one piece of memory stand for a reused address
    first, second = (torch.from_numpy(memory.numpy()).view(4, 16, 64) for _ in range(2))
    assert first.untyped_storage()._cdata != second.untyped_storage()._cdata
    _plan._mark_tiled(first, 16, 64)
    w = torch.nn.Parameter(first, requires_grad=False)
    call = _kept_call(w)
    assert call.holds() and _plan.is_tiled(w)
    del first
    w.data = second
    gc.collect()
    assert not _plan.is_tiled(w) and not call.holds()
    assert _kept_call(w).holds()


def test_layers_that_hit_outlive_calls_that_always_miss(monkeypatch):
    """Least recently USED first out: a layer called in every step keeps its block although another one's calls (fresh
    tensors each time) fill the table over and over."""
    monkeypatch.setattr(_plan, "_CALLS", type(_plan._CALLS)())
    monkeypatch.setattr(_plan, "MAX_CALLS", 4)
    w = torch.zeros(4, 16, 64)
    mine = _kept_call(w)
    _plan._keep_call("layer", mine)
    for step in range(20):
        assert _plan._kept_call("layer") is mine
        _plan._keep_call(("other", step), _kept_call(w))
    assert len(_plan._CALLS) == 4
    for step in range(4):
        _plan._keep_call(("other", step), _kept_call(w))
    assert _plan._kept_call("layer") is None


def test_workspace_keeps_no_stand_in():
    """A call under a fake-tensor mode fails, as it always did, and leaves nothing behind for the real calls after it."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from vllm_kunlun_amd._plan import _Workspace
    pool, device = _Workspace(), torch.device("cpu")
    with FakeTensorMode():
        pool.get(64, device, 1)
    real = pool.get(64, device, 1)
    assert type(real) is torch.Tensor and pool.get(32, device, 1) is real
