"""Routing where scores are equal: the way that ranks distinct keys gives up and the one that goes by expert id takes over,
per token; against the oracle, for every slot count, the most experts per token and every group size the lanes hold."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import c_oracle as co  # noqa: E402


def _logits(M, E, seed):
    """Every other token's logits on a grid of eight values, so that the chosen ones repeat; the others' distinct."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((M, E)).astype(np.float32)
    x[::2] = np.clip(np.round(x[::2] * 2) / 2, -1.5, 2)
    return x


def _run(call, M, K):
    w = torch.empty(M, K, dtype=torch.float32, device="cuda")
    ids = torch.empty(M, K, dtype=torch.int32, device="cuda")
    call(w, ids)
    return ids.cpu().numpy(), w.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("E,K", [(2, 1), (17, 16), (63, 63), (64, 63), (64, 64), (100, 8), (128, 63), (130, 64), (512, 10), (1024, 63)])
def test_softmax_routing_of_equal_scores(E, K):
    from vllm_kunlun_amd import _lib as L
    M = 13
    logits = _logits(M, E, E + K)
    w_ref, ids_ref = co.softmax_topk(logits, K, 1)
    d = torch.from_numpy(logits).cuda()
    ids, w = _run(lambda w, i: L.check(L.lib.kmoe_softmax_topk(L.ptr(d), M, E, K, 1, L.ptr(w), L.ptr(i), L.stream())), M, K)
    assert np.array_equal(ids, ids_ref) and np.array_equal(w, w_ref.view(np.uint32))


@pytest.mark.parametrize("gsize", [2, 4, 8, 16, 32, 64, 12])
@pytest.mark.parametrize("n_group", [2, 8, 15])
def test_group_routing_of_equal_scores(gsize, n_group):
    from vllm_kunlun_amd import _lib as L
    M, E, tg = 9, gsize * n_group, (n_group + 1) // 2
    K = min(8, tg * gsize)
    logits = _logits(M, E, E)
    w_ref, ids_ref = co.sigmoid_group_topk_norm(logits, None, K, n_group, tg, 2.5)
    d = torch.from_numpy(logits).cuda()
    ids, w = _run(lambda w, i: L.check(L.lib.kmoe_sigmoid_group_topk_norm(L.ptr(d), None, M, E, K, n_group, tg, 2.5, L.ptr(w), L.ptr(i),
                                                                          L.stream())), M, K)
    assert np.array_equal(ids, ids_ref) and np.array_equal(w, w_ref.view(np.uint32))


def _few_values(E, K, seed):
    """Rows whose chosen scores are mostly one value: all equal (zeros of both signs), two values, the equal ones behind K - 1
    distinct ones and behind a single one, and as many equal ones as leave some rounds without a candidate."""
    rng = np.random.default_rng(seed)
    x = np.zeros((6, E), np.float32)
    x[0, ::2] = -0.0
    x[1] = rng.integers(0, 2, E)
    x[2, rng.permutation(E)[:K - 1]] = 1 + rng.permutation(K - 1)
    x[3, rng.integers(E)] = 2
    x[4] = rng.integers(0, 3, E) * 0.25
    x[5] = np.sort(rng.standard_normal(E))[::-1].repeat(2)[:E]
    return x


@pytest.mark.parametrize("E,K", [(2, 2), (17, 16), (64, 64), (65, 64), (128, 8), (256, 64), (384, 8), (1000, 63), (1024, 64)])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_routing_of_few_values(E, K, sigmoid):
    from vllm_kunlun_amd import _lib as L
    logits = _few_values(E, K, E)
    M = len(logits)
    d = torch.from_numpy(logits).cuda()
    if sigmoid:
        w_ref, ids_ref = co.sigmoid_group_topk_norm(logits, None, K, 1, 1, 2.5)
        call = lambda w, i: L.check(L.lib.kmoe_sigmoid_group_topk_norm(L.ptr(d), None, M, E, K, 1, 1, 2.5, L.ptr(w), L.ptr(i), L.stream()))
    else:
        w_ref, ids_ref = co.softmax_topk(logits, K, 1)
        call = lambda w, i: L.check(L.lib.kmoe_softmax_topk(L.ptr(d), M, E, K, 1, L.ptr(w), L.ptr(i), L.stream()))
    ids, w = _run(call, M, K)
    assert np.array_equal(ids, ids_ref) and np.array_equal(w, w_ref.view(np.uint32))


@pytest.mark.parametrize("E,K", [(17, 17), (64, 64), (200, 8), (1024, 64)])
def test_routing_of_not_a_number(E, K):
    """Every NaN is a candidate: its experts come out once each, whatever their order."""
    from vllm_kunlun_amd import _lib as L
    bits = np.full((3, E), 0xffffffff, np.uint32)
    bits[1, ::3] = 0x7fc00000
    bits[2] = 0xfffffffe
    d = torch.from_numpy(bits.view(np.float32).copy()).cuda()
    ids, _ = _run(lambda w, i: L.check(L.lib.kmoe_softmax_topk(L.ptr(d), 3, E, K, 0, L.ptr(w), L.ptr(i), L.stream())), 3, K)
    assert all(len(set(row)) == K for row in ids.tolist()) and ids.min() >= 0 and ids.max() < E
