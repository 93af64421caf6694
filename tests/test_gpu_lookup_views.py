"""MemoryPool.lookup's buffers: the selection lists are parts of one
allocation (with the workspace behind them where it is small), the shaped
views of them are made on first access, and a result frees its memory without
a garbage collection."""

import gc

import pytest
import torch

from model_amd.memory import _WS_WITH_LISTS, MemoryPool
from model_amd import _lib
from tests.gpu_helpers import make_params, oracle_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lead", [(), (1,), (5, 7), (300,)])
@pytest.mark.parametrize("n,k,query_scale", [(40, 5, False), (512, 16, True), (700, 32, False)])
def test_views_and_lifetime(lead, n, k, query_scale):
    pool = MemoryPool(n, 4, 64, 48, k, query_scale=query_scale)
    params = make_params(pool, 0, key_std=32 ** -0.5, value_std=0.02)
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randn((*lead, 4, 64), generator=g, device="cuda")
    M = q.numel() // 256
    pool.lookup(params, q)  # the packed keys and the temperature stay with the pool
    torch.cuda.synchronize()
    gc.collect()
    gc.disable()
    try:
        before = torch.cuda.memory_allocated()
        res = pool.lookup(params, q)
        assert res["out"].shape == (*lead, 48) and res["aux"]["slots"].shape == (*lead, 4, k)
        # the lists against each other: a slot is its two stage-1 ids
        i, flat = res["sub_idx"].long(), res["flat_idx"].long()
        assert i.shape == (M, 4, 2, k) and res["sub_scores"].shape == (M, 4, 2, k)
        slots = i[:, :, 0].gather(-1, flat // k) * n + i[:, :, 1].gather(-1, flat % k)
        assert torch.equal(slots, res["slots"].long())
        assert torch.equal(res["slots"], res["aux"]["slots"].reshape(M, 4, k))
        s = res["sub_scores"]
        w = torch.softmax(s[:, :, 0].gather(-1, flat // k) + s[:, :, 1].gather(-1, flat % k), -1)
        assert float((w - res["weights"]).abs().max()) < 1e-5  # 32 fp32 terms each
        oracle_check(pool, params, q.reshape(M, 4, 64), res, min_tie_free=0.0)
        aux = res["aux"]
        del res
        assert torch.isfinite(aux["balance_loss"]) and aux["queries"].shape == (M, 4, 2, 32)
        del aux, i, flat, slots, s, w
        assert torch.cuda.memory_allocated() == before
    finally:
        gc.enable()


def test_both_workspace_places():
    """Splits of stage 1 need a workspace: at few tokens it lies behind the
    lists, at more it has an allocation of its own; the same results."""
    n, k = 2048, 16
    small, large = (_lib.lib().mpl_score_select_workspace_bytes(M, 4, n, 32, k) for M in (4, 96))
    assert 0 < small <= _WS_WITH_LISTS < large
    pool = MemoryPool(n, 4, 64, 16, k)
    params = make_params(pool, 0, key_std=32 ** -0.5, value_std=0.02)
    q = torch.randn((96, 4, 64), generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
    for M in (4, 96):
        oracle_check(pool, params, q[:M], pool.lookup(params, q[:M]), min_tie_free=0.0)


def test_stream_of_any_device_form():
    """_lib.stream_ptr takes what torch.cuda.current_stream takes, and no other
    device's stream for a CPU device."""
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for device in ("cuda", "cuda:0", 0, None, torch.device("cuda"), torch.device("cuda", 0)):
            assert _lib.stream_ptr(device) == side.cuda_stream
    with pytest.raises(ValueError):
        _lib.stream_ptr(torch.device("cpu", 0))
