"""A differentiated lookup's memory is freed with its last reference, without
a garbage collection: the autograd node keeps neither its own output nor the
aux, which refers to the tracked balance loss and so to the node."""

import gc
import weakref

import pytest
import torch

from model_amd import memory
from model_amd.memory import LazyAux, MemoryPool, _lookup_with_grad, _Result, _Views
from tests.gpu_helpers import make_params


class _Held:
    pass


class _StubPool:
    """MemoryPool's part in the autograd function, on the CPU."""
    host_pool, d_value = "", 3

    def __init__(self):
        self.held = []

    def lookup(self, params, queries, **kw):
        self.held = [_Held() for _ in range(4)]
        in_res, in_aux, in_view, noise = self.held
        self.held = [weakref.ref(h) for h in self.held]
        views = _Views({"q": lambda: (queries, in_view)})
        aux = LazyAux({"mark": in_aux}, lambda: {"balance_loss": torch.ones(()), "subkey_counts": None, "_counts": 0,
                                                 "_state": 0})
        return _Result({"out": torch.ones(5, 3), "aux": aux, "mark": in_res, "gumbel": noise, "q_len": None,
                        "k_hat": None, "packed": None, "score_code": 0, "temperature": None, "staged": None}, views)


def test_no_cycle_through_the_autograd_node(monkeypatch):
    def backward(pool, res, internal, sub_keys, values, shapes, g_out, g_balance, shuffle, need_dv):
        assert res["q"][0].shape == (5, 1, 2) and "out" not in res and "aux" not in res and "gumbel" not in res
        return torch.ones(shapes[0]), torch.ones_like(sub_keys), torch.ones(()), None
    monkeypatch.setattr(memory, "_lookup_backward", backward)
    pool = _StubPool()
    q = torch.zeros((5, 1, 2), requires_grad=True)
    params = {"sub_keys": torch.zeros((1, 2, 4, 1), requires_grad=True), "log_temperature": torch.zeros(()),
              "values": torch.zeros((16, 3))}
    gc.collect()
    gc.disable()
    try:
        out, aux = _lookup_with_grad(pool, params, q, train=True, sparse_grad=False, noise_scale=1.0,
                                     shuffle_reads=False, rngs=None)
        assert pool.held[3]() is None  # the noise went with the forward
        torch.autograd.grad(out.sum() + aux["balance_loss"], [q, params["sub_keys"]])
        assert pool.held[1]() is not None
        del out, aux
        assert [h() for h in pool.held] == [None] * 4
    finally:
        gc.enable()


@pytest.mark.gpu
@pytest.mark.parametrize("vdt,sparse", [(torch.float32, False), (torch.float16, True)])
def test_training_step_frees_its_memory(gpu_lib, vdt, sparse):
    pool = MemoryPool(64, 4, 64, 48, 8, values_dtype=vdt)
    params = {k: v.requires_grad_(not (sparse and k == "values")) for k, v in
              make_params(pool, 0, key_std=32 ** -0.5, value_std=0.02).items()}
    q = torch.randn((300, 4, 64), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    q.requires_grad_()
    leaves = [q] + [v for v in params.values() if v.requires_grad]

    def step():
        out, aux = pool.apply({"params": params}, q, train=True, sparse_grad=sparse, rngs={"routing": 3})
        torch.autograd.grad(out.square().sum() + 0.01 * aux["balance_loss"], leaves)

    step()  # the packed keys, the temperature and the constants stay with the pool
    torch.cuda.synchronize()
    gc.collect()
    gc.disable()
    try:
        before = torch.cuda.memory_allocated()
        for _ in range(3):
            step()
            assert torch.cuda.memory_allocated() == before
    finally:
        gc.enable()
