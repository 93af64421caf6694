"""Stage 1 by thresholds without noise (score_topk_kernel), which calls of many
tokens over many keys take: exact ties through its bound pass and flushes, and
its results against stage 1 by sorting (the same queries in smaller calls) and
64-bit scores.  Every case asserts the kernel it runs (mpl_score_plan), so that
a change of the plan cannot leave the kernel untested."""

import ctypes

import numpy as np
import pytest
import torch

from model_amd import _lib
from model_amd._lib import ptr

gpu = pytest.mark.gpu
F16, F32, RAW, SCALED = _lib.MPL_F16, _lib.MPL_F32, _lib.MPL_Q_RAW, _lib.MPL_Q_RAW_SCALED

CASES = [
    (4096, 4, 8192, 128, 16, F16, RAW),     # the 67M-slot keys, two splits of 128 blocks
    (8192, 4, 512, 128, 16, F16, RAW),      # the text-study keys, one split
    (512, 4, 8192, 128, 32, F16, RAW),      # k = 32, eight splits
    (33, 4, 8192, 128, 32, F16, RAW),       # few tokens, a second tile of one row, 13 splits
    (8192, 4, 300, 128, 32, F16, RAW),      # k = 32, ten blocks, the last with 12 keys
    (6001, 4, 500, 64, 8, F16, SCALED),     # k < 16, ragged keys and tokens, scores by the query's length
    (8192, 4, 1024, 128, 16, F32, RAW),     # fp32 MFMAs
    (3000, 4, 7990, 16, 9, F16, RAW),       # narrow keys, ragged
    (3000, 4, 7990, 12, 9, F32, SCALED),    # the same in fp32, a width off the pack sizes
]


def _plan(M, H, n, half, k, score):
    s, b = ctypes.c_int(), ctypes.c_int()
    kernel = _lib.lib().mpl_score_plan(M, H, n, half, k, score, 0, 1, s, b)
    return kernel, s.value, b.value


def _select(q, packed, n, k, score, mode, T):
    L = _lib.lib()
    M, H, _, half = q.shape
    o = {"ids": torch.full((M, H, 2, k), -7, dtype=torch.int32, device="cuda"),
         "scores": torch.full((M, H, 2, k), 7.0, device="cuda"),
         "flat": torch.full((M, H, k), -7, dtype=torch.int32, device="cuda"),
         "slots": torch.full((M, H, k), -7, dtype=torch.int32, device="cuda"),
         "weights": torch.full((M, H, k), 7.0, device="cuda")}
    q_len = torch.empty((M, H, 2), device="cuda") if mode == SCALED else None
    wsb = L.mpl_score_select_workspace_bytes(M, H, n, half, k)
    ws = torch.empty(max(wsb, 1), dtype=torch.uint8, device="cuda")
    _lib.check(L.mpl_score_select(ptr(q), mode, ptr(q_len), ptr(packed), M, H, n, half, k, score, ptr(T), None, None,
                                  ptr(ws), wsb, ptr(o["ids"]), ptr(o["scores"]), ptr(o["flat"]), ptr(o["slots"]),
                                  ptr(o["weights"]), _lib.stream_ptr(q.device)), "mpl_score_select")
    return o


def _pack(keys, score):
    L = _lib.lib()
    H, _, n, half = keys.shape
    packed = torch.empty(L.mpl_packed_keys_bytes(H, n, half, score), dtype=torch.uint8, device="cuda")
    _lib.check(L.mpl_pack_keys(ptr(keys), H, n, half, score, None, ptr(packed), _lib.stream_ptr(keys.device)), "pack")
    return packed


def _cosines(q, keys):
    """[M, H, 2, n] fp64, a codebook at a time."""
    qn = q.double() / (q.double().square().sum(-1, keepdim=True) + 1e-6).sqrt()
    kn = keys.double() / (keys.double().square().sum(-1, keepdim=True) + 1e-6).sqrt()
    H = q.shape[1]
    return torch.stack([torch.stack([qn[:, h, c] @ kn[h, c].t().contiguous() for c in range(2)], 1)
                        for h in range(H)], 1)


def test_plan_query():
    """On the host: the kernels of the cases here, the others' conditions, and
    sizes that the calls refuse."""
    for M, H, n, half, k, score, _ in CASES:
        kernel, splits, blocks = _plan(M, H, n, half, k, score)
        assert kernel == _lib.MPL_STAGE1_THRESHOLDS
        assert splits * blocks >= (n + 31) // 32 > (splits - 1) * blocks
    L = _lib.lib()
    assert L.mpl_score_plan(4, 4, 8192, 128, 16, F16, 0, 1, None, None) == _lib.MPL_STAGE1_DECODE
    assert L.mpl_score_plan(64, 4, 8192, 128, 16, F16, 0, 1, None, None) == _lib.MPL_STAGE1_SORT
    assert L.mpl_score_plan(4, 4, 8192, 128, 16, F16, 1, 1, None, None) == _lib.MPL_STAGE1_THRESHOLDS  # noise
    for bad in ((0, 4, 64, 32, 16, F16), (8, 4, 8, 32, 16, F16), (8, 4, 64, 200, 16, F16), (8, 4, 64, 12, 16, F16),
                (8, 4, 64, 32, 33, F16), (8, 4, 64, 32, 16, 7)):
        assert L.mpl_score_plan(*bad, 0, 1, None, None) == -1 and b"mpl_score_plan" in L.mpl_last_error()


@gpu
@pytest.mark.parametrize("M,H,n,half,k,score,mode", CASES)
def test_exact_ties_across_flushes(gpu_lib, M, H, n, half, k, score, mode):
    """Each codebook holds a few distinct vectors, each repeated at least k
    times at random places, so a query's best score is reached by many keys at
    once and the lane buffers overflow again and again.  The best k are then
    the k lowest indices that hold the best vector (lax.top_k's order,
    memory.py:34-57), with one exact score.  Checked where the best and the
    second-best vector are apart by more than the scoring error."""
    assert _plan(M, H, n, half, k, score)[0] == _lib.MPL_STAGE1_THRESHOLDS
    nv = min(16, n // (2 * k))
    rng = np.random.default_rng(n + k)
    base = torch.tensor(rng.standard_normal((H, 2, nv, half)), dtype=torch.float32, device="cuda")
    assign = np.stack([np.stack([rng.permutation(n) % nv for _ in range(2)]) for _ in range(H)])  # [H, 2, n]
    first = np.stack([np.stack([np.stack([np.nonzero(assign[h, c] == v)[0][:k] for v in range(nv)])
                                for c in range(2)]) for h in range(H)])  # [H, 2, nv, k]
    at = torch.tensor(assign, device="cuda")
    keys = base.gather(2, at[..., None].expand(-1, -1, -1, half)).contiguous()
    q = torch.tensor(rng.standard_normal((M, H, 2, half)), dtype=torch.float32, device="cuda")
    o = _select(q, _pack(keys, score), n, k, score, mode, torch.full((1,), 10.0, device="cuda"))
    two = _cosines(q, base).topk(2, -1)
    free = (two.values[..., 0] - two.values[..., 1]) > (2.0 ** -9 if score == F16 else 2e-5)  # twice the error below
    assert float(free.float().mean()) > 0.5
    want = torch.tensor(first, dtype=torch.int32, device="cuda")[None].expand(M, -1, -1, -1, -1).gather(
        3, two.indices[..., :1, None].expand(-1, -1, -1, 1, k))[..., 0, :]
    assert torch.equal(o["ids"][free], want[free])
    assert torch.equal(o["scores"][free], o["scores"][free][:, :1].expand(-1, k))


@gpu
@pytest.mark.parametrize("M,H,n,half,k,score,mode", CASES)
def test_equals_sorted_stage1_and_64_bits(gpu_lib, M, H, n, half, k, score, mode):
    """A query's result does not depend on the kernel: every output equals, bit
    for bit, that of calls of few tokens, which take stage 1 by sorting, with
    repeated keys, a NaN key and NaN queries among them.  Other rows against
    64-bit scores where the k-th and the next are apart by more than twice the
    scoring error: both rows' components rounded to fp16 move each product by
    up to 2 * 2^-11 of itself, and sum |q_i k_i| <= 1 for unit rows, so a
    cosine by 2^-10 (fp32: sums of up to 128 terms, 1e-5)."""
    assert _plan(M, H, n, half, k, score)[0] == _lib.MPL_STAGE1_THRESHOLDS
    g = torch.Generator(device="cuda").manual_seed(n + k)
    q = torch.randn((M, H, 2, half), generator=g, device="cuda")
    keys = torch.randn((H, 2, n, half), generator=g, device="cuda")
    keys[:, :, 5::97] = keys[:, :, :1]
    bad_key = keys.clone()
    bad_key[1, 0, n // 3] = float("nan")
    q[7::50, 0, 1] = float("nan")
    T = torch.full((1,), 8.0, device="cuda")  # a power of two: scaling makes no two scores equal
    packed = _pack(bad_key, score)
    o = _select(q, packed, n, k, score, mode, T)
    for _ in range(4):  # and not on the run: its key tiles are overwritten by DMA while the waves go on
        again = _select(q, packed, n, k, score, mode, T)
        assert all(torch.equal(a.view(torch.int32), o[name].view(torch.int32)) for name, a in again.items())
    few = next((m for m in (64, 128) if _plan(m, H, n, half, k, score)[0] == _lib.MPL_STAGE1_SORT))
    for r0 in (0, M // 2 + 3, M - few) if few < M else ():
        part = _select(q[r0:r0 + few].contiguous(), packed, n, k, score, mode, T)
        for name, v in part.items():
            a, b = o[name][r0:r0 + few], v
            if name == "weights":  # those of a NaN list are NaN
                a, b = a.view(torch.int32), b.view(torch.int32)
            assert torch.equal(a, b), name
    assert bool((o["ids"][7::50, 0, 1] == -1).all()) and not bool((o["ids"][:, 1, 0] == n // 3).any())
    rows = torch.ones(M, dtype=torch.bool, device="cuda")
    rows[7::50] = False
    rows[1500:] = False
    keys[1, 0, n // 3] = -keys[1, 0, n // 3]  # counts nowhere: taken out below
    cos = _cosines(q[rows], keys)
    cos[:, 1, 0, n // 3] = -2.0
    top = cos.topk(k + 1, -1)
    err = 2.0 ** -10 if score == F16 else 1e-5
    free = (top.values[..., k - 1] - top.values[..., k]) > 2 * err
    assert float(free.float().mean()) > 0.05  # k = 32 of 8,192 keys crowd the k-th score
    got = o["ids"][rows].long()
    assert torch.equal(got[free].sort(-1).values, top.indices[..., :k][free].sort(-1).values)
    scale = 8.0
    if mode == SCALED:
        scale = 8.0 * ((q[rows].double().square().sum(-1, keepdim=True) + 1e-6) / half).sqrt()
    diff = (o["scores"][rows].double() - cos.gather(-1, got.clamp(min=0)) * scale).abs() / scale
    assert float(diff.max()) < err
