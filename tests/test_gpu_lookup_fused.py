"""mpl_lookup (selection and value read in one call) against mpl_score_select
followed by mpl_gather_wsum, through the C ABI: every output bit for bit.
Covers the fused stage-2 + read kernels (H = 4: k = 16 with fp16 rows of 128,
256 and 512 elements, fp32 rows, shuffled reads, split-key plans whose lists
are merged before stage 2; k < 16 and rows of any number of 16-byte vectors up
to 64), the plans with 9-64 split lists (decode sizes), whose lists the fused
decode stage 2 (pair_decode_read_k16) reduces, and the shapes that fall back
to two launches (other H, k > 16, other rows)."""

import pytest
import torch

from model_amd import _lib
from model_amd._lib import ptr

pytestmark = pytest.mark.gpu


def _run(M, H, n, d_key, d, k, vdt, shuffle, seed):
    L = _lib.lib()
    half = d_key // 2
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn((M, H, 2, half), generator=g, device="cuda")
    keys = torch.randn((H, 2, n, half), generator=g, device="cuda") * half ** -0.5
    values = (torch.randn((n * n, d), generator=g, device="cuda") * 0.02).to(vdt)
    vcode = _lib.MPL_F16 if vdt == torch.float16 else _lib.MPL_F32
    packed = torch.empty(L.mpl_packed_keys_bytes(H, n, half, _lib.MPL_F16), dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    _lib.check(L.mpl_pack_keys(ptr(keys), H, n, half, _lib.MPL_F16, None, ptr(packed), s), "pack")
    wsb = L.mpl_score_select_workspace_bytes(M, H, n, half, k)
    T = torch.full((1,), 10.0, device="cuda")  # the clamped temperature, a device scalar
    outs = []
    for fused in (False, True):
        ws = torch.empty(max(wsb, 1), dtype=torch.uint8, device="cuda")
        o = {"sub_idx": torch.full((M, H, 2, k), -7, dtype=torch.int32, device="cuda"),
             "sub_scores": torch.full((M, H, 2, k), 7.0, device="cuda"),
             "flat_idx": torch.full((M, H, k), -7, dtype=torch.int32, device="cuda"),
             "slots": torch.full((M, H, k), -7, dtype=torch.int32, device="cuda"),
             "weights": torch.full((M, H, k), 7.0, device="cuda"),
             "out": torch.full((M, d), 7.0, device="cuda")}
        sel = (ptr(q), _lib.MPL_Q_RAW, None, ptr(packed), M, H, n, half, k, _lib.MPL_F16, ptr(T), None, None,
               ptr(ws), wsb, ptr(o["sub_idx"]), ptr(o["sub_scores"]), ptr(o["flat_idx"]), ptr(o["slots"]),
               ptr(o["weights"]))
        if fused:
            _lib.check(L.mpl_lookup(*sel, ptr(values), vcode, d, shuffle, ptr(o["out"]), s), "mpl_lookup")
        else:
            _lib.check(L.mpl_score_select(*sel, s), "mpl_score_select")
            _lib.check(L.mpl_gather_wsum(ptr(values), vcode, n * n, d, ptr(o["slots"]), ptr(o["weights"]), M,
                                         H * k, shuffle, ptr(o["out"]), s), "mpl_gather_wsum")
        outs.append(o)
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("M,H,n,d_key,d,k,vdt,shuffle", [
    (8192, 4, 512, 256, 256, 16, torch.float16, 0),   # text-study layer: fused, one split
    (777, 4, 64, 64, 128, 16, torch.float16, 0),      # ragged token count, 128-wide fp16 rows
    (1000, 4, 128, 256, 256, 16, torch.float32, 0),   # fp32 rows (fact-task layer)
    (333, 4, 128, 128, 512, 16, torch.float16, 1),    # 512-wide rows, shuffled reads
    (64, 4, 1024, 256, 256, 16, torch.float16, 0),    # split-key plan merged before stage 2
    (16, 4, 1024, 256, 256, 16, torch.float16, 1),
    (1, 4, 1024, 256, 256, 16, torch.float16, 0),     # decode: one token, 4 split lists
    (5, 4, 1024, 256, 256, 16, torch.float32, 1),     # 32 split lists, fp32 rows, shuffled reads
    (3, 4, 2048, 128, 128, 16, torch.float16, 0),     # decode: 8 split lists, 128-wide rows
    (2, 4, 4096, 256, 128, 16, torch.float16, 1),     # decode: 16 split lists, shuffled reads
    (20, 4, 4096, 256, 128, 16, torch.float16, 0),    # 64 split lists
    (9, 4, 2500, 256, 256, 16, torch.float32, 0),     # 40 split lists (ragged n), fp32 rows
    (300, 2, 128, 64, 256, 16, torch.float16, 0),     # H = 2: two launches
    (300, 4, 128, 64, 256, 8, torch.float16, 0),      # k = 8: fused, the rows moved to adjoining lanes
    (300, 4, 128, 64, 96, 16, torch.float16, 0),      # 96-wide rows: fused, 12 vectors a row
])
def test_lookup_equals_select_then_gather(gpu_lib, M, H, n, d_key, d, k, vdt, shuffle):
    ref, got = _run(M, H, n, d_key, d, k, vdt, shuffle, seed=M + n)
    for name in ref:
        assert torch.equal(ref[name], got[name]), name
    assert bool((got["slots"] >= 0).all()) and bool((got["slots"] < n * n).all())


@pytest.mark.parametrize("M,H,n,d_key,d,k,vdt,shuffle", [
    (301, 4, 100, 64, 192, 8, torch.float16, 1),     # 24 vectors a row: two rows a load, 16 lanes idle
    (77, 4, 64, 64, 24, 5, torch.float16, 0),        # 3 vectors: 21 rows a load, 20 rows a token
    (50, 4, 64, 64, 8, 1, torch.float16, 0),         # one vector a row, k = 1
    (200, 4, 64, 32, 100, 16, torch.float32, 0),     # 25 fp32 vectors
    (130, 4, 300, 128, 512, 7, torch.float16, 0),    # 64 vectors, k < 16
    (65, 4, 64, 64, 132, 16, torch.float32, 1),      # 33 vectors: one row a load, 31 lanes idle
    (9, 4, 3000, 64, 192, 16, torch.float16, 0),     # more than 8 split lists, no fused width: two launches
    (9, 4, 3000, 64, 192, 4, torch.float16, 1),      # more than 8 split lists of k < 16
    (40, 2, 200, 64, 48, 11, torch.float32, 0),      # H = 2: two launches
    (30, 8, 200, 64, 520, 8, torch.float16, 0),      # 65 vectors: a thread per column
])
def test_any_row_width_and_k(gpu_lib, M, H, n, d_key, d, k, vdt, shuffle):
    """Row widths of any number of 16-byte vectors and k < 16: the lookup
    equals the two-launch path bit for bit, and both equal the sum of the
    selected rows in 64 bits within the rounding of H*k fp32 terms (each
    product and sum rounds to 2^-24 relative: H*k * 2^-24 * sum |w v|)."""
    ref, got = _run(M, H, n, d_key, d, k, vdt, shuffle, seed=M + n)
    for name in ref:
        assert torch.equal(ref[name], got[name]), name
    N = n * n
    g = torch.Generator(device="cuda").manual_seed(M + n)  # _run's values
    torch.randn((M, H, 2, d_key // 2), generator=g, device="cuda")
    torch.randn((H, 2, n, d_key // 2), generator=g, device="cuda")
    values = (torch.randn((N, d), generator=g, device="cuda") * 0.02).to(vdt).double()
    s = got["slots"].long().reshape(M, -1)
    assert bool((s >= 0).all()) and bool((s < N).all())
    terms = got["weights"].double().reshape(M, -1, 1) * values[(s + N // 2 + 1) % N if shuffle else s]
    bound = H * k * 2.0 ** -24 * terms.abs().sum(1) + 1e-12
    assert bool(((got["out"].double() - terms.sum(1)).abs() <= bound).all())
    torch.testing.assert_close(got["weights"].double().sum(-1), torch.ones((M, H), device="cuda").double(),
                               rtol=0, atol=k * 2.0 ** -22)


def test_lookup_zero_tokens_and_errors(gpu_lib):
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    # M = 0 launches nothing and succeeds
    assert L.mpl_lookup(None, _lib.MPL_Q_RAW, None, None, 0, 4, 64, 64, 16, _lib.MPL_F16, None, None, None,
                        None, 0, None, None, None, None, None, None, _lib.MPL_F16, 256, 0, None, s) == 0
    # a bad values dtype is reported, not launched
    rc = L.mpl_lookup(None, _lib.MPL_Q_RAW, None, None, 4, 4, 64, 64, 16, _lib.MPL_F16, None, None, None,
                      None, 0, None, None, None, None, None, None, 99, 256, 0, None, s)
    assert rc != 0 and b"values_dtype" in L.mpl_last_error()


@pytest.mark.parametrize("H,k,d,vdt", [
    (4, 5, 24, torch.float16),    # fused, 21 rows an instruction: the one load reaches a row past the last
    (4, 7, 24, torch.float16),    # fused, a second load with 7 rows of 21
    (4, 9, 64, torch.float32),    # fused, 4 rows an instruction, no row past the last
    (2, 9, 24, torch.float16),    # the read alone, any width
    (2, 9, 256, torch.float16),   # the read alone, 18 rows of a batch of 64
    (1, 5, 128, torch.float32),   # the same, fp32
    (2, 9, 8, torch.float16),     # one vector a row: all 18 rows in a group of 64
    (2, 9, 1024, torch.float16),  # two vectors a lane a row
    (8, 10, 512, torch.float16),  # 64 rows and 16 more
])
def test_infinite_entries_stay_infinite(gpu_lib, H, k, d, vdt):
    """A table whose column 0 is +inf: every weight is positive, so that
    column of the result is +inf, and the others are finite.  Rows past the
    last one take no part in the sum, not even with weight 0."""
    from model_amd.memory import MemoryPool
    pool = MemoryPool(32, H, 32, d, k, values_dtype=vdt)
    params = pool.init(0)
    params["params"]["values"][:, 0] = float("inf")
    q = torch.randn((37, H, 32), generator=torch.Generator(device="cuda").manual_seed(k), device="cuda")
    res = pool.lookup(params["params"], q)
    assert float(res["weights"].min()) > 0
    assert torch.equal(res["out"][:, 0], torch.full((37,), float("inf"), device="cuda"))
    assert bool(torch.isfinite(res["out"][:, 1:]).all())
