"""mpl_scatter_rows and mpl_copy_arrays: copies, so bit for bit what torch's
index_copy_ and cat give."""

import pytest
import torch

from model_amd import _lib
from model_amd._lib import check, ptr
from model_amd.rows import _stacked

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,d,count,live", [(1, 1, 1, 1), (50, 3, 20, 20), (50, 256, 50, 31), (40000, 4, 33000, 32999),
                                            (700, 260, 300, 0), (9, 1024, 9, 9)])
def test_scatter_rows(gpu_lib, N, d, count, live):
    g = torch.Generator(device="cuda").manual_seed(N + d)
    rows = torch.randn((count, d), generator=g, device="cuda")
    rows[0, 0] = float("nan")
    idx = torch.randperm(N, generator=g, device="cuda")[:count].sort().values.to(torch.int32)
    idx[live:] = N  # padding, as a merge leaves it
    num = torch.full((1,), live, dtype=torch.int32, device="cuda")
    want = torch.zeros((N, d), device="cuda").index_copy_(0, idx[:live].long(), rows[:live])
    for count_dev in (num, None):
        out = torch.zeros((N, d), device="cuda")
        check(_lib.lib().mpl_scatter_rows(ptr(rows), ptr(idx), count, ptr(count_dev), d, N, ptr(out),
                                          _lib.stream_ptr(out.device)))
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("sizes,d", [([1, 1], 1), ([4095, 4097, 3], 1), ([7, 0, 260], 33), ([4096, 4096], 256)])
def test_stacked(gpu_lib, sizes, d):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    grads = [torch.randn((n, d), generator=g, device="cuda") for n in sizes]
    slots = [torch.randint(0, 1 << 30, (5 * n,), generator=g, device="cuda", dtype=torch.int32) for n in sizes]
    odd = [t.t().contiguous().t() for t in grads]  # other strides (d > 1): torch's own path
    for group in (grads, slots, odd):
        got, = _stacked(group)
        assert got.dtype == group[0].dtype and torch.equal(got, torch.cat(group))
    got = _stacked(slots, [s.float() for s in slots], grads)
    assert all(torch.equal(a, torch.cat(b)) for a, b in zip(got, (slots, [s.float() for s in slots], grads)))
