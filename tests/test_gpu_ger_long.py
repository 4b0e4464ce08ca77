"""Rank-one updates with more rows than one launch has threads (a grid holds fewer than 2^32):
one row of 2^32 + 5 elements, which the kernel takes as that many rows of one element, and one
column of the same. Products with a power of two are exact; the operands are filled and
compared in parts of less than 2^31 elements."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from einsums_amd import _lib

pytestmark = pytest.mark.gpu

N = 2**32 + 5
PART = 2**28


@pytest.mark.parametrize("m,n", [(1, N), (N, 1)])
def test_beyond_one_grid(m, n):
    if torch.cuda.mem_get_info()[0] < 48 << 30:
        pytest.skip("needs 40 GB of device memory")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    ramp = torch.arange(PART, device="cuda", dtype=torch.float32)
    long = torch.empty(N, dtype=torch.float32, device="cuda")
    A = torch.empty(N, dtype=torch.float32, device="cuda")
    for i, (y, a) in enumerate(zip(long.split(PART), A.split(PART))):
        y.copy_(ramp[:y.numel()]).add_(i)
        a.fill_(-1.0)
    one = torch.full((1,), 2.0, dtype=torch.float32, device="cuda")
    x, y = (one, long) if m == 1 else (long, one)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib.ein_ger_f32(m, n, 0.25, ptr(x), 1, ptr(y), 1, ptr(A), m, stream))
    wrong = [int((a != y * 0.5 - 1.0).sum().item()) for y, a in zip(long.split(PART), A.split(PART))]
    del x, y, long, A, ramp
    torch.cuda.empty_cache()
    assert wrong == [0] * len(wrong)
