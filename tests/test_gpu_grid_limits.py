"""Calls with more work than one grid has threads (fewer than 2^32; a larger one is cut to the
remainder without an error): element-wise permutes, matrix-vector products by rows and by
columns, and reductions with a wave per target, each a little beyond the limit. The values are
small integers, so the results are exact; operands are filled and compared in parts."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from einsums_amd import _lib

pytestmark = pytest.mark.gpu

PART = 2**26


def _need(gib):
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < gib << 30:
        pytest.skip(f"needs {gib} GiB of device memory")


def _pattern(n, period):
    return (torch.arange(n, device="cuda") % period).float()


def _filled(n, period):
    out = torch.empty(n, dtype=torch.float32, device="cuda")
    p = _pattern(PART + period, period)
    for i, part in enumerate(out.split(PART)):
        at = i * PART % period
        part.copy_(p[at:at + part.numel()])
    return out


def _wrong(got, expect):
    return sum(int((g != e).sum().item()) for g, e in zip(got.split(PART), expect.split(PART)))


@pytest.mark.parametrize("rows", [2**22, 2**22 + 1])
def test_identity_permute(core, rows):
    _need(40)
    cols = 1024
    A = _filled(rows * cols, 8191).view(rows, cols)
    C = torch.full((rows, cols), -1.0, dtype=torch.float32, device="cuda")
    core.permute(0.0, "ij", C, 2.0, "ij", A)
    A.mul_(2.0)
    wrong = _wrong(C.view(-1), A.view(-1))
    del A, C
    torch.cuda.empty_cache()
    assert wrong == 0


@pytest.mark.parametrize("incy", [1, -1])
@pytest.mark.parametrize("trans,m,n", [("N", 2**30 + 5, 1), ("T", 3, 2**26 + 5)])
def test_gemv(trans, m, n, incy):
    _need(16)
    length = m if trans == "N" else n
    period = 1021
    A = _filled(m * n, period)
    x = torch.ones(n if trans == "N" else m, dtype=torch.float32, device="cuda")
    y = torch.full((length,), -1.0, dtype=torch.float32, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib.ein_gemv_f32(trans.encode(), m, n, 1.0, ptr(A), m, ptr(x), 1, 0.0, ptr(y), incy, stream))
    expect = A if trans == "N" else A.view(n, m).sum(1)
    if incy < 0:
        y = y.flip(0)
    wrong = _wrong(y, expect)
    del A, y, expect
    torch.cuda.empty_cache()
    assert wrong == 0


def test_wave_per_target_reduction(core):
    _need(16)
    nt, k = 2**26 + 5, 33  # above the links that one thread takes
    row = _filled(nt, 127)
    A = torch.empty((nt, k), dtype=torch.float32, device="cuda")
    for a, r in zip(A.split(PART // 4), row.split(PART // 4)):
        a.copy_(r[:, None].expand(-1, k))
    B = torch.ones(k, dtype=torch.float32, device="cuda")
    C = torch.full((nt,), -1.0, dtype=torch.float32, device="cuda")
    core.contract("i", C, "ik", A, "k", B)
    row.mul_(k)
    wrong = _wrong(C, row)
    del A, C
    torch.cuda.empty_cache()
    assert wrong == 0
