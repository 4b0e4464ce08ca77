"""More tiles of one wave each than one launch takes (2^26 - 4): a batch of 2 x 2 products whose
last ones are in the second launch. Small integers, so every result is exact."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from einsums_amd import _lib

pytestmark = pytest.mark.gpu

PART = 2**22


def test_batch_beyond_one_launch():
    batch = 2**26 + 9
    if torch.cuda.mem_get_info()[0] < 8 << 30:
        pytest.skip("needs 5 GB of device memory")
    A, B = (torch.randint(-4, 5, (batch, 4), device="cuda", dtype=torch.int8).float() for _ in range(2))
    C = torch.full((batch, 4), 99.0, dtype=torch.float32, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib.ein_gemm_strided_batched_f32(b"N", b"N", 2, 2, 2, 1.0, ptr(A), 2, 4, ptr(B), 2, 4, 0.0, ptr(C), 2,
                                                     4, batch, stream))
    wrong = 0
    for a, b, c in zip(A.split(PART), B.split(PART), C.split(PART)):
        for i in range(2):
            for j in range(2):  # column-major: element (i, j) is word i + 2 j
                ref = a[:, i] * b[:, 2 * j] + a[:, i + 2] * b[:, 1 + 2 * j]
                wrong += int((c[:, i + 2 * j] != ref).sum().item())
    del A, B, C
    torch.cuda.empty_cache()
    assert wrong == 0
