"""A batch of more LDS tiles than one grid holds (2^24 workgroups) is refused; it used to return
success with the first few products formed. The largest batch below the limit is computed."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from einsums_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,fits", [(2**24 - 1, True), (2**24, False), (2**24 + 8, False)])
def test_batch_of_long_dots(core, batch, fits):
    k = 1025  # above what the wave kernel takes with a short side
    core.clear_gemm_tuning()
    x = torch.full((k,), 0.5, dtype=torch.float32, device="cuda")
    C = torch.zeros(batch, dtype=torch.float32, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    status = _lib.lib.ein_gemm_strided_batched_f32(b"N", b"N", 1, 1, k, 1.0, ptr(x), 1, 0, ptr(x), k, 0, 0.0, ptr(C), 1, 1,
                                                   batch, stream)
    if fits:
        assert status == _lib.EIN_SUCCESS and bool((C == 0.25 * k).all())
    else:
        assert status == _lib.EIN_ERROR_UNSUPPORTED and not bool(C.any())
