"""syev on matrices that no solver layout fits (neither stride is one): solved on a contiguous
copy, whose status is the call's. The allocator's cached blocks hold nonzero words first, so a
status that nothing writes shows. Tolerances as in test_gpu_linalg.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.helpers import dev, host
from tests.test_gpu_linalg import TOL, _check_eig, _sym

pytestmark = pytest.mark.gpu


def _dirty_cache():
    blocks = [torch.full((8,), 0x7EADBEEF, dtype=torch.int32, device="cuda") for _ in range(64)]
    del blocks


def _strided(A):
    n = A.shape[0]
    X = torch.full((2 * n, 2 * n), float("nan"), dtype=torch.from_numpy(A).dtype, device="cuda")
    X[::2, ::2] = dev(A)
    return X, X[::2, ::2]


@pytest.mark.parametrize("n", [1, 2, 5, 24, 70])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_status_values_and_vectors(core, n, dtype):
    A = _sym(n, 50 + n, dtype)
    X, view = _strided(A)
    W = torch.empty(n, dtype=X.dtype, device="cuda")
    _dirty_cache()
    info = core.syev(view, W)
    assert int(info.item()) == 0
    _check_eig(A, host(W), host(view), TOL[dtype])
    assert torch.isnan(X[1::2]).all() and torch.isnan(X[:, 1::2]).all()
    _dirty_cache()
    info = core.syev(_strided(A)[1], W, compute_vectors=False, check_info=False)
    assert int(info.item()) == 0


def test_failure_of_the_solve_is_reported(core):
    A = _sym(12, 3, np.float64)
    A[2, 7] = A[7, 2] = np.nan
    W = torch.empty(12, dtype=torch.float64, device="cuda")
    info = core.syev(_strided(A)[1], W, check_info=False)
    assert int(info.item()) == 1
    with pytest.raises(core.EinsumsError):
        core.syev(_strided(A)[1], W)
