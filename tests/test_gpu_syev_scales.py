"""The eigensolver does not depend on the scale of the matrix: entries whose squares leave the
range of the type are decomposed like those near one. Every scale is a power of two, so the
eigenvalues are those of the unscaled matrix times it. Tolerances as in test_gpu_linalg.py,
relative to the unscaled matrix."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.helpers import dev, host
from tests.test_gpu_linalg import TOL, _check_eig, _sym

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,exponents", [(np.float64, (-1000, -565, -490, 480, 565, 1000)),
                                             (np.float32, (-110, -77, -50, 50, 64, 110))])
@pytest.mark.parametrize("n", [3, 24, 63, 70, 130, 210])  # each storage of M and V
def test_power_of_two_scales(core, n, dtype, exponents):
    A = _sym(n, 17 + n, dtype)
    for e in exponents:
        dA = dev(np.ldexp(A, e))
        W = torch.empty(n, dtype=dA.dtype, device="cuda")
        info = core.syev(dA, W)
        assert int(info.item()) == 0
        _check_eig(A, np.ldexp(host(W), -e), host(dA), TOL[dtype])


@pytest.mark.parametrize("n", [4, 70])
def test_zero_and_infinite_entries(core, n):
    Z = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    W = torch.empty(n, dtype=torch.float64, device="cuda")
    core.syev(Z, W)
    assert host(W).tolist() == [0.0] * n and torch.equal(Z, torch.eye(n, dtype=Z.dtype, device="cuda"))
    # a diagonal matrix is decomposed already, an infinity beside the diagonal has no decomposition
    D = np.diag(np.arange(n, 0.0, -1.0))
    D[1, 1] = np.inf
    dD = dev(D)
    core.syev(dD, W)
    assert host(W).tolist() == sorted(np.diag(D))
    A = _sym(n, 5, np.float64)
    A[0, 2] = A[2, 0] = np.inf
    info = core.syev(dev(A), W, check_info=False)
    assert int(info.item()) == 1
