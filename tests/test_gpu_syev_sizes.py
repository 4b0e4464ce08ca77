"""The Jacobi eigensolver at the sizes where its storage and its work split change: the small
kernel up to n = 64 with launch sizes that change at 16 and 32, above it M and V in LDS up to
n = 114 (FP64) or 162 (FP32), M alone up to 198 or 282, neither beyond; odd n with the index
that never rotates. Checked as in
test_gpu_linalg.py: eigenvalues to tol * |A|, A V = V W and V^T V = I to tol * sqrt(n), with
the tolerances derived there."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.helpers import dev, host
from tests.test_gpu_linalg import TOL, _check_eig, _sym

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,sizes", [(np.float64, (4, 5, 6, 15, 16, 17, 31, 32, 33, 49, 63, 64, 65, 113, 114, 115, 198, 199)),
                                         (np.float32, (5, 32, 64, 65, 162, 163, 282, 283))])
def test_storage_and_launch_edges(core, dtype, sizes):
    for n in sizes:
        A = _sym(n, 1000 + n, dtype)
        dA = dev(A)
        W = torch.empty(n, dtype=dA.dtype, device="cuda")
        core.syev(dA, W)
        _check_eig(A, host(W), host(dA), TOL[dtype])
        dN = dev(A)
        WN = torch.empty_like(W)
        core.syev(dN, WN, compute_vectors=False)
        assert torch.equal(W, WN) and np.array_equal(host(dN), A)


@pytest.mark.parametrize("scale", [1e-170, 1e170])
def test_extreme_scales(core, scale):
    """Squares of the entries under- or overflow nowhere but in the convergence norm, which
    decides as it did with unscaled rotations: zero norm or infinite limit, no sweep."""
    n = 24
    A = _sym(n, 7, np.float64)
    dA = dev(A * 1e-140)
    W = torch.empty(n, dtype=torch.float64, device="cuda")
    core.syev(dA, W)
    assert np.abs(host(W) - 1e-140 * np.linalg.eigvalsh(A)).max() <= 1e-12 * 1e-140 * np.linalg.norm(A)
    dB = dev(A * scale)
    info = core.syev(dB, W, check_info=False)
    assert int(info.item()) == 0  # as the norm decides
