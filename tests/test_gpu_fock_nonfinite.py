"""An infinite density element in the streaming Fock build (64 < n <= 128): with positive
integrals every J and K that it reaches is +inf, in each form of the row loads (even n with
aligned rows; odd n, padded rows and unaligned rows), wherever in its row it stands. The last
column and row are what lanes and waves past the matrix read from clamped addresses."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.helpers import host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad,first", [(66, 0, 0), (67, 0, 0), (82, 1, 0), (82, 0, 1), (97, 2, 0), (127, 0, 0), (128, 1, 1)])
def test_infinite_density_gives_infinite_sums(core, n, pad, first):
    g = torch.ones((n, n, n, n), dtype=torch.float64, device="cuda")
    for c, d in ((0, n - 1), (n - 1, n - 1), (n - 1, 0), (3, 64)):
        store = torch.full((first + n * (n + pad),), float("nan"), dtype=torch.float64, device="cuda")
        D = store[first:].view(n, n + pad)[:, :n]
        D.fill_(1.0)
        D[c, d] = float("inf")
        for alpha_j, alpha_k in ((1.0, 1.0), (2.0, 0.5)):
            F = torch.zeros((n, n), dtype=torch.float64, device="cuda")
            core.fock_jk(g, D, F, alpha_j=alpha_j, alpha_k=alpha_k)
            assert np.all(host(F) == np.inf), (c, d, np.argwhere(host(F) != np.inf)[:4])
