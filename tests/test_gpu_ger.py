"""Outer products at the edges of the ger kernel's thread layout: one row or column (a rank-0
operand), extents around the 16-byte vector and the 256-thread block, unaligned and padded
outputs, and the factor on C (0, 1, other). An element is one rounded product and one rounded
update, so three units of the last place of max(|C|, |x y|) bound its error."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.helpers import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("beta", [0.0, 1.0, -0.5])
@pytest.mark.parametrize("m,n,pad", [(1, 1, 0), (1, 4099, 0), (4099, 1, 0), (1, 4096, 0), (2, 515, 0), (3, 70, 0),
                                     (70, 3, 2), (257, 65, 1), (512, 1030, 0), (1030, 512, 4), (1, 600, 3)])
def test_outer_product(core, m, n, pad, beta, dtype):
    rng = np.random.default_rng(m * 31 + n)
    x, y = rng.uniform(-1, 1, m).astype(dtype), rng.uniform(-1, 1, n).astype(dtype)
    c0 = rng.uniform(-1, 1, (m, n + pad)).astype(dtype)
    eps = np.finfo(dtype).eps
    for order in ("ij", "ji"):  # C row-major along y, then along x
        base = c0 if order == "ij" else np.ascontiguousarray(rng.uniform(-1, 1, (n, m + pad)).astype(dtype))
        dC = dev(base)
        view = dC[:, :n] if order == "ij" else dC[:, :m]
        alg = core.einsum(order, view, "i", dev(x), "j", dev(y), C_prefactor=beta, AB_prefactor=1.5)
        assert core.algorithm_name(alg) == "GER"
        prod = 1.5 * np.outer(x, y).astype(np.float64)
        prod = prod if order == "ij" else prod.T
        old = base[:, :prod.shape[1]].astype(np.float64)
        got = host(dC)
        assert np.all(np.abs(got[:, :prod.shape[1]] - (beta * old + prod)) <= 3 * eps * (np.abs(beta * old) + np.abs(prod)))
        assert np.array_equal(got[:, prod.shape[1]:], base[:, prod.shape[1]:])


def test_rank0_operand_fills_a_tensor(core):
    """dL/dt of a dot: a scalar times a tensor, C overwritten even where it holds NaN."""
    t = np.random.default_rng(3).standard_normal((3, 5, 7, 11))
    out = torch.full(t.shape, float("nan"), dtype=torch.float64, device="cuda")
    core.einsum("ijab", out, "", dev(np.array(2.0)), "ijab", dev(t), AB_prefactor=0.25)
    assert np.array_equal(host(out), 0.5 * t)
