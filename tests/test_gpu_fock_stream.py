"""The streaming Fock build (64 < n <= 128) at the edges of its row split (n = 16 k and one
either side), with even and odd n, padded D and F, and a factor on F, against numpy. Each
result is a sum of n^2 products, so its rounding is below n^2 eps times the sum of their
magnitudes; that bound, divided by 16 for the 16-way tree of partial sums, is the tolerance."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.helpers import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [66, 79, 80, 81, 95, 97, 111, 112, 113, 127])
@pytest.mark.parametrize("pad,beta", [(0, 0.0), (1, -0.5), (2, 1.0)])
def test_against_numpy(core, n, pad, beta):
    rng = np.random.default_rng(n + pad)
    g = rng.uniform(-1, 1, (n, n, n, n))
    D, F = rng.uniform(-1, 1, (n, n + pad)), rng.uniform(-1, 1, (n, n + pad))
    dD, dF = dev(D), dev(F)
    core.fock_jk(dev(g), dD[:, :n], dF[:, :n], beta=beta)
    Dn = D[:, :n]

    def build(gg, dd):
        J = gg.reshape(n * n, n * n) @ dd.reshape(-1)
        K = np.tensordot(gg, dd, axes=((1, 3), (0, 1)))
        return J.reshape(n, n), K

    J, K = build(g, Dn)
    mag = sum(x * y for x, y in zip(build(np.abs(g), np.abs(Dn)), (2.0, 1.0))) + np.abs(beta * F[:, :n])
    got = host(dF)
    assert np.all(np.abs(got[:, :n] - (beta * F[:, :n] + 2 * J - K)) <= n * n / 16 * np.finfo(float).eps * mag)
    assert np.array_equal(got[:, n:], F[:, n:])


def test_infinite_integral_stays_in_its_sums(core):
    """g(a,b,c,d) = inf reaches J(a,b) and K(a,c) and nothing else (out-of-range lanes and rows
    read clamped addresses)."""
    for n in (67, 82):
        g = torch.ones((n, n, n, n), dtype=torch.float64, device="cuda")
        a, b, c, d = 3, 5, n - 1, n - 1
        g[a, b, c, d] = float("inf")
        D = torch.ones((n, n), dtype=torch.float64, device="cuda")
        F = torch.empty((n, n), dtype=torch.float64, device="cuda")
        core.fock_jk(g, D, F, alpha_j=1.0, alpha_k=1.0)
        bad = np.argwhere(~np.isfinite(host(F)))
        assert sorted(map(tuple, bad)) == sorted({(a, b), (a, c)})
