"""The CRT split GEMM at the edges of its tiles (256 x 128), of its 64-step stages and three-deep
ring, of the 65536-step launches whose residues add up, and for every number of moduli (three or
four limbs, with and without the quotient correction above 50 bits). Operands of small integers
are held exactly by every representation, so the products have to be exact."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _ints(shape, bound, gen):
    return torch.randint(-bound, bound + 1, shape, device="cuda", generator=gen).double()


def _check(core, m, n, k, moduli, ta="N", tb="N", bound=500, pad=0):
    gen = torch.Generator(device="cuda").manual_seed(m * 5 + n * 3 + k + moduli)
    A = _ints((k, m + pad) if ta == "T" else (m, k + pad), bound, gen)
    B = _ints((n, k + pad) if tb == "T" else (k, n + pad), bound, gen)
    A = A[:, :m] if ta == "T" else A[:, :k]
    B = B[:, :k] if tb == "T" else B[:, :n]
    C = torch.full((m, n + pad), float("nan"), dtype=torch.float64, device="cuda")[:, :n]
    core.gemm_split(ta, tb, 2.0, A, B, 0.0, C, nslices=moduli, slice_type="crt")
    ref = 2.0 * ((A.T if ta == "T" else A) @ (B.T if tb == "T" else B))  # integers below 2^53: exact
    assert torch.equal(C, ref)
    C2 = C.clone()
    core.gemm_split(ta, tb, -1.0, A, B, 3.0, C2, nslices=moduli, slice_type="crt")
    assert torch.equal(C2, 3.0 * C - 0.5 * ref)


@pytest.mark.parametrize("moduli", range(8, 17))
def test_every_moduli_count(core, moduli):
    _check(core, 130, 70, 200, moduli)


@pytest.mark.parametrize("k", [1, 63, 64, 65, 128, 129, 192, 193, 256, 257, 320, 640])
def test_stage_counts(core, k):
    _check(core, 40, 30, k, 12)


@pytest.mark.parametrize("ta", "NT")
@pytest.mark.parametrize("tb", "NT")
@pytest.mark.parametrize("m,n,pad", [(1, 1, 0), (15, 17, 1), (255, 127, 0), (256, 128, 0), (257, 129, 3), (511, 383, 0),
                                     (700, 515, 2)])
def test_tile_edges(core, m, n, pad, ta, tb):
    _check(core, m, n, 70, 13, ta, tb, pad=pad)


def test_more_items_than_workgroups(core):
    _check(core, 2100, 2100, 96, 14, "T", "N")  # 9 x 17 tiles x 14 moduli


@pytest.mark.parametrize("k", [65536, 65537, 131200])
def test_several_launches(core, k):
    _check(core, 33, 20, k, 16, bound=20)
    _check(core, 33, 20, k, 9, bound=20)
