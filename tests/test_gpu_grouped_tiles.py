"""Grouped plans at the edges of their wave tiles: extents around 16, 32 and 64 rows and
columns, contractions around the 4-step MFMA and the 16-step chunk, every storage order of the
three operands, links and rows of one and of several digits (tables), batches, unaligned and
padded operands, before and after the autotuner. FP64 and FP32 sums of k products against
numpy in FP64: (k + 2) eps times the sum of the magnitudes bounds each element."""
import itertools

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from einsums_amd import blocks
from tests.helpers import host

pytestmark = pytest.mark.gpu


def _view(x, pad):
    """x in a buffer with `pad` unused elements at the start and the end of its last axis."""
    buf = torch.zeros((*x.shape[:-1], x.shape[-1] + 2 * pad), dtype=x.dtype, device="cuda")
    v = buf[..., pad:pad + x.shape[-1]]
    v.copy_(x)
    return v


def _check(terms, dtype, autotune):
    rng = np.random.default_rng(5)
    todo, refs = [], []
    for ci, ai, bi, ext, pad, beta in terms:
        A, B, C = (rng.uniform(-1, 1, [ext[x] for x in idx]).astype(dtype) for idx in (ai, bi, ci))
        dA, dB, dC = (_view(torch.from_numpy(x), pad) for x in (A, B, C))
        todo.append((ci, dC, ai, dA, bi, dB, beta, 1.5))
        k = np.prod([ext[x] for x in set(ai + bi) - set(ci)] or [1])
        A, B, C = (x.astype(np.float64) for x in (A, B, C))
        f = lambda a, b: np.einsum(f"{ai},{bi}->{ci}", a, b, optimize=True)
        refs.append((dC, beta * C + 1.5 * f(A, B), np.abs(beta * C) + 1.5 * f(np.abs(A), np.abs(B)), k))
    plan = blocks.GroupedEinsum(todo, autotune=autotune)
    plan.execute()
    for dC, ref, mag, k in refs:
        assert np.all(np.abs(host(dC) - ref) <= (k + 2) * np.finfo(dtype).eps * mag + 1e-300)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("autotune", [False, True])
def test_extents(dtype, autotune):
    sizes = [(1, 1, 1), (15, 17, 3), (16, 16, 4), (17, 15, 5), (31, 33, 15), (32, 32, 16), (33, 31, 17), (48, 20, 31),
             (64, 64, 32), (65, 63, 33), (129, 5, 48), (5, 129, 130), (127, 96, 2047)]
    orders = itertools.cycle([("ij", "ik", "kj"), ("ji", "ik", "kj"), ("ij", "ki", "jk"), ("ji", "ki", "kj"),
                              ("ij", "ik", "jk")])
    _check([(*next(orders), dict(i=m, j=n, k=k), pad, beta) for m, n, k in sizes for pad, beta in ((0, 0.0), (1, -0.5))],
           dtype, autotune)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_digits_and_batches(dtype):
    ext = dict(i=5, j=7, k=3, l=6, m=32, b=4, a=11)
    _check([("ij", "ikl", "lkj", ext, 0, 0.0),       # two link digits in different orders: table per step
            ("ij", "ilm", "mlj", ext, 1, 1.0),       # innermost link a multiple of 16: affine chunks
            ("iaj", "ika", "kj", ext, 0, 0.5),       # two row digits, split in C
            ("bij", "bik", "kbj", ext, 1, 0.0),      # batch label
            ("bij", "kbi", "bjk", ext, 0, -1.0),
            ("ai", "ia", "b", ext, 0, 0.0)], dtype, False)  # b summed alone


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_tall_tiles(dtype):
    _check([("ij", "ik", "kj", dict(i=511, j=127, k=120 + z), 0, 0.0) for z in range(24)], dtype, True)


def test_infinities_stay_in_their_row_and_column():
    """A padded row, column or step never meets another element."""
    for m, n, k in ((17, 33, 5), (33, 17, 18)):
        A = torch.ones((m, k), dtype=torch.float64, device="cuda")
        B = torch.ones((k, n), dtype=torch.float64, device="cuda")
        A[m - 1, k - 1] = float("inf")
        B[k - 1, n - 1] = float("inf")
        C = torch.empty((m, n), dtype=torch.float64, device="cuda")
        blocks.GroupedEinsum([("ij", C, "ik", A, "kj", B, 0.0, 1.0)]).execute()
        ref = (A.cpu().numpy() @ B.cpu().numpy())
        assert np.array_equal(host(C), ref)
