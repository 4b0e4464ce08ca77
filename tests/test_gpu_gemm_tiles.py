"""Dense GEMMs at the edges of the FP32 256 x 128 tile (taken from two rounds of tiles on) and of
the k-major LDS layouts that move several k-rows per instruction (FP32 and FP64 64-row tiles,
FP32 128-row tiles): extents one either side of a tile, aligned and unaligned leading
dimensions, all transposes, against the FP64 product of the same values. A sum of k products
and its update round by at most (k + 2) eps of the sum of their magnitudes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _operand(rows, cols, trans, pad, dtype, gen):
    shape = (cols, rows) if trans == "T" else (rows, cols)
    x = torch.randn((shape[0], shape[1] + pad), dtype=dtype, device="cuda", generator=gen)
    return x[:, :shape[1]]


def _check(core, m, n, k, ta, tb, pad, dtype, beta):
    gen = torch.Generator(device="cuda").manual_seed(m * 7 + n * 3 + k)
    A, B = _operand(m, k, ta, pad, dtype, gen), _operand(k, n, tb, pad, dtype, gen)
    C = _operand(m, n, "N", pad, dtype, gen)
    old = C.double().clone()
    core.gemm(ta, tb, 1.0, A, B, beta, C)
    a, b = (x.double().T if t == "T" else x.double() for x, t in ((A, ta), (B, tb)))
    ref, mag = a @ b + beta * old, a.abs() @ b.abs() + (beta * old).abs()
    assert bool(((C.double() - ref).abs() <= (k + 2) * torch.finfo(dtype).eps * mag).all())


@pytest.mark.parametrize("ta", "NT")
@pytest.mark.parametrize("tb", "NT")
@pytest.mark.parametrize("m,n,k,pad,beta", [(4096, 4096, 16, 0, 0.0), (4100, 4352, 44, 0, 1.0), (4095, 4353, 33, 0, 0.0),
                                            (8448, 2304, 17, 3, -0.5), (2304, 8448, 20, 4, 0.0)])
def test_fp32_256_rows(core, m, n, k, ta, tb, pad, beta):
    _check(core, m, n, k, ta, tb, pad, torch.float32, beta)


@pytest.mark.parametrize("ta", "NT")
@pytest.mark.parametrize("tb", "NT")
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,n,k,pad", [(60, 68, 20, 0), (64, 64, 16, 0), (124, 1024, 100, 0), (1024, 92, 300, 4),
                                       (128, 128, 128, 0), (260, 252, 64, 0), (576, 576, 1200, 0)])
def test_kmajor_groups(core, m, n, k, pad, ta, tb, dtype):
    _check(core, m, n, k, ta, tb, pad, dtype, 0.5)
