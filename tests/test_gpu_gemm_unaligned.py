"""Dense GEMMs whose operands the 16-byte DMA cannot take (odd leading dimensions and extents,
unaligned bases, strides other than one), staged through registers: every tile of the tuning
table at the edges of its rows, chunks and slabs, against the FP64 product of the same values.
A sum of k products and its update round by at most (k + 2) eps of the sum of their magnitudes
(FP64: the reference too)."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TILES = [(64, 64), (64, 128), (128, 64), (128, 128), (96, 96), (256, 128)]


def _operand(rows, cols, trans, pad, shift, dtype, gen):
    r, c = (cols, rows) if trans == "T" else (rows, cols)
    flat = torch.randn(r * (c + pad) + shift, dtype=dtype, device="cuda", generator=gen)
    return flat[shift:].view(r, c + pad)[:, :c]


def _check(C, old, A, B, ta, tb, beta, k, dtype):
    a, b = (x.double().T if t == "T" else x.double() for x, t in ((A, ta), (B, tb)))
    ref, mag = a @ b + beta * old, a.abs() @ b.abs() + (beta * old).abs()
    bound = (k + 2) * torch.finfo(dtype).eps * mag * (2 if dtype == torch.float64 else 1)
    assert bool(((C.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("bm,bn", TILES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k,pad,shift", [(129, 127, 33, 0, 0), (65, 193, 15, 1, 0), (97, 95, 47, 0, 1),
                                            (256, 128, 64, 0, 1), (255, 257, 31, 2, 1), (1, 3, 17, 0, 0)])
def test_tiles(core, tmp_path, bm, bn, dtype, m, n, k, pad, shift):
    eb = torch.finfo(dtype).bits // 8
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    table = tmp_path / "table"
    for ta in "NT":
        for tb in "NT":
            if bm == 96 and (eb != 8 or (ta, tb) != ("N", "T")) or bm == 256 and eb != 4:
                continue  # tiles of one staging class or type only
            # the normalised problem: C's contiguous extent first, then A and B swap roles
            table.write_text(f"{eb} {n} {m} {k} 1 {int(tb == 'T')} {int(ta == 'N')} : {bm} {bn} 0 0\n")
            core.clear_gemm_tuning()
            core.load_gemm_tuning(table)
            try:
                assert core.gemm_tuning_lookup(eb, n, m, k, 1, tb == "T", ta == "N") is not None
                A = _operand(m, k, ta, pad, shift, dtype, gen)
                B = _operand(k, n, tb, pad, shift, dtype, gen)
                C = _operand(m, n, "N", pad, shift, dtype, gen)
                for beta in (0.0, -0.5):
                    old = C.double().clone()
                    core.gemm(ta, tb, 1.0, A, B, beta, C)
                    _check(C, old, A, B, ta, tb, beta, k, dtype)
            finally:
                core.clear_gemm_tuning()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_strided_views(core, dtype):
    """Neither direction contiguous: elements one by one."""
    gen = torch.Generator(device="cuda").manual_seed(1)
    m, n, k = 1031, 777, 301
    A = torch.randn(m, 2 * k, dtype=dtype, device="cuda", generator=gen)[:, ::2]
    B = torch.randn(2 * k, 3 * n, dtype=dtype, device="cuda", generator=gen)[::2, ::3]
    C = torch.zeros(m, n, dtype=dtype, device="cuda")
    core.compile_plan("ij", "ik", "kj").execute(0.0, C, 1.0, A, B)
    _check(C, torch.zeros_like(C).double(), A, B, "N", "N", 0.0, k, dtype)
