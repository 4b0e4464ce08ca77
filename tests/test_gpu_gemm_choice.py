"""Mid-sized GEMMs, whose tile and schedule a cost model chooses: extents where it takes each of
its candidates (tiles of 64 x 64 split over the chip or whole, 128 x 128, 96 x 96, FP32 128 x 64),
batches and thin sides among them, against the FP64 product of the same values; and captured calls. A sum of k products and its
update round by at most (k + 2) eps of the sum of their magnitudes (FP64: the reference too)."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _data(shape, dtype, gen):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)


def _check(C, ref, mag, k, dtype):
    bound = (k + 2) * torch.finfo(dtype).eps * mag * (2 if dtype == torch.float64 else 1)
    assert bool(((C.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("ta,tb", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k", [(776, 792, 400), (728, 1200, 272), (576, 576, 5776), (980, 980, 980),
                                  (1216, 1184, 1136), (361, 361, 7744), (2025, 2025, 515), (2047, 2049, 130),
                                  (100, 4001, 1200), (3000, 65, 2100), (1449, 1451, 301)])
def test_products(core, dtype, m, n, k, ta, tb):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    A = _data((m, k) if ta == "N" else (k, m), dtype, gen)
    B = _data((k, n) if tb == "N" else (n, k), dtype, gen)
    C = _data((m, n), dtype, gen)
    a, b = (x.double().T if t == "T" else x.double() for x, t in ((A, ta), (B, tb)))
    old = C.double().clone()
    core.gemm(ta, tb, 0.5, A, B, 1.0, C)
    _check(C, 0.5 * (a @ b) + old, 0.5 * (a.abs() @ b.abs()) + old.abs(), k, dtype)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("b,m,n,k", [(5, 824, 864, 72), (28, 152, 288, 168), (9, 280, 792, 152), (3, 500, 500, 500)])
def test_batches(core, dtype, b, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(b + m)
    A, B, C = _data((b, m, k), dtype, gen), _data((b, k, n), dtype, gen), _data((b, m, n), dtype, gen)
    core.compile_plan("bij", "bik", "bkj").execute(0.0, C, 1.0, A, B)
    for z in range(b):
        x, y = A[z].double(), B[z].double()
        _check(C[z], x @ y, x.abs() @ y.abs(), k, dtype)


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 256), (2048, 2048, 320), (1216, 1184, 1136)])
def test_captured(core, m, n, k):
    """Captured after the same call has run on the stream: the same configuration, bit for bit."""
    from einsums_amd import blocks

    gen = torch.Generator(device="cuda").manual_seed(7)
    A, B = _data((m, k), torch.float64, gen), _data((k, n), torch.float64, gen)
    C, eager = torch.zeros(m, n, dtype=torch.float64, device="cuda"), torch.empty(m, n, dtype=torch.float64, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    core.gemm("N", "N", 1.0, A, B, 0.0, eager, stream=s)
    g = blocks.Graph(lambda: core.gemm("N", "N", 1.0, A, B, 0.0, C, stream=s), s)
    for _ in range(3):
        C.fill_(-1.0)
        torch.cuda.synchronize()
        g.replay()
        s.synchronize()
        assert torch.equal(C, eager)
