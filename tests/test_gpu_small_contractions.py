"""Small products and contractions, one wave per tile: extents at the edges of its tiles, of its
16-step chunks and of the split over the waves of a block, against numpy in double precision. Each element is a sum of k products, so its error is at most (k + 3) roundings of the
sum of their magnitudes, whatever the order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

DTYPES = {"f64": torch.float64, "f32": torch.float32}


def _check(got, want, mag, k, dtype):
    eps = torch.finfo(dtype).eps
    err = np.abs(got.cpu().numpy().astype(np.longdouble) - want)
    bound = (k + 3) * eps * mag + 4 * np.finfo(np.float64).tiny
    assert (err <= bound).all(), float((err / bound).max())


def _gemm_case(rng, m, n, k, ta, tb, dtype):
    A = torch.from_numpy(rng.standard_normal((m, k) if ta == "N" else (k, m))).to(dtype)
    B = torch.from_numpy(rng.standard_normal((k, n) if tb == "N" else (n, k))).to(dtype)
    a, b = A.double().numpy(), B.double().numpy()
    a, b = (a if ta == "N" else a.T), (b if tb == "N" else b.T)
    return A, B, a, b


@pytest.mark.parametrize("dtype", sorted(DTYPES))
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (1, 1, 700), (15, 17, 16), (16, 16, 63), (17, 33, 64), (33, 15, 65), (64, 64, 81),  # 4 waves from 64
    (48, 31, 511), (31, 48, 512), (5, 3, 513), (100, 7, 520), (16, 16, 3000),                     # 16 waves from 512
    (1000, 65, 20), (500, 500, 33), (700, 600, 100), (1024, 1024, 48),                            # larger tiles, 256 of 64^2
    (20000, 32, 17), (20000, 33, 17), (16, 30000, 24), (9000, 16, 1024), (9000, 16, 1025),        # a thin side
])
def test_gemm(core, dtype, m, n, k):
    rng, dt = np.random.default_rng(m + 7 * n + 11 * k), DTYPES[dtype]
    for ta, tb, beta in (("N", "N", 0.0), ("T", "N", -0.5), ("N", "T", 1.0), ("T", "T", 0.0)):
        A, B, a, b = _gemm_case(rng, m, n, k, ta, tb, dt)
        c0 = torch.from_numpy(rng.standard_normal((m, n))).to(dt)
        C = torch.full((m, n), float("nan"), dtype=dt, device="cuda") if beta == 0.0 else c0.cuda()
        core.gemm(ta, tb, 1.25, A.cuda(), B.cuda(), beta, C)
        want, mag = 1.25 * (a @ b), 1.25 * (np.abs(a) @ np.abs(b))
        if beta != 0.0:
            want, mag = want + beta * c0.double().numpy(), mag + np.abs(beta * c0.double().numpy())
        # double precision has the oracle's own rounding beside it
        _check(C, want, mag * (2 if dt == torch.float64 else 1), k, dt)


@pytest.mark.parametrize("dtype", sorted(DTYPES))
@pytest.mark.parametrize("spec,ext", [
    (("pqrs", "pmrs", "mq"), {c: 16 for c in "pqrsm"}),
    (("pqrs", "pmrs", "mq"), {"p": 5, "q": 17, "r": 6, "s": 33, "m": 64}),
    (("pqrs", "pqms", "mr"), {"p": 9, "q": 4, "r": 31, "s": 18, "m": 65}),
    (("mbej", "jnfb", "mnef"), {"m": 6, "b": 17, "e": 17, "j": 5, "n": 8, "f": 32}),   # chunks inside f
    (("mbej", "jnfb", "mnef"), {"m": 7, "b": 18, "e": 19, "j": 6, "n": 7, "f": 19}),   # and across it
    (("mbej", "jnfb", "mnef"), {"m": 3, "b": 6, "e": 6, "j": 3, "n": 23, "f": 37}),    # 16 waves to a tile
    (("jiz", "zik", "zkj"), {"z": 4, "i": 33, "j": 40, "k": 70}),                      # a batch
])
def test_einsum(core, dtype, spec, ext):
    rng, dt = np.random.default_rng(sum(ext.values())), DTYPES[dtype]
    mk = lambda s: torch.from_numpy(rng.standard_normal([ext[c] for c in s])).to(dt)
    C0, A, B = (mk(s) for s in spec)
    k = int(np.prod([e for c, e in ext.items() if c not in spec[0]]))
    a, b = A.double().numpy(), B.double().numpy()
    es = f"{spec[1]},{spec[2]}->{spec[0]}"
    prod, mag = np.einsum(es, a, b), np.einsum(es, np.abs(a), np.abs(b))
    for beta in (0.0, 1.0):
        C = C0.cuda() if beta else torch.full_like(C0, float("nan"), device="cuda")
        core.compile_plan(*spec).execute(beta, C, -0.75, A.cuda(), B.cuda())
        c0 = beta * C0.double().numpy()
        _check(C, -0.75 * prod + c0, (0.75 * mag + np.abs(c0)) * (2 if dt == torch.float64 else 1), k, dt)


def test_captured(core):
    from einsums_amd import blocks

    rng = np.random.default_rng(3)
    s = torch.cuda.Stream()
    A, B, _, _ = _gemm_case(rng, 70, 50, 600, "N", "T", torch.float64)
    A, B = A.cuda(), B.cuda()
    C = torch.zeros(70, 50, dtype=torch.float64, device="cuda")
    eager = torch.empty_like(C)
    s.wait_stream(torch.cuda.current_stream())
    core.gemm("N", "T", 1.0, A, B, 0.0, eager, stream=s)
    g = blocks.Graph(lambda: core.gemm("N", "T", 1.0, A, B, 0.0, C, stream=s), s)
    for _ in range(3):
        C.fill_(-1.0)
        torch.cuda.synchronize()
        g.replay()
        s.synchronize()
        assert torch.equal(C, eager)


def test_tuning_table(core, tmp_path):
    """One wave per tile is a configuration of the tuning table, in its file as 16 x 16."""
    f = tmp_path / "table"
    f.write_text("8 40 72 100 1 0 0 : 16 16 0 0\n")
    core.load_gemm_tuning(str(f))
    try:
        assert core.gemm_tuning_lookup(8, 40, 72, 100, 1, False, False)["bm"] == 16
        rng = np.random.default_rng(5)
        A, B, a, b = _gemm_case(rng, 72, 40, 100, "N", "N", torch.float64)
        C = torch.empty(72, 40, dtype=torch.float64, device="cuda")
        core.gemm("N", "N", 1.0, A.cuda(), B.cuda(), 0.0, C)
        _check(C, a @ b, 2 * (np.abs(a) @ np.abs(b)), 100, torch.float64)
        f.write_text("8 40 72 100 1 0 0 : 16 64 0 0\n")
        with pytest.raises(ValueError):
            core.load_gemm_tuning(str(f))
    finally:
        core.clear_gemm_tuning()
