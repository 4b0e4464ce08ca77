"""The route of a generic contraction is an estimate of packing with a dense product against the
strided gather; whichever it takes, the result is that of both. Extents either side of where the
choice turns, aligned and not, against numpy. And tiles cut into many pieces, whose sums are read
four at a time: one tile left over by whole rounds, and the counts either side of four. Each
element is a sum of k products: at most (k + 3) roundings of the sum of their magnitudes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _check(C, ref, mag, k, dtype):
    eps = torch.finfo(dtype).eps * (2 if dtype == torch.float64 else 1)
    assert bool(((C.double() - ref).abs() <= (k + 3) * eps * mag).all())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("spec,ext", [
    (("mbej", "jnfb", "mnef"), dict(m=16, b=48, e=48, j=16, n=16, f=48)),
    (("mbej", "jnfb", "mnef"), dict(m=17, b=51, e=51, j=17, n=17, f=51)),
    (("mbej", "jnfb", "mnef"), dict(m=13, b=77, e=60, j=11, n=9, f=77)),
    (("pqrs", "pmrs", "mq"), dict(p=40, q=40, r=40, s=40, m=40)),
    (("pqrs", "pmrs", "mq"), dict(p=41, q=41, r=41, s=41, m=41)),
    (("acdb", "aebf", "fced"), dict(a=25, b=23, c=27, d=23, e=21, f=19)),
])
def test_routes_agree(core, dtype, spec, ext):
    gen = torch.Generator(device="cuda").manual_seed(sum(ext.values()))
    C0, A, B = (torch.randn([ext[c] for c in s], dtype=dtype, device="cuda", generator=gen) for s in spec)
    k = int(np.prod([e for c, e in ext.items() if c not in spec[0]]))
    es = f"{spec[1]},{spec[2]}->{spec[0]}"
    a, b = A.double().cpu().numpy(), B.double().cpu().numpy()
    prod = torch.from_numpy(np.einsum(es, a, b, optimize=True)).cuda()
    mag = torch.from_numpy(np.einsum(es, np.abs(a), np.abs(b), optimize=True)).cuda()
    old = C0.double()
    for route in ("auto", "ttgt", "gather"):
        with core.contraction_route(route):
            for beta in (0.0, 1.0):
                C = C0.clone() if beta else torch.full_like(C0, float("nan"))
                core.compile_plan(*spec).execute(beta, C, 0.5, A, B)
                _check(C, 0.5 * prod + beta * old, 0.5 * mag + beta * old.abs(), k, dtype)


@pytest.mark.parametrize("bm,schedule,bpc", [(64, 0, 1), (64, 0, 0), (64, 2, 0), (128, 0, 0)])
@pytest.mark.parametrize("m,n,k", [(1216, 1672, 512), (64, 64, 4096), (129, 127, 6000), (300, 200, 9000)])
def test_many_pieces(core, tmp_path, m, n, k, bm, schedule, bpc):
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    A = torch.randn(m, k, dtype=torch.float64, device="cuda", generator=gen)
    B = torch.randn(k, n, dtype=torch.float64, device="cuda", generator=gen)
    C = torch.empty(m, n, dtype=torch.float64, device="cuda")
    table = tmp_path / "table"
    table.write_text(f"8 {n} {m} {k} 1 0 1 : {bm} {bm} {schedule} {bpc}\n")
    core.clear_gemm_tuning()
    core.load_gemm_tuning(table)
    try:
        core.gemm("N", "N", 1.0, A, B, 0.0, C)
    finally:
        core.clear_gemm_tuning()
    _check(C, A @ B, A.abs() @ B.abs(), k, torch.float64)
