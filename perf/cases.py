"""Performance cases: the einsum, GEMM, Fock, SCF, gradient and block work that programs built
on this library run, called through the public Python entry points.

A case is a dict with a "kind" and sizes:

* "wabef", "wmnij", "wmbej": one CCD W intermediate, W += prefactor * contraction, in FP64 or
  (split = "crt") with the FP64 product emulated on int8 matrix cores. o and v are the numbers
  of occupied and virtual orbitals: 2 o^2 v^4, 2 o^4 v^2 and 2 o^3 v^3 flops.
* "gemm": C = alpha op(A) op(B) + beta C on row-major matrices, FP64 or FP32.
* "reorder": what a CCD iteration does with its amplitudes beside the products: the energy
  dot, the axis swap ijab -> iajb and the transposing reorder jnfb -> jbnf.
* "hf": G = 2J - K by the two einsum calls of a Hartree-Fock program (matrix-vector and
  generic contraction); "fock": the same matrix by the one-pass fock_jk.
* "scf": one restricted Hartree-Fock iteration as the reference's HF test makes it: Fock
  build, F' = X^T F X, eigensolve, orbital coefficients, density and energy.
* "ao2mo": the four quarter transformations of the two-electron integrals to the MO basis.
* "grad": loss and dL/dt of L(t) = 1/4 t.g + 1/8 t_ijab t_klab W_klij through autograd.
* "grouped": a batch of uneven small GEMMs (the blocks of a block-sparse tensor) as one plan.
"""
import math
import random

import torch

import einsums_amd.core as core
from einsums_amd import autograd, blocks, workloads

DTYPES = {"f64": torch.float64, "f32": torch.float32}

# (C labels, A labels, B labels, prefactor) of the CCD intermediates; t and g are (o, o, v, v)
CCD = {
    "wabef": ("abef", "mnef", "mnab", 0.25),  # A = g, B = t
    "wmnij": ("mnij", "ijef", "mnef", 0.25),  # A = t, B = g
    "wmbej": ("mbej", "jnfb", "mnef", -0.5),  # A = t, B = g
}


def listed():
    return [
        # the particle ladder, the largest product of a CCD iteration: many tiles, short k
        {"name": "wabef_f64", "kind": "wabef", "o": 24, "v": 96, "split": ""},
        # the hole ladder: a small output with a contraction over all virtual pairs
        {"name": "wmnij_f64", "kind": "wmnij", "o": 24, "v": 96, "split": ""},
        # the ring term: no operand folds into a matrix, the generic contraction
        {"name": "wmbej_f64", "kind": "wmbej", "o": 24, "v": 96, "split": ""},
        # the particle ladder of a larger molecule in split precision, the largest case
        {"name": "wabef_crt", "kind": "wabef", "o": 32, "v": 128, "split": "crt"},
        # a plain matrix product in single precision
        {"name": "gemm_f32", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "ta": "N", "tb": "N", "dtype": "f32",
         "beta": 0.0},
        # a product with odd extents, nothing a multiple of a tile or of 16 bytes
        {"name": "gemm_f64_odd", "kind": "gemm", "m": 1531, "n": 1013, "k": 2047, "ta": "N", "tb": "T", "dtype": "f64",
         "beta": 1.0},
        # the memory-bound steps of a CCD iteration
        {"name": "reorder_f64", "kind": "reorder", "o": 32, "v": 128},
        # Coulomb and exchange of a medium molecule in one pass
        {"name": "fock_jk", "kind": "fock", "n": 96},
        # small molecules: a chain of short calls, where latency and launches count; the
        # iteration holds the two-call Coulomb and exchange build too
        {"name": "scf_iteration", "kind": "scf", "n": 48, "nocc": 12},
        {"name": "ao2mo", "kind": "ao2mo", "n": 24, "dtype": "f64"},
        # forward and backward of the CCD-like loss
        {"name": "grad_f64", "kind": "grad", "o": 32, "v": 128, "dtype": "f64"},
        # blocks of a block-sparse tensor: extents log-uniform in [lo, hi]
        {"name": "grouped_f64", "kind": "grouped", "count": 1024, "lo": 4, "hi": 512, "dtype": "f64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["wabef", "wmnij", "wmbej", "wabef", "gemm", "gemm", "reorder", "hf", "fock", "scf", "ao2mo",
                       "grad", "grouped"])
    if kind in CCD:
        split = "crt" if kind != "wmnij" and rng.random() < 0.4 else ""
        o = _log(rng, 8, 32)
        v = _log(rng, 32, 128 if split else 104)
        return {"kind": kind, "o": o, "v": v, "split": split}
    if kind == "gemm":
        return {"kind": "gemm", "m": _log(rng, 128, 4096), "n": _log(rng, 128, 4096), "k": _log(rng, 128, 4096),
                "ta": rng.choice("NT"), "tb": rng.choice("NT"), "dtype": rng.choice(["f64", "f32"]),
                "beta": rng.choice([0.0, 1.0])}
    if kind == "reorder":
        return {"kind": "reorder", "o": _log(rng, 8, 40), "v": _log(rng, 32, 160)}
    if kind == "hf":
        return {"kind": "hf", "n": _log(rng, 16, 110)}
    if kind == "fock":
        return {"kind": "fock", "n": _log(rng, 24, 110)}
    if kind == "scf":
        n = _log(rng, 7, 100)
        return {"kind": "scf", "n": n, "nocc": max(2, n // 4)}
    if kind == "ao2mo":
        return {"kind": "ao2mo", "n": _log(rng, 7, 64), "dtype": rng.choice(["f64", "f32"])}
    if kind == "grad":
        return {"kind": "grad", "o": _log(rng, 8, 32), "v": _log(rng, 24, 128), "dtype": rng.choice(["f64", "f32"])}
    return {"kind": "grouped", "count": _log(rng, 128, 1024), "lo": 4, "hi": _log(rng, 48, 512),
            "dtype": rng.choice(["f64", "f32"])}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, scale, dtype=torch.float64):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen).mul_(scale)


def _eri(gen, n):
    """Integrals (pq|rs) with their eight-fold symmetry."""
    g = _normal(gen, (n, n, n, n), 1.0 / n)
    g = (g + g.transpose(0, 1)).mul_(0.5)
    g = (g + g.transpose(2, 3)).mul_(0.5)
    return (g + g.permute(2, 3, 0, 1)).mul_(0.5).contiguous()


def _orthonormal(gen, n):
    return torch.linalg.qr(_normal(gen, (n, n), 1.0))[0]


def _ccd_operands(case, seed):
    """The intermediate's start value and the two operands, as workloads.ccd_inputs draws them."""
    kind = case["kind"]
    inp = workloads.ccd_inputs_device(case["o"], case["v"], seed, with_vvvv=kind == "wabef")
    if kind == "wabef":
        return inp.g_vvvv, inp.g_oovv, inp.t_oovv
    return (inp.g_oooo if kind == "wmnij" else inp.g_ovvo), inp.t_oovv, inp.g_oovv


def _gemm_operands(case, seed):
    gen, dtype = _gen(seed), DTYPES[case["dtype"]]
    m, n, k = case["m"], case["n"], case["k"]
    A = _normal(gen, (m, k) if case["ta"] == "N" else (k, m), 1.0, dtype)
    B = _normal(gen, (k, n) if case["tb"] == "N" else (n, k), 1.0, dtype)
    return A, B, _normal(gen, (m, n), 1.0, dtype)


def _scf_operands(case, seed):
    gen, n, nocc = _gen(seed), case["n"], case["nocc"]
    # a core Hamiltonian with a gap between occupied and virtual levels, so that the density
    # is well determined, a near-unit overlap and a density of nocc orbitals
    levels = torch.cat([torch.linspace(-20.0, -1.0, nocc, dtype=torch.float64),
                        torch.linspace(0.5, 6.0, n - nocc, dtype=torch.float64)]).cuda()
    Q = _orthonormal(gen, n)
    H = (Q * levels) @ Q.T
    H = ((H + H.T) / 2).contiguous()
    S = _normal(gen, (n, n), 0.05 / math.sqrt(n))
    w, U = torch.linalg.eigh(torch.eye(n, dtype=torch.float64, device="cuda") + (S + S.T) / 2)
    X = ((U * w.rsqrt()) @ U.T).contiguous()
    C = _orthonormal(gen, n)[:, :nocc]
    return _eri(gen, n), H, X, (C @ C.T).contiguous()


def _grad_operands(case, seed):
    gen, dtype, o, v = _gen(seed), DTYPES[case["dtype"]], case["o"], case["v"]

    def anti(x):
        x = (x - x.transpose(0, 1)).mul_(0.5)
        return (x - x.transpose(2, 3)).mul_(0.5).contiguous()

    s = 1.0 / math.sqrt(v)
    return (anti(_normal(gen, (o, o, v, v), 0.01, dtype)), anti(_normal(gen, (o, o, v, v), s, dtype)),
            anti(_normal(gen, (o, o, o, o), s, dtype)))


def _grouped_operands(case, seed):
    # the block extents belong to the case (a molecule's irreps), the values to the seed
    r = random.Random(case["count"] * 1000 + case["hi"])
    shapes = [tuple(_log(r, case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["count"])]
    gen, dtype = _gen(seed), DTYPES[case["dtype"]]
    A = _normal(gen, (sum(m * k for m, n, k in shapes),), 1.0, dtype)
    B = _normal(gen, (sum(k * n for m, n, k in shapes),), 1.0, dtype)
    C = torch.zeros(sum(m * n for m, n, k in shapes), dtype=dtype, device="cuda")
    return shapes, A, B, C


def _cut(flat, shapes):
    """Consecutive matrices of one buffer."""
    return [x.view(s) for x, s in zip(torch.split(flat, [a * b for a, b in shapes]), shapes)]


def _grouped_views(shapes, A, B, C):
    return (_cut(A, [(m, k) for m, n, k in shapes]), _cut(B, [(k, n) for m, n, k in shapes]),
            _cut(C, [(m, n) for m, n, k in shapes]))


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind in CCD:
        c, a, b, pre = CCD[kind]
        st["W"], st["A"], st["B"] = _ccd_operands(case, seed)
        st["plan"], st["pre"] = core.compile_plan(c, a, b), pre
    elif kind == "gemm":
        st["A"], st["B"], st["C"] = _gemm_operands(case, seed)
    elif kind == "reorder":
        o, v = case["o"], case["v"]
        inp = workloads.ccd_inputs_device(o, v, seed, with_vvvv=False)
        st["t"], st["g"] = inp.t_oovv, inp.g_oovv
        st["E"] = torch.zeros((), dtype=torch.float64, device="cuda")
        st["P"] = torch.empty((o, v, o, v), dtype=torch.float64, device="cuda")
        st["Q"] = torch.empty((o, v, o, v), dtype=torch.float64, device="cuda")
        st["plan"] = core.compile_plan("", "ijab", "ijab")
    elif kind in ("hf", "fock"):
        n, gen = case["n"], _gen(seed)
        st["g"] = _eri(gen, n)
        Q = _orthonormal(gen, n)[:, :max(1, n // 4)]
        st["D"] = (Q @ Q.T).contiguous()
        st["F"] = torch.empty((n, n), dtype=torch.float64, device="cuda")
        st["J"] = core.compile_plan("ij", "kl", "ijkl")
        st["K"] = core.compile_plan("ij", "kl", "ikjl")
    elif kind == "scf":
        st["g"], st["H"], st["X"], st["D"] = _scf_operands(case, seed)
        n = case["n"]
        for name in ("F", "tmp", "vecs", "C", "Dnew"):
            st[name] = torch.empty((n, n), dtype=torch.float64, device="cuda")
        st["W"] = torch.empty(n, dtype=torch.float64, device="cuda")
        st["E"] = torch.zeros((), dtype=torch.float64, device="cuda")
        st["plans"] = [core.compile_plan(*s) for s in (
            ("ij", "kl", "ijkl"), ("ij", "kl", "ikjl"), ("ij", "ik", "kj"), ("ij", "ki", "kj"), ("ij", "im", "jm"),
            ("", "ij", "ij"))]
    elif kind == "ao2mo":
        gen, dtype, n = _gen(seed), DTYPES[case["dtype"]], case["n"]
        st["g"] = _eri(gen, n).to(dtype)
        st["C"] = _orthonormal(gen, n).to(dtype).contiguous()
        st["t1"], st["t2"], st["out"] = (torch.empty_like(st["g"]) for _ in range(3))
        st["plans"] = [core.compile_plan(*s) for s in (
            ("pqrs", "mqrs", "mp"), ("pqrs", "pmrs", "mq"), ("pqrs", "pqms", "mr"), ("pqrs", "pqrm", "ms"))]
    elif kind == "grad":
        t, st["g"], st["W"] = _grad_operands(case, seed)
        st["t"] = t.requires_grad_(True)
    elif kind == "grouped":
        shapes, A, B, C = _grouped_operands(case, seed)
        a, b, c = _grouped_views(shapes, A, B, C)
        st["out"] = C
        st["plan"] = blocks.GroupedEinsum([("ij", z, "ik", x, "kj", y, 0.0, 1.0) for x, y, z in zip(a, b, c)])
    else:
        raise ValueError(kind)
    return st


def run(st):
    kind = st["kind"]
    if kind in CCD:
        split = {"split": "auto", "slice_type": "crt"} if st["case"]["split"] else {}
        st["plan"].execute(1.0, st["W"], st["pre"], st["A"], st["B"], **split)
        return st["W"]
    if kind == "gemm":
        c = st["case"]
        core.gemm(c["ta"], c["tb"], 1.0, st["A"], st["B"], c["beta"], st["C"])
        return st["C"]
    if kind == "reorder":
        st["plan"].execute(0.0, st["E"], 0.25, st["t"], st["g"])
        core.permute(0.0, "iajb", st["P"], 1.0, "ijab", st["t"])
        core.permute(0.0, "jbnf", st["Q"], 1.0, "jnfb", st["t"])
        return {"E": st["E"], "P": st["P"], "Q": st["Q"]}
    if kind == "hf":
        st["J"].execute(0.0, st["F"], 2.0, st["D"], st["g"])
        st["K"].execute(1.0, st["F"], -1.0, st["D"], st["g"])
        return st["F"]
    if kind == "fock":
        core.fock_jk(st["g"], st["D"], st["F"])
        return st["F"]
    if kind == "scf":
        J, K, FX, XTF, DD, dot = st["plans"]
        F, X, D, tmp, vecs, C, nocc = st["F"], st["X"], st["D"], st["tmp"], st["vecs"], st["C"], st["case"]["nocc"]
        core.permute(0.0, "ij", F, 1.0, "ij", st["H"])
        J.execute(1.0, F, 2.0, D, st["g"])
        K.execute(1.0, F, -1.0, D, st["g"])
        FX.execute(0.0, tmp, 1.0, F, X)
        XTF.execute(0.0, vecs, 1.0, X, tmp)
        core.syev(vecs, st["W"], check_info=False)
        FX.execute(0.0, C, 1.0, X, vecs)
        DD.execute(0.0, st["Dnew"], 1.0, C[:, :nocc], C[:, :nocc])
        dot.execute(0.0, st["E"], 1.0, D, F)
        dot.execute(1.0, st["E"], 1.0, D, st["H"])
        # the eigenvectors' signs are free: what a program keeps of them is the density
        return {"F": F, "W": st["W"], "D": st["Dnew"], "E": st["E"]}
    if kind == "ao2mo":
        p, C = st["plans"], st["C"]
        p[0].execute(0.0, st["t1"], 1.0, st["g"], C)
        p[1].execute(0.0, st["t2"], 1.0, st["t1"], C)
        p[2].execute(0.0, st["t1"], 1.0, st["t2"], C)
        p[3].execute(0.0, st["out"], 1.0, st["t1"], C)
        return st["out"]
    if kind == "grad":
        t, g, W = st["t"], st["g"], st["W"]
        t.grad = None
        e = autograd.einsum("", "ijab", t, "ijab", g, alpha=0.25)
        u = autograd.einsum("ijab", "klij", W, "klab", t)
        loss = e + autograd.einsum("", "ijab", t, "ijab", u, alpha=0.125)
        loss.backward()
        return {"loss": loss.detach(), "grad": t.grad}
    st["plan"].execute()
    return st["out"]


def work(case):
    kind = case["kind"]
    if kind in CCD:
        o, v = case["o"], case["v"]
        c = {"wabef": v**4, "wmnij": o**4, "wmbej": o * o * v * v}[kind]
        flops = {"wabef": 2.0 * o**2 * v**4, "wmnij": 2.0 * o**4 * v**2, "wmbej": 2.0 * o**3 * v**3}[kind]
        return {"bytes": 8.0 * (2 * o * o * v * v + 2 * c), "flops": flops}
    if kind == "gemm":
        m, n, k, e = case["m"], case["n"], case["k"], 8 if case["dtype"] == "f64" else 4
        return {"bytes": float(e) * (m * k + k * n + (2 if case["beta"] else 1) * m * n), "flops": 2.0 * m * n * k}
    if kind == "reorder":
        s = (case["o"] * case["v"]) ** 2
        return {"bytes": 8.0 * 4 * s, "flops": 2.0 * s}  # t and g read, P and Q written
    if kind in ("hf", "fock"):
        n = case["n"]
        return {"bytes": 8.0 * (n**4 + 2 * n * n), "flops": 4.0 * n**4}
    if kind == "scf":
        n = case["n"]
        return {"bytes": 8.0 * (n**4 + 6 * n * n), "flops": 4.0 * n**4 + 15.0 * n**3}
    if kind == "ao2mo":
        n, e = case["n"], 8 if case["dtype"] == "f64" else 4
        return {"bytes": float(e) * (2 * n**4 + n * n), "flops": 8.0 * n**5}
    if kind == "grad":
        o, v, e = case["o"], case["v"], 8 if case["dtype"] == "f64" else 4
        # u = W t, and W^T applied to the cotangent of u; dL/dW is not asked for
        return {"bytes": float(e) * (3 * (o * v) ** 2 + o**4), "flops": 4.0 * o**4 * v**2}
    r = random.Random(case["count"] * 1000 + case["hi"])
    shapes = [tuple(_log(r, case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["count"])]
    e = 8 if case["dtype"] == "f64" else 4
    return {"bytes": float(e) * sum(m * k + k * n + m * n for m, n, k in shapes),
            "flops": 2.0 * sum(m * n * k for m, n, k in shapes)}


def exact(case, seed):
    """The results of run() by torch in FP64 from the same inputs."""
    kind = case["kind"]
    if kind in CCD:
        W, A, B = _ccd_operands(case, seed)
        if kind == "wabef":  # W_abef += g_mnef t_mnab / 4
            W += torch.tensordot(B, A, dims=([0, 1], [0, 1])).mul_(0.25)
        elif kind == "wmnij":  # W_mnij += t_ijef g_mnef / 4
            W += torch.tensordot(B, A, dims=([2, 3], [2, 3])).mul_(0.25)
        else:  # W_mbej -= t_jnfb g_mnef / 2
            W -= torch.tensordot(B, A, dims=([1, 3], [1, 2])).permute(0, 3, 1, 2).mul(0.5)
        return W
    if kind == "gemm":
        A, B, C = (x.double() for x in _gemm_operands(case, seed))
        return (A if case["ta"] == "N" else A.T) @ (B if case["tb"] == "N" else B.T) + case["beta"] * C
    if kind == "reorder":
        inp = workloads.ccd_inputs_device(case["o"], case["v"], seed, with_vvvv=False)
        t, g = inp.t_oovv, inp.g_oovv
        return {"E": 0.25 * (t * g).sum(), "P": t.permute(0, 2, 1, 3).contiguous(), "Q": t.permute(0, 3, 1, 2).contiguous()}
    if kind in ("hf", "fock"):
        n, gen = case["n"], _gen(seed)
        g = _eri(gen, n)
        Q = _orthonormal(gen, n)[:, :max(1, n // 4)]
        return _two_electron(g, (Q @ Q.T).contiguous())
    if kind == "scf":
        g, H, X, D = _scf_operands(case, seed)
        F = H + _two_electron(g, D)
        w, U = torch.linalg.eigh((X.T @ (F @ X)).cpu())
        C = X @ U.cuda()[:, :case["nocc"]]
        return {"F": F, "W": w.cuda(), "D": C @ C.T, "E": (D * F).sum() + (D * H).sum()}
    if kind == "ao2mo":
        dtype, gen, n = DTYPES[case["dtype"]], _gen(seed), case["n"]
        x = _eri(gen, n).to(dtype).double()
        C = _orthonormal(gen, n).to(dtype).double()
        for _ in range(4):  # contracts the leading axis and puts the new one last
            x = torch.tensordot(x, C, dims=([0], [0]))
        return x
    if kind == "grad":
        t, g, W = (x.double() for x in _grad_operands(case, seed))
        o, v = case["o"], case["v"]
        tm, Wm = t.reshape(o * o, v * v), W.reshape(o * o, o * o)
        u = Wm.T @ tm
        grad = 0.25 * g.reshape(o * o, v * v) + 0.125 * (u + Wm @ tm)
        return {"loss": 0.25 * (t * g).sum() + 0.125 * (tm * u).sum(), "grad": grad.reshape(t.shape)}
    shapes, A, B, C = _grouped_operands(case, seed)
    a, b, c = _grouped_views(shapes, A.double(), B.double(), C.double())
    return torch.cat([(x @ y).reshape(-1) for x, y in zip(a, b)])


def _two_electron(g, D):
    n = D.shape[0]
    J = g.reshape(n * n, n * n) @ D.reshape(-1)
    K = torch.tensordot(g, D, dims=([1, 3], [0, 1]))
    return 2.0 * J.reshape(n, n) - K
