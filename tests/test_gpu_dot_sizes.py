"""Dots at the edges of their kernels (one workgroup to 4096 elements, chunks of 8192 above),
strides and beta included, against numpy: at most (n + 2) roundings of the sum of magnitudes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("inc", [1, 3])
@pytest.mark.parametrize("n", [1, 63, 64, 1023, 1025, 4095, 4096, 4097, 8192, 8193])
def test_dot(core, dtype, inc, n):
    rng = np.random.default_rng(n)
    x, y = (torch.from_numpy(rng.standard_normal(n * inc)).to(dtype) for _ in range(2))
    a, b = (t.double().numpy()[::inc] for t in (x, y))
    xg, yg = x.cuda()[::inc], y.cuda()[::inc]
    mag, eps = np.abs(a) @ np.abs(b), torch.finfo(dtype).eps
    plan = core.compile_plan("", "i", "i")
    for beta, start in ((0.0, float("nan")), (2.0, 0.5)):
        C = torch.full((), start, dtype=dtype, device="cuda")
        plan.execute(beta, C, -1.5, xg, yg)
        want = -1.5 * (a @ b) + (beta * start if beta else 0.0)
        scale = 1.5 * mag + abs(beta * start if beta else 0.0)
        assert abs(float(C) - want) <= (n + 2) * eps * scale * (2 if dtype == torch.float64 else 1)


@pytest.mark.parametrize("n", [100, 4096, 4097])
def test_captured(core, n):
    from einsums_amd import blocks

    s = torch.cuda.Stream()
    gen = torch.Generator(device="cuda").manual_seed(n)
    x, y = (torch.randn(n, dtype=torch.float64, device="cuda", generator=gen) for _ in range(2))
    C, eager = torch.zeros((), dtype=torch.float64, device="cuda"), torch.zeros((), dtype=torch.float64, device="cuda")
    plan = core.compile_plan("", "i", "i")
    s.wait_stream(torch.cuda.current_stream())
    plan.execute(0.0, eager, 1.0, x, y, stream=s)
    g = blocks.Graph(lambda: plan.execute(0.0, C, 1.0, x, y, stream=s), s)
    for _ in range(3):
        C.fill_(-1.0)
        torch.cuda.synchronize()
        g.replay()
        s.synchronize()
        assert float(C) == float(eager)
