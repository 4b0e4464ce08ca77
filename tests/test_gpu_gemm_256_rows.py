"""The FP32 256 x 128 tile, forced through a tuning table at the edges of a tile and with short k,
and chosen by its rule at the rule's edges (k 255 to 257, rounds of tiles just whole and not, rows
that leave half a tile empty). Tolerance as in test_gpu_gemm_tiles.py."""
import pytest

torch = pytest.importorskip("torch")

from tests.test_gpu_gemm_tiles import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta", "NT")
@pytest.mark.parametrize("tb", "NT")
@pytest.mark.parametrize("m,n,k,pad,beta", [(256, 128, 16, 0, 0.0), (257, 129, 33, 0, 1.0), (1020, 388, 44, 0, 0.0),
                                            (511, 640, 17, 3, -0.5), (640, 511, 100, 4, 0.0), (1100, 900, 300, 1, 1.0)])
def test_forced(core, tmp_path, m, n, k, ta, tb, pad, beta):
    f = tmp_path / "t.txt"
    f.write_text("".join(f"4 {x} {y} {k} 1 {a} {b} : 256 128 0 0\n" for x, y in ((m, n), (n, m)) for a in (0, 1) for b in (0, 1)))
    core.clear_gemm_tuning()
    core.load_gemm_tuning(f)
    try:
        _check(core, m, n, k, ta, tb, pad, torch.float32, beta)
    finally:
        core.clear_gemm_tuning()


@pytest.mark.parametrize("ta", "NT")
@pytest.mark.parametrize("tb", "NT")
@pytest.mark.parametrize("m,n,k", [(4096, 4096, 255), (4096, 4096, 256), (4096, 4096, 257), (2048, 8192, 260), (3200, 5120, 512),
                                   (5120, 3200, 512), (11712, 2304, 516), (2304, 11713, 512), (4224, 4096, 300)])
def test_rule(core, m, n, k, ta, tb):
    _check(core, m, n, k, ta, tb, 0, torch.float32, 0.0)
