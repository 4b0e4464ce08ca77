"""Host check of the estimated time of dense products."""
from tests.test_cpp_api import _run


def test_gemm_cost_program():
    res = _run("test_gemm_cost", 60)
    assert res.returncode == 0 and "0 failures" in res.stdout
