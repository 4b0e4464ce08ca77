"""Host check of the estimated time of permutes."""
from tests.test_cpp_api import _run


def test_permute_cost_program():
    res = _run("test_permute_cost", 60)
    assert res.returncode == 0 and "0 failures" in res.stdout
