"""Host check of the k-major LDS layouts with several k-rows per instruction."""
from tests.test_cpp_api import _run


def test_lds_layout_groups_program():
    res = _run("test_lds_layout_groups", 60)
    assert res.returncode == 0 and "0 failures" in res.stdout
