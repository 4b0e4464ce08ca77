"""Host check that long tile lists go in launches that HIP takes whole."""
from tests.test_cpp_api import _run


def test_launch_bounds_program():
    res = _run("test_launch_bounds", 60)
    assert res.returncode == 0 and "0 failures" in res.stdout
