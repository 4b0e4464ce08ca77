"""Outer products at the edges of the rule for one column a thread: 64 and 65 columns, 2^18
elements and just above, odd rows. Tolerance as in test_gpu_ger.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.test_gpu_ger import test_outer_product as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("m,n,pad", [(64, 4096, 0), (64, 4097, 0), (65, 4096, 1), (63, 2049, 0), (1, 2**18 + 1, 0), (33, 31, 2)])
def test_one_column_rule(core, m, n, pad, beta, dtype):
    _check(core, m, n, pad, beta, dtype)
