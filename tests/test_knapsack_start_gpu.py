"""The knapsack's variable fixing started at the bound max - rhs, and its
columns of up to 32768 rows on a workgroup, against the CPU oracle."""
import numpy as np
import pytest

from tests import inputs
from tests.test_prox_gpu import DTYPES, parity, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,result", DTYPES)
@pytest.mark.parametrize("m", [1, 10, 37, 129, 1000, 2049, 4097, 16384])
@pytest.mark.parametrize("op,kw", [
    ("knapsack_eq", dict(lo=0.0, hi=1.0, rhs=1.0)),
    ("knapsack_eq", dict(lo=0.0, hi=3.0, rhs=0.25)),
    ("knapsack_eq", dict(lo=0.0, hi=0.0, rhs=0.0)),
    ("knapsack_le_biased", dict(lo=0.0, hi=1.0, rhs=1.0, rho=0.5)),
])
def test_knapsack_start_at_the_maximum(cuda, oracle, op, kw, m, dtype, result):
    """lo = 0 and hi >= rhs: the fixing starts from the bound max - rhs."""
    n = 8 if m > 2048 else 60
    for name, x in [("normal", inputs.normal(n, m, dtype, 900 + m)),
                    ("small", inputs.normal(n, m, dtype, 901 + m, 1e-3)),
                    ("mixed", inputs.mixed_signs(n, m, dtype, 902 + m, -3, 3)),
                    ("edge", inputs.edge_columns(m, dtype, 903 + m))]:
        got, thr = run_gpu(op, x, result, cuda, **kw)
        parity(oracle, op, x, got, result, f"{op} {name} m={m}", nthreads=8, thr=thr, **kw)
