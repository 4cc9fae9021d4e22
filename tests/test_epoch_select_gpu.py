"""The epoch's hinge thresholds by selection (epoch_select in sdca_epoch.hip)
against the oracle: rows around the steps of its forms (the column as its own
list up to 257 classes, one to eight entries per thread, past them the sorted
column), k around the lists' ranks, examples whose top-k simplex needs the
cone search, and knapsacks with more candidates than the list holds (the
first epoch from zero).

The bar: 4 times the spread of the oracle's two roundings of the scores plus 8
ulps (the feature epoch's tests), plus what the oracle's searches round: they
add up to m values one by one, m u of a sum of magnitude one per example,
and W and the later scores collect those of n examples, n m u in all."""
import numpy as np
import pytest

from tests.test_epoch_gpu import gpu_epochs, oracle_epochs, problem

pytestmark = pytest.mark.gpu

FORMS = [(64, 1), (65, 9), (256, 10), (257, 56), (258, 3), (513, 55), (1024, 5), (1025, 17),
         (2048, 10), (2049, 2)]


def check(oracle, cuda, obj, dtype, result, n, d, m, seed):
    import libsdca_amd as sd
    X, y = problem(dtype, n, d, m, seed)
    orders = [sd.epoch_order(n, e) for e in range(2)]
    got = gpu_epochs(cuda, obj, X, y, m, result, orders)
    want = oracle_epochs(oracle, obj, X, y, m, result, orders)
    other = oracle_epochs(oracle, obj, X, y, m, result, orders, reverse=True)
    eps = float(np.finfo(dtype).eps)
    for name, g, o, v in zip("WA", got, want, other):
        scale = max(1.0, float(np.abs(o).max()))
        tol = 4 * float(np.abs(o - v).max()) + (8 + 0.5 * n * m) * eps * scale
        err = float(np.abs(g - o).max())
        assert err <= tol, f"{obj[0]} m={m} {name}: |gpu - oracle| {err:.3e} > {tol:.3e}"
    assert np.abs(want[1]).max() > 0.01


@pytest.mark.parametrize("dtype,result", [(np.float32, 0), (np.float64, 1)])
@pytest.mark.parametrize("m,k", FORMS)
@pytest.mark.parametrize("name,gamma", [("hinge_topk", 1.0), ("hinge_topk_smooth", 0.5),
                                        ("topk_hinge", 1.0), ("topk_hinge_smooth", 1.0)])
def test_epoch_select(cuda, oracle, name, gamma, m, k, dtype, result):
    check(oracle, cuda, (name, 1.0, gamma, k), dtype, result, 96, 48, m, 31 + m + k)


@pytest.mark.parametrize("dtype,result", [(np.float32, 0), (np.float64, 1)])
@pytest.mark.parametrize("m", [90, 700])
def test_epoch_select_cone(cuda, oracle, m, dtype, result):
    """Loose sums (c large): the simplex gives way to the cone."""
    check(oracle, cuda, ("hinge_topk_smooth", 8.0, 1.0, 5), dtype, result, 128, 512, m, 17 + m)
