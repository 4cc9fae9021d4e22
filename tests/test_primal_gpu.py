"""W = W0 + X A' (sdca_recompute_primal) against float64: the edges of the
64 x 64 output tiles and of the example slabs and splits, both element
types, with and without W0, host and device arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,m,d", [(1, 1, 1), (15, 64, 63), (16, 65, 64), (33, 2, 129), (127, 7, 16),
                                   (129, 63, 65), (5000, 3, 70), (20011, 37, 33), (70000, 5, 9),
                                   (700, 300, 2900), (6000, 40, 700)])
@pytest.mark.parametrize("with_w0", [False, True])
def test_recompute_primal_shapes(cuda, dtype, n, m, d, with_w0):
    import torch
    import libsdca_amd as sd
    rng = np.random.default_rng(n + m + d)
    X = rng.standard_normal((n, d)).astype(dtype)
    A = rng.standard_normal((n, m)).astype(dtype)
    W0 = rng.standard_normal((m, d)).astype(dtype) if with_w0 else None
    up = [None if a is None else torch.from_numpy(a).to(cuda) for a in (X, A, W0)]
    got = sd.recompute_primal(up[0], up[1], up[2]).cpu().numpy().astype(np.float64)
    X64, A64 = X.astype(np.longdouble), A.astype(np.longdouble)
    if n * m * d > 3e7:  # float64 is exact enough next to n u
        X64, A64 = X.astype(np.float64), A.astype(np.float64)
    want = A64.T @ X64
    bound = np.abs(A64).T @ np.abs(X64)
    if with_w0:
        want = want + W0
        bound = bound + np.abs(W0)
    # |error| <= (n + 1) u sum |a x| for any order of the sum
    u = np.finfo(dtype).eps / 2
    assert (np.abs(got - want) <= (n + 2) * u * bound).all()
    # the error of a random-sign sum is far below that bound
    rel = float(np.linalg.norm((got - want).astype(np.float64)) / np.linalg.norm(want.astype(np.float64)))
    assert rel <= 8 * u * np.sqrt(n + 1)


def test_recompute_primal_host(cuda):
    import libsdca_amd as sd
    rng = np.random.default_rng(4)
    X, A = rng.standard_normal((300, 50)), rng.standard_normal((300, 20))
    assert np.allclose(sd.recompute_primal(X, A), A.T @ X, rtol=0, atol=1e-12)
