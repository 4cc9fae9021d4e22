"""Columns of the top-k operators whose masked classes are set to a very low
value or to -inf.  A masked class ends at 0 and takes no part in the others' thresholds,
so the outputs are those of the column without it, which the CPU oracle
computes in long double.  Sizes on every path: the register kernel and its
deferred columns, the selection by wave and by workgroup, and its fallback to
the sorted column (more values at the mask than its list holds)."""
import numpy as np
import pytest

from tests.test_prox_gpu import F32, F64

pytestmark = pytest.mark.gpu

OPS = [("topk_simplex", dict(rhs=1.0)), ("topk_cone", dict()),
       ("topk_simplex_biased", dict(rhs=1.0, rho=0.5)), ("topk_cone_biased", dict(rho=0.25))]


def masked_columns(m, k, dtype, mask, seed):
    """N(0,1) columns with one label, all but some classes masked: one class,
    half of them, all but k + 1, k, k - 1, and all but the first 16 (which sit
    in few of the parts whose maxima give the selection its cut)."""
    rng = np.random.default_rng(seed)
    cols, keeps = [], []
    for kept in (m - 1, m // 2, k + 1, k, k - 1, None):
        keep = np.zeros(m, bool)
        if kept is None:
            keep[:16] = True
        else:
            keep[rng.permutation(m)[:kept]] = True
        x = (rng.standard_normal(m) * 0.7).astype(dtype)
        x[rng.integers(0, m)] += 2
        x[~keep] = mask
        cols.append(x)
        keeps.append(keep)
    return np.stack(cols), keeps


def check_masked(oracle, cuda, op, kw, m, k, dtype, mask):
    import torch
    import libsdca_amd as sd
    from oracle import binding
    x, keeps = masked_columns(m, k, dtype, mask, m + k)
    got = sd.prox(op, torch.from_numpy(x).to(cuda), k=k, **kw).cpu().numpy()
    # a threshold's rounding: 4 (m + k) u of values of unit size
    tol = 4 * (m + k) * float(np.finfo(dtype).eps)
    for j, keep in enumerate(keeps):
        want = np.zeros((1, int(keep.sum())))
        if want.shape[1] >= k:  # fewer than k classes left: the cone is {0}
            want = x[j, keep].astype(np.float64)[None, :].copy()
            oracle.prox(op, want, result=2, params=binding.make_params(k=k, **kw))
        err = np.abs(got[j, keep] - want[0]).max(initial=0.0)
        assert err <= tol, f"{op} m={m} k={k} column {j} ({int(keep.sum())} kept): error {err:.2e}"
        assert (got[j, ~keep] == 0).all(), f"{op} m={m} k={k} column {j}: a masked class is not 0"


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,k", [(40, 3), (100, 8), (300, 20), (700, 3), (1025, 8), (1500, 5),
                                 (2048, 3)])
@pytest.mark.parametrize("op,kw", OPS)
def test_masked_low(cuda, oracle, op, kw, m, k, dtype):
    """Finite masks, down to the type's lowest value."""
    for mask in (-1e9, -1e30, -np.finfo(dtype).max):
        check_masked(oracle, cuda, op, kw, m, k, dtype, dtype(mask))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,k", [(40, 20), (300, 20), (513, 3), (700, 3), (1024, 20), (1025, 8),
                                 (2048, 3), (2049, 5), (3000, 8), (10000, 20), (16384, 10)])
@pytest.mark.parametrize("op,kw", OPS)
def test_masked_inf(cuda, oracle, op, kw, m, k, dtype):
    """-inf on the selection's columns: left out like padding."""
    check_masked(oracle, cuda, op, kw, m, k, dtype, -np.inf)


@pytest.mark.parametrize("m,k", [(1500, 8), (2500, 5), (2500, 55)])
def test_masked_inf_among_ties(cuda, oracle, m, k):
    """More equal values than the selection's list holds (k < 56: its route) beside masked
    classes: the sorted column without them."""
    import torch
    import libsdca_amd as sd
    x = np.full((2, m), 0.5, np.float32)
    x[0, 400:] = -np.inf
    x[1, ::2] = -np.inf
    for op, kw in OPS:
        got = sd.prox(op, torch.from_numpy(x).to(cuda), k=k, **kw).cpu().numpy()
        for j in range(2):
            keep = x[j] > 0
            n = int(keep.sum())
            from oracle import binding
            want = x[j, keep].astype(np.float64)[None, :].copy()
            oracle.prox(op, want, result=2, params=binding.make_params(k=k, **kw))
            assert (got[j, ~keep] == 0).all()
            # one ulp of 0.5 in the threshold moves every entry together
            assert np.abs(got[j, keep] - want[0]).max() <= 4 * np.finfo(np.float32).eps, f"{op} n={n}"


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m", [2049, 3000, 16384])
@pytest.mark.parametrize("lo", [0.0, -1e-3])
def test_masked_knapsack_le_biased(cuda, m, lo, dtype):
    """knapsack_le_biased on a workgroup's columns whose sum is -inf (two
    classes or more at the type's lowest value, one at -inf):
    x = clamp(a - t, lo, 1) with t = rho sum x where that sum is at most 1,
    else sum x = 1."""
    import torch
    import libsdca_amd as sd
    rho = 0.5
    u = float(np.finfo(dtype).eps)
    for mask in (-np.inf, -np.finfo(dtype).max):
        # 3 and 4 classes at 0.3: inactive for lo = 0; 16 with a label: active
        cols = []
        for kept, scale in ((3, 0.1), (4, 0.3), (16, 1.0), (m // 2, 1.0), (m - 2, 1.0)):
            rng = np.random.default_rng(m + kept)
            x = np.full(m, mask)
            x[rng.permutation(m)[:kept]] = rng.standard_normal(kept) * scale + 0.1
            cols.append(x)
        x = np.stack(cols).astype(dtype)
        got, thr = sd.prox("knapsack_le_biased", torch.from_numpy(x).to(cuda), lo=lo, rho=rho,
                           thresholds=True)
        got, thr = got.cpu().numpy().astype(np.float64), thr.cpu().numpy()
        for j in range(len(x)):
            keep = x[j] > -1e30
            t, s = thr[j, 0], got[j].sum()
            assert (got[j, ~keep] == float(dtype(lo))).all(), (j, mask)
            # the outputs' own rounding in the sum: m u of values up to 4
            tol = 8 * m * u
            assert np.abs(got[j, keep] - np.clip(x[j, keep] - t, lo, 1.0)).max() <= 8 * u
            if s <= 1.0 - tol:
                assert abs(t - rho * s) <= tol, (j, mask, t, s)
            else:
                assert abs(s - 1.0) <= tol and t >= rho * 1.0 - tol, (j, mask, t, s)
