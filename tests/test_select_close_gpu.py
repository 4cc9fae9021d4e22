"""Workgroup-per-column float columns whose sets are a close call (a value
within rounding of t or t + hi, or none free) and the float knapsack of such
columns: the selection's and the register form's steps against the sorted
column's, which the deferred-column kernel still takes for k past the lists.
The reference values are numpy restatements of the sorted column's steps in
float32 with exactly rounded sums (knapsack_eq.h:25-109), so the thresholds
agree to one rounding of the final quotient: 4 ulps of the largest value."""
import numpy as np
import pytest

from tests.test_prox_gpu import F32, run_gpu

pytestmark = pytest.mark.gpu


def sorted_knapsack(x, hi, rhs):
    """t of the variable fixing over the sorted column, float32 throughout,
    each sum exact and rounded once."""
    f32 = np.float32
    s = np.sort(x)[::-1]
    m = len(s)
    total = lambda b, e: f32(np.sum(s[b:e].astype(np.float64)))
    eps = np.finfo(f32).eps * max(f32(1), abs(rhs))
    hi, rhs = f32(hi), f32(rhs)
    t, f, l, mc = (total(0, m) - rhs) / f32(m), 0, m, m
    for _ in range(m + 1):
        p_lo = f + int(np.sum(s[f:l] > t))
        p_hi = f + int(np.sum(s[f:p_lo] > f32(hi + t)))
        s_lo, n_lo, s_hi, n_hi = total(p_lo, l), l - p_lo, total(f, p_hi), p_hi - f
        sh = f32(n_hi) * hi
        infeas = f32(f32(f32(s_hi + s_lo) - sh) - f32(f32(n_hi + n_lo) * t))
        if n_hi > 0 and infeas > eps:
            f = p_hi
            nxt = f32(f32(f32(mc) * t - s_hi) + sh)
            mc -= n_hi
        elif n_lo > 0 and infeas < -eps:
            l = p_lo
            nxt = f32(f32(mc) * t - s_lo)
            mc -= n_lo
        else:
            f, l = p_hi, p_lo
            break
        if mc == 0:
            break
        t = f32(nxt / f32(mc))
    if l > f:
        t = f32(f32(f32(total(f, l) + f32(f) * hi) - rhs) / f32(l - f))
    return t


def close_columns(m, k, n, seed):
    """Columns with label + 2, half of them with an entry moved to the exact
    threshold, to the threshold plus hi, or with the k + 1-th more than hi
    below the k-th (none free)."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, m)).astype(np.float32)
    x[np.arange(n), rng.integers(0, m, n)] += 2
    for j in range(0, n, 2):
        t = sorted_knapsack(x[j], 1.0 / k, 1.0)
        order = np.argsort(-x[j])
        kind = (j // 2) % 3
        if kind == 0:
            x[j, order[k + 3]] = t + np.float32(rng.uniform(-1e-4, 1e-4))
        elif kind == 1:
            x[j, order[0]] = t + np.float32(1.0 / k) + np.float32(rng.uniform(-1e-4, 1e-4))
        else:
            x[j, order[:k]] += np.float32(1.5 / k)
    return x


@pytest.mark.parametrize("m,k", [(2049, 5), (4100, 10), (10000, 3), (20000, 1), (32768, 10)])
def test_close_call(cuda, m, k):
    x = close_columns(m, k, 24, 900 + m + k)
    t = np.array([sorted_knapsack(c, np.float32(1) / np.float32(k), 1.0) for c in x])
    tol = 4 * np.finfo(np.float32).eps * np.abs(x).max()
    want = np.clip(x - t[:, None], 0, np.float32(1) / np.float32(k))
    got, _ = run_gpu("topk_simplex", x, F32, cuda, k=k, rhs=1.0)
    assert np.abs(got - want).max() <= tol
    t = np.array([sorted_knapsack(c, 1.0, 1.0) for c in x])
    want = np.clip(x - t[:, None], 0, np.float32(1))
    got, _ = run_gpu("knapsack_eq", x, F32, cuda, lo=0.0, hi=1.0, rhs=1.0)
    assert np.abs(got - want).max() <= tol


@pytest.mark.parametrize("m,k", [(2049, 5), (4100, 10), (10000, 3), (20000, 1), (32768, 10)])
def test_close_call_projection(cuda, oracle, m, k):
    """How far those steps are from the projection (long double): the fixing's
    numerator is rounded to float in each of its passes, of which there are at
    most 16 here (the free set halves in each), by u sum |a| at most, over the
    values free at the end."""
    from oracle import binding
    x = close_columns(m, k, 24, 900 + m + k)
    u = np.finfo(np.float32).eps / 2
    for op, kw in (("topk_simplex", dict(k=k, rhs=1.0)), ("knapsack_eq", dict(lo=0.0, hi=1.0, rhs=1.0))):
        got, _ = run_gpu(op, x, F32, cuda, **kw)
        want = x.astype(np.float64)
        oracle.prox(op, want, result=2, params=binding.make_params(**kw), nthreads=8)
        free = ((want > 0) & (want < (1.0 / k if op == "topk_simplex" else 1.0))).sum(axis=1)
        bound = 16 * u * np.abs(x.astype(np.float64)).sum(axis=1) / np.maximum(free, 1)
        err = np.abs(got - want).max(axis=1)
        print(f"{op} m={m} k={k}: error {err.max():.1e}, at most {(err / bound).max():.2f} of the bound")
        assert (err <= bound).all()
