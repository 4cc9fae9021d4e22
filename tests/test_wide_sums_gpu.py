"""Sums that are carried beyond the Result type and rounded once: of the
columns a workgroup holds.  Against exactly rounded sums (math.fsum)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cancelling(n, m, seed):
    """Columns whose large values cancel: the exact sum is about 1e-9 of the
    values' magnitude."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, m)) * 1e3
    x[:, 1::2] = -x[:, 0:2 * (m // 2):2]
    x[:, ::7] += rng.standard_normal((n, len(range(0, m, 7)))) * 1e-6
    for j in range(n):
        x[j] = x[j, rng.permutation(m)]
    return x


@pytest.mark.parametrize("m", [2049, 5000, 16384])
@pytest.mark.parametrize("op,kw", [("knapsack_eq", {}), ("knapsack_le", {}),
                                   ("knapsack_le_biased", dict(rho=0.5))])
def test_knapsack_all_free(cuda, op, kw, m):
    """Every value free: t = (sum a - rhs) / m (or sum a / (1 / rho + m))."""
    import torch
    import libsdca_amd as sd
    x = cancelling(8, m, m)
    s = np.array([math.fsum(c) for c in x])
    rhs = 1e-8 if op == "knapsack_eq" else 0.0
    if op == "knapsack_le":
        x, s = np.where(s[:, None] < 0, -x, x), np.abs(s)  # the sum constraint acts
    _, thr = sd.prox(op, torch.from_numpy(x).to(cuda), lo=-1e6, hi=1e6, rhs=rhs, thresholds=True,
                     **kw)
    t = thr.cpu().numpy()[:, 0]
    want = (s - rhs) / m
    if op == "knapsack_le_biased":
        want = np.where(want >= 0, want, s / (2.0 + m))
    # three roundings of terms no larger than |sum| + rhs, over m
    u = np.finfo(np.float64).eps / 2
    assert (np.abs(t - want) <= 6 * u * (np.abs(s) + rhs) / m).all()


@pytest.mark.parametrize("m", [2049, 10000, 30000])
def test_knapsack_le_inactive(cuda, m):
    """knapsack_le's test of the sum constraint: the float sum is the exact
    one rounded once (sums within a few ulps of the bound)."""
    import torch
    import libsdca_amd as sd
    f32 = np.float32
    rng = np.random.default_rng(m)
    x = rng.random((64, m))
    x = (x / x.sum(axis=1, keepdims=True) * (1 + rng.uniform(0, 3e-7, (64, 1)))).astype(f32)
    _, sets = sd.prox("knapsack_le", torch.from_numpy(x).to(cuda), sets=True)
    branch = [sd.BRANCHES[int(b)] for b in sets.cpu().numpy()[:, 2]]
    active = np.array([f32(math.fsum(c)) > f32(1) + np.finfo(f32).eps for c in x])
    assert 0 < active.sum() < 64
    assert (np.array([b != "inactive" for b in branch]) == active).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m", [2049, 3000, 16384])
def test_knapsack_le_biased_small_values(cuda, m, dtype):
    """The search's t = rho sum x on values of size 1e-3, far below the
    tolerance the sum constraint's size gives."""
    import torch
    import libsdca_amd as sd
    n = 64 if m > 5000 else 400
    x = (np.random.default_rng(m).standard_normal((n, m)) * 1e-3).astype(dtype)
    _, thr = sd.prox("knapsack_le_biased", torch.from_numpy(x).to(cuda), rho=0.5, thresholds=True)
    t = thr.cpu().numpy()[:, 0]
    want = np.empty(n)
    for j in range(n):  # sum of the n largest over 1 / rho + n, the n that are above it
        a = np.sort(x[j].astype(np.longdouble))[::-1]
        r = np.cumsum(a) / (2 + np.arange(1, m + 1))
        want[j] = r[int((a > r).sum()) - 1]
    # the sum's and the quotient's rounding: 2 ulps
    assert (np.abs(t - want) <= 2 * np.finfo(dtype).eps * want).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m", [16, 40, 100, 200, 300, 512, 700, 3000])
def test_topk_constant(cuda, m, dtype):
    """The k = 12 largest equal by the projection, hi = (sum of them) / 12,
    where large values cancel in that sum."""
    import torch
    import libsdca_amd as sd
    k = 12
    rng = np.random.default_rng(m)
    x = np.full((50, m), -1e5)
    for j in range(50):
        # (their sum is 8 ulps of a value of 100 at least: above 16 eps, where
        # the zero branch ends)
        a = rng.uniform(100, 1000, k // 2).astype(np.float32)
        top = np.concatenate([a, -a[:-1], [-a[-1] + np.spacing(a[-1], dtype=np.float32) * 8]])
        x[j, rng.permutation(m)[:k]] = top
    x = x.astype(dtype)
    for op, kw, div in (("topk_cone", {}, 12.0), ("topk_cone_biased", dict(rho=0.25), 12 + 0.25 * 144)):
        _, thr = sd.prox(op, torch.from_numpy(x).to(cuda), k=k, thresholds=True, **kw)
        hi = thr.cpu().numpy()[:, 2]
        want = np.array([math.fsum(sorted(c)[-k:]) for c in x]) / div
        # the sum's rounding and the quotient's
        assert (np.abs(hi - want) <= 2 * np.finfo(dtype).eps * want).all(), op
