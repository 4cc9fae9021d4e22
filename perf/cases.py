"""The work that users of this library have it do, as cases that can be timed.

A case is one call (or one short sequence of calls) of the public Python
entry points on device data:

  prox     one batched proximal step over an n x m matrix, out of place
  eval     one evaluation pass of a data set (scores, losses, accuracy)
  refresh  the primal recomputation followed by the evaluation pass
  epoch    one pass of the SDCA solver over the training examples, on
           features or on a kernel matrix; W and A are updated in place, so
           repeated passes are the following epochs of one solve

`exact` restates every path in 64 bits with plain torch or numpy: thresholds
by bisection, with no code of the library.
"""
import math

import numpy as np
import torch

import libsdca_amd as sd

DEV = "cuda"
CHUNK = 1 << 24  # entries of a 64-bit working set in exact()


def listed():
    return [
        # The smallest call: the simplex projection of short double columns,
        # where launches and host work count.
        {"name": "simplex_small_f64", "path": "prox", "op": "knapsack_eq", "dtype": "f64",
         "m": 10, "n": 100_000},
        # The benchmark's headline: top-5 simplex over a large float batch.
        {"name": "topk_simplex_f32", "path": "prox", "op": "topk_simplex", "dtype": "f32",
         "m": 100, "n": 4_000_000, "k": 5},
        # Top-10 over a thousand classes.
        {"name": "topk_simplex_k10_f32", "path": "prox", "op": "topk_simplex", "dtype": "f32",
         "m": 1000, "n": 50_000, "k": 10},
        # Entropic projections, exp map and Lambert map, in double; the
        # second with a row count that fits no tile.
        {"name": "entropy_f64", "path": "prox", "op": "entropy", "dtype": "f64",
         "m": 1000, "n": 100_000},
        {"name": "entropy_norm_f64", "path": "prox", "op": "entropy_norm", "dtype": "f64",
         "m": 777, "n": 50_000},
        # The multilabel dual's projection, a split point per column.
        {"name": "two_simplex_f32", "path": "prox", "op": "two_simplex", "dtype": "f32",
         "m": 200, "n": 500_000},
        # Very many classes: columns far beyond one wave's registers.
        {"name": "topk_simplex_wide_f32", "path": "prox", "op": "topk_simplex", "dtype": "f32",
         "m": 10_000, "n": 4_096, "k": 5},
        # Evaluation during training, a thousand classes, dual variables given.
        {"name": "eval_multiclass_f32", "path": "eval", "dtype": "f32", "labels": "multiclass",
         "d": 4096, "m": 1000, "n": 50_000},
        # Multilabel evaluation, 1-5 labels per example.
        {"name": "eval_multilabel_f32", "path": "eval", "dtype": "f32", "labels": "multilabel",
         "d": 1024, "m": 200, "n": 200_000},
        # The accurate-math flow in double, odd sizes: W recomputed from the
        # dual variables, then evaluated, losses per example.
        {"name": "refresh_eval_f64", "path": "refresh", "dtype": "f64", "labels": "multiclass",
         "d": 513, "m": 137, "n": 20_011},
        # Training: an epoch on features (smooth top-5 hinge, a thousand
        # classes), and one on a Gaussian kernel with fewer classes.
        {"name": "epoch_features_f32", "path": "epoch", "input": "features", "dtype": "f32",
         "objective": "l2_hinge_topk_smooth", "k": 5, "d": 4096, "m": 1000, "n": 20_000},
        {"name": "epoch_kernel_f32", "path": "epoch", "input": "kernel", "dtype": "f32",
         "objective": "l2_topk_hinge_smooth", "k": 3, "d": 64, "m": 50, "n": 3_001},
    ]


PROX_SIMPLEX = ("knapsack_eq", "knapsack_le", "topk_simplex", "topk_cone", "topk_simplex_biased")
PROX_ENTROPIC = ("entropy", "entropy_norm")
EPOCH_OBJECTIVES = ("l2_hinge_topk_smooth", "l2_topk_hinge_smooth", "l2_entropy")


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.choice(["prox"] * 3 + ["entropic", "two", "eval", "eval", "refresh", "epoch", "epoch"])
    dtype = rng.choice(["f32", "f32", "f64"])
    if what in ("prox", "entropic", "two"):
        op = {"prox": rng.choice(PROX_SIMPLEX), "entropic": rng.choice(PROX_ENTROPIC),
              "two": "two_simplex"}[what]
        m = _log_uniform(rng, 7 if op == "two_simplex" else 5, 20_000)
        size = _log_uniform(rng, 300_000, 40_000_000)
        case = {"path": "prox", "op": op, "dtype": dtype, "m": m,
                "n": max(64, min(2_000_000, size // m))}
        if op.startswith("topk"):
            case["k"] = rng.randint(1, min(10, m - 1))
        return case
    if what in ("eval", "refresh"):
        d, m = _log_uniform(rng, 16, 4096), _log_uniform(rng, 7, 2_000)
        most = int(min(3e10 / (d * m) * (1.0 if dtype == "f64" else 4.0), 1e8 / (d + m)))
        n = _log_uniform(rng, 500, max(1_000, min(500_000, most)))
        labels = "multiclass" if what == "refresh" else rng.choice(["multiclass", "multilabel"])
        return {"path": what, "dtype": dtype, "labels": labels, "d": d, "m": m, "n": n}
    source = rng.choice(["features", "kernel"])
    m = _log_uniform(rng, 5, 2_000)
    return {"path": "epoch", "input": source, "dtype": dtype,
            "objective": rng.choice(EPOCH_OBJECTIVES), "k": rng.randint(1, min(10, m - 1)),
            "d": _log_uniform(rng, 16, 4096), "m": m, "n": _log_uniform(rng, 500, 6_000)}


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _label_rows(g, n, m):
    """CSR labels: 1 to 5 distinct sorted labels per example."""
    p = torch.randint(1, 6, (n,), generator=g, device=DEV)
    step = m // 6  # distinct by construction: one label in each of 5 of the strides
    first = torch.randint(0, step, (n, 5), generator=g, device=DEV)
    rows = first + step * torch.arange(5, device=DEV)[None, :]
    keep = torch.arange(5, device=DEV)[None, :] < p[:, None]
    offsets = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    offsets[1:] = torch.cumsum(p, 0)
    return rows[keep].contiguous(), offsets


def _positives(state, n, m):
    """(n, m) mask of each example's labels."""
    pos = torch.zeros((n, m), dtype=torch.bool, device=DEV)
    if state["offsets"] is None:
        pos[torch.arange(n, device=DEV), state["labels"]] = True
    else:
        off = state["offsets"]
        rows = torch.repeat_interleave(torch.arange(n, device=DEV), off[1:] - off[:-1])
        pos[rows, state["labels"]] = True
    return pos


def _prox_input(case, seed):
    g, n, m, dt = _generator(seed), case["n"], case["m"], _dtype(case)
    if case["op"] in PROX_ENTROPIC:
        return torch.rand((n, m), generator=g, device=DEV, dtype=dt) * 20 - 10, None
    a = torch.randn((n, m), generator=g, device=DEV, dtype=dt)
    if case["op"] == "two_simplex":
        return a, torch.randint(1, 6, (n,), generator=g, device=DEV, dtype=torch.int64)
    # scores of a model that has learnt something: the label's row stands out
    label = torch.randint(0, m, (n,), generator=g, device=DEV)
    a[torch.arange(n, device=DEV), label] += 2
    if case["op"] == "topk_cone":
        # margins: most classes are below the label, or the cone does nothing
        a -= math.sqrt(2 * math.log(m)) - 1
    return a, None


def _features(g, case):
    X = torch.randn((case["n"], case["d"]), generator=g, device=DEV, dtype=torch.float32)
    X /= X.norm(dim=1, keepdim=True)
    return X.to(_dtype(case))


def _eval_input(case, seed):
    """Features, weights as a few epochs leave them, and feasible dual
    variables (label entries up, the others down, sums that balance)."""
    g, n, m, dt = _generator(seed), case["n"], case["m"], _dtype(case)
    s = {"X": _features(g, case), "offsets": None}
    s["W"] = torch.randn((m, case["d"]), generator=g, device=DEV,
                         dtype=torch.float32).mul_(0.5).to(dt)
    if case["labels"] == "multilabel":
        s["labels"], s["offsets"] = _label_rows(g, n, m)
        s["objs"] = [sd.objective("l2_multilabel_hinge_smooth"), sd.objective("l2_multilabel_entropy")]
    else:
        s["labels"] = torch.randint(0, m, (n,), generator=g, device=DEV)
        s["objs"] = [sd.objective("l2_hinge_topk_smooth", k=min(5, m - 1)), sd.objective("l2_entropy")]
    pos = _positives(s, n, m)
    A = torch.rand((n, m), generator=g, device=DEV, dtype=torch.float32).pow_(8)
    A.masked_fill_(pos, 0)
    A *= -0.5 / A.sum(dim=1, keepdim=True)
    A += pos.to(A.dtype) * (0.5 / pos.sum(dim=1, keepdim=True))
    s["A"] = A.to(dt).contiguous()
    return s


def _epoch_input(case, seed):
    g, n, m, dt = _generator(seed), case["n"], case["m"], _dtype(case)
    X = _features(g, case)
    if case["input"] == "kernel":
        X = (X @ X.T).sub_(1).mul_(0.5).exp_().contiguous()  # Gaussian kernel of unit vectors
    return X, torch.randint(0, m, (n,), generator=g, device=DEV)


def prepare(case, seed):
    dt = _dtype(case)
    if case["path"] == "prox":
        a, p = _prox_input(case, seed)
        return {"path": "prox", "op": case["op"], "a": a, "out": torch.empty_like(a), "p": p,
                "k": case.get("k", 1)}
    if case["path"] in ("eval", "refresh"):
        s = _eval_input(case, seed)
        if case["path"] == "refresh":
            s["W"] = torch.empty_like(s["W"])
        return dict(s, path=case["path"])
    X, labels = _epoch_input(case, seed)
    n, m = case["n"], case["m"]
    s = {"path": "epoch", "input": case["input"], "X": X, "labels": labels, "epoch": 0,
         "A": torch.zeros((n, m), dtype=dt, device=DEV),
         "obj": sd.objective(case["objective"], k=case["k"]),
         "orders": [torch.from_numpy(sd.epoch_order(n, e)).to(DEV) for e in range(3)]}
    if case["input"] == "features":
        s["W"] = torch.zeros((m, case["d"]), dtype=dt, device=DEV)
        s["norms"] = (X * X).sum(dim=1).contiguous()
    return s


def run(state):
    if state["path"] == "prox":
        return sd.prox(state["op"], state["a"], out=state["out"], k=state["k"], col_p=state["p"],
                       check_col_p=False)
    if state["path"] == "eval":
        records, accuracy, _ = sd.eval_features(state["objs"], state["X"], state["W"],
                                                state["labels"], A=state["A"],
                                                offsets=state["offsets"])
        return {"records": records, "accuracy": accuracy}
    if state["path"] == "refresh":
        W = sd.recompute_primal(state["X"], state["A"], out=state["W"])
        records, accuracy, losses = sd.eval_features(state["objs"], state["X"], W, state["labels"],
                                                     A=state["A"], per_example=True)
        return {"records": records, "accuracy": accuracy, "losses": losses, "W": W}
    order = state["orders"][state["epoch"] % len(state["orders"])]
    state["epoch"] += 1
    if state["input"] == "kernel":
        return {"A": sd.epoch_kernel(state["obj"], state["X"], state["A"], state["labels"],
                                     order=order)}
    W, A = sd.epoch_features(state["obj"], state["X"], state["W"], state["A"], state["labels"],
                             order=order, norms=state["norms"])
    return {"W": W, "A": A}


def work(case):
    es = 4 if case["dtype"] == "f32" else 8
    n, m, d = case["n"], case["m"], case.get("d", 0)
    if case["path"] == "prox":
        return {"bytes": 2 * n * m * es + (8 * n if case["op"] == "two_simplex" else 0), "flops": 0}
    if case["path"] == "eval":
        return {"bytes": es * (n * d + m * d + n * m) + 8 * n, "flops": 2 * n * m * d}
    if case["path"] == "refresh":
        return {"bytes": es * (n * d + m * d + n * m) + 8 * n + 32 * n, "flops": 4 * n * m * d}
    if case["input"] == "kernel":
        return {"bytes": es * (n * n + 2 * n * m) + 16 * n, "flops": 2 * n * n * m}
    # scores and the rank-one update of every example
    return {"bytes": es * (n * d + 2 * m * d + 2 * n * m) + 16 * n, "flops": 4 * n * m * d}


def tolerance(case):
    """About four times the largest error seen over the drawn ranges: the
    prox against `exact`, the epochs against themselves with the features
    (or the training examples) in another order, two epochs on."""
    single = case["dtype"] == "f32"
    if case["path"] == "prox":
        if not single:
            return {"rel": 1e-14, "max": 5e-13}
        # the threshold's rounding against the small values of a wide column
        return {"rel": 3e-6, "max": 3e-3} if case["m"] <= 2048 else {"rel": 1.6e-5, "max": 1.5e-2}
    if case["path"] in ("eval", "refresh"):
        # a near tie at the label's score moves one accuracy by 1 / n
        return ({"rel": 2e-5, "max": max(1e-4, 4 / case["n"])} if single
                else {"rel": 1e-14, "max": 1e-12})
    return {"rel": 1.3e-5, "max": 5e-4} if single else {"rel": 3e-14, "max": 4e-13}


# ---------------------------------------------------------------------------
# The same values in 64 bits.
# ---------------------------------------------------------------------------
def _bisect(f, lo, hi, steps=64):
    """The root of a decreasing f in [lo, hi], per column."""
    for _ in range(steps):
        t = (lo + hi) * 0.5
        up = f(t) > 0
        lo = torch.where(up, t, lo)
        hi = torch.where(up, hi, t)
    return (lo + hi) * 0.5


def _knapsack(a, hi, rhs):
    """t with sum clamp(a - t, 0, hi) = rhs; hi and rhs (n, 1) or numbers."""
    top = a.amax(dim=1, keepdim=True)
    low = a.amin(dim=1, keepdim=True) - hi
    return _bisect(lambda t: ((a - t).clamp_(min=0).minimum(torch.as_tensor(hi).to(a))
                              .sum(dim=1, keepdim=True) - rhs), low, top)


def _clamped(a, t, hi):
    return (a - t).clamp_(min=0).minimum(torch.as_tensor(hi).to(a))


def _topk(a, k, rhs, rho):
    """argmin 0.5 |x - a|^2 + 0.5 rho <1,x>^2 over 0 <= x_i <= <1,x> / k and
    <1,x> <= rhs (None: unbounded): for a fixed bound s = <1,x> / k the
    problem is a knapsack of sum k s, and its value is convex in s with the
    slope below."""
    def slope(a, s):
        t = _knapsack(a, s, k * s)
        return k * k * rho * s - k * t - (a - t - s).clamp_(min=0).sum(dim=1, keepdim=True)

    # from this bound on the knapsack's threshold is not above 0: a slope >= 0
    top = a.clamp(min=0)
    top = torch.maximum(top.amax(dim=1, keepdim=True), top.sum(dim=1, keepdim=True) / k)
    s = top if rhs is None else torch.full_like(top, rhs / k)
    inside = (slope(a, s) > 0).squeeze(1).nonzero().squeeze(1)
    if inside.numel():
        b = a[inside]
        s[inside] = _bisect(lambda v: -slope(b, v), torch.zeros_like(s[inside]), s[inside])
    return _clamped(a, _knapsack(a, s, k * s), s)


def _w_exp(z):
    """W(e^z): Newton's method on w + log w = z."""
    w = torch.where(z > 1, z - torch.log(z.clamp(min=1)) * 0.5, torch.exp(z.clamp(max=1)) / 1.5)
    w = w.clamp_(min=1e-300)
    for _ in range(7):
        w = w * (1 + z - torch.log(w)) / (1 + w)
        w = w.clamp_(min=1e-300)
    return w


def _two_simplex(a, b, rhs):
    """The projections x of a and y of b with sum x = sum y <= rhs (rows of
    -inf entries are left out of a block)."""
    def simplex(v, r):
        top = v.amax(dim=1, keepdim=True)
        return _bisect(lambda t: (v - t).clamp_(min=0).sum(dim=1, keepdim=True) - r, top - r, top)

    ta, tb = simplex(a, rhs), simplex(b, rhs)
    free = ta + tb < 0
    top_a, top_b = a.amax(dim=1, keepdim=True), b.amax(dim=1, keepdim=True)
    low, high = -top_b, torch.maximum(top_a, -top_b)
    t = _bisect(lambda t: ((a - t).clamp_(min=0).sum(dim=1, keepdim=True)
                           - (b + t).clamp_(min=0).sum(dim=1, keepdim=True)), low, high)
    ta, tb = torch.where(free, t, ta), torch.where(free, -t, tb)
    return (a - ta).clamp_(min=0), (b - tb).clamp_(min=0)


def _prox_exact(op, a, k, p):
    if op == "knapsack_eq":
        return _clamped(a, _knapsack(a, 1.0, 1.0), 1.0)
    if op == "knapsack_le":
        t = torch.where(a.clamp(0, 1).sum(dim=1, keepdim=True) <= 1, torch.zeros_like(a[:, :1]),
                        _knapsack(a, 1.0, 1.0))
        return _clamped(a, t, 1.0)
    if op in ("topk_simplex", "topk_cone", "topk_simplex_biased"):
        return _topk(a, k, None if op == "topk_cone" else 1.0, 1.0 if op.endswith("biased") else 0.0)
    if op in PROX_ENTROPIC:
        f = torch.exp if op == "entropy" else _w_exp
        top = torch.logsumexp(a, dim=1, keepdim=True)
        low = a.amin(dim=1, keepdim=True) - 1
        t = _bisect(lambda t: f(a - t).clamp_(max=1).sum(dim=1, keepdim=True) - 1, low, top)
        return f(a - t).clamp_(max=1)
    inf = float("inf")
    first = torch.arange(a.shape[1], device=a.device)[None, :] < p[:, None]
    x, y = _two_simplex(a.masked_fill(~first, -inf), a.masked_fill(first, -inf), 1.0)
    return torch.where(first, x, y)


def _xlogx(v):
    return torch.special.xlogy(v, v)


def _losses_exact(case, S, A, pos):
    """Each objective's (primal, dual) losses and, for one label, the number
    of classes at or above it, else the rank loss."""
    inf = float("inf")
    if case["labels"] == "multilabel":
        x, y = _two_simplex((0.5 - S).masked_fill(~pos, -inf), (0.5 + S).masked_fill(pos, -inf), 1.0)
        primal = ((0.5 - S) * x + (0.5 + S) * y - 0.5 * (x * x + y * y)).sum(dim=1)
        a_pos, a_neg = (A * pos).sum(dim=1), (A * ~pos).sum(dim=1)
        count = pos.sum(dim=1).double()
        hinge = (primal, 0.5 * (a_pos - a_neg - (A * A).sum(dim=1)))
        mean = (S * pos).sum(dim=1) / count
        dual = (-(_xlogx(1 - count[:, None] * A) * pos).sum(dim=1) / count
                - (_xlogx(-A * ~pos)).sum(dim=1) + torch.log(count) * (1 - a_pos))
        entropy = (torch.logsumexp(S, dim=1) - mean, dual)
        tops = S.masked_fill(~pos, -inf).topk(5, dim=1).values
        wrong = sum(((S >= tops[:, q:q + 1]) & ~pos & (q < count[:, None])).sum(dim=1)
                    for q in range(5))
        return hinge, entropy, wrong / (count * (S.shape[1] - count))
    y = S[pos][:, None]
    a = 1 + S - y
    a = torch.where(pos, a.amin(dim=1, keepdim=True) - 1, a)  # the label takes no part
    x = _topk(a, min(5, S.shape[1] - 1), 1.0, 0.0) * ~pos
    ay, rest = A[pos], A.masked_fill(pos, 0)
    hinge = ((a * x - 0.5 * x * x).sum(dim=1), ay - 0.5 * (rest * rest).sum(dim=1))
    entropy = (torch.logsumexp(S, dim=1) - y[:, 0],
               -_xlogx(1 - ay) - _xlogx(-rest).sum(dim=1))
    return hinge, entropy, ((S >= y) & ~pos).sum(dim=1)


def _eval_exact(case, seed):
    n, m = case["n"], case["m"]
    s = _eval_input(case, seed)
    X, A, W = s["X"].double(), s["A"].double(), s["W"].double()
    if case["path"] == "refresh":
        W = A.T @ X
    pos = _positives(s, n, m)
    losses, counts = [], []
    step = max(1, CHUNK // m)
    for i in range(0, n, step):
        hinge, entropy, count = _losses_exact(case, X[i:i + step] @ W.T, A[i:i + step], pos[i:i + step])
        losses.append(torch.stack([torch.stack(hinge, 1), torch.stack(entropy, 1)], 1))
        counts.append(count)
    losses = torch.cat(losses)
    sums = losses.sum(dim=0)
    reg = 0.5 * float((W * W).sum())
    rank = 0.0
    if case["labels"] == "multilabel":
        rank = float(torch.cat(counts).mean())
    records = []
    for o in range(2):
        primal, dual = float(sums[o, 0]), float(sums[o, 1])
        records.append({"primal": primal + reg, "dual": dual - reg, "primal_loss": primal,
                        "dual_loss": dual, "primal_regularizer": reg, "dual_regularizer": reg,
                        "rank_loss": rank})
    accuracy = None
    if case["labels"] == "multiclass":
        hist = torch.bincount(torch.cat(counts), minlength=m)
        accuracy = (torch.cumsum(hist, 0).double() / n).cpu()
    if case["path"] == "refresh":
        return {"records": records, "accuracy": accuracy, "losses": losses, "W": W}
    return {"records": records, "accuracy": accuracy}


def _epoch_exact(case, seed):
    """The solver's loop, one example after the other (smooth top-k hinge of
    the sum: knapsack with the bias term)."""
    X, labels = _epoch_input(case, seed)
    X, y = X.double().cpu().numpy(), labels.cpu().numpy()
    n, m, k = case["n"], case["m"], case["k"]
    kernel = case["input"] == "kernel"
    A = np.zeros((n, m))
    W = None if kernel else np.zeros((m, X.shape[1]))
    for i in sd.epoch_order(n, 0):
        norm2 = X[i, i] if kernel else X[i] @ X[i]
        rho = norm2 / (norm2 + 1.0)
        scores = X[i] @ A if kernel else W @ X[i]
        old = A[i].copy()
        v = rho / norm2 * scores - rho * old
        v += rho / norm2 - v[y[i]]
        v[y[i]] = -np.inf
        lo, hi = v[np.isfinite(v)].min() - 2.0, max(v.max(), 0.0) + 2.0
        # total(t) = 1 has the root of the equality; with the bias t = rho * total
        for bias in (True, False):
            low, high = lo, hi
            for _ in range(60):
                t = 0.5 * (low + high)
                total = np.minimum(np.maximum(v - t, 0.0), 1.0 / k).sum()
                if (rho * total > t) if bias else (total > 1.0):
                    low = t
                else:
                    high = t
            x = np.minimum(np.maximum(v - t, 0.0), 1.0 / k)
            if x.sum() <= 1.0:
                break
        A[i] = -x
        A[i, y[i]] = min(1.0, x.sum())
        if not kernel:
            W += np.outer(A[i] - old, X[i])
    return {"A": A} if kernel else {"W": W, "A": A}


def exact(case, seed):
    if case["path"] == "prox":
        a, p = _prox_input(case, seed)
        out = torch.empty_like(a, dtype=torch.float64)
        step = max(1, CHUNK // case["m"])
        for i in range(0, case["n"], step):
            out[i:i + step] = _prox_exact(case["op"], a[i:i + step].double(), case.get("k", 1),
                                          None if p is None else p[i:i + step])
        return out
    if case["path"] in ("eval", "refresh"):
        return _eval_exact(case, seed)
    # one example after the other on the host: the small epochs only
    width = case["n"] if case["input"] == "kernel" else 3 * case["d"]
    if (case["objective"] == "l2_topk_hinge_smooth"
            and case["n"] * (1.5e-3 + width * case["m"] * 1.5e-9) < 15):
        return _epoch_exact(case, seed)
    return None
