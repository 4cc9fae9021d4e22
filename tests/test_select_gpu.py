"""The top-k operators by selection (prox_select.hip) against the CPU oracle:
the sizes around each configuration step, k around the register lists, inputs that take every way through the selection
(short lists, more candidates than the list holds, searches past the first
list, ties with zero and with the thresholds, whole-column fallback)."""
import numpy as np
import pytest

from tests import inputs
from tests.test_prox_gpu import DTYPES, F32, F64, parity, run_gpu

pytestmark = pytest.mark.gpu

OPS = [("topk_simplex", dict(rhs=1.0)), ("topk_cone", dict()),
       ("topk_simplex_biased", dict(rhs=1.0, rho=0.5)), ("topk_cone_biased", dict(rho=0.25))]


def select_inputs(m, dtype, seed, n=24):
    yield "label+2", inputs.label_shifted(n, m, dtype, seed)
    # the cone's searches: few values above zero
    margin = np.sqrt(2 * np.log(m + 1)) - 1
    yield "margins", (inputs.label_shifted(n, m, np.float64, seed + 1) - margin).astype(dtype)
    # every value a candidate of the knapsack
    yield "small", inputs.normal(n, m, dtype, seed + 2, 1e-3)
    yield "mixed", inputs.mixed_signs(n, m, dtype, seed + 3, -3, 3)
    # the largest values in one of the 64 parts
    x = inputs.normal(n, m, dtype, seed + 4, 0.1)
    x[:, ::64] += 3
    yield "one part", x
    yield "ties", np.round(inputs.normal(n, m, dtype, seed + 5) * 2).astype(dtype) / 2
    yield "edge", inputs.edge_columns(m, dtype, seed + 6)


@pytest.mark.parametrize("dtype,result", DTYPES)
@pytest.mark.parametrize("m,k", [(16, 9), (17, 15), (40, 16), (256, 20), (257, 10), (512, 16),
                                 (513, 3), (1000, 10), (1024, 15), (1025, 5), (2048, 55)])
@pytest.mark.parametrize("op,kw", OPS)
def test_select_wave(cuda, oracle, op, kw, m, k, dtype, result):
    """One wave per column."""
    for name, x in select_inputs(m, dtype, 500 + m + k):
        got, thr = run_gpu(op, x, result, cuda, k=k, **kw)
        parity(oracle, op, x, got, result, f"{op} k={k} {name} m={m}", nthreads=8, thr=thr, k=k, **kw)


@pytest.mark.parametrize("dtype,result", [(np.float32, F32), (np.float64, F64), (np.float32, F64)])
@pytest.mark.parametrize("m,k", [(2049, 10), (4096, 5), (4098, 20), (8193, 2), (16384, 12)])
@pytest.mark.parametrize("op,kw", OPS)
def test_select_workgroup(cuda, oracle, op, kw, m, k, dtype, result):
    """One workgroup per column."""
    for name, x in select_inputs(m, dtype, 600 + m + k, n=6):
        got, thr = run_gpu(op, x, result, cuda, k=k, **kw)
        parity(oracle, op, x, got, result, f"{op} k={k} {name} m={m}", nthreads=8, thr=thr, k=k, **kw)


@pytest.mark.parametrize("m,k", [(2048, 56), (300, 70), (30001, 7)])
def test_select_limits(cuda, oracle, m, k):
    """k at and past the lists' part maxima, and the widest form."""
    x = inputs.label_shifted(8, m, np.float32, 700 + m)
    for op, kw in OPS:
        got, thr = run_gpu(op, x, F32, cuda, k=k, **kw)
        parity(oracle, op, x, got, F32, f"{op} k={k} m={m}", nthreads=8, thr=thr, k=k, **kw)


@pytest.mark.parametrize("k", [3, 12])
def test_select_unaligned_and_in_place(cuda, oracle, k):
    """Columns off the 16-byte boundary (a view one element into a buffer)
    and a deferred list over several launches, in place."""
    import torch
    import libsdca_amd as sd
    for m in (300, 1028, 5000):
        x = inputs.label_shifted(40, m, np.float32, 800 + m) - np.float32(2.0)
        buf = torch.zeros(40 * m + 1, dtype=torch.float32, device=cuda)
        a = buf[1:].view(40, m)
        for _ in range(2):
            a.copy_(torch.from_numpy(x))
            out = sd.prox("topk_cone", a, k=k)
            torch.cuda.synchronize()
            parity(oracle, "topk_cone", x, out.cpu().numpy(), F32, f"unaligned m={m}", k=k)


def test_select_values_not_finite(cuda):
    """Columns that hold +inf, NaN (sorted whole; no projection is defined) or
    -inf (a masked class: test_masked_gpu.py) do not touch the others of the
    launch."""
    import torch
    import libsdca_amd as sd
    for m, k in ((300, 20), (3000, 5)):
        x = inputs.label_shifted(10, m, np.float32, 950 + m)
        want = sd.prox("topk_simplex", torch.from_numpy(x).to(cuda), k=k).cpu().numpy()
        y = x.copy()
        y[2, 5], y[4, 7], y[6, 0] = np.inf, np.nan, -np.inf
        got = sd.prox("topk_simplex", torch.from_numpy(y).to(cuda), k=k).cpu().numpy()
        keep = [0, 1, 3, 5, 7, 8, 9]
        assert (got[keep] == want[keep]).all()
