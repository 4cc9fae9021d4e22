"""Calls that need no scratch under capture: the top-k operators with
8 < k <= 15 (elsewhere they take the register kernel and its list of deferred
columns) and the biased knapsack over a workgroup's registers, on a stream
that has no scratch and on one whose list is freed after the capture."""
import numpy as np
import pytest

from tests import inputs
from tests.test_prox_gpu import F32, parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op,kw,m", [
    ("topk_simplex", dict(k=12, rhs=1.0), 100), ("topk_cone", dict(k=9), 512),
    ("topk_simplex_biased", dict(k=15, rhs=1.0, rho=0.5), 40),
    ("topk_cone_biased", dict(k=9, rho=0.25), 300),
    ("knapsack_le_biased", dict(rho=0.5), 3000)])
def test_cold_capture(cuda, oracle, op, kw, m):
    import torch
    import libsdca_amd as sd
    x = inputs.mixed_signs(64, m, np.float32, 40 + m, -2, 2)
    a = torch.from_numpy(x).to(cuda)
    out = torch.empty_like(a)
    gs = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=gs):
        sd.prox(op, a, out=out, **kw)
    for _ in range(3):
        out.fill_(-7.0)
        g.replay()
        torch.cuda.synchronize()
        parity(oracle, op, x, out.cpu().numpy(), F32, f"captured {op} m={m}", **kw)
        torch.cuda.synchronize()


@pytest.mark.parametrize("op,kw,m", [
    ("topk_simplex", dict(k=12, rhs=1.0), 100), ("topk_cone", dict(k=9), 512),
    ("topk_cone_biased", dict(k=15, rho=0.25), 40)])
def test_warm_capture(cuda, oracle, op, kw, m):
    """A capture on a stream that has a list, then a larger call there, which
    frees that list and takes another: the graph holds neither."""
    import torch
    import libsdca_amd as sd
    x = inputs.mixed_signs(64, m, np.float32, 41 + m, -2, 2)
    a = torch.from_numpy(x).to(cuda)
    out = torch.empty_like(a)
    gs = torch.cuda.Stream()
    with torch.cuda.stream(gs):
        sd.prox(op, a, out=out, **kw)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=gs):
        sd.prox(op, a, out=out, **kw)
    large = torch.from_numpy(inputs.normal(100_000, 20, np.float32, 42 + m)).to(cuda)
    torch.cuda.synchronize()
    for _ in range(3):
        with torch.cuda.stream(gs):
            sd.prox("topk_cone", large.clone(), k=5)
        torch.cuda.synchronize()
        out.fill_(-7.0)
        g.replay()
        torch.cuda.synchronize()
        parity(oracle, op, x, out.cpu().numpy(), F32, f"captured {op} m={m}", **kw)
        large = torch.cat([large, large])
