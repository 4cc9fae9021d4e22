"""More columns than one launch holds: HIP refuses 2^32 threads, and beyond
that starts the count modulo 2^32.  The selection strides over its grid, the
wide knapsack takes several launches.  Columns around the steps and at the
end give what a call of their own gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op,kw,m,n,step", [
    # a wave per column: 2^26 columns
    ("topk_simplex", dict(k=16), 17, 1 << 26, 1 << 25),
    # 512 threads per column
    ("knapsack_eq", {}, 2049, (1 << 23) + 3, (1 << 23) - 1),
])
def test_more_columns_than_a_launch(cuda, op, kw, m, n, step):
    import torch
    import libsdca_amd as sd
    if torch.cuda.mem_get_info()[0] < n * m * 4 + (4 << 30):
        pytest.skip("needs more free device memory")
    a = torch.empty((n, m), dtype=torch.float32, device=cuda)
    a.view(-1).fill_(-1.0)
    rows = torch.tensor([0, 1, step // 2, step - 4, step - 1, step, step + 1, n - 1], device=cuda)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn((len(rows), m), generator=g, device=cuda)
    a[rows] = x
    want = sd.prox(op, x.clone(), **kw)
    sd.prox(op, a, **kw)
    torch.cuda.synchronize()
    got = a[rows]
    del a
    torch.cuda.empty_cache()
    assert torch.equal(got, want)
    assert np.isfinite(want.cpu().numpy()).all()
