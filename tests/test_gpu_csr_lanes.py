"""Lanes a row and column of the CSR operator: one past 16 columns from 50000 rows times columns
on.  With one lane a column's sums do not depend on how many columns there are, with eight the
entries are added in another order: the first 18 of 40 columns (one lane) tell which it was."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,one", [(3355, True), (1845, False)])
def test_lanes_past_sixteen_columns(p, one):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    rng = np.random.default_rng(p)
    A = sp.diags([rng.standard_normal(p - abs(d)) for d in range(-13, 14)], range(-13, 14)).tocsr()
    A.sort_indices()
    op = device.KronOperator([(A.indptr + 1, A.indices + 1, A.data)] * 2, q=1)
    x = torch.as_tensor(rng.standard_normal((p, 40)), device="cuda")
    y = {}
    for c in (18, 40):
        T = op.tmat(np.ones((c, 2, 1, 1)), False)
        xc = x[:, :c].contiguous()
        y[c] = torch.full_like(xc, float("nan"))
        op.apply(T, xc, y[c], c)
    assert torch.allclose(y[18], y[40][:, :18], rtol=1e-10, atol=1e-10)
    assert torch.equal(y[18], y[40][:, :18]) == one
