"""The built-in choice between the slice and the node-group kernel of the SpMM at sizes where
they differ by 15 % or more (operators of a box of hexahedra, values at random).  The two add a
row's products in different orders, so the result's bits tell which one ran."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _box(dev, nx, ny, nz, rng):
    """Operator of nx x ny x nz nodes, each coupled to its up to 27 neighbours."""
    t = lambda n: sp.diags([np.ones(n - 1), np.ones(n), np.ones(n - 1)], [-1, 0, 1])
    P = sp.kron(sp.kron(t(nx), t(ny)), t(nz))
    K, M = (sp.kron(P, S).tocsr() for S in (np.ones((3, 3)), np.eye(3)))
    for S in (K, M):
        S.data = rng.standard_normal(S.nnz)
    return dev.KronOperator([(S.indptr + 1, S.indices + 1, S.data) for S in (K, M)], q=6)


@pytest.mark.parametrize("nodes,R,fp32,groups", [
    ((333, 30, 5), 4, False, False),      # slices / groups 79 / 102 us
    ((2777, 12, 3), 4, True, False),      # 82 / 103
    ((12, 12, 13), 32, False, False),     # 24 / 28
    ((222, 3, 3), 42, False, True),       # 34 / 22
    ((1333, 3, 3), 20, True, True),       # 45 / 32
    ((1888, 3, 3), 8, False, True),       # 55 / 41
])
def test_the_faster_kernel_runs(nodes, R, fp32, groups):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, tune
    rng = np.random.default_rng(R)
    op = _box(device, *nodes, rng)
    assert op.format == "blocks"
    dt = torch.float32 if fp32 else torch.float64
    T = op.tmat(rng.standard_normal((R, 2, 6, 6)), fp32)
    x = torch.as_tensor(rng.standard_normal(op.p * 6 * R), device="cuda").to(dt)
    y = {}
    try:
        for k in (0, 1, 2):
            tune.set_knob("spmm_group", k)
            y[k] = torch.full_like(x, float("nan"))
            op.apply(T, x, y[k], R, fp32=fp32)
    finally:
        tune.set_knob("spmm_group", 0)
    assert not torch.equal(y[1], y[2])
    assert torch.equal(y[0], y[2] if groups else y[1])
