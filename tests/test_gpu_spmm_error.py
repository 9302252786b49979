"""Rounding error of the several-case SpMM kernels (kronspmv's sum, kronecker.f90:19-85) on a
hexahedral mesh, against the sum in more bits of the same (rounded) inputs.  The node groups
add product by product, the slices a block at a time; with the group's own nodes last the
groups' sums stay the more exact ones (in a model of both in FP32: 0.78 of the slices' error
in the 2-norm on boxes of several shapes; 1.25 with the nodes in sorted order)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [True, False])
@pytest.mark.parametrize("size", [(14, 13, 5), (9, 9, 9), (30, 14, 2)])
def test_groups_no_less_exact_than_slices(size, fp32):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, fem, tune
    rng = np.random.default_rng(3)
    K, M = fem.assemble(fem.structured_hex(*size, *map(float, size)), 1.0, 0.3, 1.0)[:2]
    p, R = len(K[0]) - 1, 12
    dt, wide = (np.float32, np.float64) if fp32 else (np.float64, np.longdouble)
    A, B = rng.standard_normal((2, R, 6, 6)).astype(dt)
    x = rng.standard_normal((p, R, 6)).astype(dt)
    KX, MX = (np.asarray(sp.csr_matrix((np.asarray(S[2]).astype(dt).astype(wide),
                                        np.asarray(S[1]) - 1, np.asarray(S[0]) - 1),
                                       shape=(p, p)) @ x.astype(wide).reshape(p, R * 6))
              for S in (K, M))
    ref = (np.einsum("rij,prj->pri", A.astype(wide), KX.reshape(p, R, 6)) +
           np.einsum("rij,prj->pri", B.astype(wide), MX.reshape(p, R, 6)))
    op = device.KronOperator([K, M], q=6)
    T = op.tmat(np.stack([A, B], axis=1).astype(np.float64), fp32)
    X = torch.as_tensor(x, device="cuda")
    err = {}
    try:
        for knob in (1, 2):
            tune.set_knob("spmm_group", knob)
            y = torch.empty_like(X)
            op.apply(T, X, y, R, fp32=fp32)
            err[knob] = float(np.sqrt(((y.cpu().numpy().astype(wide) - ref) ** 2).sum()))
    finally:
        tune.set_knob("spmm_group", 0)
    assert 0 < err[2] <= err[1], err
