"""The slice SpMM kernel with the load cases packed over a slice's lanes without gaps, against
kronspmv's sum (kronecker.f90:19-85) in FP64 on the host: case counts below, at and above
powers of two, over the 64 of a launch, node counts that do not fill the last slice, on both
sides of the 256 waves from which on the packing starts."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _operator(nn, rng):
    pairs = [(a, a + d) for a in range(nn) for d in (-17, -2, -1, 0, 1, 2, 17) if 0 <= a + d < nn]
    a, b = np.array(pairs).T
    n, p = len(a), 3 * nn
    i, j = np.divmod(np.arange(9), 3)
    K = sp.csr_matrix((rng.standard_normal(9 * n), ((3 * a[:, None] + i).ravel(),
                                                     (3 * b[:, None] + j).ravel())), shape=(p, p))
    d = np.arange(3)
    M = sp.csr_matrix((rng.standard_normal(3 * n), ((3 * a[:, None] + d).ravel(),
                                                     (3 * b[:, None] + d).ravel())), shape=(p, p))
    K.sort_indices(), M.sort_indices()
    return K, M


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("nn", [1, 130, 1000, 5250])
def test_slices(nn, fp32):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, tune
    rng = np.random.default_rng(nn)
    K, M = _operator(nn, rng)
    op = device.KronOperator([(S.indptr + 1, S.indices + 1, S.data) for S in (K, M)], q=6)
    dt, eps = (torch.float32, 2.0 ** -24) if fp32 else (torch.float64, 2.0 ** -53)
    tune.set_knob("spmm_group", 1)
    try:
        for R in (2, 3, 5, 7, 8, 9, 13, 15, 17, 31, 33, 63, 64, 65, 67):
            A, B = rng.standard_normal((2, R, 6, 6))
            x, y0 = (torch.as_tensor(rng.standard_normal((3 * nn, R, 6)), device="cuda").to(dt)
                     .contiguous() for _ in range(2))
            for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
                y = y0.clone()
                op.apply(op.tmat(np.stack([A, B], axis=1), fp32), x, y, R, alpha=alpha, beta=beta,
                         fp32=fp32)
                want, size = beta * y0.double().cpu().numpy(), np.abs(beta * y0.double().cpu().numpy())
                x64 = x.double().cpu().numpy()
                for S, T in ((K, A), (M, B)):
                    Z, Za = ((Q @ X.reshape(3 * nn, -1)).reshape(x64.shape)
                             for Q, X in ((S, x64), (abs(S), np.abs(x64))))
                    want = want + alpha * np.einsum("prj,rij->pri", Z, T)
                    size = size + abs(alpha) * np.einsum("prj,rij->pri", Za, np.abs(T))
                # rounded inputs (matrix, temporal matrix), 21 + 3 spatial and 12 temporal
                # terms, alpha and beta: at most 48 roundings of the sum of magnitudes
                err = np.abs(y.double().cpu().numpy() - want)
                assert (err <= 48 * eps * size + 1e-300).all(), (R, alpha, float((err / size).max()))
    finally:
        tune.set_knob("spmm_group", 0)
