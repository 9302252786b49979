"""The node-group SpMM kernel (XT_TUNE_SPMM_GROUP: a wave reads each neighbour's rows of X
once for four consecutive nodes) against kronspmv's sum (kronecker.f90:19-85) in FP64 on
the host: node counts that do not fill the last group, irregular patterns and rows without
neighbours, case counts at the edges of the lanes of a slot (8, 16, 24, 32) and over a
chunk of 32 cases, alpha and beta, new values in place."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, tune
    yield device
    tune.set_knob("spmm_group", 0)


def _blocks(nn, kind, rng):
    """K (3 x 3 blocks) and M (diagonal blocks) on a random or banded node pattern."""
    if kind == "banded":
        pairs = [(a, a + d) for a in range(nn) for d in (-17, -16, -2, -1, 0, 1, 2, 16, 17)
                 if 0 <= a + d < nn]
    else:       # long rows next to rows of one entry, unsymmetric
        pairs = [(a, a) for a in range(nn)]
        for a in range(0, nn, 5):
            pairs += [(a, b) for b in rng.choice(nn, min(nn, 40), replace=False)]
        pairs = sorted(set((int(a), int(b)) for a, b in pairs))
    a, b = np.array(pairs).T
    n = len(a)
    rows = (3 * a[:, None, None] + np.arange(3)[None, :, None] + np.zeros((1, 1, 3), int)).ravel()
    cols = (3 * b[:, None, None] + np.arange(3)[None, None, :] + np.zeros((1, 3, 1), int)).ravel()
    K = sp.csr_matrix((rng.standard_normal(9 * n), (rows, cols)), shape=(3 * nn, 3 * nn))
    rows = (3 * a[:, None] + np.arange(3)).ravel()
    cols = (3 * b[:, None] + np.arange(3)).ravel()
    M = sp.csr_matrix((rng.standard_normal(3 * n), (rows, cols)), shape=(3 * nn, 3 * nn))
    K.sort_indices()
    M.sort_indices()
    return K, M


def _operator(dev, K, M):
    return dev.KronOperator([(S.indptr + 1, S.indices + 1, S.data) for S in (K, M)], q=6)


def _check(dev, op, K, M, R, fp32, rng, alpha=1.0, beta=0.0):
    import torch
    p = K.shape[0]
    dt, eps = (torch.float32, 2.0 ** -24) if fp32 else (torch.float64, 2.0 ** -53)
    A, B = rng.standard_normal((2, R, 6, 6))
    x, y0 = (torch.as_tensor(rng.standard_normal((p, R, 6)), device="cuda").to(dt).contiguous()
             for _ in range(2))
    y = y0.clone()
    T = op.tmat(np.stack([A, B], axis=1), fp32)
    op.apply(T, x, y, R, alpha=alpha, beta=beta, fp32=fp32)
    x64, y64 = x.double().cpu().numpy(), y0.double().cpu().numpy()

    def form(K, M, A, B, x, y, a, b):
        KX, MX = (S @ x.reshape(p, R * 6) for S in (K, M))
        return (a * (np.einsum("rij,prj->pri", A, KX.reshape(p, R, 6)) +
                     np.einsum("rij,prj->pri", B, MX.reshape(p, R, 6))) + b * y)
    ref = form(K, M, A, B, x64, y64, alpha, beta)
    mag = form(abs(K), abs(M), abs(A), abs(B), abs(x64), abs(y64), abs(alpha), abs(beta))
    # a sum of n products (n: longest row), 12 of those, alpha and beta; inputs rounded
    n = int(np.diff(K.indptr).max())
    bound = (n + 12 + 8) * eps * mag
    err = np.abs(y.double().cpu().numpy() - ref)
    assert (err <= bound).all(), (R, fp32, float((err / bound).max()))


@pytest.mark.parametrize("kind", ["banded", "irregular"])
@pytest.mark.parametrize("nn", [1, 3, 8, 37, 262])
def test_group_kernel_matches_the_sum(dev, kind, nn):
    from xtfem_amd import tune
    rng = np.random.default_rng(nn)
    K, M = _blocks(nn, kind, rng)
    op = _operator(dev, K, M)
    assert op.format == "blocks"
    tune.set_knob("spmm_group", 2)
    for R in (2, 8, 9, 16, 17, 24, 25, 32, 33, 50, 65):
        for fp32 in (False, True):
            _check(dev, op, K, M, R, fp32, rng)
    _check(dev, op, K, M, 7, False, rng, alpha=-0.5, beta=2.0)
    _check(dev, op, K, M, 32, True, rng, alpha=1.5, beta=-1.0)


def test_group_kernel_after_new_values(dev):
    import torch
    from xtfem_amd import tune
    rng = np.random.default_rng(0)
    K, M = _blocks(101, "irregular", rng)
    op = _operator(dev, K, M)
    tune.set_knob("spmm_group", 2)
    K.data, M.data = rng.standard_normal(K.nnz), rng.standard_normal(M.nnz)
    op.set_values(torch.as_tensor(K.data, device="cuda"), torch.as_tensor(M.data, device="cuda"))
    for R in (5, 32):
        for fp32 in (False, True):
            _check(dev, op, K, M, R, fp32, rng)


def test_built_in_choice_takes_groups_for_many_cases(dev):
    """Both sides of the built-in line give the sum (2000 nodes: 64 cases are above it)."""
    from xtfem_amd import tune
    rng = np.random.default_rng(1)
    K, M = _blocks(2000, "banded", rng)
    op = _operator(dev, K, M)
    tune.set_knob("spmm_group", 0)
    for R in (2, 20, 64):
        _check(dev, op, K, M, R, False, rng)
