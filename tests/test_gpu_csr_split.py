"""The multi-term CSR operator (kronspmv's sum, kronecker.f90:19-85) with 8 lanes a row and
column (few rows times columns) and with one, against the sum in FP64 on the host: rows of 0
to 70 entries, a term without any entry, 1 to 3 terms, 2 to 8 temporal functions."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    return device


def _matrix(p, kind, rng):
    if kind == "none":
        return sp.csr_matrix((p, p))
    n = rng.integers(0, 8, p)
    n[rng.integers(0, p, 5)] = min(p, 70)
    n[0] = n[p - 1] = 0
    cols = [rng.choice(p, k, replace=False) for k in n]
    S = sp.csr_matrix((rng.standard_normal(n.sum()), np.concatenate([np.sort(c) for c in cols]),
                       np.concatenate([[0], np.cumsum(n)])), shape=(p, p))
    return S


@pytest.mark.parametrize("p", [1, 31, 1000, 20011])
@pytest.mark.parametrize("terms", ["a", "aa", "a none", "none a", "aaa"])
def test_csr_operator_matches_the_sum(dev, p, terms):
    import torch
    rng = np.random.default_rng(p)
    kinds = [k for k in (terms.split() if " " in terms else terms)]
    mats = [_matrix(p, "none" if k == "none" else "a", rng) for k in kinds]
    nt = len(mats)
    for q, R in ((3, 1), (3, 9), (2, 5), (6, 1), (8, 4), (8, 5), (5, 30)):
        op = dev.KronOperator([(S.indptr + 1, S.indices + 1, S.data) for S in mats], q=q)
        if op.format != "csr":
            op.format = "csr"
        Ts = rng.standard_normal((R, nt, q, q))
        for fp32, eps in ((False, 2.0 ** -53), (True, 2.0 ** -24)):
            dt = torch.float32 if fp32 else torch.float64
            x, y0 = (torch.as_tensor(rng.standard_normal((p, R, q)), device="cuda").to(dt)
                     .contiguous() for _ in range(2))
            y = y0.clone()
            op.apply(op.tmat(Ts, fp32), x, y, R, alpha=0.5, beta=-2.0, fp32=fp32)
            x64, y64 = x.double().cpu().numpy(), y0.double().cpu().numpy()

            def form(M, T, x, y, a, b):
                z = sum(np.einsum("rij,prj->pri", T[:, k], (M[k] @ x.reshape(p, -1)).reshape(p, R, q))
                        for k in range(nt))
                return a * z + b * y
            ref = form(mats, Ts, x64, y64, 0.5, -2.0)
            mag = form([abs(S) for S in mats], abs(Ts), abs(x64), abs(y64), 0.5, 2.0)
            # 70 products a row at most, q nt of those; inputs rounded to FP32
            bound = (70 + q * nt + 8) * eps * mag
            assert (np.abs(y.double().cpu().numpy() - ref) <= bound).all(), (q, R, fp32)
