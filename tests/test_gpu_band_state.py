"""What a banded factor keeps from one call to the next: its captured sweeps, the scratch of
a factorization and the library handle with its stream.  Reference: sparse LU in FP64
(scipy).  The strips are clamped along their long side, so cond(K) is about 1e3: FP64
agrees to 1e3 x a few hundred eps, 1e-10; FP32 to 1e-3."""
import numpy as np
import pytest

from test_gpu_band_twisted import check, strip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    return device


def on_device(K):
    import torch
    return tuple(torch.as_tensor(np.ascontiguousarray(v), device="cuda") for v in K)


def coupled(K, reach):
    """K with every DOF also coupled to the one reach before it, diagonally dominant."""
    import scipy.sparse as sp
    p = len(K[0]) - 1
    S = sp.csr_matrix((K[2], K[1] - 1, K[0] - 1), shape=(p, p))
    far = sp.diags([np.full(p - reach, -1.0)], [reach], shape=(p, p))
    W = (S + far + far.T + sp.diags(np.full(p, 2.0))).tocsr()
    W.sort_indices()
    return W.indptr.astype(np.int32) + 1, W.indices.astype(np.int32) + 1, W.data


@pytest.mark.parametrize("block", [256, 512])
def test_captured_sweeps_follow_the_band(dev, block):
    """The same column counts before and after each refactorization with a wider band: the
    arrays of the factor change their layout, wherever the allocator puts them."""
    K = strip(6 * block // 12)
    pr = dev.BandPreconditioner(K, block=block)
    check(dev, pr, K, (3, 60), 0)
    for reach in (100, 180, block - 6):
        W = coupled(K, reach)
        pr.refactor(*on_device(W))
        check(dev, pr, W, (3, 60), reach)
