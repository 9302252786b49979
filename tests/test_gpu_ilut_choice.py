"""Which sweep kernel a small ILUT factor gets: factors of few wide levels the one with a
barrier a level, those of many narrow ones two columns a workgroup.  The second is built for
factors up to 4096 rows only, and the two add a row's products in different orders, so the same
system with 4200 rows (the others uncoupled) gives the same bits where the first runs in both."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _levels(p, n, rng, more):
    """p rows in n levels, each row coupled to six of the level before (the drop tolerance keeps
    most of the fill out), and more uncoupled rows."""
    w = p // n
    r = np.repeat(np.arange(w, n * w), 6)
    c = (r // w - 1) * w + rng.integers(0, w, r.size)
    A = sp.coo_matrix((rng.uniform(-0.6, -0.5, r.size), (r, c)), shape=(p, p)).tocsr()
    A = A + A.T + 20.0 * sp.eye(p)
    A = sp.block_diag([A, sp.eye(more)]).tocsr() if more else A.tocsr()
    A.sort_indices()
    return A.indptr.astype(np.int32) + 1, A.indices.astype(np.int32) + 1, A.data


@pytest.mark.parametrize("p,n,wide", [(4000, 40, True), (3900, 1300, False)])
@pytest.mark.parametrize("fp32", [False, True])
def test_wide_levels_go_to_one_workgroup(p, n, wide, fp32):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    y = []
    for more in (0, 4200 - p):
        K = _levels(p, n, np.random.default_rng(1), more)
        pr = device.IlutPreconditioner(K, 12, 0.02)
        lo, up = pr.levels()
        assert (lo < 60 and up < 100) if wide else (lo > 1000 and up > 1000)
        g = torch.Generator(device="cpu").manual_seed(5)
        x = torch.randn((4200, 6), generator=g, dtype=torch.float64)[:p + more].cuda()
        x = x.to(torch.float32 if fp32 else torch.float64).contiguous()
        out = torch.full_like(x, float("nan"))
        pr.apply(None, x, out, 6, q=1, fp32=fp32)
        y.append(out[:p].clone())
    assert torch.allclose(*y, rtol=1e-4 if fp32 else 1e-12)
    assert torch.equal(*y) == wide
