"""The banded factor eliminated from both ends: block counts around the smallest ones (no
chain, one chain, both), blocks wider than twice the band (chains on the band's rows only),
column counts around the tile widths, and refactorizations of a wider band and from every
block on.  Reference: sparse LU in FP64 (scipy).  The strip is clamped along its long side,
so cond(K) is about 1e3: FP64 agrees to 1e3 x a few hundred eps, 1e-10; FP32 to 1e-3."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    return device


def strip(n):
    """n x 1 x 1 elements clamped on y = 0 (12 DOFs a section, half-bandwidth below 64)."""
    from xtfem_amd import fem
    mesh = fem.structured_hex(n, 1, 1, float(n), 1.0, 1.0)
    K, *_ = fem.assemble(mesh, 2.0e5, 0.3, 7.85e-9)
    return fem.applybc(K, fem.clamp_mask(mesh, 1, [0.0]))


def lu(K):
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    p = len(K[0]) - 1
    return sl.splu(sp.csr_matrix((K[2], K[1] - 1, K[0] - 1), shape=(p, p)).tocsc())


def check(dev, pr, K, columns, seed):
    import torch
    p = len(K[0]) - 1
    F = lu(K)
    rng = np.random.default_rng(seed)
    for c in columns:
        X = rng.standard_normal((p, c))
        want = F.solve(X)
        for dt, tol in ((torch.float64, 1e-10), (torch.float32, 1e-3)):
            x = torch.as_tensor(X, device="cuda").to(dt).contiguous()
            y = torch.full_like(x, float("nan"))
            pr.apply(None, x, y, c, q=1, fp32=dt == torch.float32)
            got = y.double().cpu().numpy()
            assert rel(got, want) < tol, (c, dt, rel(got, want))


@pytest.mark.parametrize("block", [64, 128, 192])
@pytest.mark.parametrize("nblocks", [1, 2, 3, 4, 5, 12])
def test_block_counts(dev, block, nblocks):
    K = strip((nblocks * block) // 12 - 2 if nblocks < 12 else nblocks * block // 12 - 1)
    pr = dev.BandPreconditioner(K, block=block)
    assert pr.nblocks == nblocks and pr.block == block
    check(dev, pr, K, (1, 16, 17, 48), 10 * nblocks + block)


@pytest.mark.parametrize("columns", [(6, 32, 33), (64, 66, 96), (97, 144, 160), (192, 246, 252)])
def test_column_counts(dev, columns):
    K = strip(200)
    check(dev, dev.BandPreconditioner(K, block=256), K, columns, columns[0])
    check(dev, dev.BandPreconditioner(K), K, columns, columns[1])


@pytest.mark.parametrize("first", [0, 1, 4, 5, 6, 9])
def test_refresh_from_block(dev, first):
    """K changed from a row of block `first` of 10 on: before, in and past the middle block."""
    import torch
    K = strip(105)
    ia, ja, a = (np.asarray(v) for v in K)
    p, b = len(ia) - 1, 128
    pr = dev.BandPreconditioner(K, block=b)
    assert pr.nblocks == 10
    r0 = first * b + 7 if first else 0
    rows = np.repeat(np.arange(p), np.diff(ia))
    K2 = (ia, ja, a * np.where((rows >= r0) & (ja - 1 >= r0), 1.3, 1.0))
    t = lambda v, d: torch.as_tensor(np.ascontiguousarray(v, dtype=d), device="cuda")
    pr.refactor(t(ia, np.int32), t(ja, np.int32), t(K2[2], np.float64), first_row=r0)
    check(dev, pr, K2, (6, 192), first)


def test_refactor_with_a_wider_band(dev):
    """A K whose couplings reach further than those the factor was built for, within its
    blocks: refactored and refreshed."""
    import scipy.sparse as sp
    import torch
    K = strip(120)
    p, b = len(K[0]) - 1, 256
    S = sp.csr_matrix((K[2], K[1] - 1, K[0] - 1), shape=(p, p))
    far = sp.diags([np.full(p - 200, -1.0)], [200], shape=(p, p))
    W = (S + far + far.T + sp.diags(np.full(p, 2.0))).tocsr()
    W.sort_indices()
    K2 = (W.indptr.astype(np.int32) + 1, W.indices.astype(np.int32) + 1, W.data)
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device="cuda")
    for first in (0, 300):
        pr = dev.BandPreconditioner(K, block=b)
        pr.refactor(*(t(v) for v in K2), first_row=first)
        check(dev, pr, K2, (3, 60), first)


def test_failed_refactor_keeps_the_factor(dev):
    """An indefinite K of a wider band is refused and the factor still solves with the old one;
    a good K afterwards refactors in place, several times."""
    import torch
    from xtfem_amd.api import XtError
    K = strip(60)
    ia, ja, a = (np.asarray(v) for v in K)
    t = lambda v, d: torch.as_tensor(np.ascontiguousarray(v, dtype=d), device="cuda")
    pr = dev.BandPreconditioner(K, block=256)
    p = len(ia) - 1
    bad = (np.arange(1, p + 2), np.arange(1, p + 1), np.full(p, -1.0))
    bad[0][p] += 1                       # last row: also couples 200 columns back
    bad = (bad[0], np.concatenate([bad[1][:-1], [p - 200, p]]), np.full(p + 1, -1.0))
    with pytest.raises(XtError, match="code -3"):
        pr.refactor(t(bad[0], np.int32), t(bad[1], np.int32), t(bad[2], np.float64))
    check(dev, pr, K, (6, 60), 1)
    for scale in (1.5, 0.7, 1.1):
        K2 = (ia, ja, a * scale)
        pr.refactor(t(ia, np.int32), t(ja, np.int32), t(K2[2], np.float64))
        check(dev, pr, K2, (6, 60), 2)
