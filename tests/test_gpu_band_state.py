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


def test_scratch_is_kept_from_the_first_refactorization_on(dev):
    """A factor that is only built holds its matrices and no scratch; a second refactorization
    takes no more memory than the first.  The scratch is the diagonal and the sub-diagonal
    blocks in FP64, 16 bytes b^2 a block; memory is counted to half of it."""
    import torch
    b, nb = 1024, 24
    K = strip(nb * b // 12 - 2)
    small = dev.BandPreconditioner(strip(20))      # (the library's own first allocations)
    small.refactor(*on_device(strip(20)))
    torch.cuda.synchronize()
    Kd = on_device(K)

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    scratch = 16 * b * b * nb
    start = used()
    pr = dev.BandPreconditioner(K, block=b)
    assert pr.nblocks == nb
    built = used()
    # D and D^T in both precisions; G and H are narrow here (64 of 1024 columns)
    assert built - start < 24 * b * b * nb + scratch // 2
    pr.refactor(*Kd)
    once = used()
    assert once - built > scratch // 2
    pr.refactor(*Kd)
    assert used() - once < scratch // 8


def test_refactorizations_on_streams_that_come_and_go(dev):
    """Each refactorization on a stream of its own that is destroyed afterwards: what the
    factor keeps refers to none of them."""
    import ctypes as C
    import torch
    from xtfem_amd._lib import check as ok, lib
    hip = lib()                      # (its symbols include those of the runtime it links)
    K = strip(60)
    pr = dev.BandPreconditioner(K, block=128)
    for scale in (1.5, 0.7, 1.1):
        K2 = (K[0], K[1], K[2] * scale)
        ia, ja, a = on_device(K2)
        torch.cuda.synchronize()
        s = C.c_void_p()
        assert hip.hipStreamCreate(C.byref(s)) == 0
        ok(lib().xt_prec_refactor_band(pr.h, ia.data_ptr(), ja.data_ptr(), a.data_ptr(), s),
           "refactor")
        assert hip.hipStreamDestroy(s) == 0
        check(dev, pr, K2, (6, 60), 3)


@pytest.mark.parametrize("block,fp32", [(768, False), (64, True)])
def test_work_is_counted_on_the_band(dev, block, fp32):
    """Algorithmic bytes and flops of an apply without pairing levels against those of its
    launches (bytes within 2 %: the launches read the middle block's vector once for both
    chains and a chain's own vectors twice where its rows are split), and the bytes of the
    matrices: blocks of 768 rows with a band of 64, and blocks all band."""
    import ctypes as C
    import torch
    from xtfem_amd import tune
    from xtfem_amd._lib import check as ok, lib
    nb, c, kw = 9, 32, 64
    pr = dev.BandPreconditioner(strip(nb * block // 12 - 2), block=block)
    assert pr.nblocks == nb
    sv, dt = (4, torch.float32) if fp32 else (8, torch.float64)
    assert pr.matrix_bytes(fp32) == sv * (2 * nb * block * block + 2 * (nb - 1) * block * kw)
    x = torch.ones(pr.p * c, device="cuda", dtype=dt)
    y = torch.empty_like(x)
    kind = tune.XT_PROF_BAND if fp32 else tune.XT_PROF_BAND64
    v = [C.c_double() for _ in range(5)]
    n = C.c_longlong()
    tune.set_knob("band_pair", 1)
    try:
        ok(lib().xt_prof_enable(1 << kind))
        pr.apply(None, x, y, c, q=1, fp32=fp32)
        ok(lib().xt_prof_read(kind, C.addressof(v[0]), C.addressof(n), C.addressof(v[1]),
                              C.addressof(v[2])))
        ok(lib().xt_prof_read_alg(kind, C.addressof(v[3]), C.addressof(v[4])))
    finally:
        ok(lib().xt_prof_enable(0))
        tune.set_knob("band_pair", 0)
    _, byts, flops, alg_bytes, alg_flops = (u.value for u in v)
    assert alg_flops == pytest.approx(flops, rel=1e-9)
    assert alg_bytes == pytest.approx(byts, rel=0.02)


@pytest.mark.parametrize("row", [5, 300, 640, 700, 1271, 1280])
def test_indefinite_row_is_named(dev, row):
    """An uncoupled row with a negative diagonal (0-based; blocks of 128, the middle block
    from 640 on) is named in K's order, whichever end its elimination starts from."""
    from xtfem_amd.api import XtError
    ia, ja, a = strip(106)
    p = len(ia) - 1
    assert p == 1284
    rows = np.repeat(np.arange(p), np.diff(ia))
    hit = (rows == row) | (ja - 1 == row)
    a = np.where(hit, np.where(rows == ja - 1, -1.0, 0.0), a)
    with pytest.raises(XtError, match=rf"code -3.*elimination of row {row}\)"):
        dev.BandPreconditioner((ia, ja, a), block=128)
