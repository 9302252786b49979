"""Sweeps of more rows and cases than one launch has threads (2^32): the vectors go to and from
the factor's order in several launches."""
import numpy as np
import pytest

from test_gpu_band_twisted import lu, strip

pytestmark = pytest.mark.gpu


def test_more_rows_and_cases_than_a_launch_holds():
    """65544 rows with 65536 columns, sixteen of them in turn: the first sixteen against the
    sparse LU (cond(K) about 1e3: FP32 agrees to 1e-3), the others equal to them."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    K = strip(5461)
    p, n = len(K[0]) - 1, 65536
    assert p * n >= 2 ** 32
    if torch.cuda.mem_get_info()[0] < 5 * 4 * p * n:
        pytest.skip("needs 86 GB of device memory")
    pr = device.BandPreconditioner(K, fp32_only=True)
    X = np.random.default_rng(0).standard_normal((p, 16))
    x = torch.as_tensor(X, device="cuda").float().repeat(1, n // 16)
    y = torch.full_like(x, float("nan"))
    pr.apply(None, x, y, n, q=1, fp32=True)
    first = y[:, :16].clone()
    want = lu(K).solve(X)
    assert np.abs(first.double().cpu().numpy() - want).max() < 1e-3 * np.abs(want).max()
    y = y.view(p, n // 16, 16)
    for r in range(0, p, 4096):
        assert (y[r:r + 4096] == first[r:r + 4096, None]).all()
    del x, y
    torch.cuda.empty_cache()


@pytest.mark.parametrize("cases", [1, 7])
def test_few_cases_take_one_launch_each_way(cases):
    """The nodes of a captured apply on 12012 rows: a launch each way and those of the sweeps,
    not one for every row."""
    import ctypes as C
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    from xtfem_amd._lib import check, lib
    hip = lib()                           # (its symbols include those of the runtime it links)
    pr = device.BandPreconditioner(strip(1000), block=512)
    x = torch.ones((pr.p, cases), device="cuda", dtype=torch.float64)
    y = torch.empty_like(x)
    pr.apply(None, x, y, cases, q=1)      # (sizes the workspace)
    torch.cuda.synchronize()
    s, graph, n = C.c_void_p(), C.c_void_p(), C.c_size_t(0)
    assert hip.hipStreamCreate(C.byref(s)) == 0
    assert hip.hipStreamBeginCapture(s, 1) == 0            # thread-local
    check(lib().xt_prec_apply(pr.h, cases, 1, None, x.data_ptr(), y.data_ptr(), 0, s))
    assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(s) == 0
    assert 4 <= n.value < 100
