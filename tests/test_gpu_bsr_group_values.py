"""When the node groups of the SpMM (XT_TUNE_SPMM_GROUP) hold values of their own: only from
the first apply that takes them, per precision; kept up to date by set_values; and a first
apply under graph capture, which may not allocate, takes the slices."""
import numpy as np
import pytest

from test_gpu_bsr_group import _blocks, _check, _operator

pytestmark = pytest.mark.gpu


@pytest.fixture
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, tune
    yield device
    tune.set_knob("spmm_group", 0)


def _used():
    import torch
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_values_only_where_the_groups_run(dev):
    """A second copy of the values is 96 bytes a block in FP64 and 48 in FP32; memory is
    counted to a third of that."""
    import torch
    from xtfem_amd import tune
    rng = np.random.default_rng(0)
    tune.set_knob("spmm_group", 2)
    K, M = _blocks(37, "banded", rng)
    for f in (False, True):                           # (the kernels' own first launches)
        _check(dev, _operator(dev, K, M), K, M, 2, f, rng)
    op = _operator(dev, *_blocks(120000, "banded", rng))
    n = 9 * 120000 - 2 * (1 + 2 + 16 + 17)            # blocks
    x = {f: torch.ones(360000 * 12, device="cuda", dtype=torch.float32 if f else torch.float64)
         for f in (False, True)}
    y = {f: torch.empty_like(v) for f, v in x.items()}
    T = {f: op.tmat(rng.standard_normal((2, 2, 6, 6)), f) for f in (False, True)}
    apply = lambda f: op.apply(T[f], x[f], y[f], 2, fp32=f)
    tune.set_knob("spmm_group", 1)
    for f in (False, True):
        apply(f)
    slices = _used()
    tune.set_knob("spmm_group", 2)
    for f, size in ((False, 96 * n), (True, 48 * n)):
        before = _used()
        apply(f)
        assert _used() - before > size * 2 // 3
        apply(f)
        assert _used() - before < size * 4 // 3
    assert _used() - slices < 144 * n * 4 // 3


def test_new_values_reach_groups_in_use(dev):
    import torch
    from xtfem_amd import tune
    rng = np.random.default_rng(1)
    K, M = _blocks(262, "irregular", rng)
    op = _operator(dev, K, M)
    tune.set_knob("spmm_group", 2)
    for _ in range(3):
        for fp32 in (False, True):
            _check(dev, op, K, M, 9, fp32, rng)
        K.data, M.data = rng.standard_normal(K.nnz), rng.standard_normal(M.nnz)
        op.set_values(torch.as_tensor(K.data, device="cuda"), torch.as_tensor(M.data, device="cuda"))
    for fp32 in (False, True):
        _check(dev, op, K, M, 9, fp32, rng)


@pytest.mark.parametrize("warm", [False, True])
def test_captured_applies_follow_new_values(dev, warm):
    """Captured before the groups hold values (the slices run) and after; replays see the
    values that set_values wrote in between."""
    import torch
    from xtfem_amd import tune
    rng = np.random.default_rng(2)
    K, M = _blocks(262, "banded", rng)
    op = _operator(dev, K, M)
    tune.set_knob("spmm_group", 2)
    R = 9
    A = rng.standard_normal((R, 2, 6, 6))
    T = op.tmat(A, False)
    x = torch.as_tensor(rng.standard_normal((786, R, 6)), device="cuda")
    y = torch.empty_like(x)
    if warm:
        op.apply(T, x, y, R)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.apply(T, x, y, R)
    for _ in range(3):
        K.data, M.data = rng.standard_normal(K.nnz), rng.standard_normal(M.nnz)
        op.set_values(torch.as_tensor(K.data, device="cuda"), torch.as_tensor(M.data, device="cuda"))
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        X = x.cpu().numpy().reshape(786, R * 6)
        form = lambda K, M, A, X: sum(
            np.einsum("rij,prj->pri", A[:, t], (S @ X).reshape(786, R, 6))
            for t, S in enumerate((K, M)))
        bound = (9 * 3 + 20) * 2.0 ** -53 * form(abs(K), abs(M), abs(A), abs(X))
        assert (np.abs(y.cpu().numpy() - form(K, M, A, X)) <= bound).all()
        _check(dev, op, K, M, R, False, rng)           # (an eager apply in between)
