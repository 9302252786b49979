"""The ILUT sweeps of two columns a workgroup (results that are their own flags, the last
entry of a row kept apart, 32 entries a slot and longer rows behind them) and their
neighbours in the dispatch (a barrier a level, a launch a level) against the substitution of
lusol (ilut.f:2383-2432) on the host: sizes at the ends of the slots' range, odd column
counts, rows without entries, full rows, wide levels, NaN and infinities."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device
    return device


def _factor(n, kind, rng):
    """L (strictly lower), U (strictly upper) and the inverse diagonal, rows of small sum."""
    L, U = {}, {}
    for i in range(n):
        if kind == "chain":          # one level a row, up to 18 entries
            lo = range(max(0, i - 18), i)
            hi = range(i + 1, min(n, i + 19))
        elif kind == "wide":         # two levels
            lo = range(0, min(i, 1) if i % 2 else 0)
            hi = range(n - 1, n) if i < n - 1 and i % 3 == 0 else range(0)
        else:                        # long rows (32, 33, 34 and all entries) among short ones
            k = {0: 32, 1: 33, 2: 34, 3: n}.get(i % 11, 2)
            lo = sorted(rng.choice(i, min(i, k), replace=False)) if i else []
            m = n - 1 - i
            hi = sorted(i + 1 + rng.choice(m, min(m, k), replace=False)) if m else []
        lo, hi = list(lo), list(hi)
        L[i] = (lo, rng.uniform(-1, 1, len(lo)) / max(len(lo), 1))
        U[i] = (hi, rng.uniform(-1, 1, len(hi)) / max(len(hi), 1))
    return L, U, rng.uniform(0.5, 1.0, n)


def _msr(L, U, dinv):
    n = len(dinv)
    size = n + 1 + sum(len(L[i][0]) + len(U[i][0]) for i in range(n))
    alu, jlu, ju = np.zeros(size), np.zeros(size, np.int32), np.zeros(n, np.int32)
    alu[:n] = dinv
    at = n + 1
    for i in range(n):
        jlu[i] = at + 1
        for cols, vals, up in ((*L[i], False), (*U[i], True)):
            if up:
                ju[i] = at + 1
            alu[at:at + len(cols)] = vals
            jlu[at:at + len(cols)] = np.array(cols, np.int32) + 1
            at += len(cols)
    jlu[n] = at + 1
    return alu, jlu, ju


def _solve(L, U, dinv, b, fabs=False):
    """The two substitutions; fabs: of absolute values, sums added (an error's growth)."""
    n = len(dinv)
    x = b.copy()
    for i in range(n):
        c, v = L[i]
        if len(c):
            x[i] = x[i] + abs(v) @ x[c] if fabs else x[i] - v @ x[c]
    for i in range(n - 1, -1, -1):
        c, v = U[i]
        if len(c):
            x[i] = x[i] + abs(v) @ x[c] if fabs else x[i] - v @ x[c]
        x[i] = dinv[i] * x[i]
    return x


def _apply(dev, msr, b, fp32):
    import ctypes as C
    import torch
    from xtfem_amd._lib import check, lib
    n, c = b.shape
    h = C.c_void_p()
    check(lib().xt_prec_create(n, *[a.ctypes.data for a in msr], C.addressof(h)), "prec_create")
    try:
        dt = torch.float32 if fp32 else torch.float64
        x = torch.as_tensor(b, device="cuda").to(dt).contiguous()
        y = torch.full_like(x, 7.0)
        check(lib().xt_prec_apply(h, c, 1, None, x.data_ptr(), y.data_ptr(), int(fp32),
                                  torch.cuda.current_stream().cuda_stream), "prec_apply")
        torch.cuda.synchronize()
        return y.double().cpu().numpy()
    finally:
        lib().xt_prec_destroy(h)


@pytest.mark.parametrize("n,kind", [(1, "chain"), (2, "chain"), (40, "long"), (257, "chain"),
                                    (600, "long"), (1500, "wide"), (4096, "chain"),
                                    (4097, "chain")])
def test_ilut_sweeps_match_the_substitution(dev, n, kind):
    rng = np.random.default_rng(n)
    L, U, dinv = _factor(n, kind, rng)
    msr = _msr(L, U, dinv)
    width = 1 + max(max(len(L[i][0]), len(U[i][0])) for i in range(n))
    for c in (1, 2, 3, 6, 13, 64):
        if n > 4000 and c > 13:
            continue
        b = rng.standard_normal((n, c))
        for fp32, eps in ((False, 2.0 ** -53), (True, 2.0 ** -24)):
            b0 = b.astype(np.float32).astype(float) if fp32 else b
            ref = _solve(L, U, dinv, b0)
            # backward error of the substitutions: each result's terms off by width + 4
            # roundings (entries rounded once more in FP32), carried on by the absolute values
            grow = _solve(L, U, dinv, abs(b0), True)
            bound = 2 * (width + 6) * eps * _solve(L, U, dinv, _solve(L, U, dinv, abs(b0), True), True)
            y = _apply(dev, msr, b0, fp32)
            assert (abs(y - ref) <= bound + (width + 6) * eps * grow).all(), \
                (c, fp32, float((abs(y - ref) / bound).max()))


def test_ilut_sweeps_not_finite(dev):
    rng = np.random.default_rng(5)
    L, U, dinv = _factor(300, "chain", rng)
    msr = _msr(L, U, dinv)
    b = rng.standard_normal((300, 6))
    # a NaN of any payload and an infinity end the column they stand in, no other
    b[150, 1] = np.inf
    b[20, 3] = np.array([0x7FFADEAD00000000], np.uint64).view(np.float64)[0]
    y, z = _apply(dev, msr, b, False), _apply(dev, msr, np.nan_to_num(b), False)
    assert np.isnan(y[:, 3]).all() and not np.isfinite(y[150, 1])
    keep = [0, 2, 4, 5]
    assert np.array_equal(y[:, keep], z[:, keep])
