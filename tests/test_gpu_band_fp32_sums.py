"""How the FP32 sweeps with few columns add up a row.  K = L L^T with L = 1 on the diagonal and
-1 below it, so D = L^-1 is all ones, exactly, and the last entry of K^-1 x is the sum of x:
one large entry, 1, and the others 2^-27, which are lost where they are added to it in FP32
(also four at a time).  Of the 4096 entries a wave of `waves` takes a share, in four sums, so
at most 4096 / waves / 4 - 1 are lost, an eighth of a unit roundoff u = 2^-24 each; three more
roundings follow and one is kept for the result.  (One sum a wave loses four times as many.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [1, 6, 16])
@pytest.mark.parametrize("waves,knobs", [(8, dict(band_smallc=1)), (4, dict(band_smallc=2)),
                                         (4, dict(band_smallc=1, band_chain_few=2))])
def test_small_entries_are_not_lost_to_one_large(waves, knobs, columns):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, tune
    p = 4096
    rows = np.repeat(np.arange(p), [1] + [2] * (p - 1))
    ia = np.concatenate([[0], np.cumsum(np.bincount(rows))]) + 1
    ja = np.concatenate([[0]] + [[i - 1, i] for i in range(1, p)]) + 1
    a = np.concatenate([[1.0]] + [[-1.0, 2.0]] * (p - 1))
    pr = device.BandPreconditioner((ia, ja, a), block=p)
    assert pr.nblocks == 1
    x = torch.full((p, columns), 2.0 ** -27, device="cuda", dtype=torch.float32)
    x[0] = 1.0
    y = torch.empty_like(x)
    try:
        for k, v in knobs.items():
            tune.set_knob(k, v)
        pr.apply(None, x, y, columns, q=1, fp32=True)
    finally:
        for k in knobs:
            tune.set_knob(k, 0)
    want = 1.0 + (p - 1) * 2.0 ** -27
    err = np.abs(y[-1].double().cpu().numpy() - want).max() / 2.0 ** -24
    assert err <= (p // waves // 4 - 1) / 8 + 4, err
