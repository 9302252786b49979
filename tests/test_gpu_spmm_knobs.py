"""Which SpMM kernel the tuning knobs select: with the node groups asked for
(XT_TUNE_SPMM_GROUP 2) the LDS-staged kernel (XT_TUNE_SPMM_LDS 2) is not taken, so the
autotuner, which leaves the better of lds 1 and 2 set, times the groups themselves.  The two
kernels add a row's products in different orders, so random values tell them apart."""
import numpy as np
import pytest

from test_gpu_bsr_group import _blocks, _operator

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
def test_groups_asked_for_are_taken_before_the_staged_kernel(fp32):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import device, tune
    rng = np.random.default_rng(3)
    R, dt = 8, torch.float32 if fp32 else torch.float64
    op = _operator(device, *_blocks(37, "banded", rng))
    T = op.tmat(rng.standard_normal((R, 2, 6, 6)), fp32)
    x = torch.as_tensor(rng.standard_normal((111, 6 * R)), device="cuda").to(dt).contiguous()

    def apply(lds, group):
        tune.set_knob("spmm_lds", lds)
        tune.set_knob("spmm_group", group)
        y = torch.full_like(x, float("nan"))
        op.apply(T, x, y, R, fp32=fp32)
        return y
    try:
        groups, staged, both = apply(1, 2), apply(2, 1), apply(2, 2)
    finally:
        tune.set_knob("spmm_lds", 0)
        tune.set_knob("spmm_group", 0)
    assert not torch.equal(groups, staged)
    assert torch.equal(both, groups)
