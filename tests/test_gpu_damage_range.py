"""The damage kernel's quotients by reciprocals, its yield test on the squared stress and
the terms it keeps until the damage changes, bit for bit against the oracle's functor
(kokkos_kernel.h:44-344) where they could differ from it: displacements of zero, subnormal,
tiny and huge size next to ordinary ones in one wave, a damaged start, other fatigue limits,
and temporal tables of 1, 2 and 3 points."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS6 = ("eps_old", "eps_pl", "sig_eff", "sig_back")
SIZES = np.array([1.0, 0.0, 1e-311, 3e-303, 1e-150, 1e-6, 1e-2, 3.0, 1e60, 1e160, 1e305])


@pytest.fixture(scope="module")
def block():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from xtfem_amd import fem
    mesh = fem.structured_hex(11, 3, 2, 11.0, 3.0, 2.0)   # 528 points: the last wave is not full
    _, _, Nx, Ny, Nz = fem.assemble(mesh, 2.0e5, 0.3, 7.85e-9)
    return mesh, Nx, Ny, Nz


@pytest.mark.parametrize("nip", [1, 2, 3, 130])
@pytest.mark.parametrize("sigf", [180.0, 350.0, 1e-3, 1e200])
@pytest.mark.parametrize("order", ["mixed", "by wave"])
def test_damage_bitexact_over_the_range(block, oracle_lib, nip, sigf, order):
    from xtfem_amd import slab
    mesh, Nx, Ny, Nz = block
    ne, nn, ngp = mesh.ne, mesh.nn, 8 * mesh.ne
    params = np.array([sigf, 1.2 * sigf + 200.0, 0.08, 1740.0, 0.2, 0.5, 0.5])
    rng = np.random.default_rng(nip)
    # a displacement field of strains about 0.006; the points' derivatives carry the sizes
    x = mesh.xcoord
    sol = np.zeros((6, nn, 3))
    for k in range(6):
        w = rng.uniform(0.5, 1.0)
        sol[k, :, 0] = 0.006 * w * x[:, 0] * (1 + 0.3 * x[:, 1])
        sol[k, :, 1] = -0.002 * w * x[:, 1] + 0.001 * w * x[:, 0] ** 2
        sol[k, :, 2] = -0.002 * w * x[:, 2]
    e = np.arange(ne)
    size = SIZES[(e if order == "mixed" else e // 8) % len(SIZES)]
    scale = np.repeat(size, 8)[:, None]
    N = [(v.reshape(ngp, 8) * scale).ravel() for v in (Nx, Ny, Nz)]
    Nt = slab.damage_nt(np.array([0.0, 0.25, 0.5]), 2 * np.pi * 20, 130)[-nip:]
    state = {k: np.zeros(6 * ngp) for k in FIELDS6}
    state.update({k: np.zeros(ngp) for k in ("p", "D", "ws", "del_po", "sig_d")})
    state["D"][::3] = rng.uniform(0.0, 0.6, len(state["D"][::3]))      # damaged points
    state["D"][1::7] = -0.0
    state["ws"][::3] = params[2] * (params[1] - params[0])             # at the threshold
    state["sig_d"][:] = rng.uniform(0.0, 300.0, ngp)
    args = (ne, nn, nip, np.repeat(mesh.xconn, 8, axis=0).ravel(), *N, Nt.ravel(), sol.ravel(),
            np.full(ngp, 1.97e5), rng.uniform(0.0, 0.45, ngp))
    oracle_lib.damage_params(params)
    try:
        want = oracle_lib.kokkos_host(*args, state)
        want = oracle_lib.kokkos_host(*args, want)
    finally:
        oracle_lib.damage_params(None)
    got = _device(mesh, args, state, params)
    for k in want:
        assert np.array_equal(got[k], want[k], equal_nan=True), \
            (k, np.flatnonzero(~((got[k] == want[k]) | (np.isnan(got[k]) & np.isnan(want[k]))))[:8])


def _device(mesh, args, state, params):
    import torch
    from xtfem_amd._lib import check, lib
    ne, nn, nip = args[:3]
    dev = [torch.as_tensor(np.ascontiguousarray(a, dtype=np.int32 if i == 0 else np.float64),
                           device="cuda") for i, a in enumerate(args[3:])]
    st = {k: torch.as_tensor(v.copy(), device="cuda") for k, v in state.items()}
    keys = ("eps_old", "eps_pl", "sig_eff", "sig_back", "p", "D", "ws", "del_po", "sig_d")
    for _ in range(2):
        check(lib().xt_damage_device_params(ne, nn, nip, *[t.data_ptr() for t in dev],
                                            *[st[k].data_ptr() for k in keys],
                                            params.ctypes.data,
                                            torch.cuda.current_stream().cuda_stream), "damage")
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in st.items()}
