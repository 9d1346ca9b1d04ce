"""Fused directions with rho*theta outside the power's table (64 .. 1024)."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def _run(p, start, tuning, nsteps):
    import pyminiweather_amd.solve as S
    from pyminiweather_amd import _lib
    from pyminiweather_amd._lib import ptr
    from pyminiweather_amd.data import initialize_fields
    from pyminiweather_amd.ics import init
    from pyminiweather_amd.mesh import MeshData
    f = initialize_fields(p)
    init(f, p, MeshData(p))
    f.state += start
    inj = p["ic_type"] == "injection"
    flag = ctypes.c_int(0)
    _lib.call("pmw_evolve_ex", ptr(f.state), ptr(f.state_tmp), ptr(f.state_work),
              ptr(f.hy_dens_cell), ptr(f.hy_dens_theta_cell), ptr(f.hy_dens_int),
              ptr(f.hy_dens_theta_int), ptr(f.hy_pressure_int), None, int(inj),
              ptr(f.inj_rows) if inj else None, f.nx, f.nz, p["dx"], p["dz"], p["dt"],
              S.hv_coeff(p["dx"], p["dt"]), S.hv_coeff(p["dz"], p["dt"]), ctypes.byref(flag),
              nsteps, (ctypes.c_int * 3)(*tuning), _lib.stream_of(), None)
    torch.cuda.synchronize()
    return f.state.cpu().numpy(), f.state_tmp.cpu().numpy()


@pytest.mark.parametrize("nx,nz,ic", [(60, 40, "collision"), (130, 20, "injection"),
                                      (700, 120, "collision"), (2000, 180, "collision"),
                                      (2717, 260, "collision")])
@pytest.mark.parametrize("value", [1500.0, 30.0])
def test_rare_powers_bitwise_equal_per_stage(nx, nz, ic, value):
    """One cell whose rho*theta lies in another binade than the table's, in the
    middle of waves and tiles, at a wall and at the row's ends: states after one
    short step equal the per-stage kernels' bit for bit (waves and tiles of
    every size, most of which hold no such cell). Near the top 30 makes
    rho*theta negative: its NaNs have to be in the same places."""
    p = O.make_params(nx, nz, ic, cfl=0.05, max_speed=450.0)
    start = torch.zeros((4, nz + 4, nx + 4), dtype=torch.float64, device="cuda")
    for k, i in ((nz // 2, nx // 2), (0, 3), (nz - 1, nx - 1), (nz // 3, 0)):
        start[3, k + 2, i + 2] = value - 300.0
    want = _run(p, start, (1, 256, 8096), 1)
    got = _run(p, start, (0, 512, 8096), 1)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])


def test_rare_powers_in_an_ensemble_bitwise_equal_single():
    """Members of the large z tiles, one with such a cell."""
    import pyminiweather_amd.solve as S
    from pyminiweather_amd.ensemble import Ensemble
    params = [O.make_params(nx, nz, "thermal", cfl=0.05, max_speed=450.0)
              for nx, nz in ((800, 400), (400, 200), (400, 100))]
    ens = Ensemble(params)
    ens.fields[1].state[3, 102, 202] = 1200.0
    singles = [f.state.clone() for f in ens.fields]
    ens.evolve(2)
    for p, f, s in zip(params, ens.fields, singles):
        from pyminiweather_amd.data import initialize_fields
        from pyminiweather_amd.ics import init
        from pyminiweather_amd.mesh import MeshData
        g = initialize_fields(p)
        init(g, p, MeshData(p))
        g.state.copy_(s)
        S.reverse_direction = False
        S.run(p, g, None, 2)
        assert torch.all(torch.isfinite(g.state))
        np.testing.assert_array_equal(f.state[:, 2:-2, 2:-2].cpu().numpy(),
                                      g.state[:, 2:-2, 2:-2].cpu().numpy())
    S.reverse_direction = False
