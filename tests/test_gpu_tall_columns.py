"""Fused directions over columns up to the top of their background, and with
arguments outside the power's table in the two-cell inflow waves."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def _run(p, spots, tuning):
    import pyminiweather_amd.solve as S
    from pyminiweather_amd import _lib
    from pyminiweather_amd._lib import ptr
    from pyminiweather_amd.data import initialize_fields
    from pyminiweather_amd.ics import init
    from pyminiweather_amd.mesh import MeshData
    f = initialize_fields(p)
    init(f, p, MeshData(p))
    for k, i, v in spots:
        f.state[3, k + 2, i + 2] += v
    inj = p["ic_type"] == "injection"
    flag = ctypes.c_int(1)  # x first
    _lib.call("pmw_evolve_ex", ptr(f.state), ptr(f.state_tmp), ptr(f.state_work),
              ptr(f.hy_dens_cell), ptr(f.hy_dens_theta_cell), ptr(f.hy_dens_int),
              ptr(f.hy_dens_theta_int), ptr(f.hy_pressure_int), None, int(inj),
              ptr(f.inj_rows) if inj else None, f.nx, f.nz, p["dx"], p["dz"], p["dt"],
              S.hv_coeff(p["dx"], p["dt"]), S.hv_coeff(p["dz"], p["dt"]), ctypes.byref(flag),
              2, (ctypes.c_int * 3)(*tuning), _lib.stream_of(), None)
    torch.cuda.synchronize()
    return f.state.cpu().numpy(), f.state_tmp.cpu().numpy()


def _check(p, spots, tunings):
    want = _run(p, spots, (1, 512, 8096))
    assert all(np.isfinite(w).mean() > 0.8 for w in want)
    for tuning in tunings:
        got = _run(p, spots, tuning)
        np.testing.assert_array_equal(got[0], want[0], err_msg=str(tuning))
        np.testing.assert_array_equal(got[1], want[1], err_msg=str(tuning))


@pytest.mark.parametrize("nx,nz,ic", [(130, 60, "collision"), (130, 60, "injection"),
                                      (600, 130, "gravity"), (3301, 95, "thermal"),
                                      (700, 450, "injection"), (2717, 260, "collision")])
@pytest.mark.parametrize("zlen", [2.0e4, 2.8e4, 3.05e4])
def test_tall_columns_bitwise_equal_per_stage(nx, nz, ic, zlen):
    """Two short steps; 30.5 km lie below the table's last entry at the top, so
    whole waves and tiles there take the general power; where the halo rows above
    them have no pressure left their NaNs are in the same places."""
    p = O.make_params(nx, nz, ic, cfl=0.02, max_speed=450.0, zlen=zlen)
    _check(p, (), [(0, x, 8096) for x in (256, 512, 1512)])


@pytest.mark.parametrize("nx,nz", [(130, 20), (113, 21), (1003, 301)])
def test_rare_powers_in_inflow_waves(nx, nz):
    """Cells whose rho*theta exceeds the table beside the inflow, in the middle of
    a row and at its end: the wave runs again from the halos that its first run
    read, with one and with two cells per lane."""
    p = O.make_params(nx, nz, "injection", cfl=0.05, max_speed=450.0)
    rows = [k for k in (nz // 2, int(nz * 0.75), nz - 1)]
    spots = [(k, i, 1200.0) for k in rows for i in (1, nx // 2, nx - 1)]
    _check(p, spots, [(0, 256, 8096), (0, 1512, 8096)])
