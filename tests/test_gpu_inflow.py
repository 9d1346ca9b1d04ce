"""The injection inflow's fused x direction against the per-stage kernels."""
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
    f.state += torch.from_numpy(start[0]).cuda()
    f.state_tmp += torch.from_numpy(start[1]).cuda()
    flag = ctypes.c_int(0)
    _lib.call("pmw_evolve_ex", ptr(f.state), ptr(f.state_tmp), ptr(f.state_work),
              ptr(f.hy_dens_cell), ptr(f.hy_dens_theta_cell), ptr(f.hy_dens_int),
              ptr(f.hy_dens_theta_int), ptr(f.hy_pressure_int), None, 1, ptr(f.inj_rows),
              f.nx, f.nz, p["dx"], p["dz"], p["dt"], S.hv_coeff(p["dx"], p["dt"]),
              S.hv_coeff(p["dz"], p["dt"]), ctypes.byref(flag), nsteps,
              (ctypes.c_int * 3)(*tuning), _lib.stream_of(), None)
    torch.cuda.synchronize()
    return f.state.cpu().numpy(), f.state_tmp.cpu().numpy()


@pytest.mark.parametrize("nx,nz", [(15, 9), (16, 9), (17, 40), (41, 20), (102, 33), (112, 33),
                                   (113, 21), (1003, 117)])
@pytest.mark.parametrize("tuning", [(0, 256, 8096), (0, 1512, 8096), (0, 512, 18096)])
def test_fused_inflow_bitwise_equals_per_stage(nx, nz, tuning):
    """From random states whose halos are nonzero and differ between state
    and state_tmp, three steps of the fused directions leave both buffers
    whole (halos and corners too) as one launch per RK stage does: rows below
    and at the fused minimum, rows of just one wave window and one more, odd
    rows, several waves per row."""
    p = O.make_params(nx, nz, "injection", cfl=1.0, max_speed=450.0)
    rng = np.random.default_rng(nx * 1000 + nz)
    scale = np.array([1e-3, 2.0, 2.0, 0.5])[:, None, None]
    start = [scale * rng.standard_normal((4, nz + 4, nx + 4)) for _ in range(2)]
    want = _run(p, start, (1, 256, 8096), 3)
    got = _run(p, start, tuning, 3)
    assert all(np.all(np.isfinite(w)) for w in want)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
