"""The z tiles and column waves against the per-stage kernels, bit for bit."""
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
    f.state_tmp += start.flip(1)
    flag = ctypes.c_int(0)
    src = ptr(f.src_w) if p["ic_type"] == "gravity" else None
    _lib.call("pmw_evolve_ex", ptr(f.state), ptr(f.state_tmp), ptr(f.state_work),
              ptr(f.hy_dens_cell), ptr(f.hy_dens_theta_cell), ptr(f.hy_dens_int),
              ptr(f.hy_dens_theta_int), ptr(f.hy_pressure_int), src, 0, None,
              f.nx, f.nz, p["dx"], p["dz"], p["dt"], S.hv_coeff(p["dx"], p["dt"]),
              S.hv_coeff(p["dz"], p["dt"]), ctypes.byref(flag), nsteps,
              (ctypes.c_int * 3)(*tuning), _lib.stream_of(), None)
    torch.cuda.synchronize()
    return f.state.cpu().numpy(), f.state_tmp.cpu().numpy()


# just over 300000 cells: four-wave tiles from their smallest column (46 rows),
# two to three tiles a column (80 / 81 rows), past the eight-wave tiles'
# smallest (94); then sizes whose eight-wave tiles fill the GPU's last round:
# two tiles of 96 rows exactly, three, five; the last column tile is ragged
@pytest.mark.parametrize("nx,nz", [(6547, 46), (6451, 47), (3877, 80), (3829, 81), (3301, 94),
                                   (3265, 95), (8190, 176), (8177, 171), (2717, 260),
                                   (2719, 261), (1601, 400)])
@pytest.mark.parametrize("ic", ["collision", "gravity"])
def test_three_row_tiles_bitwise_equal_per_stage(nx, nz, ic):
    """Two steps from random states with nonzero halos: state and state_tmp
    whole, halos and corners included."""
    p = O.make_params(nx, nz, ic, cfl=1.0, max_speed=450.0)
    g = torch.Generator(device="cuda").manual_seed(nx * 1000 + nz)
    scale = torch.tensor([1e-3, 2.0, 2.0, 0.5], dtype=torch.float64, device="cuda")
    start = scale[:, None, None] * torch.randn((4, nz + 4, nx + 4), dtype=torch.float64,
                                               device="cuda", generator=g)
    want = _run(p, start, (1, 256, 8096), 2)
    got = _run(p, start, (0, 512, 8096), 2)
    assert all(np.all(np.isfinite(w)) for w in want)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])


# one wave per column up to 60 rows, two to 112, then one more every 52; up to
# 512 waves share nothing, up to 4096 pass their columns through LDS four by
# four (the last group ragged), 4097 are one too many
@pytest.mark.parametrize("nx,nz", [(17, nz) for nz in (2, 3, 4, 57, 58, 59, 60, 61, 62, 63, 111,
                                                       112, 113, 164, 165, 217)] +
                         [(2, 9), (3, 70), (512, 60), (513, 60), (307, 61), (515, 113), (271, 217),
                          (4096, 60), (4097, 60)])
@pytest.mark.parametrize("ic", ["collision", "gravity"])
def test_column_waves_bitwise_equal_per_stage(nx, nz, ic):
    """Three steps from random states with nonzero halos, as above."""
    p = O.make_params(nx, nz, ic, cfl=1.0, max_speed=450.0)
    g = torch.Generator(device="cuda").manual_seed(nx * 1000 + nz)
    scale = torch.tensor([1e-3, 2.0, 2.0, 0.5], dtype=torch.float64, device="cuda")
    start = scale[:, None, None] * torch.randn((4, nz + 4, nx + 4), dtype=torch.float64,
                                               device="cuda", generator=g)
    want = _run(p, start, (1, 256, 8096), 3)
    got = _run(p, start, (0, 512, 8096), 3)
    assert all(np.all(np.isfinite(w)) for w in want)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
