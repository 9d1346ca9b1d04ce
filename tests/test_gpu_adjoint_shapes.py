"""The fused adjoint directions against the per-stage adjoint kernels."""
import ctypes

import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

# Both sides evaluate the same sums in other orders: about 30 roundings of
# u = 2^-53 a stage, six stages, terms up to four times the result.
TOL = 30 * 6 * 4 * 2.0 ** -53


def _check(nx, nz, members, tuning):
    from pyminiweather_amd import _lib
    from pyminiweather_amd.data import initialize_fields
    from pyminiweather_amd.ics import init
    from pyminiweather_amd.mesh import MeshData
    from pyminiweather_amd.solve import hv_coeff
    ptr, st = _lib.ptr, _lib.stream_of()
    p = O.make_params(nx, nz, "collision", cfl=1.5, max_speed=450.0)
    f = initialize_fields(p)
    init(f, p, MeshData(p))
    g = torch.Generator(device="cpu").manual_seed(nx * 1000 + nz)
    scale = torch.tensor([1e-3, 2.0, 2.0, 0.5], dtype=torch.float64)[:, None, None]
    shape = (7, members) + tuple(f.shape)
    tape = (scale * torch.randn(shape, generator=g, dtype=torch.float64)).cuda() + f.state
    lam = torch.randn(shape[1:], generator=g, dtype=torch.float64).cuda()
    hy = (f.hy_dens_cell, f.hy_dens_theta_cell, f.hy_dens_int, f.hy_dens_theta_int)
    hvs = [hv_coeff(p[d], p["dt"]) for d in ("dx", "dz")]

    got, ws = lam.clone(), torch.empty_like(lam)
    _lib.call("pmw_tape_adjoint", ptr(tape), tape.numel(), members, ptr(got), ptr(ws),
              ws.numel(), *map(ptr, hy), nx, nz, p["dx"], p["dz"], p["dt"], hvs[0], hvs[1],
              0, 1, (ctypes.c_int * 2)(*tuning), st)
    for m in range(members):
        cur = lam[m].clone()
        for slot, d in ((3, 0), (0, 1)):  # z ran first: x is reversed first
            lams = [cur]
            for s, frac in ((2, 1), (1, 2), (0, 3)):
                out = torch.empty_like(cur)
                acc = lams if s == 0 else []
                acc = [ptr(q) for q in acc] + [None] * (3 - len(acc))
                _lib.call("pmw_adjoint_stage", d, ptr(tape[slot + s, m]), ptr(lams[-1]),
                          p["dt"] / frac, *acc, ptr(out), *map(ptr, hy), nx, nz,
                          p["dx"] if d == 0 else p["dz"], hvs[d], st)
                lams.append(out)
            cur = lams[-1]
        want = cur[:, 2:-2, 2:-2]
        err = (got[m][:, 2:-2, 2:-2] - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)
        assert torch.all(err <= TOL), f"member {m}: {err.tolist()}"


@pytest.mark.parametrize("tuning", [(256, 8512), (384, 8512)])
@pytest.mark.parametrize("nx", [2, 3, 36, 37, 49, 50, 51, 64, 100, 113, 114, 115, 229, 513])
def test_x_waves_match_stages(nx, tuning):
    """Rows shorter than a wave, of one wave's cells and one more or less,
    several rows and members per block, one and two cells per lane."""
    _check(nx, 5, 2, tuning)


@pytest.mark.parametrize("tuning", [(256, 8512), (256, 4256), (256, 2256)])
@pytest.mark.parametrize("nz", [2, 3, 4, 17, 18, 19, 36, 37, 49, 50, 51, 100, 101])
def test_z_tiles_match_stages(nz, tuning):
    """Columns of a few rows (both walls in one thread's reach), of one tile's
    rows and one more or less, of two tiles, with a ragged last column group."""
    _check(21, nz, 2, tuning)
