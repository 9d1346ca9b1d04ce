"""Kernels that the rules by size choose for few grids, against the per-stage
kernels bit for bit."""
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def _tiles(nx, nz, waves):
    """Three-row z tiles of a grid (zt_tiles and zt_blocks, pmw_fused.hip)."""
    c, ce = 12 * waves - 12, 12 * waves - 8
    return (nx + 15) // 16 * (2 if nz <= 2 * ce else 2 + (nz - 2 * ce + c - 1) // c)


def _eight_waves(grids):
    """The choice of zt_waves for one launch over these grids."""
    cost = [w + -(-w // 4096) * 4096
            for w in (k * sum(_tiles(nx, nz, k) for nx, nz in grids) for k in (4, 8))]
    return min(nz for _, nz in grids) >= 94 and 10 * cost[0] > 11 * cost[1]


def _fields(p):
    from pyminiweather_amd.data import initialize_fields
    from pyminiweather_amd.ics import init
    from pyminiweather_amd.mesh import MeshData
    f = initialize_fields(p, intermediates=False)
    init(f, p, MeshData(p))
    return f


def _disturb(f, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    for v, scale in enumerate((1e-3, 2.0, 2.0, 0.5)):
        f.state[v] += scale * torch.randn(f.state.shape[1:], dtype=torch.float64, device="cuda",
                                          generator=g)


def _staged(p, start, start_tmp, steps):
    """State and state_tmp after `steps` steps of one launch per RK stage."""
    f = _fields(p)
    f.state.copy_(start)
    f.state_tmp.copy_(start_tmp)
    return _run(p, f, (1, 512, 8096), steps)


def _run(p, f, tuning, steps):
    import pyminiweather_amd.solve as S
    S.set_tuning(f.nx, f.nz, tuning)
    S.reverse_direction = False
    try:
        S.run(p, f, None, steps)
    finally:
        S._tuning_table.clear()
        S.reverse_direction = False
    return f.state, f.state_tmp


def _same(got, want):
    assert all(bool(torch.isfinite(w).all()) for w in want)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


EIGHT = [((1601, 400),), ((1601, 400), (37, 94), (1876, 261)),
         tuple([(800, 400)] * 3 + [(400, 200)] * 2 + [(203, 101)] * 4)]


@pytest.mark.parametrize("grids", EIGHT, ids=str)
def test_ensemble_of_eight_wave_tiles(grids):
    """Members lists whose launch takes z tiles of eight waves: one member, uneven
    ones with columns of the tiles' smallest height, many."""
    from pyminiweather_amd.ensemble import Ensemble
    assert _eight_waves(grids) and sum(nx * nz for nx, nz in grids) > 300000
    params = [O.make_params(nx, nz, "thermal", cfl=0.8, max_speed=450.0) for nx, nz in grids]
    ens = Ensemble(params)
    for q, f in enumerate(ens.fields):
        _disturb(f, q)
    starts = [(f.state.clone(), f.state_tmp.clone()) for f in ens.fields]
    ens.evolve(2)
    for p, f, s in zip(params, ens.fields, starts):
        _same((f.state, f.state_tmp), _staged(p, *s, 2))


# above 300000 cells three-row tiles need columns of 46 rows and rows below 2^22
# cells; others take one-cell tiles of 96 rows (from 41 rows on) or of 32
@pytest.mark.parametrize("nx,nz", [(7400, 41), (6701, 45), (7700, 40), ((1 << 22) - 1, 46),
                                   (1 << 22, 46)])
def test_one_cell_tiles_of_large_grids(nx, nz):
    p = O.make_params(nx, nz, "thermal", cfl=0.8, max_speed=450.0)
    f = _fields(p)
    _disturb(f, nx + nz)
    start = f.state.clone(), f.state_tmp.clone()
    got = _run(p, f, (0, 512, 8096), 2)
    _same(got, _staged(p, *start, 2))


@pytest.mark.parametrize("grids", [((7400, 41), (150, 200)), ((2100, 45), (1999, 96), (60, 300)),
                                   ((900, 20), (1000, 300))], ids=str)
def test_ensemble_of_one_cell_tiles(grids):
    """The lowest member's 41 to 45 rows decide for all of them: tiles of 96 rows
    also for members that are higher; 20 rows: tiles of 32."""
    from pyminiweather_amd.ensemble import Ensemble
    assert sum(nx * nz for nx, nz in grids) > 300000
    params = [O.make_params(nx, nz, "thermal", cfl=0.8, max_speed=450.0) for nx, nz in grids]
    ens = Ensemble(params)
    for q, f in enumerate(ens.fields):
        _disturb(f, q)
    starts = [(f.state.clone(), f.state_tmp.clone()) for f in ens.fields]
    ens.evolve(2)
    for p, f, s in zip(params, ens.fields, starts):
        _same((f.state, f.state_tmp), _staged(p, *s, 2))
