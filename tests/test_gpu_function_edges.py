"""The per-function kernels at the edges of their threads' rows."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(2, 2), (3, 6), (5, 7), (2, 8), (255, 9), (256, 14), (257, 15),
                                   (33, 16), (1000, 3)])
def test_per_function_chain_bitwise_equals_fused_stage(nx, nz):
    """Interpolation of both directions against the four taps bit for bit
    (columns of one thread's faces and one more or less), and discrete_step by
    functions against the fused stage, also where the output is the forcing."""
    import pyminiweather_amd.solve as S
    from pyminiweather_amd.data import initialize_fields
    from pyminiweather_amd.ics import Directions, init, set_bc_x, set_bc_z
    from pyminiweather_amd.mesh import MeshData
    p = O.make_params(nx, nz, "collision", cfl=1.0, max_speed=450.0)
    f = initialize_fields(p)
    init(f, p, MeshData(p))
    rng = np.random.default_rng(nx * 100 + nz)
    scale = np.array([1e-3, 2.0, 2.0, 0.5])[:, None, None]
    start = f.state + torch.from_numpy(scale * rng.standard_normal(f.shape)).cuda()

    s = start.clone()
    set_bc_x(p, f, s, "collision")
    set_bc_z(p, f, s, "collision")
    S.interpolate_x(p, f, s)
    S.interpolate_z(p, f, s)
    h = s.cpu().numpy()
    w4 = (-1.0 / 12, 7.0 / 12, 7.0 / 12, -1.0 / 12)
    for vals, d3, q in (
            (f.vals_x, f.d3_vals_x, [h[:, 2:-2, j:j + nx + 1] for j in range(4)]),
            (f.vals_z, f.d3_vals_z, [h[:, j:j + nz + 1, 2:-2] for j in range(4)])):
        for got, c in ((vals, w4), (d3, (-1.0, 3.0, -3.0, 1.0))):
            want = ((q[0] * c[0] + q[1] * c[1]) + q[2] * c[2]) + q[3] * c[3]
            np.testing.assert_array_equal(got.cpu().numpy(), want)

    for d in (Directions.X, Directions.Z):
        for alias in (False, True):
            outs = []
            for fused in (True, False):
                forcing = start.clone()
                out = forcing if alias else torch.zeros_like(start)
                S.discrete_step(p, f, None, start, forcing, out, p["dt"] / 2, d, fused=fused)
                outs.append(out[:, 2:-2, 2:-2].cpu().numpy())
            assert np.all(np.isfinite(outs[0]))
            np.testing.assert_array_equal(outs[0], outs[1])
