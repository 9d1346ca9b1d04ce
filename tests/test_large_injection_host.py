"""What pmw_evolve_ex answers for an injection grid past the dense codes' slots."""
import ctypes

import pytest
import torch

from pyminiweather_amd import _lib


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="launches, on addresses that are none")
@pytest.mark.parametrize("x_code", [256, 512, 1256, 1512])
@pytest.mark.parametrize("bc", [0, 1])
def test_dense_x_codes_refuse_periodic_rows_only(bc, x_code):
    """2^30 slots (rows with their 6 cells on either side) bound the codes 1256
    and 1512 of periodic rows; the injection boundary takes every code at every
    size. Without a device an accepted call ends at its launch, with HIP's error."""
    nx, nz = 32768, 32800
    assert nz * (nx + 12) > 1 << 30
    fake = [ctypes.c_void_p(4096 * (i + 1)) for i in range(9)]
    flag = ctypes.c_int(1)  # x first
    rc = _lib.load().pmw_evolve_ex(
        *fake[:8], None, bc, fake[8] if bc else None, nx, nz, 1.0, 1.0, 0.1, -0.1, -0.1,
        ctypes.byref(flag), 1, (ctypes.c_int * 3)(0, x_code, 8096), None, None)
    PMW_EINVAL = -1
    assert (rc == PMW_EINVAL) == (bc == 0 and x_code > 1000)
    assert rc != 0
