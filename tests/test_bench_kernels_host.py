"""The kernels under whose names bench.py looks up the committed counters."""
import shutil
import subprocess
import sys

import pytest

from conftest import REPO

sys.path.insert(0, REPO)
import bench  # noqa: E402


@pytest.fixture(scope="module")
def kernels():
    from pyminiweather_amd import _lib
    _lib.load()
    if shutil.which("nm") is None:
        pytest.skip("nm not available")
    return subprocess.run(["nm", "-C", _lib.LIB_PATH], capture_output=True, text=True,
                          check=True).stdout


def test_every_code_names_a_kernel_of_the_library(kernels):
    """Every accepted x and z code on the profiled grid."""
    names = set()
    for xb in (256, 448, 512, 1256, 1512):
        for zs in (8, 16, 24, 32, 48, 64, 8064, 4128, 8096, 8128, 18128, 18096):
            names.update(bench.launched_kernels((0, xb, zs), 2000, 1000))
    assert len(names) == 5
    for n in names:
        assert f"__device_stub__{n}(" in kernels, n


def test_same_kernels_have_the_same_counts():
    """Codes that run the default's kernels find its counts; other grids find
    none, as the counts are those of one launch at 2000 x 1000."""
    default = bench.launched_kernels((0, 512, 8096), 2000, 1000)
    assert bench.launched_kernels((0, 1512, 8128), 2000, 1000) == default
    for k in default:
        assert bench.traffic_from_profile(k) and bench.valu_from_profile(k)
    for k in bench.launched_kernels((0, 512, 8096), 400, 200):
        assert bench.traffic_from_profile(k) is None and bench.valu_from_profile(k) is None


def test_autotuner_times_each_kernel_once():
    """No two candidates of a direction run the same kernel."""
    from pyminiweather_amd.autotune import X_BLOCKS, Z_SEGMENTS
    x = [bench.launched_kernels((0, xb, 8096), 2000, 1000)[0] for xb in X_BLOCKS]
    z = [bench.launched_kernels((0, 512, zs), 2000, 1000)[1] for zs in Z_SEGMENTS]
    assert len(set(x)) == len(x) == 2 and len(set(z)) == len(z) == 3
