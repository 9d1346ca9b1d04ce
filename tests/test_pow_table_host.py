"""The range of the flux power's table: rho*theta of whole columns."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle as O
from conftest import REPO

CSRC = os.path.join(REPO, "pyminiweather_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("powt") / "pow_table_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC,
                    os.path.join(REPO, "tests", "pow_table_check.cpp"), "-o", exe,
                    "-lquadmath"], check=True)
    return exe


@pytest.mark.parametrize("zlen", [1.0e4, 1.6e4, 2.0e4, 2.8e4])
@pytest.mark.parametrize("ic", ["thermal", "gravity"])
def test_columns_lie_in_the_table(checker, ic, zlen):
    """Every level of a column of up to 28 km, 30 K colder or warmer than its
    background: the fused kernels, which compute a wave or tile again when an
    argument lies outside, do so for none of it. At the intervals' edges the
    powers are correctly rounded but for ~1e-5 of them."""
    f = O.init_state(O.make_params(2, 200, ic, zlen=zlen))
    rt = np.concatenate([f["hy_dens_theta_cell"][2:-2], f["hy_dens_theta_int"]])
    rho = np.concatenate([f["hy_dens_cell"][2:-2], f["hy_dens_int"]])
    args = np.concatenate([rt, rt - 30.0 * rho, rt + 30.0 * rho])
    assert np.all(args > 0.0)
    out = subprocess.run([checker, *map(repr, args.tolist())], capture_output=True, text=True,
                         check=True).stdout.split()
    outside, bad, edges = (int(v) for v in out)
    assert outside == 0
    assert bad <= max(1, 1e-5 * edges), (bad, edges)
