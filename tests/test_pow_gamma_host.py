"""pow_gamma (the flux's power, pyminiweather_amd/csrc/pmw_pow.h) built for the
host and checked against 113-bit quadmath."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

CSRC = os.path.join(REPO, "pyminiweather_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("powg") / "pow_gamma_check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC,
                        os.path.join(REPO, "tests", "pow_gamma_check.cpp"), "-o", exe,
                        "-lquadmath"], capture_output=True, text=True)
    if r.returncode != 0:
        pytest.skip("quadmath not available: " + r.stderr[-200:])
    return exe


@pytest.mark.parametrize("lo,hi", [(50.0, 2000.0), (1e-3, 1e5), (1e-180, 1e200)])
def test_pow_gamma_is_correctly_rounded_almost_always(checker, lo, hi):
    """The value before rounding is within 5e-22 relative of the power, so a
    result can miss the correctly rounded one only that close to a midpoint
    between doubles: at most about 2 * 5e-22 / 2^-53 ~ 1e-5 of the arguments
    (random ones and the edges of the table intervals). Special arguments
    give what pow gives. x^(gamma-1) is within 3 ulp: two table factors and
    their product (1.5 ulp) and the series' last step."""
    out = subprocess.run([checker, "200000", str(lo), str(hi)], capture_output=True, text=True,
                         check=True).stdout.split()
    n, bad, special = (int(v) for v in out[:3])
    assert float(out[3]) <= 3 * 2.0 ** -52, out[3]
    assert special == 0
    assert bad <= 1e-5 * (n + 53 * 512 * 3), bad
