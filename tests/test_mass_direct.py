"""Masses and their look-up indices without pow and log (mass_direct) against the
reference's chain (mass_chain), on the host: wherever the direct form says that it
holds, both indices equal the chain's, from the smallest to the largest number of
bins, at and around every kind of tie and beyond both ends of the range.  P(k)'s
index, from the short logarithm away from ties, equals the library chain's everywhere.

The chain's argument L nb / ln(mmax / mmin) carries the roundings of m and of L, 2^-53
of ln-values up to 40 each and a few of its own: below 40 x 6 x 1.2e-16 nb / ln(mmax /
mmin), 1e-10 at most here, a tenth of the margin to a tie.  The mass: half a unit in
the last place and the carried parts' roundings, below 1.5 x 2^-53."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("mass") / "mass_probe")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip",
                        "--offload-arch=gfx950", "-Wno-unused-command-line-argument",
                        os.path.join(ROOT, "tests", "cxx", "mass_probe.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode:
        pytest.skip("hipcc host build unavailable: " + r.stderr[-300:])
    return exe


@pytest.mark.parametrize("nb,lo,hi", [(2, 10, 17), (16, 10, 17), (128, 10, 17), (128, 3, 16.5),
                                      (256, 9.7, 16.1), (1000, 11, 12), (46340, 8, 17)])
def test_indices(probe, nb, lo, hi):
    out = subprocess.run([probe, str(nb), str(lo), str(hi), "5"], capture_output=True, text=True,
                         check=True).stdout
    taken, wrong, far, err, special, kwrong = out.split()
    print(out)
    assert int(taken) > 100000
    assert int(wrong) == 0
    assert float(far) < 1e-10
    assert float(err) < 1.5 * 2.0 ** -53
    assert int(special) == 0
    assert int(kwrong) == 0
