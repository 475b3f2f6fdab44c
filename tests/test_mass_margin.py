"""The mass look-ups without pow and log (mass_direct) on tables whose bins are so fine
that the rounding of ln m is a visible part of one: the margin to a tie within which
the reference's chain decides has to grow with the number of bins per unit of ln m.
Host build, as in test_mass_direct; wherever the direct form says that it holds, both
indices equal the chain's, also for masses far from one (ln m of up to 600)."""
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


@pytest.mark.parametrize("nb,lo,hi", [(46340, 11, 12), (46340, 11, 11.01), (46340, 11, 11.0001),
                                      (1000, 11, 11.001), (2, 11, 11.000001),
                                      (128, -250, -249.99), (16, 250, 250.001)])
def test_indices(probe, nb, lo, hi):
    out = subprocess.run([probe, str(nb), str(lo), str(hi), "5"], capture_output=True, text=True,
                         check=True).stdout
    taken, wrong, far, err, special, kwrong = out.split()
    print(out)
    assert int(taken) > 100000
    assert int(wrong) == 0
    # the argument's bound, half the margin's
    assert float(far) < 1e-12 * nb / ((hi - lo) * 2.302585092994046)
    assert float(err) < 1.5 * 2.0 ** -53
    assert int(special) == 0
    assert int(kwrong) == 0
