"""ln(1 + c) of the NFW normalisation (P64::nfw_norm), built for the host, against 64-bit
mantissas: over the concentrations of the tables and prior draws (0.04 to 25) and beyond
on both sides its error is no larger than the library logarithm's of the rounded 1 + c,
and neither is that of F = ln(1 + c) - c / (1 + c).

The largest error: half a unit of the last addition, and at most a fifth of one from
the polynomial's part, a third of the result, with three roundings."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ln1p") / "ln1p_probe")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip",
                        "--offload-arch=gfx950", "-Wno-unused-command-line-argument",
                        os.path.join(ROOT, "tests", "cxx", "ln1p_probe.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode:
        pytest.skip("hipcc host build unavailable: " + r.stderr[-300:])
    return exe


@pytest.mark.parametrize("lo,hi", [(-0.9, -0.1), (0.001, 0.04), (0.04, 0.3), (0.3, 1), (1, 3),
                                   (3, 25), (25, 300)])
def test_no_further_off_than_the_library(probe, lo, hi):
    out = subprocess.run([probe, str(lo), str(hi), "7"], capture_output=True, text=True,
                         check=True).stdout
    print(out)
    rms, worst, lib_rms, lib_worst, rms_f, lib_rms_f, nan = map(float, out.split())
    assert rms <= lib_rms
    assert worst <= lib_worst
    assert worst < 0.75
    assert rms_f <= lib_rms_f
    assert nan == 4
