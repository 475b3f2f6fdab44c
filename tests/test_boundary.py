"""The boundary of a Gladwell batch as k_select and k_onedim find it (find_boundary of
select_wave.h), compiled for the host with a wave of 64 lanes run one after the other,
against popping the sorted errors one by one (the loop of src/hcubature.cpp:971-985).

1 to 2048 regions, at and beside the sizes where another number of keys per lane or
another search begins; errors all equal, over 300 octaves, whole numbers with
tolerances at a partial sum and one unit beside it (closer than a 32-bit sum resolves),
a few values and zeros, equal in their high words, and denormal; budgets of one region,
half and all; and searches among part of the errors, which have to say when the
boundary is not among them."""
import os
import subprocess

from conftest import ROOT


def test_boundary_is_that_of_the_sorted_errors(tmp_path):
    exe = str(tmp_path / "boundary_probe")
    cxx = os.path.join(ROOT, "tests", "cxx")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O2", "-Wno-attributes",
                    "-I", os.path.join(cxx, "hostwave"),
                    os.path.join(cxx, "boundary_probe.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe, "1"], capture_output=True, text=True, check=True).stdout
    searches, wrong, silent = map(int, out.split()[-3:])
    assert searches > 1500
    assert (wrong, silent) == (0, 0), out
