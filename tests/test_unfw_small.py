"""u_NFW's polynomial branch (a2 < 4) of the FP64 policy at the edges of its
range, built for the host and checked against the transform at 40 digits: a2
just below 4 and beside it the next branch, a2 down to 1e-6, concentrations
0.04 (the prior's smallest f with the tables' smallest c) to 25.

u = 1 + rest / F with F = ln(1+c) - c/(1+c) formed from terms about 2/c times
larger than itself (F ~ c^2/2 for small c), in rest as in F: a few roundings
of each, 16 here, give a relative error below 8 eps (1 + 2/c)^2.  It must also not
exceed the per-piece form's by more than its own rounding."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from test_unfw_forms import _hex, _run, _u_exact

mpmath = pytest.importorskip("mpmath")


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("unfw") / "unfw_probe")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip",
                        "--offload-arch=gfx950", "-Wno-unused-command-line-argument",
                        os.path.join(ROOT, "tests", "cxx", "unfw_probe.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode:
        pytest.skip("hipcc host build unavailable: " + r.stderr[-300:])
    return exe


@pytest.mark.parametrize("c", [0.04, 0.3, 1.0, 4.0, 25.0])
def test_polynomial_branch(probe, c):
    mpmath.mp.dps = 40
    a2 = np.concatenate([4.0 - 4.0 ** -np.arange(1, 20), np.linspace(0.05, 3.95, 60),
                         10.0 ** np.linspace(-6, -1.3, 25)])
    a1 = a2 / (1 + c)
    rows = _run(probe, [f"u {_hex(x)} {_hex(c)}" for x in a1])
    eps = 2.0 ** -52
    for x, (u, u0) in zip(a1, rows):
        t = _u_exact(x, c)
        e, e0 = float(abs((u - t) / t)), float(abs((u0 - t) / t))
        assert e <= 8 * eps * (1 + 2 / c) ** 2, (x, e, e0)
        assert e <= 2 * e0 + 2 * eps * (1 + 2 / c) ** 2, (x, e, e0)
