"""The plain driver sends halves to the device in runs of 2048 and holds up to
32768 of them (from 4096, doubled when they run out) before it waits; against the
oracle's heap, which knows none of this: the same count of evaluations, and the
value within the parity tests' bound.

Budgets: the root alone; batches up to a run's length; batches beyond a run, the
first and the largest buffer."""
import numpy as np
import pytest

from conftest import ARCMIN, T, say

pytestmark = pytest.mark.gpu

TOL = 1e-4   # of test_gpu_parity.py


@pytest.mark.parametrize("stat,maxeval", [(0, 1), (0, 380_000), (1, 3_000_000), (0, 20_000_000)])
def test_plain_chunks(tables, oracle_model, stat, maxeval):
    from g3lhalo_amd import _lib
    ctx = _lib.Context(tables)
    sid = ctx.hodset(T.FIDUCIAL_HOD, T.FIDUCIAL_HOD)
    th = np.array([1.0, 2.0, 8.0]) * ARCMIN
    say(f"plain chunks: stat {stat}, maxeval {maxeval}")
    r = ctx.eval_plain(_lib.make_request(stat, 1, th, hodset=sid, reltol=1e-9, maxeval=maxeval))
    o = oracle_model.eval_term(stat, 1, th, 1, 2, 1e-9, maxeval)
    print(r.value, o["value"], r.neval, o["neval"])
    assert r.neval == o["neval"]
    assert abs(r.value - o["value"]) <= TOL * abs(o["value"])
    ctx.close()
