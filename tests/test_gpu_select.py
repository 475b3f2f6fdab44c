"""The selection kernel at the edges of its forms: one wave up to 64 and 256
regions, a block beyond, with 1024 threads for up to 512 integrals and 256
threads for more, and chunks of four slots per thread.

Each integral's evaluation budget ends its refinement near one of those region
counts.  The same integrals run alone (the wide block) and among 600 (the
narrow one): both have to give the same bits, since an integral's result does
not depend on what else is in flight, and the oracle's evaluation count and
value.  The oracle's points differ from the device's by about 1e-15 (median)
and a total adds at most 2e4 of one sign in another order, 2e4 half-ulps, so
the bound on the values is 1e-11."""
import numpy as np
import pytest

from conftest import ARCMIN, T, say

pytestmark = pytest.mark.gpu

PTS = {1: 93, 2: 149, 3: 241}


@pytest.fixture(scope="module")
def ctx(tables):
    from g3lhalo_amd import _lib
    c = _lib.Context(tables)
    assert c.hodset(T.FIDUCIAL_HOD, T.FIDUCIAL_HOD) == 0
    yield c
    c.close()


@pytest.mark.parametrize("stat,term", [(0, 1), (0, 2), (1, 1), (1, 3)])
def test_forms_agree(ctx, oracle_model, stat, term):
    from g3lhalo_amd import _lib
    theta = np.array([2.0, 4.0, 8.0]) * ARCMIN
    regions = (1, 2, 63, 64, 65, 128, 255, 256, 257, 700, 1024, 1025, 4095, 4097, 9000)
    # a budget of one point more than n regions' (2 n - 1 evaluated) lets one
    # more region be cut
    budgets = [PTS[term] * (2 * n - 1) + d for n in regions for d in (0, 1)]
    reqs = [_lib.make_request(stat, term, theta, reltol=1e-7, maxeval=b) for b in budgets]
    say(f"select: stat={stat} term={term}, {len(reqs)} integrals alone")
    alone = ctx.eval_batch(reqs)
    say("select: among 600")
    many = ctx.eval_batch((reqs * (600 // len(reqs) + 1))[:600])[:len(reqs)]
    for b, x, y in zip(budgets, alone, many):
        assert (x.value, x.raw, x.err, x.neval, x.rounds, x.status) == \
               (y.value, y.raw, y.err, y.neval, y.rounds, y.status), b
    for b, x in zip(budgets[::3], alone[::3]):
        o = oracle_model.eval_term(stat, term, list(theta), 1, 2, 1e-7, b)
        assert x.neval == o["neval"], b
        assert x.value == pytest.approx(o["value"], rel=1e-11), b
