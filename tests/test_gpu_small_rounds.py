"""Small rounds, evaluated in one launch for all kinds and queued before the
last one's outcome is known, against rounds the host waits for: the
allocation-free entry point runs every round kind by kind, with the same kernels
otherwise, so the two have to agree bit for bit.

Sizes: one integral of one kind, one of each kind, and 40 mixed ones, whose
rounds pass from queued to single to separate launches; budgets that end at the
root, after a queued round, and beyond; a tolerance that a queued round meets
while later ones are already on their way."""
import numpy as np
import pytest

from conftest import ARCMIN, T, say

pytestmark = pytest.mark.gpu

KINDS = [(0, 1), (0, 2), (0, 3), (1, 1), (1, 2), (1, 3)]


@pytest.mark.parametrize("kinds,maxeval,reltol", [
    ([(0, 2)], 1, 1e-4), ([(0, 3)], 40000, 1e-4), ([(1, 1)], 400000, 1e-4),
    (KINDS, 300, 1e-4), (KINDS, 20000, 1e-4), (KINDS, 150000, 1e-4),
    (KINDS, 150000, 0.5), (KINDS * 6 + KINDS[:4], 30000, 1e-3)])
def test_small_rounds_agree(tables, kinds, maxeval, reltol):
    from g3lhalo_amd import _lib
    ctx = _lib.Context(tables)
    sid = ctx.hodset(T.FIDUCIAL_HOD, T.FIDUCIAL_HOD)
    rng = np.random.default_rng(len(kinds) + maxeval)
    reqs = [_lib.make_request(st, t, 0.5 * 64.0 ** rng.uniform(0, 1, 3) * ARCMIN, hodset=sid,
                              reltol=reltol, maxeval=maxeval) for st, t in kinds]
    say(f"small rounds: {len(reqs)} integrals, maxeval {maxeval}, reltol {reltol}")
    a, b = ctx.eval_batch(reqs), ctx.eval_batch_noalloc(reqs)
    for x, y in zip(a, b):
        assert (x.value, x.raw, x.err, x.neval, x.rounds, x.status) == \
               (y.value, y.raw, y.err, y.neval, y.rounds, y.status)
    st = ctx.last_stats()
    assert st.rounds == max(y.rounds for y in b)
    ctx.close()
