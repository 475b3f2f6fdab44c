"""One-dimensional integrals refined several to a block against the same integrals in
other company: the number of integrals that share a block (and its nodes) must not
show in any of them, so all comparisons are bit for bit.

A block takes up to eight integrals of a group.  The HOD sets and bin counts below
give it every count, as a unit's size and as a group's remainder: 3, 5, 6 and 7, which
divide neither a wave nor the 32 regions that are reduced together, beside the
powers of two; with and without the table of the tree's top; and, at 300 and 400 bins,
trees that outgrow the nodes that a block keeps (one of the sets at 300 bins needs more
regions than an integral may hold, and the call that has it is refused like that set
alone).  One set alone has one integral per block."""
import numpy as np
import pytest

from conftest import T, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbins,sets", [
    # integrals per unit (a group's remainder)
    (128, 6), (128, 10), (128, 12), (128, 14),   # 3 (2), 5 (3), 6 (2), 7 (2)
    (400, 2),                                    # 3 (1), under the table of the top
    (125, 17), (127, 17), (99, 21), (62, 40),    # 8 (5), 8 (7), 8 (3), 8 (6)
    (300, 5), (300, 6), (300, 8),                # 5 (0), 7 (6), 8 (4)
])
def test_densities_do_not_depend_on_company(nbins, sets):
    from g3lhalo_amd import _lib
    t = T.make_tables(nbins)
    h1 = T.hod_prior_draws(sets, seed=nbins)
    h2 = T.hod_prior_draws(sets, seed=nbins + 1)
    ctx = _lib.Context(t)
    say(f"units: {sets} sets of {nbins} bins in one call")

    def densities(a, b):
        """Of each set, or the status the call is refused with."""
        try:
            first = ctx.hodsets(a, b)
        except _lib.G3LError as e:
            return e.rc
        return [ctx.densities(first + i) for i in range(len(a))]

    many = densities(h1, h2)
    alone = [densities(h1[i:i + 1], h2[i:i + 1]) for i in range(sets)]
    if isinstance(many, int):
        assert many in alone
    else:
        for i, (got, one) in enumerate(zip(many, alone)):
            for name, x, y in zip(("rho_bar", "n_bar1", "n_bar2"), got, one[0]):
                np.testing.assert_array_equal(x, y, err_msg=f"set {i} {name}")
    ctx.close()


@pytest.mark.parametrize("n", [6, 7, 10, 11, 12, 13, 14])
def test_precomputation_does_not_depend_on_company(n):
    """Every fourth bin of a grid of 4 n bins is the grid of n bins, with the same bits
    (bin widths differ by a power of two): units of 3, 5, 6 and 7 integrals against
    units of 8."""
    from g3lhalo_amd import _lib
    cosmo = {"Omega_m": 0.3, "Omega_Lambda": 0.7, "Omega_b": 0.046, "sigma8": 0.8, "H0": 70.0,
             "ns": 0.96}
    z = np.linspace(0.01, 3.0, 40)
    nz = z ** 2 * np.exp(-(z / 0.5) ** 1.5)
    args = (cosmo, 0.001, 2.0, 1e10, 1e17, 1e-4, 1e4)
    say(f"units: precomputation at {n} and {4 * n} bins")
    a, b = _lib.precompute(*args, n, z, nz), _lib.precompute(*args, 4 * n, z, nz)
    for key, x in a.items():
        x, y = np.asarray(x), np.asarray(b[key])
        y = y[::4, ::4] if x.ndim == 2 else y[::4]
        np.testing.assert_array_equal(x, y, err_msg=key)


def test_more_integrals_than_one_launch_takes():
    """2^20 integrals and 400 more (every set has four of them), in two launches: each
    set's densities are those of its parameters, whichever launch it is in."""
    from g3lhalo_amd import _lib
    t = T.make_tables(2)
    h = T.hod_prior_draws(7, seed=3)
    n = (1 << 18) + 100
    ctx = _lib.Context(t)
    say(f"units: {n} sets of 2 bins in one call")
    alone = [ctx.densities(ctx.hodset(x, x)) for x in h]
    first = ctx.hodsets([h[i % 7] for i in range(n)])
    for i in [*range(0, n, 997), *range((1 << 18) - 8, n)]:
        for x, y in zip(ctx.densities(first + i), alone[i % 7]):
            np.testing.assert_array_equal(x, y, err_msg=f"set {i}")
    ctx.close()
