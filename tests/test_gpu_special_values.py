"""Bit patterns of results where a quotient is zero, infinite, not a number or next to a rounding boundary."""
import numpy as np
import pytest

from fvleg_2d_amd import SchemeConfig, Solver
from fvleg_2d_amd.problems import uniform_nodes, wavy_nodes

pytestmark = pytest.mark.gpu

FLUXES = ["AUSMPW+", "SLAU", "SLAU2", "SD-SLAU", "SD-SLAU2", "Roe", "AUSM+", "HLLC", "M-AUSMPW+"]
OPEN = ("zero_gradient",) * 4


def same_bits(got, want):
    return np.array_equal(np.ascontiguousarray(got).view(np.int64), np.ascontiguousarray(want).view(np.int64))


def interior_rates(oracle, prims, nodes, flux, limiter, bcs=OPEN, tile=-1):
    """(got, want): the rates of the interior cells from Solver.residual and from the oracle."""
    cfg = SchemeConfig(flux=flux, limiter=limiter, bcs=bcs, tile=tile)
    nh, (ni, nj) = cfg.n_ghost, prims[0].shape
    x, y = nodes(ni, nj, nh)
    ocfg = oracle.Config(ni, nj, flux=flux, limiter=limiter, bcs=bcs)
    halo = [np.asfortranarray(np.pad(a, nh)) for a in prims]
    with Solver(cfg, x, y) as s:
        got = s.residual(*[a.copy(order="F") for a in halo])
    want = oracle.solve(ocfg, oracle.Geometry(ocfg, x, y), *halo)
    return [a[nh:-nh, nh:-nh] for a in got], [a[nh:-nh, nh:-nh] for a in want]


# a flow at rest, a uniform one and a contact in it: balances that are zero in most cells, whose rate is the -0 that
# dividing -0 by the volume gives, on volumes that are no power of two and on quadrilateral cells
@pytest.mark.parametrize("tile", [-1, 0])
@pytest.mark.parametrize("nodes", [uniform_nodes, wavy_nodes], ids=["uniform", "wavy"])
@pytest.mark.parametrize("flux", FLUXES)
def test_zero_rates_keep_their_sign(oracle, flux, nodes, tile):
    one = np.ones((21, 18))
    for speed, jump in ((0.0, 0.0), (0.3, 0.0), (0.3, 1.0)):
        rho = one + jump * (np.arange(21) >= 9)[:, None]
        prims = [rho, speed * one, -0.5 * speed * one, one]
        got, want = interior_rates(oracle, prims, nodes, flux, "van_leer", tile=tile)
        if jump == 0.0 and nodes is uniform_nodes:
            assert all((w == 0.0).all() and np.signbit(w).all() for w in want)
        for g, w in zip(got, want):
            assert same_bits(g, w)
