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


def next_to_ties(b, count=4):
    """53-bit numerators whose quotients by the odd b lie next to the middle of two doubles."""
    out = []
    for k in (53, 54):  # quotients above and below 1
        inv = pow(1 << k, -1, b)
        for r in range(1, 2 * count, 2):
            out += [a for a in ((r * inv) % b, (-r * inv) % b) if a >= 1 << 52]
            out += [a + b for a in ((r * inv) % b, (-r * inv) % b) if a + b < 1 << 53]
    return [a for a in out if a + 1 < 1 << 53]


# denominators whose reciprocal, formed in too few steps, is the wrong neighbour of a tie, with numerators whose
# quotient that reciprocal then rounds the wrong way; and denominators over the binade
HARD = {0x1FFFFFF4AFB0DD: [0x183AE850BC9D36], 0x1FFFFFF4AFB0D5: [0x1D5DEB16A5FF7B],
        0x1FFFFFF4AFB0D3: [0x1535056D46796C], 0x1FFFFFF4AFB0D1: [0x19011D77ED891A],
        0x1FFFFFE95F61A9: [0x12AC9245C236D8], 0x1FFFFFE95F61A3: [0x1B5CC4B3FB7470],
        0x1FFFFFCEAF47DF: [0x1278331DCFC0B9], 0x1FFFFFCAEF1B07: [0x127C54DE819F71],
        0x1FFFFFC64FA9AD: [0x14053B8C4F89D1], 0x1FFFFFD66E47C1: [0x1620CE4E284F57]}
SPREAD = [int(b) | 1 for b in np.random.default_rng(8).integers(1 << 52, 1 << 53, 12)]


def two_columns(b1, b2, nj):
    """Nodes of two columns of cells, b1 2^-52 and b2 2^-52 wide, nj cells of height 1 (and ghost cells)."""
    def nodes(ni, rows, nh):
        x = np.concatenate([-b1 * 2.0 ** -52 - np.arange(2 * nh, 0, -2), [-b1 * 2.0 ** -52, 0.0, b2 * 2.0 ** -52],
                            b2 * 2.0 ** -52 + np.arange(2, 2 * nh + 1, 2)])
        g = np.meshgrid(x, np.arange(-nh, nj + nh + 1, dtype=np.float64), indexing="ij")
        return [np.asfortranarray(c) for c in g]
    return nodes


@pytest.mark.parametrize("tile", [-1, 0])
def test_quotients_of_fluxes_next_to_ties(oracle, tile):
    """The flux balance divides by the larger flux: pressures b and 2 a - b beside each other make the fluxes b and a,
    exactly.  (Not with the b of fewer than 2^5 ulp below 2, where the compiler's own division, whose operations these
    are, rounds some quotients the wrong way.)"""
    pairs = [(n, b) for b in list(HARD) + SPREAD for n in HARD.get(b, []) + next_to_ties(b) if n < b]
    a, b = (np.array(c, dtype=np.float64) * 2.0 ** -52 for c in zip(*pairs))
    p = np.asfortranarray(np.stack([b, 2.0 * a - b]))
    one, zero = np.ones(p.shape), np.zeros(p.shape)
    got, want = interior_rates(oracle, [one, zero, zero, p], two_columns(1 << 52, 1 << 52, len(pairs)), "AUSM+", "minmod",
                               tile=tile)
    assert np.array_equal(want[1][0], -((a / b - 1.0) * b))
    for g, w in zip(got, want):
        assert same_bits(g, w)


@pytest.mark.parametrize("tile", [-1, 0])
def test_quotients_by_the_volume_next_to_ties(oracle, tile):
    """d / volume in two columns of cells: a pressure jump of a 2^-53 between them makes d = a 2^-54, exactly."""
    widths = list(HARD) + SPREAD + [(1 << 53) - k for k in (1, 3, 5)]
    for b1, b2 in zip(widths, widths[1:] + widths[:1]):
        a = [n for b in (b1, b2) for n in HARD.get(b, []) + next_to_ties(b)]
        nj = len(a)
        lo = np.full(nj, 2.0 ** -53)
        p = np.asfortranarray(np.stack([np.array(a, dtype=np.float64) * 2.0 ** -53 + lo, lo]))
        one, zero = np.ones((2, nj)), np.zeros((2, nj))
        got, want = interior_rates(oracle, [one, zero, zero, p], two_columns(b1, b2, nj), "AUSM+", "minmod", tile=tile)
        d = np.array(a, dtype=np.float64) * 2.0 ** -54
        assert np.array_equal(want[1], np.stack([d / (b1 * 2.0 ** -52), d / (b2 * 2.0 ** -52)]))
        for g, w in zip(got, want):
            assert same_bits(g, w)


# Roe's sensor next to pressures that are not a number or minus infinity: neighbours whose other terms are all 0
@pytest.mark.parametrize("odd", [np.nan, -np.inf, np.inf, -2.0])
def test_sensor_of_odd_pressures(oracle, odd):
    cfg = SchemeConfig(flux="Roe", limiter="minmod", bcs=OPEN)
    ni, nj, nh = 21, 18, cfg.n_ghost
    x, y = uniform_nodes(ni, nj, nh)
    ocfg = oracle.Config(ni, nj, flux="Roe", limiter="minmod", bcs=OPEN)
    rng = np.random.default_rng(7)
    p = np.full((ni + 2 * nh, nj + 2 * nh), -1.0, order="F")
    p[nh::4, nh::4] = odd
    edges = [np.asfortranarray(rng.uniform(0.3, 1.5, (2, ni + 1, nj + 1))) for _ in range(8)]
    one = np.ones_like(p)
    with np.errstate(all="ignore"):
        want = oracle.edge_fluxes(ocfg, oracle.Geometry(ocfg, x, y), one, one, one, p, edges)
        with Solver(cfg, x, y) as s:
            got = s.edge_fluxes(edges, p)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


# AUSM+ where twice a finite Mach number is infinite: half of that over the Mach number is infinite, not 1, and
# times a zero normal not a number
def test_mach_numbers_near_the_largest_double(oracle):
    cfg = SchemeConfig(flux="AUSM+", limiter="minmod", bcs=OPEN)
    ni, nj, nh = 5, 4, cfg.n_ghost
    x, y = uniform_nodes(ni, nj, nh)
    ocfg = oracle.Config(ni, nj, flux="AUSM+", limiter="minmod", bcs=OPEN)
    shape = (2, ni + 1, nj + 1)
    # [0]: the left, [1]: the right state of an edge; a sound speed near 2e-162 beside speeds that make Mach numbers
    # on both sides of 2^1022 and 2^1023
    speed = np.array([1.0, 9.0, 11.0, 19.0, 21.0, 29.0])[:, None] * 1e145 * np.ones((1, nj + 1))
    for side, sign in ((0, 1.0), (1, -1.0)):
        e = [np.ones(shape, order="F") for _ in range(8)]
        for k in (2, 3, 4, 5):
            e[k][:] = 0.0
        for k in (2, 5):  # u on the i-edges, v on the j-edges
            e[k][side] = sign * speed
        for k in (3, 4):  # the other component, so that no mass flux meets a zero speed
            e[k][side] = 1.0
        for k in (6, 7):
            e[k][1 - side] = 5e-324
        one = np.ones((ni + 2 * nh, nj + 2 * nh), order="F")
        with np.errstate(all="ignore"):
            want = oracle.edge_fluxes(ocfg, oracle.Geometry(ocfg, x, y), one, one, one, one, e)
            with Solver(cfg, x, y) as s:
                got = s.edge_fluxes(e, one)
        assert np.isinf(want[0]).any() and np.isnan(want[0]).any()
        for g, w in zip(got, want):
            assert np.array_equal(g, w, equal_nan=True)
