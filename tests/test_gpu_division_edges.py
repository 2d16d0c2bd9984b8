"""Where divisions are left out or share a reciprocal: the operands at which they would differ from IEEE ones."""
import numpy as np
import pytest

from fvleg_2d_amd import SchemeConfig, Solver
from fvleg_2d_amd.problems import uniform_nodes

pytestmark = pytest.mark.gpu

NI, NJ = 21, 18


def states(seed, scale=1.0, speed=1.0):
    rng = np.random.default_rng(seed)
    f = [rng.uniform(0.2, 2.0, (NI, NJ)), rng.uniform(-1, 1, (NI, NJ)), rng.uniform(-1, 1, (NI, NJ)),
         rng.uniform(0.2, 2.0, (NI, NJ))]
    return [np.asfortranarray(x) for x in (f[0], speed * f[1], speed * f[2], scale * f[3])]


def both_residuals(oracle, flux, limiter, prims, size=(1.0, 1.0), tile=-1):
    cfg = SchemeConfig(flux=flux, limiter=limiter, bcs=("zero_gradient",) * 4, tile=tile)
    nx, ny = uniform_nodes(NI, NJ, cfg.n_ghost, (0.0, size[0]), (0.0, size[1]))
    ocfg = oracle.Config(NI, NJ, flux=flux, limiter=limiter, bcs=cfg.bcs)
    halo = [np.asfortranarray(np.pad(a, cfg.n_ghost)) for a in prims]
    with Solver(cfg, nx, ny) as s:
        got = s.residual(*[a.copy(order="F") for a in halo])
    return got, oracle.solve(ocfg, oracle.Geometry(ocfg, nx, ny), *halo)


# the flux balance's normalisation by the larger flux: pressures that put the fluxes on both sides of 2^1000,
# where the shared reciprocal gives way to IEEE divisions, and where one flux vanishes beside the other
@pytest.mark.parametrize("tile", [-1, 0])
@pytest.mark.parametrize("scale", [2.0 ** 998, 2.0 ** 1000, 2.0 ** 1003, 2.0 ** 1020, 1e-300])
def test_flux_balance_scales(oracle, scale, tile):
    with np.errstate(all="ignore"):
        got, want = both_residuals(oracle, "AUSM+", "minmod", states(1, scale), tile=tile)
    for g, w in zip(got, want):
        assert np.array_equal(g, w, equal_nan=True)


# cell volumes on both sides of the range in which the four variables share a reciprocal ([2^-400, 2^400])
@pytest.mark.parametrize("tile", [-1, 0])
@pytest.mark.parametrize("side", [3e-61, 1e-60, 1e-10, 7.0, 1e60, 3e61])
def test_cell_volumes(oracle, side, tile):
    got, want = both_residuals(oracle, "SLAU", "van_leer", states(2), size=(side, 0.9 * side), tile=tile)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


# speeds on both sides of Mach 1 in both directions (the supersonic splits without a division)
@pytest.mark.parametrize("flux", ["AUSM+", "SLAU", "SLAU2", "SD-SLAU"])
@pytest.mark.parametrize("speed", [0.0, 1.0, 2.0, 30.0])
def test_supersonic_splits(oracle, flux, speed):
    for tile in (-1, 0):
        got, want = both_residuals(oracle, flux, "superbee", states(3, speed=speed), tile=tile)
        for g, w in zip(got, want):
            assert np.array_equal(g, w)


# the pressure ratios of Roe's sensor and of AUSMPW+: equal, nearly equal, twice as large, zero, negative,
# infinite and NaN cell and edge pressures
@pytest.mark.parametrize("flux", ["Roe", "AUSMPW+", "M-AUSMPW+"])
def test_pressure_ratios(oracle, flux):
    cfg = SchemeConfig(flux=flux, limiter="minmod", bcs=("zero_gradient",) * 4)
    nh = cfg.n_ghost
    nx, ny = uniform_nodes(NI, NJ, nh)
    ocfg = oracle.Config(NI, NJ, flux=flux, limiter="minmod", bcs=cfg.bcs)
    og = oracle.Geometry(ocfg, nx, ny)
    rng = np.random.default_rng(4)
    odd = np.array([1.0, 1.0 + 2.0 ** -52, 1.0 - 2.0 ** -53, 2.0, 2.0 + 2.0 ** -51, 2.0 - 2.0 ** -52, 0.5, 0.0, -0.0,
                    -1e-16, -1.0, 1e-16, 5e-324, 1e308, np.inf, np.nan])
    p = np.asfortranarray(rng.choice(odd, (NI + 2 * nh, NJ + 2 * nh)))
    halo = [np.asfortranarray(np.pad(a, nh, mode="edge")) for a in states(5)[:3]]
    n = 16 if flux == "M-AUSMPW+" else 8
    edges = [np.asfortranarray(rng.uniform(0.3, 1.5, (2, NI + 1, NJ + 1))) for _ in range(n)]
    for k in range(6, n, 8):  # the pressure states of both directions
        for q in (k, k + 1):
            edges[q] = np.asfortranarray(rng.choice(odd, edges[q].shape))
    with np.errstate(all="ignore"):
        want = oracle.edge_fluxes(ocfg, og, *halo, p, edges)
        with Solver(cfg, nx, ny) as s:
            got = s.edge_fluxes(edges, p)
    for g, w in zip(got, want):
        assert np.array_equal(g, w, equal_nan=True)


# in-range cells (speeds below 2^20, densities and pressures in [2^-20, 2^20]) whose sound speed is lost beside
# the flow speed: AUSMPW+'s normal enthalpy and Roe's c^2 cancel, to zero or a negative number on some edges
@pytest.mark.parametrize("tile", [-1, 0])
@pytest.mark.parametrize("limiter", ["minmod", "van_leer", "MLP5"])
@pytest.mark.parametrize("flux", ["Roe", "AUSMPW+", "AUSM+", "HLLC"])
def test_cancelled_sound_speeds(oracle, flux, limiter, tile):
    rng = np.random.default_rng(6)
    shape = (NI, NJ)
    prims = [rng.uniform(1e5, 9e5, shape), rng.choice([0.0, 3.0, 9e5, -9e5], shape) * rng.choice([1.0, 1 + 1e-9], shape),
             rng.choice([1.0, 9e5, 9.1e5, -8e5], shape), rng.uniform(1e-6, 3e-6, shape)]
    with np.errstate(all="ignore"):
        got, want = both_residuals(oracle, flux, limiter, [np.asfortranarray(a) for a in prims], tile=tile)
    for g, w in zip(got, want):
        assert np.array_equal(g, w, equal_nan=True)
