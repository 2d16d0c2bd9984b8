"""The latency layout of small grids (the library's own tile choice) against the 32 x 8 tiles and the oracle."""
import numpy as np
import pytest

from fvleg_2d_amd import SchemeConfig, Solver
from fvleg_2d_amd.problems import uniform_nodes, wavy_nodes
from error_cases import ERROR_CASES, NI, NJ, error_case_fields

pytestmark = pytest.mark.gpu

FLUXES = ["AUSMPW+", "SLAU", "SLAU2", "SD-SLAU", "SD-SLAU2", "Roe", "AUSM+", "HLLC", "M-AUSMPW+"]
OPEN = ("zero_gradient",) * 4


def solver(ni, nj, flux, limiter, integrator="ssp_rk3", precision="fp64", bcs=OPEN, tile=-1, wavy=False):
    cfg = SchemeConfig(flux=flux, limiter=limiter, integrator=integrator, bcs=bcs, cfl=0.3, precision=precision,
                       tile=tile, bc_pressure=0.8)
    s = Solver(cfg, *(wavy_nodes if wavy else uniform_nodes)(ni, nj, cfg.n_ghost))
    rng = np.random.default_rng([ni, nj])
    x, y = np.meshgrid((np.arange(ni) + 0.5) / ni, (np.arange(nj) + 0.5) / nj, indexing="ij")
    jump = x + 0.4 * y > 0.6
    s.set_primitive(np.where(jump, 0.5, 1.3) + 0.02 * rng.random((ni, nj)), np.where(jump, 0.2, -0.3) + 0.1 * y,
                    0.2 * np.sin(6.0 * x), np.where(jump, 0.4, 1.1) + 0.02 * rng.random((ni, nj)))
    return s


def after(steps, *args, **kw):
    with solver(*args, **kw) as s:
        done = s.run(1e300, steps)
        return done, s.conserved() + s.primitive()


def same(a, b):
    assert a[0] == b[0]
    for x, y in zip(a[1], b[1]):
        assert np.array_equal(x, y)


# every scheme (its states in one launch of items) on partial tiles, quadrilateral cells too
@pytest.mark.parametrize("precision", ["fp64", "fp32_flux"])
@pytest.mark.parametrize("limiter", ["minmod", "superbee", "van_leer", "MLP3", "MLP5"])
@pytest.mark.parametrize("flux", FLUXES)
def test_equals_the_32x8_tiles(flux, limiter, precision):
    same(after(12, 37, 21, flux, limiter, precision=precision),
         after(12, 37, 21, flux, limiter, precision=precision, tile=0))


# smallest grids, one tile, tile edges, and the largest grid of the layout (1280 tiles)
@pytest.mark.parametrize("ni,nj", [(3, 3), (8, 8), (9, 7), (16, 24), (65, 3), (320, 256)])
def test_sizes(ni, nj):
    same(after(9, ni, nj, "HLLC", "MLP5"), after(9, ni, nj, "HLLC", "MLP5", tile=0))


# steps that close each other, 32 to a graph: fewer, one graph, one graph and a rest, with the error of a
# failing step, every number of stages, and each boundary that a step may read
@pytest.mark.parametrize("steps", [1, 2, 31, 33, 34, 70])
@pytest.mark.parametrize("integrator", ["ssp_rk2", "ssp_rk3", "rk(1,4)", "rk(2,5)"])
def test_chained_steps(steps, integrator):
    bcs = ("outflow", "symmetry", "periodic", "periodic")
    same(after(steps, 40, 33, "SLAU", "van_leer", integrator, bcs=bcs),
         after(steps, 40, 33, "SLAU", "van_leer", integrator, bcs=bcs, tile=0))


# the constructed failures of error_cases.py, in the device loop at their constant dt
@pytest.mark.parametrize("name", sorted(ERROR_CASES))
@pytest.mark.parametrize("steps", [5, 40])
def test_chained_steps_end_on_an_error_and_leave_no_flags(steps, name):
    """A step that fails ends the run with the same code and count; the flags it set are gone from the next."""
    c, got = ERROR_CASES[name], []
    for tile in (-1, 0):
        cfg = SchemeConfig(flux="SLAU", limiter="minmod", integrator=c["integrator"], bcs=OPEN, tile=tile)
        with Solver(cfg, *uniform_nodes(NI, NJ, cfg.n_ghost)) as s:
            s.set_primitive(*error_case_fields(name))
            first = s.run(1e300, steps, constant_dt=c["dt"])
            one = np.ones((NI, NJ), order="F")
            s.set_primitive(one, 0.1 * one, 0.0 * one, one)
            got.append((first[0], first[2], s.step(1e-4), s.run(1e300, 3)[2]))
    assert got[0] == got[1] and got[0][1] != 0 and got[0][2:] == (0, 0)


def test_chained_steps_end_on_max_time():
    for kw in ({}, {"wavy": True, "bcs": ("periodic",) * 4}):
        ends = []
        for tile in (-1, 0):
            with solver(48, 40, "SLAU", "van_leer", tile=tile, **kw) as s:
                ends.append((s.run(0.03, 0, 0.011), s.conserved()))
        same(*ends)
