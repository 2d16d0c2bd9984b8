"""Boundary fill and flux solver on halo'd host fields: leading dimensions, strips, every ghost cell."""
import ctypes as C

import numpy as np
import pytest

from fvleg_2d_amd import SchemeConfig, Solver
from fvleg_2d_amd import _native as N
from fvleg_2d_amd.problems import uniform_nodes

pytestmark = pytest.mark.gpu
DP = C.POINTER(C.c_double)


def fields(ni, nj, nh, ld, seed=5):
    """Four fields of nj + 2 nh rows of ld values: random interiors, NaN in every ghost cell and beyond it."""
    rng = np.random.default_rng(seed)
    out = [np.full((nj + 2 * nh, ld), np.nan) for _ in range(4)]
    for k, f in enumerate(out):
        f[nh:nh + nj, nh:nh + ni] = rng.uniform(0.5, 1.5, (nj, ni)) - (1.0 if k in (1, 2) else 0.0)
    return out


BCS = [("zero_gradient",) * 4, ("periodic",) * 4, ("outflow", "symmetry", "symmetry", "zero_gradient"),
       ("pressure_input", "zero_gradient", "symmetry", "symmetry")]


# the interior's smallest sizes, strips, one tile more than a row of tiles; rows as wide as the halo'd field and
# wider (the values beyond it are the caller's); a first call, and a larger and a smaller one on the same solver
@pytest.mark.parametrize("limiter", ["minmod", "MLP5"])
@pytest.mark.parametrize("bcs", BCS, ids=lambda b: b[0])
@pytest.mark.parametrize("ni,nj", [(3, 3), (40, 3), (3, 37), (33, 25)])
@pytest.mark.parametrize("pad", [0, 5])
def test_leading_dimension(oracle, ni, nj, bcs, limiter, pad):
    cfg = SchemeConfig(flux="SLAU", limiter=limiter, bcs=bcs, bc_pressure=0.9, bc_density=0.8)
    nh = cfg.n_ghost
    nx, ny = uniform_nodes(ni, nj, nh)
    ocfg = oracle.Config(ni, nj, flux="SLAU", limiter=limiter, bcs=bcs, bc_pressure=0.9)
    og = oracle.Geometry(ocfg, nx, ny)
    ref = [np.asfortranarray(f[:, :ni + 2 * nh].T) for f in fields(ni, nj, nh, ni + 2 * nh)]
    with Solver(cfg, nx, ny) as s:
        want = s.residual(*ref)
        for ld in (ni + 2 * nh + pad, ni + 2 * nh + 2 * pad, ni + 2 * nh + pad):
            a, d = fields(ni, nj, nh, ld), [np.full((nj + 2 * nh, ld), 7.0) for _ in range(4)]
            beyond = [f[:, ni + 2 * nh:].copy() for f in a]
            ptr = [x.ctypes.data_as(DP) for x in a + d]
            N.check(s.lib.cato_residual(s.h, *ptr, ld), "residual")
            for k in range(4):
                assert np.array_equal(a[k][:, :ni + 2 * nh].T, ref[k])
                assert np.array_equal(a[k][:, ni + 2 * nh:], beyond[k], equal_nan=True)
                assert np.array_equal(d[k][:, :ni + 2 * nh].T, want[k]) and not d[k][:, ni + 2 * nh:].any()
            b = fields(ni, nj, nh, ld)
            N.check(s.lib.cato_apply_bc(s.h, *[x.ctypes.data_as(DP) for x in b], ld), "apply_bc")
            for x, y in zip(a, b):
                assert np.array_equal(x, y, equal_nan=True)
    if bcs[0] != "pressure_input":  # its inlet calls pow: parity has a test of its own, with a tolerance
        q = [np.asfortranarray(f[:, :ni + 2 * nh].T) for f in fields(ni, nj, nh, ni + 2 * nh)]
        for x, y in zip(want, oracle.solve(ocfg, og, *q)):
            assert np.array_equal(x, y)
        for x, y in zip(ref, q):
            assert np.array_equal(x, y)
