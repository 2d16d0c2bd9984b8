"""What the operator calls leave behind: device memory, and rates in the caller's own arrays."""
import ctypes as C

import numpy as np
import pytest
import torch

from fvleg_2d_amd import SchemeConfig, Solver
from fvleg_2d_amd import _native as N
from fvleg_2d_amd.problems import uniform_nodes

pytestmark = pytest.mark.gpu
DP = C.POINTER(C.c_double)
MIB = 1 << 20


def halo_fields(s, nh, seed=11):
    rng = np.random.default_rng(seed)
    return [np.asfortranarray(rng.uniform(0.5, 1.5, (s.ni + 2 * nh, s.nj + 2 * nh)) - (1.0 if k in (1, 2) else 0.0))
            for k in range(4)]


# a field is 8 MiB: the boundary fill and the flux solver take none of their own, and of the 26 fields that the edge
# fluxes take nothing beyond 64 MiB is kept (4 MiB: the granularity of the device's allocations)
def test_operator_calls_give_their_memory_back():
    cfg = SchemeConfig(flux="SLAU", limiter="minmod", bcs=("zero_gradient",) * 4)
    nh = cfg.n_ghost
    with Solver(cfg, *uniform_nodes(1024, 1024, nh)) as s:
        halo = halo_fields(s, nh)
        s.set_primitive(*[np.asfortranarray(a[nh:-nh, nh:-nh]) for a in halo])
        s.step(1e-9)
        free = torch.cuda.mem_get_info()[0]
        s.residual(*halo)
        s.apply_bc(*halo)
        assert free - torch.cuda.mem_get_info()[0] <= 4 * MIB
        edges = [e for q in halo for e in s.interpolate_edges(q)]
        s.edge_fluxes(edges, halo[3])
        assert free - torch.cuda.mem_get_info()[0] <= 68 * MIB


# narrow grids and wide rows, whose fields do not fit what a context has free, and sizes on both sides of that
@pytest.mark.parametrize("ni,nj,pad", [(400, 4, 0), (4, 400, 0), (16, 16, 0), (33, 25, 0), (33, 25, 40), (33, 25, 400)])
def test_operator_calls_leave_the_state_alone(ni, nj, pad):
    cfg = SchemeConfig(flux="SLAU", limiter="MLP5", bcs=("zero_gradient",) * 4, cfl=0.3)
    nh, ld = cfg.n_ghost, ni + 2 * cfg.n_ghost + pad
    states = []
    for operators in (False, True):
        with Solver(cfg, *uniform_nodes(ni, nj, nh)) as s:
            halo = halo_fields(s, nh)
            s.set_primitive(*[np.asfortranarray(a[nh:-nh, nh:-nh]) for a in halo])
            for k in range(3):
                if operators:
                    wide = [np.asfortranarray(np.pad(a, ((0, pad), (0, 0)))) for a in halo]
                    rates = [np.full_like(a, 7.0) for a in wide]
                    N.check(s.lib.cato_residual(s.h, *[a.ctypes.data_as(DP) for a in wide + rates], ld), "residual")
                    s.interpolate_edges(halo[0])
                s.run(1e300, 2)
            states.append(s.conserved() + s.primitive())
    for x, y in zip(*states):
        assert np.array_equal(x, y)


# the free sets after a subcycled step has swapped them
def test_residual_after_subcycled_steps():
    got = []
    for sub in (False, True):
        for integrator in ("ssp_rk2", "ssp_rk3"):
            cfg = SchemeConfig(flux="SLAU", limiter="minmod", integrator=integrator, bcs=("zero_gradient",) * 4)
            nh = cfg.n_ghost
            with Solver(cfg, *uniform_nodes(40, 33, nh)) as s:
                halo = halo_fields(s, nh)
                s.set_primitive(*[np.asfortranarray(a[nh:-nh, nh:-nh]) for a in halo])
                s.set_subcycle(sub, 1e300)
                for _ in range(3):
                    s.step(1e-4)
                    got.append(s.residual(*halo))
                got.append(s.conserved())
    half = len(got) // 2
    for a, b in zip(got[:half], got[half:]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


def test_rates_in_the_primitives_own_arrays():
    """Every value of a rate array is the rate (0 in the halo), also where it is one of the primitives' arrays."""
    cfg = SchemeConfig(flux="SLAU", limiter="minmod", bcs=("zero_gradient",) * 4)
    with Solver(cfg, *uniform_nodes(33, 25, cfg.n_ghost)) as s:
        halo = halo_fields(s, cfg.n_ghost)
        want = s.residual(*[a.copy(order="F") for a in halo])
        ptr = [a.ctypes.data_as(DP) for a in halo]
        N.check(s.lib.cato_residual(s.h, *ptr, *ptr, s.halo_shape()[0]), "residual")
        for x, y in zip(halo, want):
            assert np.array_equal(x, y)
