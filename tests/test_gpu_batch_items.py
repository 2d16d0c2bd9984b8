"""Work list of the batched stage kernel: item counts around the number of its slices and workgroups."""
import numpy as np
import pytest

from fvleg_2d_amd import Solver
from fvleg_2d_amd.batch import Batch
from fvleg_2d_amd.problems import riemann2d

pytestmark = pytest.mark.gpu


# sides in 32 x 8 tiles of each solve of a batch: 1, 7, 8 and 9 items (fewer than, as many as and one more
# than the slices), 1024 and 1025 (as many items as workgroups, and one more), 2100 (cursors and helpers)
@pytest.mark.parametrize("tiles", [[(1, 1)], [(1, 3), (2, 2)], [(2, 4)], [(3, 3)], [(16, 64)], [(16, 64), (1, 1)],
                                   [(16, 64), (1, 50), (6, 171)]], ids=lambda t: str(sum(a * b for a, b in t)))
@pytest.mark.parametrize("precision", ["fp64", "fp32_flux"])
def test_every_item_runs_once(tiles, precision):
    """Each solve of the batch is bit-identical to solving alone on the same tile, whatever the item count."""
    schemes = [("HLLC", "minmod"), ("AUSM+", "MLP5"), ("Roe", "van_leer")]
    pbs = [riemann2d(n=32 * a, nj=8 * b, seed=k, flux=schemes[k][0], limiter=schemes[k][1], precision=precision)
           for k, (a, b) in enumerate(tiles)]
    with Batch(pbs, precision=precision, tile=0) as b:
        for k, pb in enumerate(pbs):
            b.set_primitive(k, pb.rho, pb.u, pb.v, pb.p)
        it, _, err = b.run(1e300, 1e300, max_iterations=5)
        got = [b.conserved(k) for k in range(len(pbs))]
    assert list(it) == [5] * len(pbs) and not err.any()
    for pb, g in zip(pbs, got):
        pb.cfg.tile = 0
        with Solver(pb.cfg, pb.node_x, pb.node_y) as s:
            s.set_primitive(pb.rho, pb.u, pb.v, pb.p)
            s.run(1e300, 5)
            want = s.conserved()
        for x, y in zip(g, want):
            assert np.array_equal(x, y)
