"""The dense inverse of the coarsest level at the edges of its blocks: meshes that are one level
(the cycle is then the inverse itself), with 8 to 150 nodes, so with one to four 32-node blocks and
on the global-memory path beyond 128.  Random coefficients, one operator and sets.  The bound is
the rounding of an elimination, condition number (below 1e4 here) times 1e-16, with a factor 100."""

import numpy as np
import pytest

from tests._helpers import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 3, 1), (7, 1, 1), (10, 2, 1), (3, 3, 3),
                                   (4, 4, 3), (7, 3, 2), (5, 4, 3), (4, 4, 4), (7, 3, 3),
                                   (5, 4, 4)])
def test_single_level_cycle_is_the_inverse(gpu, shape, bc):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(sum(shape))
    h = [rng.uniform(5.0, 15.0, n) for n in shape]
    eng = NodalEngine(h, np.zeros(3), bc_type=bc, coarse_max=200)
    x = rng.standard_normal((eng.nN, 3))
    if bc == "Neumann":
        x[0] = 0.0
    sig = np.exp(rng.standard_normal((2, eng.nC))) * 0.01
    for k in range(2):
        eng.set_sigma(sig[k])
        b = eng.apply(eng.to_block(x))
        assert rel(eng.from_block(eng.vcycle(b)), x) < 1e-10
    eng.set_sigma_sets(sig)
    cols = np.repeat(np.array([0, 1], np.int32), 8)
    q = rng.standard_normal((eng.nN, 16))
    if bc == "Neumann":
        q[0] = 0.0
    u, res = eng.solve_sets(eng.to_block(q), cols, mode="fp64")
    assert res.converged and res.iters <= 2
    eng.close()
