"""The register inverse of the coarsest level away from its full sizes: 16 wavefronts hold the rows
k + 16 i, 64 lanes the columns (two each above 64 nodes), in three kernels for up to 32, 64 and 128
nodes.  One-level meshes with a remainder in the rows, the columns or both and with an early end of
the pivots in each kernel; the cycle is then the inverse itself.  Bound: as for the full sizes,
condition number (below 1e4 here) times 1e-16, with a factor 100."""

import numpy as np
import pytest

from tests._helpers import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
@pytest.mark.parametrize("shape,nodes", [((2, 1, 1), 12), ((3, 1, 1), 16), ((2, 2, 1), 18),
                                         ((2, 2, 2), 27), ((8, 1, 1), 36), ((4, 2, 2), 45),
                                         ((5, 3, 1), 48), ((6, 2, 2), 63), ((16, 1, 1), 68),
                                         ((8, 2, 2), 81), ((27, 1, 1), 112), ((6, 5, 2), 126)])
def test_remainders(gpu, shape, nodes, bc):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(nodes)
    h = [rng.uniform(5.0, 15.0, n) for n in shape]
    eng = NodalEngine(h, np.zeros(3), bc_type=bc)
    assert eng.nN == nodes and eng.levels == 1
    x = rng.standard_normal((nodes, 3))
    if bc == "Neumann":
        x[0] = 0.0
    for k in range(2):
        eng.set_sigma(np.exp(rng.standard_normal(eng.nC)) * 0.01)
        b = eng.apply(eng.to_block(x))
        assert rel(eng.from_block(eng.vcycle(b)), x) < 1e-10
        z = eng.from_block(eng.vcycle(b.float()).double())
        assert rel(z, x) < 1e4 * 2.0 ** -24 * 10  # fp32: the rounding of b and of the result
    eng.close()
