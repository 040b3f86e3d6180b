"""The automatic choice between V- and W-cycle at its line, 262,144 nodes: the cycle it runs is the
one of the explicit level, and the W step inside the coarse tail, now only run on request on
small meshes, follows the fp64 cycle of separate launches (1e-5: some 100 fp32 operations)."""

import numpy as np
import pytest
import torch

from tests._helpers import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,bc,level", [((63, 63, 62), "Robin", 0), ((63, 63, 63), "Robin", 1),
                                            ((63, 63, 62), "Neumann", 1)])
def test_automatic_level(gpu, shape, bc, level):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(3)
    eng = NodalEngine([np.full(n, 10.0) for n in shape], np.zeros(3), bc_type=bc)
    eng.set_sigma(np.exp(0.5 * rng.standard_normal(eng.nC)) * 0.01)
    b = eng.to_block(rng.standard_normal((eng.nN, 2)))
    out = {}
    for w in (-1, 0, 1):
        eng.set_params(wcycle_level=w)
        out[w] = eng.from_block(eng.vcycle(b))
    assert np.array_equal(out[-1], out[level])
    assert not np.array_equal(out[0], out[1])
    eng.close()


@pytest.mark.parametrize("shape", [(12, 11, 12), (15, 15, 15), (31, 15, 15)])
@pytest.mark.parametrize("level", [1, 2])
def test_w_step_in_the_tail(gpu, shape, level):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(sum(shape))
    h = [rng.uniform(5.0, 15.0, n) for n in shape]
    eng = NodalEngine(h, np.zeros(3), params={"vcycle_bf16": 0, "wcycle_level": level},
                      coarse_max=30)
    eng.set_sigma(np.exp(rng.standard_normal(eng.nC)) * 0.01)
    a = rng.standard_normal((eng.nN, 3))
    ref = eng.from_block(eng.vcycle(eng.to_block(a)))
    out = eng.from_block(eng.vcycle(eng.to_block(a, torch.float32)).double())
    assert rel(out, ref) < 1e-5
    eng.close()


def test_columns_choose_the_cycle_of_a_solve(gpu):
    """Few columns on a large mesh take the V-cycle, many the W-cycle, whatever was solved and
    recorded before: the potentials are those of the explicit levels."""
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(4)
    eng = NodalEngine([np.full(63, 10.0)] * 3, np.zeros(3))
    eng.set_sigma(np.exp(0.5 * rng.standard_normal(eng.nC)) * 0.01)
    q = eng.to_block(rng.standard_normal((eng.nN, 33)))
    cases = {3: 0, 31: 0, 33: 1}  # 2^18 nodes x 32 columns = 2^23
    ref = {}
    for n, level in cases.items():
        eng.set_params(wcycle_level=level)
        ref[n] = eng.solve(q[:n].contiguous(), n)
    eng.set_params(wcycle_level=-1)
    for _ in range(2):
        for n in cases:
            u, r = eng.solve(q[:n].contiguous(), n)
            assert r.converged and r.iters == ref[n][1].iters
            assert torch.equal(u, ref[n][0]), n
    eng.close()
