"""The single-launch coarse tail at the edges of its sizes: top levels of just under, exactly and
just over 2, 4 and 8 nodes per work-item (the last one starts below the finest level), odd and
thin shapes with random widths, both interpolations, V- and W-cycle, operator sets.  The fp32
cycle has to agree with the fp64 one, which always runs as separate launches, to the accumulated
rounding of some 100 fp32 operations (1e-5, as for the fp32 cycle of separate launches)."""

import numpy as np
import pytest
import torch

from tests._helpers import rel

pytestmark = pytest.mark.gpu

SHAPES = [(12, 11, 12), (15, 15, 7), (16, 15, 7), (15, 15, 15), (16, 15, 15), (31, 15, 15),
          (32, 15, 15), (40, 1, 3), (23, 9, 30)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
def test_fp32_cycle_matches_fp64(gpu, shape, bc):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(sum(shape))
    h = [rng.uniform(5.0, 15.0, n) for n in shape]
    eng = NodalEngine(h, np.zeros(3), bc_type=bc, params={"vcycle_bf16": 0})
    eng.set_sigma(np.exp(rng.standard_normal(eng.nC)) * 0.01)
    a = rng.standard_normal((eng.nN, 3))
    if bc == "Neumann":
        a[0] = 0.0
    for interp in (1, 0):
        for wlevel in (-1, 0):
            eng.set_params(interp=interp, wcycle_level=wlevel)
            ref = eng.from_block(eng.vcycle(eng.to_block(a)))
            out = eng.from_block(eng.vcycle(eng.to_block(a, torch.float32)).double())
            assert rel(out, ref) < 1e-5, (interp, wlevel)
    eng.close()


@pytest.mark.parametrize("shape", [(15, 15, 15), (31, 15, 15), (32, 15, 15)])
def test_operator_sets_and_new_models(gpu, shape):
    """Each column group follows its own set's image, and a new model replaces every image."""
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(1 + sum(shape))
    h = [rng.uniform(5.0, 15.0, n) for n in shape]
    eng = NodalEngine(h, np.zeros(3))
    q = rng.standard_normal((eng.nN, 24))
    sets = np.repeat([0, 1, 2], 8)
    for _ in range(2):
        sig = np.exp(rng.standard_normal((3, eng.nC))) * 0.01
        eng.set_sigma_sets(sig)
        u, res = eng.solve_sets(eng.to_block(q), sets)
        assert res.converged and res.fp64_iters == 0
        for k in range(3):
            eng.set_sigma(sig[k])
            v, one = eng.solve(eng.to_block(q[:, 8 * k:8 * k + 8]))
            assert one.converged
            # both at a residual of 1e-10 of their right-hand side
            assert rel(u[8 * k:8 * k + 8, :eng.nN].cpu().numpy(),
                       v[:, :eng.nN].cpu().numpy()) < 1e-7
            eng.set_sigma_sets(sig)
    eng.close()
