"""The grid transfers at the edges of their indexing: axes of one cell, odd and even counts, axes
that are not coarsened at first, column counts around the column groups.  The cycle of separate
launches with the y and z restriction in one launch has to equal the one with the 27-point
restriction, and be symmetric (the prolongation is the restriction's transpose), both in fp64 to
the rounding of a sum over some 10^4 nodes (1e-11); a column may not depend on how many columns
run beside it beyond the rounding of a differently compiled sum (1e-13),
and the cycle on fp32 vectors has to follow to some 100 fp32 operations (1e-5)."""

import numpy as np
import pytest
import torch

from tests._helpers import rel

pytestmark = pytest.mark.gpu

SHAPES = [((1, 9, 12), (1, 1, 1)), ((12, 1, 7), (1, 1, 1)), ((13, 10, 1), (1, 1, 1)),
          ((21, 16, 9), (1, 1, 1)), ((22, 17, 10), (2, 1, 1)), ((19, 18, 12), (1, 2, 1)),
          ((24, 13, 11), (1, 1, 2))]


@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
@pytest.mark.parametrize("shape,scale", SHAPES)
def test_transfers_are_transposes(gpu, shape, scale, bc):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(sum(shape))
    h = [10.0 * s * rng.uniform(0.8, 1.2, n) for n, s in zip(shape, scale)]
    eng = NodalEngine(h, np.zeros(3), bc_type=bc,
                      params={"fused_tail": 0, "wcycle_level": 0, "vcycle_bf16": 0})
    eng.set_sigma(np.exp(rng.standard_normal(eng.nC)) * 0.01)
    a = rng.standard_normal((eng.nN, 9))
    if bc == "Neumann":
        a[0] = 0.0
    for interp in (1, 0):
        out = {}
        for sep in (1, 0):
            eng.set_params(interp=interp, xfer_separable=sep)
            out[sep] = eng.from_block(eng.vcycle(eng.to_block(a)))
            g = a.T @ out[sep]
            assert np.abs(g - g.T).max() < 1e-11 * np.abs(g).max(), (interp, sep)
        assert rel(out[1], out[0]) < 1e-11
        eng.set_params(xfer_separable=1)
        for n in (1, 2, 3, 5):
            one = eng.from_block(eng.vcycle(eng.to_block(a[:, :n])))
            assert rel(one, out[1][:, :n]) < 1e-13, (interp, n)
            f32 = eng.from_block(eng.vcycle(eng.to_block(a[:, :n], torch.float32)))
            assert rel(f32, one) < 1e-5, (interp, n)
    eng.close()
