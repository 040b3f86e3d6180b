"""The sums behind beta and alpha, taken inside the kernels that use them, at the edges: one
block, exactly and just over 256 blocks (65,536 nodes; beyond, separate launches), column counts
around the column groups, one and several iterations per host read, the column loop.  Potentials
agree with the fp64 solver's: both have residuals of 1e-10."""

import numpy as np
import pytest

from tests._helpers import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7, 6, 3), (15, 63, 63), (15, 63, 64)])
@pytest.mark.parametrize("ncol,check_every,col_loop", [(1, 1, 1), (3, 2, 1), (9, 1, 1), (9, 1, 8),
                                                       (17, 2, 16)])
def test_inline_sums(gpu, shape, ncol, check_every, col_loop):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(ncol)
    h = [rng.uniform(8.0, 12.0, n) for n in shape]
    eng = NodalEngine(h, np.zeros(3), params={"check_every": check_every, "col_loop": col_loop})
    eng.set_sigma(np.exp(0.5 * rng.standard_normal(eng.nC)) * 0.01)
    q = eng.to_block(rng.standard_normal((eng.nN, ncol)))
    if ncol == 9:
        q[4] = 0.0
    u, r = eng.solve(q)
    v, r64 = eng.solve(q, mode="fp64")
    assert r.converged and r.fp64_iters == 0 and r.iters <= r64.iters + 4, (r, r64)
    a, b = (x[:ncol, :eng.nN].cpu().numpy() for x in (u, v))
    for c in range(ncol):
        if b[c].any():
            assert rel(a[c], b[c]) < 1e-8, c
        else:
            assert not a[c].any()
    eng.close()
