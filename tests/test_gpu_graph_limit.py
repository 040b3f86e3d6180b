"""More column counts than the cache of recorded iterations has room for (64 graphs, six per count
in the mixed solver): solves in whose middle the cache starts over give the bits of solves
without recording, and so do the counts that have to be recorded again."""

import numpy as np
import pytest

from tests._helpers import tiny_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["mixed", "fp64"])
def test_solves_while_the_cache_starts_over(gpu, mode):
    from simpeg_amd import maps
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh, survey, m = tiny_problem(seed=3, nsrc=4)
    sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh))
    eng = sim.engine
    eng.set_sigma(np.exp(m))
    rng = np.random.default_rng(5)
    # six graphs per count, or (fp64) the first cycle and one iteration
    counts = list(range(1, 15 if mode == "mixed" else 37))
    q = eng.to_block(rng.standard_normal((eng.nN, counts[-1])))
    ref = {}
    eng.set_params(graph=0)
    for n in counts:  # (also the workspace of the most columns)
        ref[n] = eng.solve(q[:n].contiguous(), n, mode=mode)
    eng.set_params(graph=1)
    for n in counts + [3, 1, 14, 2]:
        u, r = eng.solve(q[:n].contiguous(), n, mode=mode)
        assert (r.iters, r.converged) == (ref[n][1].iters, True)
        a, b = (x[:n, :eng.nN].cpu().numpy() for x in (u, ref[n][0]))
        assert np.array_equal(a, b), n
