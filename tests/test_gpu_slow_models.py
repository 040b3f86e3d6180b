"""Models on which every iteration gains little, in fp64 as well: 30 % of the cells, at random, 1,000
times as conductive as the rest.  The mixed solver must not give them up for the fp64 solver,
whose iterations cost more and gain no more."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("core,npad", [((24, 24, 12), 5), ((64, 48, 32), 7)])
@pytest.mark.parametrize("columns", [8, 48])
def test_mixed_solver_stays(gpu, core, npad, columns):
    from simpeg_amd import maps, workloads as W
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh = W.padded_mesh(core, npad=npad)
    survey = W.grid_survey(4, 12, 2, spacing=10.0, y_span=200.0)
    sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh))
    eng = sim.engine
    rng = np.random.default_rng(1)
    eng.set_sigma(np.where(rng.random(eng.nC) < 0.3, 10.0, 0.01))
    q = sim._source_block()[:columns].contiguous()
    _, r64 = eng.solve(q, columns, mode="fp64")
    for _ in range(2):
        _, r = eng.solve(q, columns)
        print(r64.iters, r)
        assert r.converged and r.fp64_iters == 0, (r, r64)
        assert r.iters <= 1.5 * r64.iters + 2, (r, r64)
