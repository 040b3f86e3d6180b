"""One iteration between two host reads (the host launches what the decision's note asks for)
against several (the same kernels are always launched and test the control block): the kernels
that do work are the same, so the potentials, iterations and updates are too; the edges are an
iteration limit of one, right-hand sides without any source and zero columns beside others."""

import numpy as np
import pytest

from tests._helpers import tiny_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["mixed", "fp64"])
@pytest.mark.parametrize("max_iter", [1, 2, 200])
@pytest.mark.parametrize("zero", ["none", "some", "all"])
def test_notes_and_control_block_agree(gpu, mode, max_iter, zero):
    from simpeg_amd import maps
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh, survey, m = tiny_problem(seed=2, nsrc=4)
    sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh))
    eng = sim.engine
    ns = survey.nSrc
    q = sim._source_block().clone()
    if zero == "some":
        q[1:3] = 0.0
    elif zero == "all":
        q[:] = 0.0
    out = []
    for check_every in (1, 3):
        eng.set_params(check_every=check_every)
        eng.set_sigma(np.exp(m))  # forgets a stalled solve
        u, r = eng.solve(q, ns, mode=mode, max_iter=max_iter, raise_on_fail=False)
        out.append((u[:ns, :eng.nN].cpu().numpy(), r))
    (a, ra), (b, rb) = out
    assert np.array_equal(a, b)
    assert (ra.iters, ra.outer, ra.converged, ra.fp64_iters) == \
        (rb.iters, rb.outer, rb.converged, rb.fp64_iters)
    assert ra.max_rel_res == rb.max_rel_res
    if zero == "all":
        assert ra.converged and not a.any()
