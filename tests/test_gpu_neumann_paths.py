"""Every path of a mixed solve on a Neumann operator aims at the same residual, tol / 32: the shift
of the potentials that a residual at the tolerance can hide is then below ten times the tolerance
(against an fp64 solve to 1e-13), also when an earlier solve gave the operator up for fp64."""

import numpy as np
import pytest

from tests._helpers import rel

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _problem(npad, seed):
    from simpeg_amd import maps, workloads as W
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh = W.padded_mesh((28, 24, 16), npad=npad)
    m = np.log(0.01) + W.gaussian_random_field(mesh, std=1.0, corr=60.0, seed=seed)
    survey = W.grid_survey(2, 4, 4, spacing=20.0, y_span=100.0)
    sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh), bc_type="Neumann")
    sim.model = m
    sim._ensure_sigma()
    q, n = sim._source_block(), survey.nSrc
    ref, _ = sim.engine.solve(q, n, mode="fp64", tol=1e-13)
    return sim.engine, q, n, ref[:n, :sim.engine.nN].cpu().numpy()


@pytest.mark.parametrize("npad", [3, 4, 6])
@pytest.mark.parametrize("seed", [0, 1])
def test_solves_after_a_stalled_one(gpu, npad, seed):
    eng, q, n, ref = _problem(npad, seed)
    eng.solve(q, n, max_iter=1, raise_on_fail=False)  # one iteration: given up
    u, r = eng.solve(q, n, tol=TOL)
    assert r.converged and r.iters == 0 and r.fp64_iters > 0, r  # fp64 from the start
    assert r.max_rel_res <= 1.01 * TOL / 32, r
    assert rel(u[:n, :eng.nN].cpu().numpy(), ref) < 1e-9


@pytest.mark.parametrize("npad", [3, 4, 6])
@pytest.mark.parametrize("seed", [0, 1])
def test_iterative_refinement(gpu, npad, seed):
    eng, q, n, ref = _problem(npad, seed)
    _, r64 = eng.solve(q, n, mode="fp64", tol=TOL)
    u, r = eng.solve(q, n, mode="mixed_ir", tol=TOL)
    print(r64, r)
    assert r.converged and r.max_rel_res <= TOL / 32, r
    assert r.iters <= 2 * r64.iters, (r, r64)
    assert rel(u[:n, :eng.nN].cpu().numpy(), ref) < 1e-9
