"""Potentials of mixed Neumann solves at the default tolerance: only the grounded corner holds the
constant, so a small residual alone does not bound the shift that u has.  Against an fp64 solve to
1e-13 the potentials have to agree to 1e-9, ten times the tolerance."""

import pytest

from tests._helpers import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npad", [3, 4, 6])
@pytest.mark.parametrize("seed", [0, 1])
def test_potentials_without_a_shift(gpu, npad, seed):
    import numpy as np

    from simpeg_amd import maps, workloads as W
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh = W.padded_mesh((28, 24, 16), npad=npad)
    m = np.log(0.01) + W.gaussian_random_field(mesh, std=1.0, corr=60.0, seed=seed)
    survey = W.grid_survey(2, 4, 4, spacing=20.0, y_span=100.0)
    u = {}
    for precision, rtol in (("mixed", 1e-10), ("fp64", 1e-13)):
        sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh),
                                bc_type="Neumann", precision=precision, rtol=rtol)
        f = sim.fields(m)
        assert sim.last_solve.converged and sim.last_solve.max_rel_res <= 1e-10
        u[precision] = f.u_block[:survey.nSrc, :sim.engine.nN].cpu().numpy()
    assert rel(u["mixed"], u["fp64"]) < 1e-9
