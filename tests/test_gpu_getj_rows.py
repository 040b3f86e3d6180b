"""The dense sensitivity of a diagonal map derivative, whose rows are scaled on the GPU, against
the sparse product on the host: the same products in the same order, so the same numbers."""

import numpy as np
import pytest

from tests._helpers import tiny_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jchunk", [1, 5, 64])
@pytest.mark.parametrize("kind", ["exp", "identity", "rho"])
def test_scaled_rows_match_the_sparse_product(gpu, kind, jchunk, monkeypatch):
    from simpeg_amd import maps
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh, survey, m = tiny_problem(seed=4, nsrc=3)
    kw = {"exp": {"sigmaMap": maps.ExpMap(mesh)}, "identity": {"sigmaMap": maps.IdentityMap(mesh)},
          "rho": {"rhoMap": maps.IdentityMap(mesh)}}[kind]
    if kind != "exp":
        m = np.exp(m if kind == "identity" else -m)
    out = []
    for general in (False, True):
        sim = Simulation3DNodal(mesh, survey=survey, **kw)
        sim.jchunk = jchunk
        if general:
            monkeypatch.setattr(sim, "_sigma_deriv_diagonal", lambda: None)
        else:
            sim.model = m
            assert sim._sigma_deriv_diagonal() is not None
        J = sim.getJ(m)
        assert J.flags.c_contiguous and J.dtype == np.float64
        out.append(J)
    assert np.array_equal(out[0], out[1])
