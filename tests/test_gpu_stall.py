"""The mixed solver on operators whose smoothest mode is nearly free: large padded Neumann meshes
(one pinned node) and layered models on stretched padding, where fp32 rounding of the operator's
diagonal or bf16 rounding of the multigrid vectors outweighs the mode's own energy.  The fp32
phase has to converge by itself within a few iterations of the fp64 solver's count (its operator
is summed over differences, and Neumann vectors are fp32), and the fp32 operator must map a
constant to the Robin term alone, to fp32 rounding of that term."""

import numpy as np
import pytest
import torch

from tests._helpers import rel

pytestmark = pytest.mark.gpu


def _problem(bc):
    from simpeg_amd import maps, workloads as W
    from simpeg_amd.resistivity import Simulation3DNodal

    wl = W.layered_ellipsoid_model(0, core=(37, 29, 19), npad=7, nlines=1, nsrc_per_line=5, nrx=3)
    return wl, lambda **kw: Simulation3DNodal(
        wl.mesh, survey=wl.survey, sigmaMap=maps.ExpMap(wl.mesh), bc_type=bc, **kw)


@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
def test_mixed_phase_keeps_up_with_fp64(gpu, bc):
    wl, make = _problem(bc)
    u, its = {}, {}
    for precision in ("mixed", "fp64"):
        sim = make(precision=precision)
        f = sim.fields(wl.model)
        res = sim.last_solve
        assert res.converged and res.max_rel_res <= 1e-10 and res.fp64_iters == 0, res
        u[precision], its[precision] = f.u_block.cpu().numpy(), res.iters
    assert its["mixed"] <= 1.5 * its["fp64"] + 2, its
    for c in range(wl.survey.nSrc):
        assert rel(u["mixed"][c], u["fp64"][c]) < 1e-8


@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
def test_fp32_operator_of_a_constant(gpu, bc):
    """A 1 = the Robin diagonal: in fp32 the edge terms of a constant cancel exactly, so what is
    left agrees with fp64 to one rounding per term; nodes off the boundary give exactly 0 (the
    identity row of a pinned node gives 1)."""
    wl, make = _problem(bc)
    sim = make()
    sim.model = wl.model
    sim._ensure_sigma()
    eng = sim.engine
    ones = np.ones((wl.mesh.n_nodes, 3))
    a32 = eng.from_block(eng.apply(eng.to_block(ones, torch.float32)).double())
    a64 = eng.from_block(eng.apply(eng.to_block(ones)))
    assert np.abs(a32 - a64).max() <= 2.0 ** -23 * np.abs(a64).max()
    n1 = [n + 1 for n in wl.mesh.shape_cells]
    inner = a32[:, 0].reshape(n1, order="F")[1:-1, 1:-1, 1:-1]
    assert np.all(inner == 0.0)
