"""Errors of solves at the default parameters and tolerance against those with the W step on the
first level of at most a quarter of the nodes, on Robin meshes where the automatic cycle can be
the V-cycle (below 262,144 nodes, and few columns on a larger mesh): the V-cycle leaves more of
the smooth error at the same residual, so its solves have to work towards a smaller one.  A single
pair depends on where the last iteration lands, so the geometric mean over the models and columns
is compared."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["mixed", "fp64"])
@pytest.mark.parametrize("core,npad,columns,wlevel", [((24, 24, 12), 5, (2, 8), 2),
                                                      ((48, 40, 26), 6, (2, 8), 1),
                                                      ((72, 64, 40), 7, (1, 8), 1)])
def test_errors_not_above_those_of_the_w_cycle(gpu, mode, core, npad, columns, wlevel):
    from simpeg_amd import maps, workloads as W
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh = W.padded_mesh(core, npad=npad)
    survey = W.grid_survey(2, 4, 2, spacing=20.0, y_span=100.0)
    sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh))
    eng = sim.engine
    q = sim._source_block()
    ratio = []
    for seed in range(3):
        m = np.log(0.01) + W.gaussian_random_field(mesh, std=1.0, corr=60.0, seed=seed)
        for n in columns:
            b = q[:n].contiguous()
            eng.set_sigma(np.exp(m))
            ref, _ = eng.solve(b, n, mode="fp64", tol=2e-14)
            err = {}
            for level in (-1, wlevel):
                eng.set_params(wcycle_level=level)
                u, r = eng.solve(b, n, mode=mode)
                assert r.converged and r.max_rel_res <= 1e-10, r
                d = (u[:n, :eng.nN] - ref[:n, :eng.nN]).norm(dim=1) / ref[:n, :eng.nN].norm(dim=1)
                err[level] = float(d.max())
            eng.set_params(wcycle_level=-1)
            ratio.append(err[-1] / err[wlevel])
    print(mode, core, ["%.2f" % v for v in ratio])
    assert np.exp(np.mean(np.log(ratio))) <= 1.0


@pytest.mark.parametrize("core,npad,std,columns", [((24, 24, 12), 5, 4.0, 8),
                                                   ((64, 48, 32), 7, 4.0, 8)])
def test_rough_models(gpu, core, npad, std, columns):
    """White noise of standard deviation 4 in the log conductivity: default mixed solves converge
    within the default iteration limit and agree with fp64 ones (which the W-cycle does not
    reach on the larger mesh)."""
    from simpeg_amd import maps, workloads as W
    from simpeg_amd.resistivity import Simulation3DNodal

    mesh = W.padded_mesh(core, npad=npad)
    survey = W.grid_survey(2, 4, 2, spacing=10.0, y_span=100.0)
    sim = Simulation3DNodal(mesh, survey=survey, sigmaMap=maps.ExpMap(mesh))
    eng = sim.engine
    eng.set_sigma(0.01 * np.exp(std * np.random.default_rng(1).standard_normal(eng.nC)))
    q = sim._source_block()[:columns].contiguous()
    u, res = eng.solve(q, columns)
    assert res.converged and res.max_rel_res <= 1e-10, res
    ref, _ = eng.solve(q, columns, mode="fp64", tol=1e-12)
    d = (u - ref)[:columns, :eng.nN].norm(dim=1) / ref[:columns, :eng.nN].norm(dim=1)
    print(res, float(d.max()))
    assert float(d.max()) < 1e-6  # a contrast of e^30 amplifies the residual
