"""One handle used for solves and for single V-cycles in turn.  The two may run the coarse tail from
different levels on and keep their vectors in different types (Neumann solves always fp32), but
neither may undo what the other has in hand: same bits as on handles of their own, and a V-cycle
between solves stays a mere sequence of launches, so that a caller can record it in a graph."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# the finest level inside the tail (5,832 nodes), and above it (27,000)
SHAPES = [(17, 17, 17), (29, 29, 29)]


def _engine(shape, bc, seed=0, **params):
    from simpeg_amd.engine import NodalEngine

    rng = np.random.default_rng(seed)
    eng = NodalEngine([rng.uniform(5.0, 15.0, n) for n in shape], np.zeros(3), bc_type=bc,
                      params=params or None)
    sig = np.exp(rng.standard_normal((2, eng.nC))) * 0.01
    x = rng.standard_normal((eng.nN, 5))
    if bc == "Neumann":
        x[0] = 0.0
    return eng, sig, x


def _record(eng, b):
    """eng.vcycle(b) as a graph: (graph, its output)."""
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        z = eng.vcycle(b)
    return g, z


@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
@pytest.mark.parametrize("shape", SHAPES)
def test_solves_and_cycles_in_turn(gpu, shape, bc):
    ref = {}
    for kind in ("solve", "cycle", "both"):
        eng, sig, x = _engine(shape, bc)
        eng.set_sigma(sig[0])
        q = eng.to_block(x)
        b = q.float()
        if kind == "both":
            eng.vcycle(b)
            eng.solve(q, 5)
            g, z = _record(eng, b)
        for _ in range(3):
            if kind != "cycle":
                u, r = eng.solve(q, 5)
                got = (u[:5, :eng.nN].cpu().numpy(), r.iters)
                if kind == "solve":
                    ref[kind] = got
                else:
                    assert got[1] == ref["solve"][1] and np.array_equal(got[0], ref["solve"][0])
            if kind != "solve":
                c = eng.vcycle(b)[:, :eng.nN].cpu().numpy()
                if kind == "cycle":
                    ref[kind] = c
                else:
                    assert np.array_equal(c, ref["cycle"])
                    g.replay()
                    assert np.array_equal(z[:, :eng.nN].cpu().numpy(), ref["cycle"])
        torch.cuda.synchronize()
        if kind == "both":
            del g
        eng.close()
