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


@pytest.mark.parametrize("params", [{}, {"vcycle_bf16": 0}, {"vcycle_bf16": 0, "interp": 0}])
@pytest.mark.parametrize("shape", SHAPES)
def test_recorded_cycle_follows_the_operator(gpu, shape, params):
    """A recorded V-cycle runs on the operator that is set when it is replayed, and recording one
    leaves later calls as they are, also when the operator was set between the two."""
    eng, sig, x = _engine(shape, "Robin", seed=1, **params)
    b = eng.to_block(x).float()
    ref = []
    for s in sig:
        eng.set_sigma(s)
        ref.append(eng.vcycle(b)[:, :eng.nN].cpu().numpy())
    g, z = _record(eng, b)
    for k in (0, 1, 0):
        eng.set_sigma(sig[k])
        g.replay()
        assert np.array_equal(z[:, :eng.nN].cpu().numpy(), ref[k])
        eng.set_sigma(sig[1 - k])
        h, y = _record(eng, b)
        assert np.array_equal(eng.vcycle(b)[:, :eng.nN].cpu().numpy(), ref[1 - k])
        h.replay()
        assert np.array_equal(y[:, :eng.nN].cpu().numpy(), ref[1 - k])
        del h
    torch.cuda.synchronize()
    del g
    eng.close()


@pytest.mark.parametrize("bf16", [1, 3])
@pytest.mark.parametrize("bc", ["Robin", "Neumann"])
def test_recorded_cycle_before_the_first_solve(gpu, bc, bf16):
    """A solve of no more columns leaves the memory of a recorded V-cycle where it is, though it
    keeps its vectors in another type."""
    eng, sig, x = _engine((17, 17, 17), bc, seed=3, vcycle_bf16=bf16)
    eng.set_sigma(sig[0])
    q = eng.to_block(x)
    b = q.float()
    ref = eng.vcycle(b)[:, :eng.nN].cpu().numpy()
    g, z = _record(eng, b)
    hold = []
    for _ in range(3):
        eng.solve(q, 5)
        hold.append(torch.full((64 << 20,), float("nan"), device=eng.device))  # what was freed
        g.replay()
        assert np.array_equal(z[:, :eng.nN].cpu().numpy(), ref)
    torch.cuda.synchronize()
    del g
    eng.close()


def test_recorded_cycle_beside_solves_and_sets(gpu):
    """The same with solves and operator sets on the handle between two replays."""
    eng, sig, x = _engine((17, 17, 17), "Robin", seed=2)
    q = eng.to_block(np.tile(x, (1, 4))[:, :16])
    b = q[:5].float().contiguous()
    colset = np.repeat(np.array([0, 1], np.int32), 8)
    eng.set_sigma_sets(sig)
    eng.solve_sets(q, colset)
    ref = eng.vcycle(b)[:, :eng.nN].cpu().numpy()  # set 0
    g, z = _record(eng, b)
    for _ in range(2):
        eng.set_sigma(sig[1])
        eng.solve(q, 5)
        eng.set_params(interp=0)
        eng.solve(q, 5)
        eng.set_params(interp=1)
        eng.set_sigma_sets(sig)
        u, r = eng.solve_sets(q, colset)
        assert r.converged
        eng.vcycle(b)
        g.replay()
        assert np.array_equal(z[:, :eng.nN].cpu().numpy(), ref)
    torch.cuda.synchronize()
    del g
    eng.close()
