"""The BILU0 application as a replayed graph (GPU): the bits of its launches, level by level
and persistent, with either precision of the factors, over repeated replays with other
device work between them and after a new ordering with another number of levels."""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1], ids=["levels", "persistent"])
@pytest.mark.parametrize("prec", [1, 0], ids=["fp64", "fp32"])
@pytest.mark.parametrize("kind,nc,p", [("tri", 4, 2), ("tet", 2, 3)], ids=["tri4p2", "tet2p3"])
def test_replays_equal_launches(kind, nc, p, prec, mode):
    from hfem_amd.lib import HDGContext
    prob = make_problem(kind, nc, p, seed=4, angle=0.3, elevation=0.2)
    ctx = HDGContext(prob)
    ctx.assemble_linear_system()
    xs = [np.random.default_rng(s).standard_normal(prob.UH.size) for s in range(3)]
    ctx.set_bilu0_sweep(mode)
    levels = []
    for order in (0, 1, 0):
        ctx.compute_ordering(order)
        levels.append(ctx.get_ordering()[1])
        ctx.set_apply_graph(False)
        ctx.compute_preconditioner(0, prec_precision=prec)
        want = [ctx.apply_preconditioner(x) for x in xs]
        hist = ctx.gmres(restart=10, tol=1e-9, maxit=30)
        ctx.set_apply_graph(True)
        for rep in range(3):
            for x, w in zip(xs, want):
                assert np.array_equal(ctx.apply_preconditioner(x), w), (order, rep)
            ctx.bsr_matvec(xs[rep])
        again = ctx.gmres(restart=10, tol=1e-9, maxit=30)
        assert hist[:2] == again[:2] and np.array_equal(hist[2], again[2])
        # a graph of the factors before is not replayed for the new ones
        ctx.compute_preconditioner(0, prec_precision=prec)
        assert np.array_equal(ctx.apply_preconditioner(xs[1]), want[1])
    assert levels[0] != levels[1]
    ctx.close()
