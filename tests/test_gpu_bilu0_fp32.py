"""Single-precision BILU0 factors against double precision (GPU).

The single-precision factorisation rounds like the unblocked elimination, so its error in
M^-1 x stays at a few hundred roundings (6e-8) over the block sizes 8 to 75 on these
meshes, and does not depend on how the rows are scheduled.
"""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nc,p", [("tri", 4, 1), ("tri", 8, 2), ("tri", 5, 3), ("tri", 6, 4), ("tri", 4, 5),
                                       ("tet", 2, 1), ("tet", 3, 2), ("tet", 3, 3), ("tet", 2, 4), ("hex", 3, 2),
                                       ("hex", 5, 1)])
def test_error_against_double(kind, nc, p):
    from hfem_amd.lib import HDGContext
    kw = dict(state="taylor_green", amp=1e-3) if kind == "hex" else dict(angle=0.3, elevation=0.2)
    prob = make_problem(kind, nc, p, seed=3, **kw)
    ctx = HDGContext(prob)
    if kind == "hex":
        ctx.set_physics(10.0, 1.0, 1)
    ctx.assemble_linear_system()
    ctx.compute_ordering(1)
    x = np.random.default_rng(2).standard_normal(prob.UH.size)
    ctx.compute_preconditioner(0, 1)
    want = ctx.apply_preconditioner(x)
    got = []
    for mode in (0, 1):
        ctx.set_bilu0_sweep(mode)
        ctx.compute_preconditioner(0, 0)
        got.append(ctx.apply_preconditioner(x))
    err = np.linalg.norm(got[1] - want) / np.linalg.norm(want)
    print(f"{kind}{nc} p{p}: {err:.2e}", flush=True)
    assert np.array_equal(got[0], got[1])
    assert err < 300 * 2.0 ** -24
    ctx.close()


def test_precision_after_the_other():
    """Factors of either precision after those of the other, in the same and in a new ordering:
    the bits of a context that has only ever had the one."""
    from hfem_amd.lib import HDGContext
    prob = make_problem("tet", 2, 3, seed=3, angle=0.3, elevation=0.2)
    x = np.random.default_rng(2).standard_normal(prob.UH.size)

    def context():
        c = HDGContext(prob)
        c.assemble_linear_system()
        return c

    ctx, before = context(), None
    for order, prec in [(1, 1), (1, 0), (0, 0), (1, 0), (0, 1), (0, 0), (1, 1)]:
        fresh = context()
        for c in (ctx, fresh):
            if c is fresh or order != before:
                c.compute_ordering(order)
            c.compute_preconditioner(0, prec)
        before = order
        print(f"ordering {order} precision {prec}", flush=True)
        assert np.array_equal(ctx.apply_preconditioner(x), fresh.apply_preconditioner(x))
        fresh.close()
    ctx.close()
