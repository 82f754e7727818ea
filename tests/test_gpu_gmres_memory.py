"""GMRES after a Krylov basis that did not fit into device memory (GPU): the call reports it,
and the next one allocates its own basis and returns what a fresh context returns, bit
for bit."""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", [0, 5], ids=["first", "after_a_solve"])
def test_retry_after_failed_allocation(before):
    from hfem_amd.lib import HDGContext, HfemError
    prob = make_problem("tri", 2, 1, seed=5, angle=0.3, elevation=0.2)
    out = []
    for fail in (False, True):
        ctx = HDGContext(prob)
        ctx.assemble_linear_system()
        ctx.compute_preconditioner(2)
        if before:
            ctx.gmres(restart=before, maxit=before)
        if fail:
            # (2^31 - 2 vectors of at least 100 doubles: 1.7 TB and more)
            assert prob.UH.size >= 100
            with pytest.raises(HfemError):
                ctx.gmres(restart=2 ** 31 - 2, maxit=10)
        for restart in (20, 3):
            out.append((ctx.gmres(restart=restart, tol=1e-10, maxit=40), ctx.trace_solution()))
        ctx.close()
    for (a, x), (b, y) in zip(out[:2], out[2:]):
        assert a[:2] == b[:2] and np.array_equal(a[2], b[2]) and np.array_equal(x, y)
