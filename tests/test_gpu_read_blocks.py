"""Element blocks read back through the packing kernels (GPU): any range of elements is
the same bits as that range of the whole, and one output alone as all together."""
import ctypes

import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nc,p", [("tri", 2, 1), ("tri", 3, 5), ("tet", 2, 2), ("tet", 1, 4), ("hex", 3, 2)])
def test_ranges_and_single_outputs(kind, nc, p):
    from hfem_amd.lib import HDGContext, load
    prob = make_problem(kind, nc, p, seed=8)
    ctx = HDGContext(prob)
    ctx.assemble_element_matrix_vector()
    el = ctx.read_elements()
    ctx.schur_element_matrix_vector()
    ctx.sync()
    co = ctx.read_condensed()
    for e0, n in [(0, 1), (1, 2), (prob.ne - 3, 3), (prob.ne // 2, 1), (0, prob.ne - 1)]:
        print(f"{kind}{nc} p{p}: elements {e0}..{e0 + n - 1} of {prob.ne}", flush=True)
        part = ctx.read_condensed(e0, n)
        for k in co:
            assert np.array_equal(part[k], co[k][e0:e0 + n]), k
        for i, k in enumerate(["DinvRu", "DinvF", "AH", "FH"]):
            out = np.full_like(part[k], -1.0)
            args = [None] * 4
            args[i] = out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
            assert load().hfem_read_condensed(ctx.h, e0, n, *args, None) == 0
            assert np.array_equal(out, part[k]), k
    # the last column and the transposed ones against each other: D (DinvF, DinvRu) = (F, Ru)
    d = prob.dims
    na, nb = d["na"], d["nb"]
    e = prob.ne - 1
    D = el["D"][e].reshape(na, na).T
    for got, want in [(co["DinvF"][e].reshape(nb, na).T, el["F"][e].reshape(nb, na).T), (co["DinvRu"][e], el["Ru"][e])]:
        # (backward error of an explicit inverse: cond(D) * 2^-53, cond(D) < 1e6 here)
        assert np.abs(D @ got - want).max() <= 1e-9 * np.abs(want).max()
    ctx.close()
