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


def test_reads_of_several_chunks():
    """162 p=4 tets: 8.5 M doubles of DinvF and 14.6 M of AH, more than the staging buffer
    takes at once.  Elements at the chunks' edges read one by one give the same bits, also
    with the buffer sized by a smaller read before, and D DinvF = F either side of an edge."""
    from hfem_amd.lib import HDGContext, load
    prob = make_problem("tet", 3, 4, seed=8)
    na, nb, ne = prob.dims["na"], prob.dims["nb"], prob.ne
    cap = 1 << 22
    ctx = HDGContext(prob)
    ctx.assemble_element_matrix_vector()
    fh = np.zeros((2, nb))
    ctx.schur_element_matrix_vector()
    ctx.sync()
    assert load().hfem_read_condensed(ctx.h, 0, 2, None, None, None, fh.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                      None) == 0
    whole = ctx.read_condensed()
    assert np.array_equal(fh, whole["FH"][:2])
    edges = {0, ne - 1}
    for per in (na * nb, nb * nb):
        m = cap // per
        assert 1 < m < ne and ne % m
        edges |= {e for e in range(m - 1, ne, m)} | {e for e in range(m, ne, m)}
    for e in sorted(edges):
        print(f"element {e} of {ne}", flush=True)
        one = ctx.read_condensed(e, 1)
        for k in whole:
            assert np.array_equal(one[k][0], whole[k][e]), k
    ctx.assemble_element_matrix_vector()
    for e in (cap // (na * nb) - 1, cap // (na * nb)):
        el = ctx.read_elements(e, 1)
        D, F = el["D"][0].reshape(na, na).T, el["F"][0].reshape(nb, na).T
        # (backward error of an explicit inverse: cond(D) * 2^-53, cond(D) < 1e6 here)
        assert np.abs(D @ whole["DinvF"][e].reshape(nb, na).T - F).max() <= 1e-9 * np.abs(F).max()
    ctx.close()
