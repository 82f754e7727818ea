"""Trace graphs a caller may pass beyond the mesh's own (GPU): rows in any order, further
blocks on one side of the diagonal only, a column or the diagonal listed twice.

BILU0 takes a row's neighbours in the order of their numbers and the first block of a
column (kernel/computeBILU0.m), MDF weights count pairs of unnumbered neighbours
(kernel/computeMDFordering.m), a block the graph does not have being zero: against those in
numpy, to 1e-10 relative, the tolerance of the other preconditioner tests, and the same
permutation.
"""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


def widened(mesh, rng, extra, twice):
    """The mesh's graph with `extra` further columns a row, its rows shuffled, and again at
    the end of every other row its entry `twice` (0: the diagonal, None: none)."""
    start, cols = [0], []
    for i in range(mesh.nf):
        row = list(mesh.ent2ent[mesh.ent2entStart[i] + 1:mesh.ent2entStart[i + 1]])
        row += list(rng.permutation(np.setdiff1d(np.arange(mesh.nf), row + [i]))[:extra])
        cols += [i] + list(rng.permutation(row))
        if twice is not None and i % 2:
            cols.append(cols[start[-1] + twice])
        start.append(len(cols))
    mesh.ent2entStart, mesh.ent2ent = np.array(start, dtype=np.int64), np.array(cols, dtype=np.int64)


def first_in_row(rp, ci, row, col):
    return next((m for m in range(rp[row] + 1, rp[row + 1]) if ci[m] == col), -1)


def bilu0(rp, ci, o2u, u2o, B):
    for r in o2u:
        lower = [k for k in range(rp[r] + 1, rp[r + 1]) if u2o[ci[k]] < u2o[r]]
        for k in sorted(lower, key=lambda k: u2o[ci[k]]):
            B[k] = B[k] @ B[rp[ci[k]]]
            for l in range(rp[r], rp[r + 1]):
                m = first_in_row(rp, ci, ci[k], ci[l])
                if m >= 0 and (l == rp[r] or u2o[ci[l]] > u2o[ci[k]]):
                    B[l] -= B[k] @ B[m]
        B[rp[r]] = np.linalg.inv(B[rp[r]])


def bilu0_solve(rp, ci, o2u, u2o, B, x):
    v = x.reshape(len(o2u), -1).copy()
    for r in o2u:
        for k in range(rp[r] + 1, rp[r + 1]):
            if u2o[ci[k]] < u2o[r]:
                v[r] -= B[k] @ v[ci[k]]
    for r in o2u[::-1]:
        for k in range(rp[r] + 1, rp[r + 1]):
            if u2o[ci[k]] > u2o[r]:
                v[r] -= B[k] @ v[ci[k]]
        v[r] = B[rp[r]] @ v[r]
    return v.reshape(-1)


def mdf(rp, ci, H):
    n = len(rp) - 1
    C = np.array([np.linalg.norm(np.linalg.solve(H[rp[i]], H[k])) for i in range(n) for k in range(rp[i], rp[i + 1])])
    numbered = np.zeros(n, bool)

    def weight(k):
        s = 0.0
        nbr = [m for m in range(rp[k] + 1, rp[k + 1]) if not numbered[ci[m]]]
        for i in nbr:
            back = first_in_row(rp, ci, ci[i], k)
            near = set(ci[rp[ci[i]]:rp[ci[i] + 1]])
            for j in nbr:
                if j != i and ci[j] not in near and back >= 0:
                    s += (C[back] * C[j]) ** 2
        return np.sqrt(s)

    w, order = np.array([weight(k) for k in range(n)]), []
    for _ in range(n):
        p = int(np.argmin(np.where(numbered, np.inf, w)))
        order.append(p)
        numbered[p] = True
        for k in ci[rp[p] + 1:rp[p + 1]]:
            if not numbered[k]:
                w[k] = weight(k)
    return np.array(order)


@pytest.mark.parametrize("extra,twice", [(3, None), (0, 1), (3, 1), (0, 0)],
                         ids=["one_sided", "twice", "both", "diagonal"])
@pytest.mark.parametrize("kind,nc,p,seed", [("tri", 3, 2, 0), ("tri", 4, 1, 1), ("tet", 1, 2, 2)])
def test_bilu0(kind, nc, p, seed, extra, twice):
    from hfem_amd.lib import HDGContext
    rng = np.random.default_rng(seed)
    prob = make_problem(kind, nc, p, seed=3, angle=0.3, elevation=0.2)
    widened(prob.mesh, rng, extra, twice)
    rp, ci, n = prob.mesh.ent2entStart, prob.mesh.ent2ent, prob.mesh.nf
    ctx = HDGContext(prob)
    ctx.assemble_linear_system()
    bsz = prob.UH.size // n
    B = ctx.read_system()[0].reshape(-1, bsz, bsz).transpose(0, 2, 1).copy()
    x = rng.standard_normal(n * bsz)
    o2u = rng.permutation(n)
    u2o = np.argsort(o2u)
    bilu0(rp, ci, o2u, u2o, B)
    want = bilu0_solve(rp, ci, o2u, u2o, B, x)
    for mode in (0, 1):
        ctx.set_bilu0_sweep(mode)
        ctx.set_ordering(o2u)
        ctx.compute_preconditioner(0)
        err = np.linalg.norm(ctx.apply_preconditioner(x) - want) / np.linalg.norm(want)
        print(f"{kind}{nc} p{p} mode {mode}: {n} rows, relative error {err:.1e}", flush=True)
        assert err < 1e-10
    ctx.close()


@pytest.mark.parametrize("extra,twice", [(0, None), (3, None), (0, 1), (3, 1), (0, 0)],
                         ids=["shuffled", "one_sided", "twice", "both", "diagonal"])
@pytest.mark.parametrize("kind,nc,p,seed", [("tri", 3, 2, 0), ("tri", 4, 1, 1), ("tet", 1, 2, 2)])
def test_mdf_ordering(kind, nc, p, seed, extra, twice):
    from hfem_amd.lib import HDGContext
    prob = make_problem(kind, nc, p, seed=3, angle=0.3, elevation=0.2)
    widened(prob.mesh, np.random.default_rng(seed), extra, twice)
    ctx = HDGContext(prob)
    ctx.assemble_linear_system()
    bsz = prob.UH.size // prob.mesh.nf
    H = ctx.read_system()[0].reshape(-1, bsz, bsz).transpose(0, 2, 1)
    ctx.compute_ordering(1)
    print(f"{kind}{nc} p{p}: {prob.mesh.nf} rows", flush=True)
    assert np.array_equal(ctx.get_ordering()[0], mdf(prob.mesh.ent2entStart, prob.mesh.ent2ent, H))
    ctx.close()


@pytest.mark.parametrize("column", [-1, 33, 2 ** 31 - 1], ids=["negative", "rows", "largest"])
def test_column_out_of_range_is_refused(column):
    """A further block with such a column is refused, and the mesh set before stays in use."""
    from hfem_amd.lib import HDGContext, HfemError, _d, _f64, _i, _i32, load
    prob = make_problem("tri", 3, 2, seed=3, angle=0.3, elevation=0.2)
    mesh = prob.mesh
    assert mesh.nf == 33
    mesh.ent2entStart[-1] += 1
    mesh.ent2ent = np.append(mesh.ent2ent, 0)
    ctx = HDGContext(prob)
    ctx.assemble_linear_system()
    ctx.compute_preconditioner(0)
    x = np.random.default_rng(0).standard_normal(prob.UH.size)
    want = ctx.apply_preconditioner(x)
    mesh.ent2ent[-1] = column
    with pytest.raises(HfemError, match="column"):
        HDGContext(prob)
    rc = load().hfem_set_mesh(ctx.h, _d(_f64(prob.dgnodes_ref())), _i(_i32(mesh.elcon)), _i(_i32(mesh.bf)),
                              _i(_i32(mesh.t2f)), _i(_i32(mesh.ent2entStart)), _i(_i32(mesh.ent2ent)), len(mesh.ent2ent))
    assert rc != 0
    assert np.array_equal(ctx.apply_preconditioner(x), want)
    ctx.close()
