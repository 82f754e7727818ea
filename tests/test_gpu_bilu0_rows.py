"""BILU0 factorisation and sweeps over every block size's kernel shape (GPU).

Block sizes 8 to 75 (triangles p=1-5, tets p=1-4, hexes p=1-2), rows with no, few and
more neighbours than a sweep keeps in registers.  Against the CPU oracle to 1e-10
relative, the tolerance of the other preconditioner tests (different summation
orders); the one-launch and level-launched forms bit for bit.
"""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu

FAMILIES = [("tri", 3, 1), ("tri", 3, 2), ("tri", 3, 3), ("tri", 2, 4), ("tri", 2, 5), ("tet", 2, 1), ("tet", 1, 2),
            ("tet", 1, 3), ("tet", 1, 4), ("hex", 3, 1), ("hex", 3, 2)]


@pytest.fixture(scope="module", params=FAMILIES, ids=lambda c: f"{c[0]}{c[1]}p{c[2]}")
def solver(request, oracle_mod):
    from hfem_amd.lib import HDGContext
    kind, nc, p = request.param
    kw = dict(state="taylor_green", amp=1e-3) if kind == "hex" else dict(angle=0.3, elevation=0.2)
    prob = make_problem(kind, nc, p, seed=6, **kw)
    ctx = HDGContext(prob)
    if kind == "hex":
        ctx.set_physics(10.0, 1.0, 1)
    ctx.assemble_linear_system()
    M = oracle_mod.BSR.from_problem(prob, ctx.read_system()[0])
    o2u, u2o = oracle_mod.mdf_order(M)
    ctx.set_ordering(o2u)
    print(f"{kind}{nc} p{p}: block {M.bsz}, rows {M.nrows}, levels {ctx.get_ordering()[1]}", flush=True)
    yield ctx, M, o2u, u2o
    ctx.close()


def test_application_matches_oracle(oracle_mod, solver):
    ctx, M, o2u, u2o = solver
    ctx.compute_preconditioner(0)
    Mg, _ = oracle_mod.bilu0_factor(M, o2u, u2o)
    x = np.random.default_rng(1).standard_normal(M.nrows * M.bsz)
    want = oracle_mod.bilu0_apply(M, o2u, u2o, Mg, x)
    got = ctx.apply_preconditioner(x)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"  relative error {err:.2e}", flush=True)
    assert err < 1e-10


@pytest.mark.parametrize("prec", [1, 0], ids=["fp64", "fp32"])
def test_one_launch_equals_levels(solver, prec):
    ctx, M, _, _ = solver
    xs = [np.random.default_rng(s).standard_normal(M.nrows * M.bsz) for s in range(2)]
    # NaN and infinity travel as in the level launches; one is the pattern that marks a
    # vector entry as not yet written
    xs.append(xs[0].copy())
    xs[2][[0, M.nrows * M.bsz // 2]] = np.nan, np.inf
    xs.append(xs[1].copy())
    xs[3].view(np.uint64)[3] = 0x7ff4dead5eed0001
    try:
        ctx.set_bilu0_sweep(0)
        ctx.compute_preconditioner(0, prec_precision=prec)
        ref = [ctx.apply_preconditioner(x) for x in xs]
        ctx.set_bilu0_sweep(1)
        ctx.compute_preconditioner(0, prec_precision=prec)
        for rep in range(3):
            for x, r in zip(xs, ref):
                assert np.array_equal(ctx.apply_preconditioner(x), r, equal_nan=True), rep
    finally:
        ctx.set_bilu0_sweep(1)
