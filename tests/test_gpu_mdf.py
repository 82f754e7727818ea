"""MDF ordering on the device's block weights (GPU): the oracle's permutation over block
sizes 8 to 75, one per shape of the weight kernel, exactly (the states are perturbed at
random, so no two rows' weights are within rounding of each other)."""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nc,p", [("tri", 4, 1), ("tri", 5, 2), ("tri", 3, 4), ("tri", 2, 5), ("tet", 2, 2),
                                       ("tet", 2, 3), ("tet", 1, 4), ("hex", 3, 1), ("hex", 3, 2)])
def test_ordering_matches_oracle(oracle_mod, kind, nc, p):
    from hfem_amd.lib import HDGContext
    kw = dict(state="taylor_green", amp=1e-1) if kind == "hex" else dict(angle=0.3, elevation=0.2)
    prob = make_problem(kind, nc, p, seed=9, **kw)
    ctx = HDGContext(prob)
    ctx.assemble_linear_system()
    M = oracle_mod.BSR.from_problem(prob, ctx.read_system()[0])
    ctx.compute_ordering(1)
    o2u, nlev = ctx.get_ordering()
    print(f"{kind}{nc} p{p}: block {M.bsz}, rows {M.nrows}, levels {nlev}", flush=True)
    assert np.array_equal(o2u, oracle_mod.mdf_order(M)[0])
    ctx.close()
