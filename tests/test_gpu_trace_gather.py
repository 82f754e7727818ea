"""The gathered trace matrix against the oracle's scatter (GPU): block sizes 8 to 75,
interior, boundary and periodic faces.  FP64 sums of at most two terms: 1e-10 of the largest
entry, the condensation's tolerance."""
import numpy as np
import pytest

from hfem_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nc,p", [("tri", 1, 1), ("tri", 3, 2), ("tri", 2, 5), ("tet", 1, 2), ("tet", 1, 4),
                                       ("hex", 3, 1), ("hex", 3, 2)])
def test_matrix_matches_oracle(oracle_mod, kind, nc, p):
    from hfem_amd.lib import HDGContext
    kw = dict(state="taylor_green", amp=1e-2) if kind == "hex" else dict(angle=0.3, elevation=0.2)
    prob = make_problem(kind, nc, p, seed=4, **kw)
    ctx = HDGContext(prob)
    print(f"{kind}{nc} p{p}: {prob.ne} elements, {prob.mesh.nf} faces", flush=True)
    ctx.assemble_linear_system()
    Hg, Rg = ctx.read_system()
    M, R, _, _ = oracle_mod.trace_system(prob)
    assert np.abs(Hg.reshape(-1) - M.blocks).max() <= 1e-10 * np.abs(M.blocks).max()
    assert np.abs(Rg.reshape(-1) - np.asarray(R).reshape(-1)).max() <= 1e-10 * np.abs(R).max()
    ctx.close()
