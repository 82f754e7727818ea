"""Condensation of a caller's blocks over shapes at the edges of the product kernel's tiles
(GPU): na (the contraction) around multiples of 4 and 8, na and nb around the 32- and
64-wide wave blocks, one to a few elements, against numpy in FP64.  Tolerance: the
blocks are diagonally dominant (condition below 10), so an entry's error is a few na
roundings of its sums: 1e-12 relative to the largest entry.
"""
import numpy as np
import pytest

from test_zz_no_alloc import DeviceBuffers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb,n", [(1, 1, 1), (3, 2, 2), (4, 7, 1), (5, 31, 3), (8, 32, 9), (15, 33, 2), (31, 63, 4),
                                     (32, 64, 1), (33, 65, 17), (60, 60, 8), (64, 127, 3), (65, 128, 2), (100, 200, 5),
                                     (135, 270, 3), (176, 300, 2)])
def test_condense_shapes(na, nb, n):
    from hfem_amd.lib import load
    rng = np.random.default_rng(na * 1000 + nb)
    ldx = nb + 1 + na % 3
    D = rng.standard_normal((n, na, na)) / na + 2 * np.eye(na)          # [e, column, row]
    Fx = rng.standard_normal((n, na, ldx))
    K = rng.standard_normal((n, na, nb))
    H = rng.standard_normal((n, nb + 1, nb))
    X0 = np.full((n, na, ldx), 7.0)
    buf = DeviceBuffers()
    p = {k: buf.upload(v) for k, v in dict(D=D, Fx=Fx, K=K, H=H, X=X0, info=np.zeros(n, np.int32)).items()}
    print(f"na {na} nb {nb} n {n}", flush=True)
    assert load().hfem_condense_noalloc(na, nb, ldx, n, p["D"], p["Fx"], p["K"], p["H"], p["X"], p["info"], None) == 0
    got, gotH, info = buf.download(p["X"], X0), buf.download(p["H"], H), buf.download(p["info"], np.zeros(n, np.int32))
    buf.free()
    want = np.linalg.solve(D.transpose(0, 2, 1), Fx[:, :, :nb + 1])
    assert not info.any()
    assert np.abs(got[:, :, :nb + 1] - want).max() <= 1e-12 * np.abs(want).max()
    assert (got[:, :, nb + 1:] == 7.0).all()
    wantH = H - np.einsum("eai,eaj->eij", want, K)
    assert np.abs(gotH - wantH).max() <= 1e-12 * na * np.abs(wantH).max()
