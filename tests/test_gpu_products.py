"""Condensation of a caller's blocks over shapes at the edges of the product kernel's tiles
(GPU): na (the contraction) around multiples of 4 and 8, na and nb around the 32- and
64-wide wave blocks, one to a few elements, against numpy in FP64.  Tolerance: the
blocks are diagonally dominant (condition below 10), so an entry's error is a few na
roundings of its sums: 1e-12 relative to the largest entry.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb,n", [(1, 1, 1), (3, 2, 2), (4, 7, 1), (5, 31, 3), (8, 32, 9), (15, 33, 2), (31, 63, 4),
                                     (32, 64, 1), (33, 65, 17), (60, 60, 8), (64, 127, 3), (65, 128, 2), (100, 200, 5),
                                     (135, 270, 3), (176, 300, 2)])
def test_condense_shapes(na, nb, n):
    import torch
    from hfem_amd.lib import load
    rng = np.random.default_rng(na * 1000 + nb)
    ldx = nb + 1 + na % 3
    D = rng.standard_normal((n, na, na)) / na + 2 * np.eye(na)          # [e, column, row]
    Fx = rng.standard_normal((n, na, ldx))
    K = rng.standard_normal((n, na, nb))
    H = rng.standard_normal((n, nb + 1, nb))
    t = {k: torch.from_numpy(v.copy()).cuda() for k, v in dict(D=D, Fx=Fx, K=K, H=H).items()}
    X = torch.full((n, na, ldx), 7.0, dtype=torch.float64, device="cuda")
    info = torch.zeros(n, dtype=torch.int32, device="cuda")
    print(f"na {na} nb {nb} n {n}", flush=True)
    rc = load().hfem_condense_noalloc(na, nb, ldx, n, *[ctypes.c_void_p(t[k].data_ptr()) for k in ("D", "Fx", "K", "H")],
                                      ctypes.c_void_p(X.data_ptr()), ctypes.c_void_p(info.data_ptr()),
                                      torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    want = np.linalg.solve(D.transpose(0, 2, 1), Fx[:, :, :nb + 1])
    got = X.cpu().numpy()
    assert not info.cpu().numpy().any()
    assert np.abs(got[:, :, :nb + 1] - want).max() <= 1e-12 * np.abs(want).max()
    assert (got[:, :, nb + 1:] == 7.0).all()
    wantH = H - np.einsum("eai,eaj->eij", want, K)
    assert np.abs(t["H"].cpu().numpy() - wantH).max() <= 1e-12 * na * np.abs(wantH).max()
