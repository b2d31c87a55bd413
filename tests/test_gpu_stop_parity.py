"""Solves that stop at every place of a batch of iterations: the stop flags alternate with the iteration,
so the iteration that converges must be found, and nothing changed after it, whether it is the first or
the last, an even or an odd one of its batch.  The iterations are the same launches whatever the batch:
equal counts and equal bits."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DP = [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]  # elastic here: symmetric, and not taken by the bricks


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("el_type,n", [("C3D8", (1, 1, 1)), ("C3D8", (5, 4, 3)), ("C3D20R", (3, 2, 2))])
def test_folded_pcg_stops_at_the_same_iteration_in_any_batch(el_type, n, precision):
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    prec = _lib.EFE_FP64 if precision == "fp64" else _lib.EFE_FP32
    pm = device_model(n, (1.0, 1.0, 1.0), el_type, "druckerprager", DP, jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, "druckerprager", np.array(DP))
    sysm.set_dirichlet(pm.dofsOfNodeSet("gen_bottom"))
    sysm.compute_elements(sysm.zeros(), sysm.zeros(), sysm.zeros(), precision=prec)
    b = torch.as_tensor(np.random.default_rng(4).standard_normal(sysm.n_dof), device="cuda")
    seen = set()
    for rtol in (5e-1, 2e-1, 1e-1, 5e-2, 2e-2, 1e-2, 1e-3, 1e-4):
        want = None
        for check_every in (2, 4, 6, 32):
            x = sysm.zeros()
            info = sysm.linsolve(b, x, precision=prec, rtol=rtol, check_every=check_every)
            assert info.status == 0
            got = (info.iterations, info.residual, x.cpu().numpy().tobytes())
            want = want or got
            assert got == want
            seen.add(info.iterations % 4)
    sysm.close()
    assert len(seen) >= 3


@pytest.mark.parametrize("n", [1, 300, 20000])
def test_csr_cg_stops_at_the_same_iteration_in_any_batch(n):
    import ctypes

    import scipy.sparse as sp

    from edelweissfe_amd import _lib

    rng = np.random.default_rng(n)
    i, j = rng.integers(0, n, 6 * n), rng.integers(0, n, 6 * n)
    A = sp.coo_matrix((rng.uniform(-1, 1, i.size), (i, j)), shape=(n, n)).tocsr()
    A = A + A.T
    A = A - sp.diags(A.diagonal())
    A = sp.csr_matrix(A + sp.diags(1.05 * np.asarray(abs(A).sum(axis=1)).ravel() + 0.01))
    A.sort_indices()
    ip, ix = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    b = rng.standard_normal(n)
    seen = set()
    for rtol in (5e-1, 2e-1, 1e-1, 3e-2, 1e-2, 1e-3, 1e-5, 1e-10):
        want = None
        for check_every in (1, 2, 3, 5, 32):
            x = np.empty(n)
            o = _lib.SolveOpts(solver=_lib.EFE_SOLVER_CG, max_iter=2000, check_every=check_every, rtol=rtol)
            info = _lib.SolveInfo()
            _lib.check(_lib.load().efe_csr_linsolve(n, ip.ctypes.data, ix.ctypes.data, A.data.ctypes.data,
                                                    b.ctypes.data, x.ctypes.data, ctypes.byref(o),
                                                    ctypes.byref(info)), "efe_csr_linsolve")
            assert info.status == 0
            got = (info.iterations, info.residual, x.tobytes())
            want = want or got
            assert got == want
            seen.add(info.iterations % 2)
    assert n == 1 or len(seen) == 2
