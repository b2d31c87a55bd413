"""Meshes with a node that belongs to no element: its row has a diagonal block without contributions.
A solve with zero load there gives zero on that node and elsewhere what the mesh without it gives.

Device memory of the size of the block-Jacobi inverse is filled with NaN and freed before each context,
so that a block nobody writes is not finite by chance.  Both meshes take four iterations from x = 0, the
same operations summed in other groups: 1e-12 relative in FP64; in FP32, whose products round by 6e-8
each, 1e-4."""

import ctypes

import numpy as np
import pytest

from helpers import device_model, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

J2 = [210000.0, 0.3, 250.0, 1000.0, 0.0, 0.0]


def _dirty(n_nodes):
    from edelweissfe_amd import _lib

    hip = ctypes.CDLL(_lib.LIB_PATH)  # its handle resolves the HIP runtime it is linked with
    held = []
    for size in (72 * n_nodes, 36 * n_nodes):
        for _ in range(128):
            p = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0
            assert hip.hipMemcpy(p, b"\xff" * size, ctypes.c_size_t(size), 1) == 0
            held.append(p)
    assert hip.hipDeviceSynchronize() == 0
    for p in held:
        assert hip.hipFree(p) == 0


def _mesh(n, el_type, extra):
    pm = device_model(n, (1.0, 1.0, 1.0), el_type, "vonmises", J2, jitter=0.1, seed=3)
    coords, conn = pm.coordinates, pm.connectivity
    dirs = np.r_[pm.dofsOfNodeSet("gen_bottom"), pm.dofsOfNodeSet("gen_top", [1])]
    if extra is None:
        return coords, conn, dirs
    return (np.insert(coords, extra, [0.5, 0.5, 3.0], axis=0), conn + (conn >= extra),
            dirs + 3 * (dirs // 3 >= extra))


def _solve(n, el_type, extra, precision, solver, batched):
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    coords, conn, dirs = _mesh(n, el_type, extra)
    N = len(coords)
    kw = dict(specimen_of_node=np.zeros(N, dtype=np.int32), n_specimens=1) if batched else {}
    _dirty(N)
    sysm = DeviceSystem(coords, np.ascontiguousarray(conn), el_type, "vonmises", J2, **kw)
    sysm.set_dirichlet(dirs)
    rng = np.random.default_rng(5)
    n_dof = 3 * N - (0 if extra is None else 3)
    dU, b = rng.uniform(-1, 1, n_dof) * 5e-4, rng.standard_normal(n_dof)
    if extra is not None:
        dU, b = (np.insert(v.reshape(-1, 3), extra, 0.0, axis=0).ravel() for v in (dU, b))
    dU, b = torch.as_tensor(dU, device="cuda"), torch.as_tensor(b, device="cuda")
    x, P, F = sysm.zeros(), sysm.zeros(), sysm.zeros()
    sysm.compute_elements(dU, P, F, precision=precision)
    if batched:
        info, _ = sysm.linsolve_batched(b, x, np.zeros(1), precision=precision, max_iter=4, check_every=2)
    else:
        info = sysm.linsolve(b, x, solver=solver, precision=precision, rtol=0.0, max_iter=4, check_every=2)
    sysm.close()
    assert info.status == _lib.EFE_NOT_CONVERGED
    return x.cpu().numpy()


@pytest.mark.parametrize("form", ["cg", "gmres", "batched"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("el_type,n", [("C3D8", (4, 3, 3)), ("C3D20R", (3, 2, 2))])
@pytest.mark.parametrize("where", ["first", "inside", "last"])
def test_an_unattached_node_takes_no_part(form, precision, el_type, n, where):
    from edelweissfe_amd import _lib

    prec, tol = (_lib.EFE_FP64, 1e-12) if precision == "fp64" else (_lib.EFE_FP32, 1e-4)
    N = len(_mesh(n, el_type, None)[0])
    at = {"first": 0, "inside": N // 2, "last": N}[where]
    solver = _lib.EFE_SOLVER_GMRES if form == "gmres" else _lib.EFE_SOLVER_CG
    want = _solve(n, el_type, None, prec, solver, form == "batched")
    got = _solve(n, el_type, at, prec, solver, form == "batched").reshape(-1, 3)
    assert np.isfinite(got).all()
    assert (got[at] == 0.0).all()
    assert rel_err(np.delete(got, at, axis=0).ravel(), want) < tol


@pytest.mark.parametrize("form", ["cg", "batched"])
@pytest.mark.parametrize("el_type,n", [("C3D8", (4, 3, 3)), ("C3D20R", (3, 2, 2))])
@pytest.mark.parametrize("where", ["first", "inside", "last"])
def test_an_unattached_node_takes_no_part_matrix_free(form, el_type, n, where):
    from edelweissfe_amd import _lib

    N = len(_mesh(n, el_type, None)[0])
    at = {"first": 0, "inside": N // 2, "last": N}[where]
    args = (_lib.EFE_FP32_MATFREE, _lib.EFE_SOLVER_CG, form == "batched")
    want = _solve(n, el_type, None, *args)
    got = _solve(n, el_type, at, *args).reshape(-1, 3)
    assert np.isfinite(got).all()
    assert (got[at] == 0.0).all()
    assert rel_err(np.delete(got, at, axis=0).ravel(), want) < 1e-4
