"""The PCG on assembled systems around the size up to which its direction rides in the product (28000
nodes): the true residual of the FP64 solve, the FP32 solve against it, and solves whose last allowed
iteration is the one that converges.

The recurrence's residual, at most 1e-10 ||b||, is the true one up to the round-off of some hundred
iterations, below 1e-12 ||b||.  The FP32 solve stops at 1e-5 on an operator rounded to 6e-8: with a
condition number below 1e4 its solution is within 1e-1; the stop test at 1e-5 leaves 1e-2 typically,
so the bound checks the system, not the rounding."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DP = [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]  # elastic here: symmetric, and not taken by the bricks


def _system(n, el_type):
    from edelweissfe_amd.device import DeviceSystem

    pm = device_model(n, (1.0, 1.0, 1.0), el_type, "druckerprager", DP, jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, "druckerprager", np.array(DP))
    sysm.set_dirichlet(np.r_[pm.dofsOfNodeSet("gen_bottom"), pm.dofsOfNodeSet("gen_top", [1])])
    return sysm


def _assemble(sysm, precision):
    sysm.compute_elements(sysm.zeros(), sysm.zeros(), sysm.zeros(), precision=precision)


@pytest.mark.parametrize("el_type,n", [
    ("C3D8", (1, 1, 1)),
    ("C3D8", (5, 4, 3)),
    ("C3D8", (29, 29, 30)),   # 27900 nodes
    ("C3D8", (29, 30, 30)),   # 28830
    ("C3D20R", (3, 2, 2)),
])
def test_pcg_reaches_the_true_residual(el_type, n):
    from edelweissfe_amd import _lib

    sysm = _system(n, el_type)
    b = torch.as_tensor(np.random.default_rng(2).standard_normal(sysm.n_dof), device="cuda")
    x, x32, y = sysm.zeros(), sysm.zeros(), sysm.zeros()
    _assemble(sysm, _lib.EFE_FP32)
    i32 = sysm.linsolve(b, x32, precision=_lib.EFE_FP32, rtol=1e-5)
    _assemble(sysm, _lib.EFE_FP64)
    info = sysm.linsolve(b, x, rtol=1e-10)
    sysm.spmv(x, y)
    sysm.close()
    assert info.status == 0 and i32.status == 0
    assert info.residual <= 1e-10 * info.rhs_norm
    assert float(torch.linalg.norm(y - b) / torch.linalg.norm(b)) < 1.02e-10
    assert float(torch.linalg.norm(x32 - x) / torch.linalg.norm(x)) < 1e-1


@pytest.mark.parametrize("rtol", [1e-2, 1e-3, 1e-4, 1e-6, 1e-8])
def test_last_allowed_iteration_converges(rtol):
    sysm = _system((5, 4, 3), "C3D8")
    from edelweissfe_amd import _lib

    _assemble(sysm, _lib.EFE_FP64)
    b = torch.as_tensor(np.random.default_rng(4).standard_normal(sysm.n_dof), device="cuda")
    x, xl = sysm.zeros(), sysm.zeros()
    info = sysm.linsolve(b, x, rtol=rtol, check_every=32)
    last = sysm.linsolve(b, xl, rtol=rtol, check_every=2, max_iter=info.iterations)
    short = sysm.linsolve(b, sysm.zeros(), rtol=rtol, check_every=2, max_iter=max(2, info.iterations - 3))
    sysm.close()
    assert info.status == 0 and last.status == 0
    assert last.iterations == info.iterations and torch.equal(x, xl)
    assert short.status != 0 or info.iterations <= 3
