"""What a PCG solve of a small assembled system (whose iterations test the result of the one before)
says at its limits: NaN of the very last allowed iteration, tolerances whose square overflows.

With rtol = 0 and a right-hand side near the smallest FP32 numbers the residual underflows until p.q is
0: alpha is infinite, the residual NaN.  Which iteration that is depends on the scale of b; with as many
iterations allowed, in batches of two, the NaN is the last one's."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DP = [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]  # elastic here: symmetric, and not taken by the bricks


def _system(n, el_type, precision):
    from edelweissfe_amd.device import DeviceSystem

    pm = device_model(n, (1.0, 1.0, 1.0), el_type, "druckerprager", DP, jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, "druckerprager", np.array(DP))
    sysm.set_dirichlet(pm.dofsOfNodeSet("gen_bottom"))
    sysm.compute_elements(sysm.zeros(), sysm.zeros(), sysm.zeros(), precision=precision)
    return sysm


@pytest.mark.parametrize("el_type,n", [("C3D8", (3, 2, 2)), ("C3D20R", (2, 1, 1))])
def test_nan_of_the_last_allowed_iteration(el_type, n):
    from edelweissfe_amd import _lib

    sysm = _system(n, el_type, _lib.EFE_FP32)
    b0 = np.random.default_rng(4).standard_normal(sysm.n_dof)
    found = 0
    for e in np.arange(-42.0, -30.0, 0.25):
        b = torch.as_tensor(b0 * 10.0 ** e, device="cuda")
        kw = dict(precision=_lib.EFE_FP32, rtol=0.0, check_every=2)
        info = sysm.linsolve(b, sysm.zeros(), max_iter=2000, **kw)
        if info.status != _lib.EFE_NAN or info.iterations % 2:
            continue
        found += 1
        last = sysm.linsolve(b, sysm.zeros(), max_iter=info.iterations, **kw)
        assert last.status == _lib.EFE_NAN and last.iterations == info.iterations
        if info.iterations > 2:  # not yet
            assert sysm.linsolve(b, sysm.zeros(), max_iter=info.iterations - 2, **kw).status == _lib.EFE_NOT_CONVERGED
    sysm.close()
    assert found


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("atol", [1e200, np.inf])
def test_a_tolerance_whose_square_overflows_stops_after_one_iteration(atol, precision):
    """Every tolerance above ||b|| ends the solve after its first iteration, also one whose square is
    not a number that FP64 holds: the same launches as with one that is, so the same bits."""
    from edelweissfe_amd import _lib

    prec = _lib.EFE_FP64 if precision == "fp64" else _lib.EFE_FP32
    sysm = _system((3, 2, 2), "C3D8", prec)
    b = torch.as_tensor(np.random.default_rng(4).standard_normal(sysm.n_dof), device="cuda")
    x, y = sysm.zeros(), sysm.zeros()
    want = sysm.linsolve(b, x, precision=prec, rtol=0.0, atol=1e6)
    got = sysm.linsolve(b, y, precision=prec, rtol=0.0, atol=atol)
    sysm.close()
    assert want.status == 0 and want.iterations == 1 and float(x.abs().max()) > 0
    assert got.status == 0 and got.iterations == 1 and got.residual == want.residual
    assert torch.equal(x, y)


@pytest.mark.parametrize("el_type,n", [
    ("C3D8", (1, 1, 1)),
    ("C3D8", (5, 4, 3)),
    ("C3D8", (29, 29, 30)),   # 27900 nodes: the most of the folded iteration
    ("C3D8", (29, 30, 30)),   # 28830
    ("C3D20R", (3, 2, 2)),
])
def test_every_row_of_the_fp32_solve_is_solved(el_type, n):
    """The FP32 solve by the residual of every row under the FP64 operator.  The recurrence's own is at
    most rtol ||b||; each iteration may add a rounding of K x to a row, 2^-24 of its |K| |x|, and so does
    the operator's own rounding.  A row that takes no part is left with its b, of order 1."""
    import scipy.sparse as sp

    from edelweissfe_amd import _lib

    sysm = _system(n, el_type, _lib.EFE_FP32)
    b = torch.as_tensor(np.random.default_rng(2).standard_normal(sysm.n_dof), device="cuda")
    x, y = sysm.zeros(), sysm.zeros()
    info = sysm.linsolve(b, x, precision=_lib.EFE_FP32, rtol=1e-5)
    assert info.status == 0
    sysm.compute_elements(sysm.zeros(), sysm.zeros(), sysm.zeros(), precision=_lib.EFE_FP64)
    sysm.spmv(x, y)
    indptr, indices = sysm.csr_pattern()
    K = sp.csr_matrix((sysm.export_csr_values().cpu().numpy(), indices, indptr))
    sysm.close()
    scale = (abs(K) @ abs(x.cpu().numpy())).max()
    bound = 1e-5 * info.rhs_norm + (info.iterations + 1) * 2.0 ** -24 * scale
    assert bound < 0.1
    assert float((y - b).abs().max()) <= bound
