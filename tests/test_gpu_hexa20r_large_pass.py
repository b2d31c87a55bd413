"""hexa20R tangent passes on both sides of the size from which FP64 ones keep to 11 workgroups per CU
(25000 workgroups of two elements): the forces against the residual-only pass, bit for bit, and the
operator against the one of the FP32 pass, whose blocks and products round by 6e-8 each: 1e-5."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(36, 37, 37), (37, 37, 37)])  # 24642 and 25327 workgroups
@pytest.mark.parametrize("material,props", [("druckerprager", [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]),
                                            ("linearelastic", [180000.0, 0.25])])
def test_large_hexa20r_pass(n, material, props):
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    pm = device_model(n, (1.0, 1.0, 1.0), "C3D20R", material, props, jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, "C3D20R", material, np.array(props))
    rng = np.random.default_rng(5)
    dU = torch.as_tensor(rng.uniform(-1, 1, sysm.n_dof) * 1e-3 / max(n), device="cuda")
    x = torch.as_tensor(rng.standard_normal(sysm.n_dof), device="cuda")
    P, F, Pr, Fr, y = (sysm.zeros() for _ in range(5))
    sysm.compute_elements(dU, P, F)
    sysm.spmv(x, y)
    sysm.compute_residual(dU, Pr, Fr)
    assert torch.equal(P, Pr) and torch.equal(F, Fr)
    sysm.compute_elements(dU, Pr, Fr, precision=_lib.EFE_FP32)
    k64 = y.cpu().numpy()
    k32 = sysm.export_csr_values().cpu().numpy()
    indptr, indices = sysm.csr_pattern()
    sysm.close()
    import scipy.sparse as sp

    K = sp.csr_matrix((k32, indices, indptr))
    xh = x.cpu().numpy()
    scale = abs(K) @ abs(xh)
    assert (abs(K @ xh - k64) <= 1e-5 * scale.max()).all()
    assert np.linalg.norm(k64) > 0
