"""Element passes and assembly at the edges of their tiles: hexa8 takes 8 elements per wavefront
(1, 7, 8, 9 and 18 elements), the assembly shares a slice of 64 rows out over 4 or 8 wavefronts by
blocks (rows of 8 to 81 blocks).  K, P and the Dirichlet correction against the oracle's element
matrices, assembled densely: 1e-12 relative in FP64 (sums of at most 216 terms of round-off 1e-16,
on strains of relative round-off 1e-14), 3e-6 in FP32 (the bound of the matrix-free operator
test).  The residual-only pass equals the tangent pass bit for bit."""

import numpy as np
import pytest

from helpers import device_model, oracle_model, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

PROPS = {"linearelastic": [210000.0, 0.3], "vonmises": [210000.0, 0.3, 250.0, 1000.0, 0.0, 0.0],
         "druckerprager": [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]}


@pytest.mark.parametrize("material", sorted(PROPS))
@pytest.mark.parametrize("el_type,n", [("C3D8", (1, 1, 1)), ("C3D8", (7, 1, 1)), ("C3D8", (2, 2, 2)),
                                       ("C3D8", (3, 3, 1)), ("C3D8", (2, 3, 3)), ("C3D20", (1, 1, 1)),
                                       ("C3D20", (2, 2, 2)), ("C3D20R", (3, 1, 2))])
def test_pass_and_assembly_at_tile_edges(material, el_type, n):
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    om = oracle_model(n, (1.0, 1.0, 1.0), el_type, material, PROPS[material], jitter=0.1, seed=6)
    pm = device_model(n, (1.0, 1.0, 1.0), el_type, material, PROPS[material], jitter=0.1, seed=6)
    rng = np.random.default_rng(8)
    dU = rng.uniform(-1, 1, om.nDof) * 2e-3
    dm = om.elements.dof_map
    Ke, Pe, _ = om.elements.compute(dU[dm], om.state, om.material)
    D = om.nDof
    K, P = np.zeros((D, D)), np.zeros(D)
    for e in range(dm.shape[0]):
        K[np.ix_(dm[e], dm[e])] += Ke[e]
        np.add.at(P, dm[e], Pe[e])
    dirs = np.unique(pm.dofsOfNodeSet("gen_bottom"))
    v = np.zeros(D)
    v[dirs] = rng.uniform(-1, 1, dirs.size)
    corr = K @ v
    corr[dirs] = 0.0
    Ke_el = K.copy()
    Ke_el[dirs] = 0.0
    Ke_el[:, dirs] = 0.0
    Ke_el[dirs, dirs] = 1.0

    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, material, PROPS[material])
    sysm.set_dirichlet(dirs)
    td, tv = torch.as_tensor(dU, device="cuda"), torch.as_tensor(v, device="cuda")
    ip, ix = sysm.csr_pattern()
    rows = np.repeat(np.arange(D), np.diff(ip))
    for prec, tol in ((_lib.EFE_FP64, 1e-12), (_lib.EFE_FP32, 3e-6)):
        Pd, Fd, cd, Pr, Fr = (sysm.zeros() for _ in range(5))
        sysm.compute_elements(td, Pd, Fd, dir_values=tv, dir_correction=cd, precision=prec)
        Kd = np.zeros((D, D))
        Kd[rows, ix] = sysm.export_csr_values().cpu().numpy()
        sysm.compute_residual(td, Pr, Fr, precision=prec)
        assert rel_err(Pd.cpu().numpy(), P) < 1e-12
        assert rel_err(Kd, Ke_el) < tol
        assert rel_err(cd.cpu().numpy(), corr) < tol
        assert torch.equal(Pd, Pr) and torch.equal(Fd, Fr)
    sysm.close()
