"""hexa20R element passes take two elements per wavefront: 1, 3 and 5 elements leave half a
wavefront empty in the last workgroup.  Same comparison and bounds as at the other tile edges
(1e-12 in FP64, 3e-6 in FP32 against the oracle's element matrices)."""

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import device_model, oracle_model, rel_err

torch = pytest.importorskip("torch")
import test_gpu_pass_edges as edges  # noqa: E402

from edelweissfe_amd import _lib  # noqa: E402
from edelweissfe_amd.device import DeviceSystem  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("material", sorted(edges.PROPS))
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 1), (1, 5, 1)])
def test_hexa20r_odd_element_counts(material, n):
    edges.test_pass_and_assembly_at_tile_edges(material, "C3D20R", n)


@pytest.mark.parametrize("material", ["vonmises", "druckerprager"])
@pytest.mark.parametrize("el_type,n", [("C3D20", (16, 8, 6)), ("C3D20", (769, 1, 1)), ("C3D20R", (16, 12, 8)),
                                       ("C3D20R", (53, 29, 1))])
def test_workgroup_size_boundary(material, el_type, n):
    """Tangent passes of up to 768 workgroups run in larger workgroups: 768 and 769 of one
    (hexa20) or two (hexa20R) elements, K and P against the oracle's, assembled sparsely."""
    om = oracle_model(n, n, el_type, material, edges.PROPS[material], jitter=0.1, seed=6)
    pm = device_model(n, n, el_type, material, edges.PROPS[material], jitter=0.1, seed=6)
    dU = np.random.default_rng(8).uniform(-1, 1, om.nDof) * 2e-3
    dm = om.elements.dof_map
    Ke, Pe, _ = om.elements.compute(dU[dm], om.state, om.material)
    P = np.zeros(om.nDof)
    np.add.at(P, dm, Pe)
    K = sp.coo_matrix((Ke.ravel(), (np.repeat(dm, dm.shape[1], 1).ravel(), np.tile(dm, dm.shape[1]).ravel())),
                      (om.nDof, om.nDof)).tocsr()
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, material, edges.PROPS[material])
    ip, ix = sysm.csr_pattern()
    for prec, tol in ((_lib.EFE_FP64, 1e-12), (_lib.EFE_FP32, 3e-6)):
        Pd, Fd = sysm.zeros(), sysm.zeros()
        sysm.compute_elements(torch.as_tensor(dU, device="cuda"), Pd, Fd, precision=prec)
        Kd = sp.csr_matrix((sysm.export_csr_values().cpu().numpy(), ix, ip), K.shape)
        assert rel_err(Pd.cpu().numpy(), P) < 1e-12
        assert abs(Kd - K).max() < tol * abs(K).max()
    sysm.close()
