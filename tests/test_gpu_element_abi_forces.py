"""efe_element_compute without Ke, whose workgroups are others than with it (hexa8: 4 elements in lists of
up to 65536, 8 in longer ones): the same residuals and states as the call with Ke, bit for bit, for
lists around the workgroups' numbers of elements and on both sides of the line."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

PROPS = {"linearelastic": [210000.0, 0.3], "vonmises": [210000.0, 0.15, 355.0, 1000.0, 200.0, 1400.0],
         "druckerprager": [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]}


@pytest.mark.parametrize("el_type,n,counts,material", [
    ("C3D8", (3, 3, 2), (1, 3, 4, 5, 17), "vonmises"),
    ("C3D8", (41, 40, 40), (65536, 65537, 65600), "vonmises"),
    ("C3D8", (41, 40, 40), (65536, 65537), "druckerprager"),
    ("C3D20R", (3, 2, 2), (1, 2, 3, 11), "druckerprager"),
    ("C3D20", (3, 2, 2), (1, 2, 11), "linearelastic"),
])
def test_forces_without_ke(el_type, n, counts, material):
    from edelweissfe_amd.device import DeviceSystem

    pm = device_model(n, (1.0, 1.0, 1.0), el_type, material, PROPS[material], jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, material, np.array(PROPS[material]))
    nd = 3 * pm.connectivity.shape[1]
    rng = np.random.default_rng(3)
    f64 = dict(dtype=torch.float64, device="cuda")
    for m in counts:
        els = rng.permutation(pm.connectivity.shape[0])[:m].astype(np.int32)
        dQ = torch.as_tensor(rng.uniform(-1, 1, (m, nd)) * 2e-3 / max(n), device="cuda")
        ref = torch.zeros((m, sysm.n_qp, sysm.n_state), **f64)
        s1, s2 = torch.full_like(ref, float("nan")), torch.full_like(ref, float("nan"))
        P1, P2 = (torch.full((m, nd), float("nan"), **f64) for _ in range(2))
        Ke = torch.empty((m, nd, nd), **f64)
        sysm.element_compute(els, dQ, ref, s1, P1, Ke)
        sysm.element_compute(els, dQ, ref, s2, P2, None)
        assert torch.isfinite(P1).all() and float(P1.abs().max()) > 0
        assert torch.equal(P1, P2) and torch.equal(s1, s2)
    sysm.close()
