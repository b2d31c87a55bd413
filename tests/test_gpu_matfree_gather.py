"""The matrix-free hexa20 PCG with its gather and its vector kernels in workgroups of their own sizes:
meshes below and above the 4096 nodes up to which the vector kernels take one wavefront, with ragged
last workgroups, at the sizes it chooses and at set ones.

Four iterations from x = 0 against the FP64 assembled operator: the tangents, products and sums of the
FP32 side round by 6e-8 each, 1e-4 in all."""

import numpy as np
import pytest

from helpers import device_model, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

J2 = [210000.0, 0.3, 250.0, 1000.0, 0.0, 0.0]


@pytest.mark.parametrize("el_type,n", [
    ("C3D20", (1, 1, 1)),
    ("C3D20R", (5, 4, 3)),
    ("C3D20R", (10, 9, 9)),    # 4080 nodes
    ("C3D20", (10, 10, 9)),    # 4499
])
def test_matrix_free_pcg_at_every_workgroup_size(el_type, n):
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    pm = device_model(n, (1.0, 1.0, 1.0), el_type, "vonmises", J2, jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, el_type, "vonmises", np.array(J2))
    sysm.set_dirichlet(np.r_[pm.dofsOfNodeSet("gen_bottom"), pm.dofsOfNodeSet("gen_top", [1])])
    rng = np.random.default_rng(7)
    dU = torch.as_tensor(rng.uniform(-1, 1, sysm.n_dof) * 1e-3 / max(n), device="cuda")
    b = torch.as_tensor(rng.standard_normal(sysm.n_dof), device="cuda")
    P, F, want, x = sysm.zeros(), sysm.zeros(), sysm.zeros(), sysm.zeros()
    kw = dict(rtol=0.0, max_iter=4, check_every=2)
    sysm.compute_elements(dU, P, F)
    sysm.linsolve(b, want, **kw)
    sysm.compute_elements(dU, P, F, precision=_lib.EFE_FP32_MATFREE)
    for block in (0, 64, 256, 128, 512):  # 0: as chosen by size
        sysm.set_launch(0, block)
        x.fill_(float("nan"))
        info = sysm.linsolve(b, x, precision=_lib.EFE_FP32_MATFREE, **kw)
        assert info.iterations == 4
        assert rel_err(x.cpu().numpy(), want.cpu().numpy()) < 1e-4, block
    sysm.close()
