"""A specimen has the same bricks, reductions and stops in a context of its own as in a batch: the batched
PCG gives it the same bits in both, whatever stands beside it (one specimen, many, smaller and larger ones,
some of them not solved)."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

J2 = [210000.0, 0.3, 250.0, 1000.0, 0.0, 0.0]


def _solve(parts, dU, b, act, precision, rtol):
    from edelweissfe_amd.device import DeviceSystem

    off = np.concatenate([[0], np.cumsum([m.nNodes for m in parts])])
    sysm = DeviceSystem(np.concatenate([m.coordinates for m in parts]),
                        np.concatenate([m.connectivity + o for m, o in zip(parts, off)]), "C3D8", "vonmises", J2,
                        n_specimens=len(parts),
                        specimen_of_node=np.repeat(np.arange(len(parts)), np.diff(off)).astype(np.int32))
    sysm.set_dirichlet(np.concatenate([np.r_[m.dofsOfNodeSet("gen_bottom"), m.dofsOfNodeSet("gen_top", [1])] + 3 * o
                                       for m, o in zip(parts, off)]))
    P, F, x = sysm.zeros(), sysm.zeros(), sysm.zeros()
    sysm.compute_elements(torch.as_tensor(np.concatenate(dU), device="cuda"), P, F, precision=precision)
    info, its = sysm.linsolve_batched(torch.as_tensor(np.concatenate(b), device="cuda"), x, np.zeros(len(parts)),
                                      np.asarray(act, dtype=np.uint8), precision=precision, rtol=rtol, check_every=8)
    sysm.close()
    assert info.status == 0
    x = x.cpu().numpy()
    return [x[3 * off[i]:3 * off[i + 1]] for i in range(len(parts))], its


@pytest.mark.parametrize("precision", ["fp64", "matfree"])
@pytest.mark.parametrize("sizes", [(1,), (3, 1, 7), (9, 4, 13, 8)])
def test_a_specimen_has_the_same_bits_alone(sizes, precision):
    from edelweissfe_amd import _lib

    prec, rtol = (_lib.EFE_FP64, 1e-12) if precision == "fp64" else (_lib.EFE_FP32_MATFREE, 1e-6)
    parts = [device_model((m, m, m + 1), (1.0, 1.0, 1.0), "C3D8", "vonmises", J2, jitter=0.1, seed=i)
             for i, m in enumerate(sizes)]
    rng = np.random.default_rng(7)
    dU = [rng.uniform(-1, 1, 3 * m.nNodes) * 1e-3 for m in parts]
    b = [rng.standard_normal(3 * m.nNodes) for m in parts]
    act = [not (len(sizes) > 2 and i == 1) for i in range(len(sizes))]
    x, its = _solve(parts, dU, b, act, prec, rtol)
    for i, m in enumerate(parts):
        if act[i]:
            one, it = _solve([m], [dU[i]], [b[i]], [True], prec, rtol)
            assert it[0] == its[i] > 0
            assert np.array_equal(one[0], x[i])
