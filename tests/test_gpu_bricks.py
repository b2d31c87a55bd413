"""The FP64 CG on the hexa8 bricks against the CG on the assembled operator of the same pass, over the
forms and sizes the bricks take.  Setting the Dirichlet DOFs again after the pass leaves the
assembled operator as the only one of that set, so the same system is solved both ways.  Both
stop at ||r|| <= 1e-13 ||b||: their solutions differ by at most the condition number (below 1e4 at
these sizes) times that, 1e-9 relative."""

import numpy as np
import pytest

from helpers import device_model, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

J2 = [210000.0, 0.3, 250.0, 1000.0, 0.0, 0.0]
LE = [180000.0, 0.25]


# a context of one specimen takes the bricks at any size (without specimens, small meshes do not)
_ALONE = lambda pm: dict(specimen_of_node=np.zeros(pm.coordinates.shape[0], dtype=np.int32), n_specimens=1)


def _sections(E):
    names = np.where(np.arange(E) % 3 == 0, "linearelastic", "vonmises").tolist()
    rows = np.tile(J2, (E, 1))
    rows[::3] = LE + [0.0] * 4
    return names, rows


@pytest.mark.parametrize("n,material,perm", [
    ((1, 1, 1), "vonmises", False),       # one element
    ((4, 8, 8), "vonmises", False),       # a full brick
    ((257, 1, 1), "vonmises", False),     # one more than a brick in a row
    ((20, 4, 4), "linearelastic", False),
    ((9, 7, 5), "sections", False),
    ((12, 11, 13), "lognormal", False),
    ((12, 11, 10), "vonmises", True),     # elements in random order
])
def test_fp64_bricks_solve_the_assembled_system(n, material, perm):
    from edelweissfe_amd.device import DeviceSystem

    pm = device_model(n, (1.0, 1.0, 1.0), "C3D8", "vonmises", J2, jitter=0.1, seed=3)
    E = pm.connectivity.shape[0]
    rng = np.random.default_rng(5)
    conn = pm.connectivity[rng.permutation(E)] if perm else pm.connectivity
    name, props = "vonmises", np.array(J2)
    if material == "linearelastic":
        name, props = material, np.array(LE)
    elif material == "sections":
        name, props = _sections(E)
    elif material == "lognormal":
        props = np.tile(J2, (E, 1))
        props[:, 0] *= np.exp(0.1 * rng.standard_normal(E))
        props[:, 2] *= np.exp(0.1 * rng.standard_normal(E))
    sysm = DeviceSystem(pm.coordinates, np.ascontiguousarray(conn), "C3D8", name, props, **_ALONE(pm))
    dirs = np.r_[pm.dofsOfNodeSet("gen_bottom"), pm.dofsOfNodeSet("gen_top", [1])]
    sysm.set_dirichlet(dirs)
    dU = torch.as_tensor(rng.uniform(-1, 1, sysm.n_dof) * 2e-3 / max(n), device="cuda")
    b = torch.as_tensor(rng.standard_normal(sysm.n_dof), device="cuda")
    P, F = sysm.zeros(), sysm.zeros()
    sysm.compute_elements(dU, P, F)
    xb, xa = sysm.zeros(), sysm.zeros()
    ib = sysm.linsolve(b, xb, rtol=1e-13)
    sysm.set_dirichlet(dirs)
    ia = sysm.linsolve(b, xa, rtol=1e-13)
    y = sysm.zeros()
    sysm.spmv(xb, y)
    sysm.close()
    assert ib.status == 0 and ia.status == 0
    assert rel_err(xb.cpu().numpy(), xa.cpu().numpy()) < 1e-9
    d = torch.as_tensor(np.unique(dirs), device="cuda")
    assert torch.equal(xb[d], b[d])
    assert rel_err(y.cpu().numpy(), b.cpu().numpy()) < 1e-9


def test_fp64_bricks_follow_a_changed_dirichlet_set():
    """A set changed after the pass is not the operator's: the solve keeps the elimination of the
    pass, and a new pass takes the new set."""
    pm = device_model((5, 4, 6), (1.0, 1.0, 1.0), "C3D8", "vonmises", J2, jitter=0.1, seed=3)
    from edelweissfe_amd.device import DeviceSystem

    sysm = DeviceSystem(pm.coordinates, pm.connectivity, "C3D8", "vonmises", J2, **_ALONE(pm))
    rng = np.random.default_rng(6)
    b = torch.as_tensor(rng.standard_normal(sysm.n_dof), device="cuda")
    P, F, x, y = (sysm.zeros() for _ in range(4))
    for dirs in (pm.dofsOfNodeSet("gen_bottom"), np.r_[pm.dofsOfNodeSet("gen_bottom"), pm.dofsOfNodeSet("gen_left")]):
        sysm.set_dirichlet(dirs)
        sysm.compute_elements(sysm.zeros(), P, F)
        assert sysm.linsolve(b, x, rtol=1e-13).status == 0
        sysm.spmv(x, y)
        assert rel_err(y.cpu().numpy(), b.cpu().numpy()) < 1e-9
    sysm.set_dirichlet(pm.dofsOfNodeSet("gen_bottom"))
    free = np.setdiff1d(np.arange(sysm.n_dof), dirs)
    assert sysm.linsolve(b, x, rtol=1e-13).status == 0
    sysm.spmv(x, y)
    sysm.close()
    assert rel_err(y.cpu().numpy()[free], b.cpu().numpy()[free]) < 1e-9


@pytest.mark.parametrize("precision", ["fp64", "matfree"])
@pytest.mark.parametrize("sizes", [(1,), (3, 1, 7), (9, 4, 6, 8)])
def test_batched_bricks_solve_every_specimen_as_alone(sizes, precision):
    """The batched PCG on the bricks against each specimen's own context, which runs the same
    bricks: the same solutions to round-off (FP64: both to 1e-13 of b, 1e-9 as above; FP32: 1e-7
    of b, within 2e-4 = condition number times that), excluded specimens zero; in FP64 also against
    the assembled operator, which a set of Dirichlet DOFs set after the pass leaves."""
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    prec, rtol, tol = ((_lib.EFE_FP64, 1e-13, 1e-9) if precision == "fp64" else (_lib.EFE_FP32_MATFREE, 1e-7, 2e-4))
    models = [device_model((m, m, m), (1.0, 1.0, 1.0), "C3D8", "vonmises", J2, jitter=0.1, seed=i)
              for i, m in enumerate(sizes)]
    S = len(models)
    off = np.concatenate([[0], np.cumsum([m.nNodes for m in models])])
    coords = np.concatenate([m.coordinates for m in models])
    conn = np.concatenate([m.connectivity + o for m, o in zip(models, off)])
    batch = DeviceSystem(coords, conn, "C3D8", "vonmises", J2, n_specimens=S,
                         specimen_of_node=np.repeat(np.arange(S), np.diff(off)).astype(np.int32))
    rng = np.random.default_rng(7)
    dirs = [np.r_[m.dofsOfNodeSet("gen_bottom"), m.dofsOfNodeSet("gen_top", [1])] for m in models]
    alld = np.concatenate([d + 3 * o for d, o in zip(dirs, off)])
    dU = rng.uniform(-1, 1, batch.n_dof) * 1e-3
    b = rng.standard_normal(batch.n_dof)
    act = np.ones(S, np.uint8)
    if S > 2:
        act[1] = 0

    def solve():
        x = batch.zeros()
        info, its = batch.linsolve_batched(torch.as_tensor(b, device="cuda"), x, np.zeros(S), act, precision=prec,
                                           rtol=rtol, check_every=7)
        assert info.status == 0 and (its[act != 0] > 0).all()
        return x.cpu().numpy()

    P, F = batch.zeros(), batch.zeros()
    batch.set_dirichlet(alld)
    batch.compute_elements(torch.as_tensor(dU, device="cuda"), P, F, precision=prec)
    x = solve()
    if precision == "fp64":
        batch.set_dirichlet(alld)
        xa = solve()
    for s, m in enumerate(models):
        sl = slice(3 * off[s], 3 * off[s + 1])
        free = np.ones(3 * m.nNodes, bool)
        free[np.unique(dirs[s])] = False
        if not act[s]:
            assert (x[sl][free] == 0.0).all()
            continue
        one = DeviceSystem(m.coordinates, m.connectivity, "C3D8", "vonmises", J2)
        one.set_dirichlet(dirs[s])
        P1, F1, x1 = one.zeros(), one.zeros(), one.zeros()
        one.compute_elements(torch.as_tensor(dU[sl], device="cuda"), P1, F1, precision=prec)
        assert one.linsolve(torch.as_tensor(b[sl], device="cuda"), x1, precision=prec, rtol=rtol).status == 0
        one.close()
        assert rel_err(x[sl], x1.cpu().numpy()) < tol
        if precision == "fp64":
            assert rel_err(xa[sl], x1.cpu().numpy()) < tol
    batch.close()


@pytest.mark.parametrize("n,material", [
    ((1, 1, 1), "vonmises"),
    ((33, 1, 1), "linearelastic"),   # one more than a split brick in a row
    ((9, 7, 5), "vonmises"),
    ((9, 7, 5), "druckerprager"),
    ((24, 32, 32), "vonmises"),      # the most elements of split bricks, and more
    ((24, 32, 32), "linearelastic"),
    ((25, 32, 32), "vonmises"),
    ((25, 32, 32), "linearelastic"),
])
def test_split_and_whole_bricks_step_as_the_assembled_operator(n, material):
    """Three PCG iterations from x = 0 (six products' worth of round-off, far from convergence) on the
    FP32 bricks (split ones, then whole ones), on what the FP64 CG takes after a pass (the assembled
    operator, then bricks) and on the assembled operator: 1e-12 relative in FP64; in FP32 the tangents'
    and products' rounding, 1e-4.  (Drucker-Prager at an elastic state, whose tangent is symmetric.)"""
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    props = {"vonmises": J2, "linearelastic": LE, "druckerprager": [30000.0, 0.2, 30.0, 10.0, 10.0, 0.0]}[material]
    pm = device_model(n, (1.0, 1.0, 1.0), "C3D8", material, props, jitter=0.1, seed=3)
    sysm = DeviceSystem(pm.coordinates, pm.connectivity, "C3D8", material, np.array(props))
    dirs = np.r_[pm.dofsOfNodeSet("gen_bottom"), pm.dofsOfNodeSet("gen_top", [1])]
    sysm.set_dirichlet(dirs)
    rng = np.random.default_rng(7)
    scale = 1e-6 if material == "druckerprager" else 2e-3
    dU = torch.as_tensor(rng.uniform(-1, 1, sysm.n_dof) * scale / max(n), device="cuda")
    b = torch.as_tensor(rng.standard_normal(sysm.n_dof), device="cuda")
    P, F = sysm.zeros(), sysm.zeros()
    x32, xb, xa = sysm.zeros(), sysm.zeros(), sysm.zeros()
    sysm.compute_elements(dU, P, F, precision=_lib.EFE_FP32_MATFREE)
    sysm.linsolve(b, x32, precision=_lib.EFE_FP32_MATFREE, rtol=0.0, max_iter=3)
    sysm.compute_elements(dU, P, F)
    sysm.linsolve(b, xb, rtol=0.0, max_iter=3)
    sysm.set_dirichlet(dirs)  # leaves the assembled operator as the only one of its set
    sysm.linsolve(b, xa, rtol=0.0, max_iter=3)
    sysm.close()
    xa = xa.cpu().numpy()
    assert np.linalg.norm(xa) > 0
    assert rel_err(xb.cpu().numpy(), xa) < 1e-12
    assert rel_err(x32.cpu().numpy(), xa) < 1e-4
