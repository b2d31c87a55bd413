"""The GMRES kernels at the edges of their splits: block ILU(0) sweeps of one-element meshes, ragged
colors and rows far longer than a slice's own steps (a fan of elements around one edge), against a
dense block ILU(0) in the same elimination order; Gram-Schmidt at basis sizes around the groups of
its kernels, by the true residual.

After one iteration from x = 0 the solution is a multiple of M^-1 b, which the dense factor gives.
Both sides round each entry of a triangular solve of a matrix with a condition number below 1e4: the
directions agree to 1e4 times the unit roundoff, 1e-10 in FP64 with a margin and 1e-3 in FP32."""

import numpy as np
import pytest

from helpers import device_model

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LE = [180000.0, 0.25]


def _fan(k, axis_last):
    """k hexa8 around the z axis, whose two nodes then have 4 k neighbours and more."""
    ang = np.linspace(0.0, 2 * np.pi, 2 * k, endpoint=False)
    r = np.where(np.arange(2 * k) % 2 == 0, 1.0, 1.1)
    ring = np.c_[r * np.cos(ang), r * np.sin(ang)]
    xy = np.r_[[[0.0, 0.0]], ring]
    coords = np.r_[np.c_[xy, np.zeros(len(xy))], np.c_[xy, np.full(len(xy), 0.5)]]
    n = len(xy)
    el = []
    for e in range(k):
        q = [0, 1 + 2 * e, 2 + 2 * e, 1 + (2 * e + 2) % (2 * k)]
        el.append(q + [m + n for m in q])
    conn = np.array(el)
    if axis_last:
        order = np.r_[np.setdiff1d(np.arange(2 * n), [0, n]), [0, n]]
        new = np.empty(2 * n, dtype=int)
        new[order] = np.arange(2 * n)
        coords, conn = coords[order], new[conn]
    return coords, np.ascontiguousarray(conn, dtype=np.int32)


def _ilu0_apply(K, conn, b):
    """M^-1 b with the block ILU(0) of K in the order of the greedy coloring, colors then nodes."""
    N = K.shape[0] // 3
    nb = [set() for _ in range(N)]
    for e in conn:
        for i in e:
            nb[i].update(int(j) for j in e)
    color = -np.ones(N, dtype=int)
    for n in range(N):
        used = {color[m] for m in nb[n] if m != n}
        c = 0
        while c in used:
            c += 1
        color[n] = c
    order = np.lexsort((np.arange(N), color))
    pos = np.empty(N, dtype=int)
    pos[order] = np.arange(N)
    row = [sorted(pos[j] for j in nb[n]) for n in order]
    B = lambda i, j: K[3 * order[i]:3 * order[i] + 3, 3 * order[j]:3 * order[j] + 3]
    F = [{j: B(i, j).copy() for j in row[i]} for i in range(N)]
    Dinv = [None] * N
    for i in range(N):
        for k in row[i]:
            if k >= i:
                break
            F[i][k] = F[i][k] @ Dinv[k]
            for j in row[k]:
                if j > k and j in F[i]:
                    F[i][j] = F[i][j] - F[i][k] @ F[k][j]
        Dinv[i] = np.linalg.inv(F[i][i])
    z = np.zeros((N, 3))
    for i in range(N):
        z[i] = b[3 * order[i]:3 * order[i] + 3] - sum((F[i][k] @ z[k] for k in row[i] if k < i), np.zeros(3))
    for i in range(N - 1, -1, -1):
        z[i] = Dinv[i] @ (z[i] - sum((F[i][j] @ z[j] for j in row[i] if j > i), np.zeros(3)))
    out = np.empty(3 * N)
    out.reshape(-1, 3)[order] = z
    return out


def _assemble(sysm, precision):
    sysm.compute_elements(sysm.zeros(), sysm.zeros(), sysm.zeros(), precision=precision)


def _prepared(coords, conn, etype, precision, rng):
    from edelweissfe_amd import _lib
    from edelweissfe_amd.device import DeviceSystem

    sysm = DeviceSystem(coords, conn, etype, "linearelastic", np.array(LE))
    z = coords[:, 2]
    fixed = np.flatnonzero(z < z.min() + 1e-9)
    dirs = np.sort(np.r_[3 * fixed, 3 * fixed + 1, 3 * fixed + 2])
    sysm.set_dirichlet(dirs)
    prec = _lib.EFE_FP64 if precision == "fp64" else _lib.EFE_FP32
    b = rng.standard_normal(sysm.n_dof)
    b[dirs] = 0.0
    return sysm, prec, b


def _mesh(mesh):
    if mesh[0] == "fan":
        return (*_fan(mesh[1], mesh[2]), "C3D8")
    pm = device_model(mesh[1], (1.0, 1.0, 1.0), mesh[0], "linearelastic", LE, jitter=0.0, seed=1)
    return pm.coordinates, pm.connectivity, mesh[0]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mesh", [
    ("C3D8", (1, 1, 1)),
    ("C3D8", (5, 4, 3)),
    ("C3D20R", (1, 1, 1)),
    ("C3D20", (3, 2, 2)),
    ("fan", 30, False),   # rows of 120 blocks after the diagonal
    ("fan", 90, False),   # 360: more steps than a color's own levels
    ("fan", 90, True),    # 360 before the diagonal
])
def test_ilu0_sweeps_match_a_dense_factor(mesh, precision):
    from edelweissfe_amd import _lib

    coords, conn, etype = _mesh(mesh)
    sysm, prec, b = _prepared(coords, conn, etype, precision, np.random.default_rng(2))
    _assemble(sysm, _lib.EFE_FP64)
    K = np.empty((sysm.n_dof, sysm.n_dof))
    unit, y = sysm.zeros(), sysm.zeros()
    for i in range(sysm.n_dof):
        unit.zero_()
        unit[i] = 1.0
        sysm.spmv(unit, y)
        K[:, i] = y.cpu().numpy()
    if precision == "fp32":
        _assemble(sysm, prec)
    x = sysm.zeros()
    sysm.linsolve(torch.as_tensor(b, device="cuda"), x, solver=_lib.EFE_SOLVER_GMRES, precond=_lib.EFE_PRECOND_ILU0,
                  precision=prec, rtol=0.0, max_iter=1, restart=4)
    got = x.cpu().numpy()
    sysm.close()
    want = _ilu0_apply(K, conn, b)
    got, want = got / np.linalg.norm(got), want / np.linalg.norm(want)
    assert min(np.linalg.norm(got - want), np.linalg.norm(got + want)) < (1e-10 if precision == "fp64" else 1e-3)


@pytest.mark.parametrize("restart", [1, 7, 8, 9, 24, 25, 70, 256])
def test_gmres_restart_lengths_reach_the_residual(restart):
    from edelweissfe_amd import _lib

    pm = device_model((6, 5, 4), (1.0, 1.0, 1.0), "C3D20R", "linearelastic", LE, jitter=0.0, seed=1)
    sysm, prec, b = _prepared(pm.coordinates, pm.connectivity, "C3D20R", "fp64", np.random.default_rng(3))
    _assemble(sysm, prec)
    pc = _lib.EFE_PRECOND_BLOCK_JACOBI if restart > 9 else _lib.EFE_PRECOND_ILU0
    bd, x, y = torch.as_tensor(b, device="cuda"), sysm.zeros(), sysm.zeros()
    info = sysm.linsolve(bd, x, solver=_lib.EFE_SOLVER_GMRES, precond=pc, rtol=1e-8, max_iter=6000, restart=restart)
    sysm.spmv(x, y)
    sysm.close()
    assert info.status == 0
    # the recurrence's residual is the true one up to its rounding
    assert float(torch.linalg.norm(y - bd) / torch.linalg.norm(bd)) < 1.1e-8
