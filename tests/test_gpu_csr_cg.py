"""CG of the CSR solve at the edges of its product: one row, rows of more entries than a lane takes in
one step, empty prescribed rows between free ones, more rows than the product's workgroups hold at
once; by the residual of the whole system.  The stop test is ||r|| <= 1e-13 ||b_f|| on the free block,
and a few tens of iterations round r by some 1e-16 of |A| |x| each: 1e-12 of | |A| |x| | bounds both."""

import numpy as np
import pytest
import scipy.sparse as sp

pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _system(n, dense_rows, fixed_every, seed):
    rng = np.random.default_rng(seed)
    i = rng.integers(0, n, 6 * n)
    j = rng.integers(0, n, 6 * n)
    A = sp.coo_matrix((rng.uniform(-1, 1, i.size), (i, j)), shape=(n, n)).tolil()
    for r in dense_rows:
        A[r, :] = rng.uniform(-1, 1, n) / n
    A = A.tocsr()
    A = A + A.T
    A = A - sp.diags(A.diagonal())
    A = A + sp.diags(1.5 * np.asarray(abs(A).sum(axis=1)).ravel() + 1.0)
    b = rng.standard_normal(n)
    if fixed_every:  # unit rows, the columns stay
        keep = np.ones(n)
        keep[::fixed_every] = 0.0
        A = sp.diags(keep) @ A + sp.diags(1.0 - keep)
    A = A.tocsr()
    A.eliminate_zeros()
    A.sort_indices()
    return A, b


@pytest.mark.parametrize("n,dense_rows,fixed_every", [
    (1, (), 0),
    (5, (), 2),
    (300, (0, 7, 299), 0),    # rows of 300 entries: four steps of 96
    (1000, (3,), 7),
    (40000, (), 11),          # more rows than 2048 workgroups of 16
])
def test_csr_cg_solves_the_system(n, dense_rows, fixed_every):
    from edelweissfe_amd.config.linsolve import csr_solve

    A, b = _system(n, dense_rows, fixed_every, seed=n)
    x, _ = csr_solve(A, b, rtol=1e-13)
    assert np.linalg.norm(A @ x - b) <= 1e-12 * np.linalg.norm(abs(A) @ abs(x))
    if fixed_every:
        assert np.array_equal(x[::fixed_every], b[::fixed_every])
