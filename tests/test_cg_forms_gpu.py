"""CG in its three forms (one workgroup, two launches and four launches per
iteration) around the sizes where they change, against the same recurrence in
numpy: the iterate after a fixed number of iterations, and the iteration at
which the tolerance is met.

Tolerance: iterates of one recurrence with sums in another order part by
eps times the growth of CG's rounding errors; after 7 iterations on these
matrices (condition below 1e5 after diagonal scaling) 1e-10 of the largest
entry.  The iteration counts may differ where the residual sits near the
tolerance, and by rounding in long runs: 2 and 2 %."""
import numpy as np
import pytest
import scipy.sparse as sp

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu


def pcg(A, b, d, tol, maxit):
    x, r = np.zeros_like(b), b.copy()
    z = r / d
    p, rz, it = z.copy(), r @ z, 0
    while it < maxit and np.linalg.norm(r) > tol * np.linalg.norm(b):
        q = A @ p
        al = rz / (p @ q)
        x, r = x + al * p, r - al * q
        z = r / d
        rz, old = r @ z, rz
        p = z + (rz / old) * p
        it += 1
    return x, it


# 2-D Q1: one workgroup to 70^2; 3-D Q1 to 12^3; two launches to 65,536 rows at
# four lanes
CASES = [(1, (2, 2)), (1, (31, 32)), (1, (70, 70)), (1, (71, 71)), (2, (20, 11)), (3, (9, 7)), (1, (2, 3, 1)),
         (1, (12, 12, 12)), (1, (13, 13, 13)), (2, (4, 4, 3)), (2, (5, 4, 4)), (1, (255, 254)), (1, (256, 256))]


@pytest.mark.parametrize("precond", ["none", "jacobi"])
@pytest.mark.parametrize("order,n", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else f"p{v}")
def test_matches_numpy(order, n, precond):
    from mrhyde_amd import Mhx

    print(f"[cg] p{order} {n} {precond}", flush=True)
    rng = np.random.default_rng(order + sum(n))
    g = Mhx(Problem(dim=len(n), order=order, quadrature=2 * order, n=n, k0=np.exp(0.3 * rng.standard_normal(np.prod(n))),
                    dbc_sides=1))
    _, j = g.assembleJacRes(np.zeros(g.n_dof))
    rp, ci = g.crs_pattern()
    A = sp.csr_matrix((j, ci, rp), shape=(g.n_dof, g.n_dof))
    b = rng.standard_normal(g.n_dof)
    b[np.asarray(g.dirichlet_mask(), bool)] = 0.0  # (fixed rows are unit rows: the rest is symmetric)
    d = A.diagonal() if precond == "jacobi" else np.ones(g.n_dof)
    ref, it7 = pcg(A, b, d, 1e-14, 7)
    x, st = g.linearSolver(j, b, solver="cg", precond=precond, tol=1e-14, max_iters=it7)
    assert np.abs(x - ref).max() <= 1e-10 * np.abs(ref).max()
    if g.n_dof < 10000:
        ref, it = pcg(A, b, d, 1e-9, 1500)
        x, st = g.linearSolver(j, b, solver="cg", precond=precond, tol=1e-9, max_iters=1500)
        assert abs(st["iters"] - it) <= 2 + it // 50
        assert np.linalg.norm(b - A @ x) <= 1.01e-9 * np.linalg.norm(b)
    g.close()


@pytest.mark.parametrize("order,n", [(4, (6, 6)), (5, (4, 4)), (6, (3, 3)), (6, (2, 3))],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else f"p{v}")
def test_long_rows_match_numpy(order, n):
    """Rows of 81 to 169 entries, on both sides of the longest that one
    workgroup takes: the iterate after 7 iterations, and the solution."""
    from mrhyde_amd import Mhx

    print(f"[cg] p{order} {n} jacobi", flush=True)
    rng = np.random.default_rng(order + sum(n))
    g = Mhx(Problem(dim=2, order=order, quadrature=2 * order, n=n, k0=np.exp(0.3 * rng.standard_normal(np.prod(n))),
                    dbc_sides=1))
    _, j = g.assembleJacRes(np.zeros(g.n_dof))
    rp, ci = g.crs_pattern()
    A = sp.csr_matrix((j, ci, rp), shape=(g.n_dof, g.n_dof))
    b = rng.standard_normal(g.n_dof)
    b[np.asarray(g.dirichlet_mask(), bool)] = 0.0
    ref, it = pcg(A, b, A.diagonal(), 1e-14, 7)
    x, st = g.linearSolver(j, b, solver="cg", precond="jacobi", tol=1e-14, max_iters=it)
    assert np.abs(x - ref).max() <= 1e-10 * np.abs(ref).max()
    x, st = g.linearSolver(j, b, solver="cg", precond="jacobi", tol=1e-9, max_iters=3000)
    assert np.linalg.norm(b - A @ x) <= 1.01e-9 * np.linalg.norm(b)
    g.close()
