"""The dense inverse of the coarsest multigrid operator on both sides of the
size where its kernel changes (128 rows: registers; above: global memory).

A hierarchy stops at 128 rows or at ten levels, so only a strip of more than
2.5 M elements, whose levels shrink three times each, ends above 128.

Tolerance: Gauss-Jordan elimination with partial pivoting leaves |I - C A|
within about n eps cond(A); 8 times that."""
import numpy as np
import pytest
import scipy.linalg as sl

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(12, 9), (30, 30), (33, 33), (36, 30), (45, 40), (60, 55), (66, 60), (9, 9, 9),
                               (15, 15, 15), (18, 15, 12), (21, 21, 18)], ids=lambda n: "x".join(map(str, n)))
def test_inverse_of_coarsest_operator(n):
    from mrhyde_amd import Mhx

    rng = np.random.default_rng(sum(n))
    g = Mhx(Problem(dim=len(n), order=1, quadrature=2, n=n, k0=np.exp(rng.standard_normal(int(np.prod(n)))), dbc_sides=3))
    _, j = g.assembleJacRes(np.zeros(g.n_dof))
    levels = g.buildAMGPreconditioner(j)
    assert levels >= 2
    A = g.amg_level(levels - 1, "A")[0].toarray()
    C, meta = g.amg_level(levels - 1, "Cinv")
    print(f"[amg coarse] {n}: {levels} levels, {meta['rows']} rows", flush=True)
    tol = 8 * len(A) * np.finfo(float).eps * np.linalg.cond(A)
    assert np.abs(C @ A - np.eye(len(A))).max() <= tol
    g.close()


def test_inverse_above_128_rows():
    from mrhyde_amd import Mhx

    nx = 2_600_000
    g = Mhx(Problem(dim=2, order=1, quadrature=2, n=(nx, 1), hi=(float(nx), 1.0), dbc_sides=3,
                    k0=np.exp(0.5 * np.random.default_rng(1).standard_normal(nx))))
    _, j = g.assembleJacRes(np.zeros(g.n_dof))
    levels = g.buildAMGPreconditioner(j)
    A = g.amg_level(levels - 1, "A")[0].toarray()
    C, meta = g.amg_level(levels - 1, "Cinv")
    print(f"[amg coarse] strip: {levels} levels, {meta['rows']} rows", flush=True)
    assert meta["rows"] > 128
    tol = 8 * len(A) * np.finfo(float).eps * np.linalg.cond(A)
    assert np.abs(C @ A - np.eye(len(A))).max() <= tol
    g.close()


@pytest.mark.parametrize("n,mu", [((8, 7, 6), 0.01), ((6, 6, 6), 0.01), ((30, 24), 1e-3)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_inverse_with_pivots_off_the_diagonal(n, mu):
    """Stabilised Navier-Stokes: an unsymmetric operator whose elimination
    exchanges rows."""
    from mrhyde_amd import Mhx

    dim = len(n)
    g = Mhx(Problem(dim=dim, order=1, quadrature=2, n=n, physics=2, mu=mu, supg=True, pspg=True,
                    dbc_sides=(1 | 2 | 4 | 16 | 32) if dim == 3 else (1 | 2 | 4), lid_sides=8,
                    lid_u=(1.0,) + (0.0,) * (dim - 1), pin_pressure=True))
    u = g.setDirichlet(1e-3 * np.random.default_rng(3).standard_normal(g.n_dof))
    _, j = g.assembleJacRes(u)
    levels = g.buildAMGPreconditioner(j)
    A = g.amg_level(levels - 1, "A")[0].toarray()
    C, meta = g.amg_level(levels - 1, "Cinv")
    piv = sl.lu_factor(A)[1]
    print(f"[amg coarse] {n}: {meta['rows']} rows, {np.count_nonzero(piv != np.arange(len(piv)))} exchanged", flush=True)
    assert (piv != np.arange(len(piv))).any()
    tol = 8 * len(A) * np.finfo(float).eps * np.linalg.cond(A)
    assert np.abs(C @ A - np.eye(len(A))).max() <= tol
    g.close()
