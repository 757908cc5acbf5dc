"""The dense inverse of the coarsest multigrid operator on both sides of the
size where its kernel changes (128 rows: registers; above: global memory).

Tolerance: an inverse by elimination without pivoting of a symmetric positive
definite matrix leaves |I - C A| within about n eps cond(A); 8 times that."""
import numpy as np
import pytest

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
