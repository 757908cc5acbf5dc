"""The residual-only kernel of Q2 box meshes (a wavefront owns 7 x 7 element
blocks and walks z) at the edges of its tiles and walks, against the residual of
the Jacobian's kernel: the two take the same operations in the same order, so
the bits agree, overwriting and accumulating."""
import numpy as np
import pytest

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu

MESHES = [(1, 1, 1), (6, 7, 1), (7, 6, 2), (8, 8, 3), (13, 14, 5), (14, 13, 9), (15, 1, 4), (1, 15, 16), (2, 3, 40),
          (31, 29, 33), (48, 47, 49)]


@pytest.mark.parametrize("n", MESHES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("full", [True, False])
def test_same_bits_as_jacobian_kernel(n, full):
    from mrhyde_amd import Mhx

    print(f"[q2res] {n}", flush=True)
    rng = np.random.default_rng(sum(n))
    ne = int(np.prod(n))
    kw = dict(k0=np.exp(rng.standard_normal(ne)), src_elem=rng.standard_normal(ne), diff_u2=0.8) if full else {}
    g = Mhx(Problem(dim=3, order=2, quadrature=4, n=n, lo=(-1.0, 0.0, 0.5), hi=(1.0, 3.0, 0.7), dbc_sides=9, **kw))
    u, r0 = rng.standard_normal(g.n_dof), rng.standard_normal(g.n_dof)
    r, _ = g.assembleJacRes(u)
    np.testing.assert_array_equal(g.assembleRes(u), r)
    ra, _ = g.assemble(u, r0.copy(), np.zeros(g.nnz), accumulate=True)
    rb, _ = g.assemble(u, r0.copy(), None, accumulate=True)
    np.testing.assert_array_equal(ra, rb)
    g.close()
