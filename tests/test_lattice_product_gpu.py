"""The order-2 lattice product (8 lanes per vertex / interior row pair, x from
an LDS tile): every mesh whose element counts end inside, at or past a tile
(8 elements along x, 1 or 2 along y), against a plain sum over the oracle's
CRS pattern, with the columns from the tile and from the index stream.

Tolerance: a row of m entries summed in any order is within m eps of the sum
of its terms' magnitudes (m <= 125)."""
import numpy as np
import pytest

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu

MESHES = [(1, 1), (2, 5), (7, 3), (8, 4), (9, 17), (1, 1, 1), (2, 1, 3), (7, 2, 2), (8, 3, 1), (16, 5, 4), (17, 2, 5)]


@pytest.mark.parametrize("n", MESHES, ids=lambda n: "x".join(map(str, n)))
def test_product_matches_pattern_sum(n):
    from mrhyde_amd import Mhx

    g = Mhx(Problem(dim=len(n), order=2, quadrature=4, n=n))
    rp, ci = g.crs_pattern()
    rng = np.random.default_rng(sum(n))
    a, x = rng.standard_normal(g.nnz), rng.standard_normal(g.n_dof)
    rows = np.repeat(np.arange(g.n_dof), np.diff(rp))
    ref, mag = np.zeros(g.n_dof), np.zeros(g.n_dof)
    np.add.at(ref, rows, a * x[ci])
    np.add.at(mag, rows, np.abs(a * x[ci]))
    tol = 2 * np.diff(rp) * np.finfo(float).eps * mag
    y = g.apply(a, x)
    assert (np.abs(y - ref) <= tol).all()
    g.set_option("krylov.lattice_columns", 0)
    np.testing.assert_array_equal(g.apply(a, x), y)
    g.close()


def test_gmres_same_bits_twice():
    """The fused Gram-Schmidt sweep reads w before any wavefront updates it:
    two solves of the same system give the same bits."""
    from mrhyde_amd import Mhx

    n = (24, 24, 24)
    rng = np.random.default_rng(3)
    g = Mhx(Problem(dim=3, order=2, quadrature=4, n=n, k0=np.exp(0.5 * rng.standard_normal(24 ** 3)), diff_u2=1.0,
                    dbc_sides=3))
    r, j = g.assembleJacRes(g.setDirichlet(rng.random(g.n_dof)))
    xs = [g.linearSolver(j, r, solver="gmres", restart=50, tol=1e-14, max_iters=30)[0] for _ in range(3)]
    np.testing.assert_array_equal(xs[0], xs[1])
    np.testing.assert_array_equal(xs[0], xs[2])
    g.close()
