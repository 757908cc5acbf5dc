"""The lattice product with four unknowns per node (3-D Q1 Navier-Stokes; 16
lanes per node): meshes from one element up, with the columns in closed form
and from the index stream, against a plain sum over the CRS pattern.

Tolerance: a row of m entries summed in any order is within m eps of the sum
of its terms' magnitudes (m <= 108); 2 m eps here."""
import numpy as np
import pytest

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu

MESHES = [(1, 1, 1), (2, 1, 1), (1, 2, 3), (3, 3, 3), (5, 4, 2), (4, 7, 1), (9, 2, 6), (16, 3, 5)]


@pytest.mark.parametrize("n", MESHES, ids=lambda n: "x".join(map(str, n)))
def test_product_matches_pattern_sum(n):
    from mrhyde_amd import Mhx

    print(f"[node4] {n}", flush=True)
    g = Mhx(Problem(dim=3, order=1, quadrature=2, n=n, physics=2, mu=0.1, supg=True, pspg=True, dbc_sides=63))
    rp, ci = g.crs_pattern()
    rng = np.random.default_rng(sum(n))
    a, x = rng.standard_normal(g.nnz), rng.standard_normal(g.n_dof)
    rows = np.repeat(np.arange(g.n_dof), np.diff(rp))
    ref, mag = np.zeros(g.n_dof), np.zeros(g.n_dof)
    np.add.at(ref, rows, a * x[ci])
    np.add.at(mag, rows, np.abs(a * x[ci]))
    y = g.apply(a, x)
    assert (np.abs(y - ref) <= 2 * np.diff(rp) * np.finfo(float).eps * mag).all()
    g.set_option("krylov.lattice_columns", 0)
    np.testing.assert_array_equal(g.apply(a, x), y)
    g.close()
