"""Row sums of FP32 products (the inner solves of iterative refinement) are
formed in FP64 and rounded once: the order-2 lattice product and the
one-workgroup CG.

Two CG iterations from zero on b = s (signs) return u s + v q with q = A s.
Every row of A has entries up to 256 that cancel to (A s)_i = d_i between 1
and 2, all multiples of 1/1024 with at most 24 bits, so the FP64 sum is exact;
a sum in FP32 is off by some 1e-5.

Tolerance: x is rounded after each of the two updates, r and p once, each to
half a unit of 2^-23 of at most the largest entry: 4 x 2^-24 of it, twice that
here."""
import numpy as np
import pytest

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu

# one workgroup (2-D Q1, 2-D Q2 and Q3, 3-D Q1); the lattice product (3-D and 2-D Q2, past the two-launch sizes)
CASES = [(1, (31, 32)), (2, (20, 11)), (3, (9, 7)), (1, (12, 12, 12)), (2, (16, 17, 16)), (2, (150, 149))]


@pytest.mark.parametrize("order,n", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else f"p{v}")
def test_rows_sum_in_64_bits(order, n):
    from mrhyde_amd import Mhx

    print(f"[fp32 sums] p{order} {n}", flush=True)
    rng = np.random.default_rng(order + sum(n))
    g = Mhx(Problem(dim=len(n), order=order, quadrature=2 * order, n=n, dbc_sides=0))
    rp, ci = g.crs_pattern()
    rows = np.repeat(np.arange(g.n_dof), np.diff(rp))
    s = rng.choice([-1.0, 1.0], g.n_dof)
    d = s * (1.0 + rng.integers(0, 1024, g.n_dof) / 1024)
    a = rng.integers(-256 * 1024, 256 * 1024, g.nnz) / 1024
    diag = ci == rows
    a[diag] = 0.0
    rest = np.zeros(g.n_dof)
    np.add.at(rest, rows, a * s[ci])
    a[diag] = (d - rest) * s
    assert np.abs(a).max() < 2.0 ** 14  # (a multiple of 2^-10: exact in FP32)
    x, st = g.linearSolver(a, s.copy(), solver="cg", precond="none-fp32", tol=1e-30, max_iters=2, inner_iters=2,
                           inner_tol=1e-30)
    assert st["iters"] == 2
    basis = np.stack([s, d], 1)
    fit = basis @ np.linalg.lstsq(basis, x, rcond=None)[0]
    err, tol = np.abs(x - fit).max(), 8 * 2.0 ** -24 * np.abs(x).max()
    print(f"  error {err:.2e}, tolerance {tol:.2e}, largest {np.abs(x).max():.2e}", flush=True)
    assert err <= tol
    g.close()
