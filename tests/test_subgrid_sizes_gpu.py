"""Batched subgrid solves at every size per axis (each has its own columns per
thread), both workgroup sizes and precisions, cubes and boxes with sources,
against the residual of the oracle's system; and the transfer of large results
through staging buffers against the same instances in small batches.

Tolerance: the solver's own (1e-10), with a factor two for the residual that the
oracle's matrix gives in another order of sums."""
import numpy as np
import pytest

from conftest import spmv_np
from mrhyde_amd.abi import Problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def systems():
    from oracle import Oracle

    rng = np.random.default_rng(8)
    out = {}
    for box in (False, True):
        n_axis = np.arange(2, 17, dtype=np.int32)
        k, g, src, ext, orc = [], [], [], [], []
        for n in n_axis:
            ne, nn = int(n) ** 3, (int(n) + 1) ** 3
            k.append(np.exp(0.5 * rng.standard_normal(ne)))
            g.append(rng.uniform(-1, 1, nn))
            src.append(rng.standard_normal(ne))
            ext.append(rng.uniform(0.5, 2.0, 3) if box else np.ones(3))
            o = Oracle(Problem(dim=3, order=1, quadrature=2, n=(int(n),) * 3, hi=tuple(ext[-1]), k0=k[-1],
                               src_elem=src[-1] if box else None, dbc_values=g[-1]))
            u0 = o.setDirichlet(np.zeros(o.n_dof))
            orc.append((u0, *o.assembleJacRes(u0), *o.crs_pattern()))
        out[box] = (n_axis, np.concatenate(k), np.concatenate(g), dict(extent=np.array(ext), src=np.concatenate(src))
                    if box else {}, orc)
    return out


@pytest.mark.parametrize("box", [False, True])
@pytest.mark.parametrize("wg", [512, 1024])
@pytest.mark.parametrize("precision", ["fp64", "fp32-refined"])
def test_every_size(systems, precision, wg, box):
    from mrhyde_amd import SubgridBatch

    n_axis, k, g, kw, orc = systems[box]
    b = SubgridBatch(n_axis, k, g, tol=1e-10, precision=precision, wg_size=wg, **kw)
    b.solve()
    x, _, rel, _ = b.results()
    for i, (u0, res, jac, rp, ci) in enumerate(orc):
        r = res - spmv_np(rp, ci, jac, b.instance(x, i) - u0)
        assert rel[i] <= 1e-10 and np.linalg.norm(r) <= 2e-10 * np.linalg.norm(res), (int(n_axis[i]), rel[i])
    b.close()


def test_result_buffers_outlive_batches_and_are_given_back():
    from mrhyde_amd import SubgridBatch, release_host_buffers

    rng = np.random.default_rng(5)
    n_axis = np.full(300, 16, dtype=np.int32)  # 11.8 MB of results
    args = n_axis, np.exp(0.3 * rng.standard_normal(300 * 16 ** 3)), rng.uniform(-1, 1, 300 * 17 ** 3)
    release_host_buffers()
    xs = []
    for keep in (True, True, False):
        b = SubgridBatch(*args, wg_size=512)
        b.solve()
        xs.append(b.results()[0])
        if not keep:  # given back in the batch's life: the next copy allocates anew
            assert release_host_buffers() == 8 << 20
            xs.append(b.results()[0])
        b.close()
    for x in xs[1:]:
        np.testing.assert_array_equal(x, xs[0])
    assert release_host_buffers() == 8 << 20
    assert release_host_buffers() == 0


def test_results_in_chunks_equal_small_batches():
    """10.4 MB through the buffers (chunks that do not divide it), and sizes on
    both sides of the line, below which no buffers are taken."""
    from mrhyde_amd import SubgridBatch, release_host_buffers

    rng = np.random.default_rng(7)
    n_axis = np.full(265, 16, dtype=np.int32)
    k, g = np.exp(0.3 * rng.standard_normal((265, 16 ** 3))), rng.uniform(-1, 1, (265, 17 ** 3))
    release_host_buffers()
    out = {}
    for m, held in ((60, 0), (93, 0), (94, 8 << 20), (265, 8 << 20)):  # 2.25, 3.49, 3.52 and 9.93 MiB
        b = SubgridBatch(n_axis[:m], k[:m].ravel(), g[:m].ravel(), wg_size=512)
        b.solve()
        out[m] = b.results()[0]
        b.close()
        assert release_host_buffers() == held
    for m in (60, 93, 94):
        np.testing.assert_array_equal(out[m], out[265][:m * 17 ** 3])


def test_pinned_destination_needs_no_buffers():
    import torch

    from mrhyde_amd import SubgridBatch, capi, release_host_buffers

    rng = np.random.default_rng(6)
    n_axis = np.full(300, 16, dtype=np.int32)
    b = SubgridBatch(n_axis, np.exp(0.3 * rng.standard_normal(300 * 16 ** 3)), rng.uniform(-1, 1, 300 * 17 ** 3),
                     wg_size=512)
    b.solve()
    out = torch.zeros(b.total_nodes, dtype=torch.float64, pin_memory=True)
    release_host_buffers()
    assert capi.lib.mhx_batch_results(b._h, out.data_ptr(), None, None, None) == 0
    assert release_host_buffers() == 0
    np.testing.assert_array_equal(out.numpy(), b.results()[0])
    b.close()


def test_large_results_equal_small_batches():
    from mrhyde_amd import SubgridBatch

    rng = np.random.default_rng(4)
    n_axis = np.full(70, 16, dtype=np.int32)  # 2.75 MB of results
    k = np.exp(0.3 * rng.standard_normal((70, 16 ** 3)))
    g = rng.uniform(-1, 1, (70, 17 ** 3))
    big = SubgridBatch(n_axis, k.ravel(), g.ravel())
    big.solve()
    x = big.results()[0]
    np.testing.assert_array_equal(big.results()[0], x)
    for lo, hi in ((0, 10), (37, 47), (60, 70)):  # below 1 MiB each
        s = SubgridBatch(n_axis[lo:hi], k[lo:hi].ravel(), g[lo:hi].ravel())
        s.solve()
        np.testing.assert_array_equal(s.results()[0], x[lo * 17 ** 3:hi * 17 ** 3])
        s.close()
    big.close()
