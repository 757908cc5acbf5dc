"""Assembly through element matrices in scratch memory and a gather per row
(the default of small general thermal meshes) against element colouring on the
same problem, to the bit (the same element kernels, the contributions of an
entry in the order of the colours): meshes of one element and up, odd counts,
every order and rule, Dirichlet rows on some and all sides, perturbed and box
elements, residual alone and accumulation.  The memory and the options around
it, in contexts and in the server."""
import numpy as np
import pytest

from mrhyde_amd import Problem

pytestmark = pytest.mark.gpu

CASES = [(1, 2, (1, 1), 0.0, 15), (1, 0, (5, 3), 0.0, 1), (1, 4, (17, 9), 0.1, 3), (2, 2, (3, 1), 0.0, 2),
         (2, 4, (9, 14), 0.1, 15), (2, 6, (2, 2), 0.0, 4), (3, 6, (5, 4), 0.1, 8), (4, 8, (3, 2), 0.0, 1),
         (5, 10, (2, 3), 0.0, 15), (6, 12, (1, 2), 0.0, 3), (1, 0, (3, 2, 1), 0.0, 3), (1, 2, (1, 1, 1), 0.0, 0),
         (1, 2, (9, 7, 5), 0.1, 63), (1, 4, (4, 3, 2), 0.0, 16), (2, 2, (2, 3, 4), 0.0, 32), (2, 4, (1, 1, 1), 0.1, 3),
         (2, 4, (5, 4, 3), 0.1, 63), (2, 6, (2, 1, 3), 0.0, 3), (2, 4, (193, 121), 0.0, 3), (2, 4, (25, 24, 24), 0.1, 3)]


@pytest.mark.parametrize("order,quad,n,perturb,dbc", CASES,
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_matches_colouring(order, quad, n, perturb, dbc):
    from mrhyde_amd import Mhx

    print(f"[element store] p{order} q{quad} {n}", flush=True)
    rng = np.random.default_rng(order + quad + sum(n))
    ne = int(np.prod(n))
    p = Problem(dim=len(n), order=order, quadrature=quad, n=n, k0=np.exp(rng.standard_normal(ne)), diff_u2=0.7,
                src_elem=rng.standard_normal(ne), modes=[(1.3, (2.0, 0.0, 3.0)[:len(n)])], dbc_sides=dbc, dbc_const=0.3,
                perturb=perturb)
    g, c = Mhx(p), Mhx(p)
    c.set_option("assembly.element_store", 0)
    assert g.get_option("assembly.colouring") == 0
    u = rng.standard_normal(g.n_dof)
    rc, jc = c.assembleJacRes(u)
    r, j = g.assembleJacRes(u)
    r2, j2 = g.assembleJacRes(u)
    np.testing.assert_array_equal(j, j2)
    np.testing.assert_array_equal(r, r2)
    np.testing.assert_array_equal(r, rc)
    np.testing.assert_array_equal(j, jc)
    np.testing.assert_array_equal(g.assembleRes(u), c.assembleRes(u))
    r0, j0 = rng.standard_normal(g.n_dof), rng.standard_normal(g.nnz)
    ra, ja = g.assemble(u, r0.copy(), j0.copy(), accumulate=True)
    rb, jb = c.assemble(u, r0.copy(), j0.copy(), accumulate=True)
    np.testing.assert_array_equal(ra, rb)
    np.testing.assert_array_equal(ja, jb)
    g.close(), c.close()


def _routes(g, u):
    """Names of the kernels that one assembly of residual and Jacobian runs."""
    g.profile_reset()
    g.profile(True)
    g.assembleJacRes(u)
    g.profile(False)
    return {k for k, v in g.profile_read().items() if k.startswith("k_") and v[1]}


PROBLEMS = {"general": dict(dim=2, order=1, quadrature=2, n=(9, 8)), "box": dict(dim=3, order=2, quadrature=4, n=(3, 2, 2)),
            "navier-stokes": dict(dim=2, order=1, quadrature=2, n=(6, 5), physics=2, mu=0.1, supg=True, pspg=True)}


@pytest.mark.parametrize("kind", list(PROBLEMS))
def test_assembly_options_survive_a_round_trip(kind):
    """Reading the assembly options and setting them to what was read, before
    and after other values, leaves the route of the default."""
    from mrhyde_amd import Mhx

    g = Mhx(Problem(**PROBLEMS[kind]))
    u = np.random.default_rng(1).standard_normal(g.n_dof)
    first = _routes(g, u)
    assert ("k_gather_rows" in first) == (kind == "general"), first
    names = ("assembly.colouring", "assembly.element_store")
    saved = {k: g.get_option(k) for k in names}
    for k in names:
        g.set_option(k, saved[k])
    assert _routes(g, u) == first
    g.set_option("assembly.colouring", 1)
    g.set_option("assembly.element_store", 0)
    assert "k_gather_rows" not in _routes(g, u)
    for k in names:
        g.set_option(k, saved[k])
    assert _routes(g, u) == first and {k: g.get_option(k) for k in names} == saved
    g.close()


def _free():
    import gc

    import torch

    gc.collect()  # (contexts that earlier tests left)
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_scratch_is_held_only_while_the_assembly_uses_it():
    """512^2 Q1: 40 MiB.  Another route or a time state gives them back, the way
    back to the steady default takes them again, with the same sums throughout."""
    from mrhyde_amd import Mhx

    g = Mhx(Problem(dim=2, order=1, quadrature=2, n=(512, 512), k0=np.linspace(1, 2, 512 * 512)))
    u = np.random.default_rng(1).standard_normal(g.n_dof)
    r, j = g.assembleJacRes(u)
    g.set_time_state(0.1, 1, [u])  # (the time state's own buffers, which it keeps)
    g.set_time_state(0.1, 0)
    size, held = 512 * 512 * (16 + 4) * 8, _free()
    steps = [(("assembly.colouring", 1), ("assembly.colouring", 0)),
             (("assembly.element_store", 0), ("assembly.element_store", 1))]
    for off, on in steps:
        g.set_option(*off)
        assert _free() >= held + size
        ro, jo = g.assembleJacRes(u)
        assert np.abs(ro - r).max() <= 1e-12 * np.abs(r).max() and np.abs(jo - j).max() <= 1e-12 * np.abs(j).max()
        g.set_option(*on)
        assert _free() < held + size
        rn, jn = g.assembleJacRes(u)
        np.testing.assert_array_equal(rn, r), np.testing.assert_array_equal(jn, j)
    g.set_time_state(0.1, 1, [u])
    assert _free() >= held + size
    g.assembleJacRes(u)
    g.set_time_state(0.1, 0)
    assert _free() < held + size
    np.testing.assert_array_equal(g.assembleJacRes(u)[1], j)
    g.close()


def test_captured_assembly_keeps_its_scratch():
    """A captured graph holds the scratch memory's address: the memory stays
    while options and the time state change, and replays keep their results."""
    import torch

    from mrhyde_amd import Mhx

    g = Mhx(Problem(dim=2, order=2, quadrature=4, n=(24, 17), perturb=0.1, perturb_seed=2, diff_u2=0.5))
    rng = np.random.default_rng(2)
    u = torch.from_numpy(rng.standard_normal(g.n_dof)).cuda()
    res, jac = torch.zeros(g.n_dof, dtype=torch.float64).cuda(), torch.zeros(g.nnz, dtype=torch.float64).cuda()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        g.assemble(u, res, jac)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        g.assemble(u, res, jac)
    for change in (None, ("assembly.colouring", 1), ("assembly.element_store", 0), "time"):
        if change == "time":
            g.set_time_state(0.1, 1, [u.cpu().numpy()])
        elif change:
            g.set_option(*change)
        u.copy_(torch.from_numpy(rng.standard_normal(g.n_dof)))
        filler = [torch.full((1 << 20,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        f = Mhx(Problem(dim=2, order=2, quadrature=4, n=(24, 17), perturb=0.1, perturb_seed=2, diff_u2=0.5))
        r, j = f.assembleJacRes(u.cpu().numpy())
        f.close()
        np.testing.assert_array_equal(res.cpu().numpy(), r)
        np.testing.assert_array_equal(jac.cpu().numpy(), j)
        del filler
    g.close()


def test_segment_survives_a_round_trip():
    """assembly.segment read and set to what was read stays automatic: it still
    follows the kernel (sine modes leave room for fewer workgroups)."""
    from mrhyde_amd import Mhx

    modes = [(1.0, (np.pi, np.pi, np.pi))]
    kw = dict(dim=3, order=2, quadrature=4, n=(192, 2, 6))
    ref = {m: Mhx(Problem(**kw, modes=modes if m else [])).get_option("assembly.segment") for m in (False, True)}
    assert ref[False] != ref[True], ref
    g = Mhx(Problem(**kw))
    g.set_option("assembly.segment", g.get_option("assembly.segment"))
    g.update(Problem(**kw, modes=modes))
    assert g.get_option("assembly.segment") == ref[True]
    g.set_option("assembly.segment", 6)
    assert g.get_option("assembly.segment") == 6
    g.set_option("assembly.segment", ref[True])
    g.update(Problem(**kw))
    assert g.get_option("assembly.segment") == ref[False]
    g.close()


def test_server_budget_without_scratch():
    """A budget that holds a request only without the scratch memory still
    admits it, with the same bits."""
    from mrhyde_amd import Server

    p = Problem(dim=3, order=1, quadrature=2, n=(12, 11, 10), modes=[(1.0, (np.pi, np.pi, np.pi))], diff_u2=0.5)
    need = Server.footprint(p)[2]
    xs = []
    for budget in (need, need - 8 * 64 * p.n_elem):
        s = Server(max_active=1, max_cached=1, hbm_budget=budget)
        xs.append(s.poll(s.submit(p))[0])
        s.close()
    np.testing.assert_array_equal(xs[0], xs[1])


def test_server_evicts_nothing_for_scratch():
    """A budget that holds two contexts only if one does without its scratch
    memory keeps both: the third request finds the first one's context."""
    from mrhyde_amd import Server

    a = Problem(dim=3, order=1, quadrature=2, n=(12, 11, 10), modes=[(1.0, (np.pi, np.pi, np.pi))])
    b = Problem(dim=3, order=1, quadrature=2, n=(11, 11, 10), modes=[(1.0, (np.pi, np.pi, np.pi))])
    s = Server(max_active=1, max_cached=4)
    alone = s.poll(s.submit(b))[0]
    s.close()
    s = Server(max_active=1, max_cached=4, hbm_budget=Server.footprint(a)[2] + Server.footprint(b)[2] - 8)
    s.poll(s.submit(a))
    x = s.poll(s.submit(b))[0]
    s.poll(s.submit(a))
    info = s.info()
    assert info["created"] == 2 and info["reused"] == 1 and info["bytes_held"] <= info["budget"], info
    np.testing.assert_array_equal(x, alone)
    s.close()
