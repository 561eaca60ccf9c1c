"""The kept lists of close pairs: what displaces what, what they hold of device
memory (8 bytes per listed pair, in the trial mesh's byte count), and what a
call does that has none."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nb():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    from nihu_amd import nbem
    return nbem


def sphere(level=2, move=0.0, seed=0):
    from nihu_amd.mesh import jittered_icosphere
    nodes, tris = jittered_icosphere(level, seed=seed)
    return nodes + np.array([move, 0.0, 0.0]), tris


def operator(nb, test, trial, form, ny=0, pol=None, dtype="complex64"):
    import torch
    out = nb.colmajor(test.dofs(form, "test"), trial.dofs(form, "trial"), dtype)
    nb.assemble(test, trial, out, nb.NB_HELMHOLTZ, 0, ny, 3.0, pol=pol, accumulate=False, formalism=form)
    torch.cuda.synchronize()
    return out


def test_other_lists_leave_the_sweeps_resident(nb):
    # Galerkin calls and collocation against other meshes, more than eight of
    # each: the mesh's own near list, which the allocation-free sweep takes, stays
    import torch
    m = nb.Mesh(*sphere())
    ks = np.array([2.0, 3.0])
    A, B = (torch.zeros((2, m.n, m.n), dtype=torch.complex64, device="cuda").transpose(1, 2) for _ in range(2))
    nb.assemble_sweep(m, ks, A, B)
    want = A.clone(), B.clone()
    others = [nb.Mesh(*sphere(1, 0.1 * i)) for i in range(5)]
    for t in others:
        for ny in (0, 1):
            operator(nb, t, m, "galerkin_linear", ny)
            operator(nb, t, m, "collocation", ny, nb.policy("nihu", limit=1.5 + 0.01 * ny))
    # the sweep's own thresholds again: the last policy above had others
    operator(nb, others[0], m, "collocation", 0, nb.policy("nihu"))
    nb.assemble_sweep(m, ks, A, B, noalloc=True)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(A), torch.view_as_real(want[0]))
    assert torch.equal(torch.view_as_real(B), torch.view_as_real(want[1]))


@pytest.mark.parametrize("form", ["collocation", "galerkin"])
def test_lists_of_many_test_meshes(nb, form):
    # twelve test meshes in turn: all their lists stay (a second round builds
    # nothing), and leave once their mesh is gone
    m = nb.Mesh(*sphere())
    tests = [nb.Mesh(*sphere(1, 0.05 * i)) for i in range(12)]
    operator(nb, tests[0], m, form)          # tables
    base, seen = m.device_bytes(), []
    for t in tests[1:]:
        operator(nb, t, m, form)
        seen.append(m.device_bytes())
    grown = np.diff([base] + seen)
    assert (grown >= 0).all() and grown.sum() > 0
    for t in tests:
        operator(nb, t, m, form)
        assert m.device_bytes() == seen[-1]
    tests.clear()
    del t
    operator(nb, m, m, form)
    own = m.device_bytes()
    operator(nb, nb.Mesh(*sphere(1, 40.0)), m, form)      # far away: an empty list
    assert m.device_bytes() == own
    fresh = nb.Mesh(*sphere())
    operator(nb, fresh, fresh, form)
    assert own == fresh.device_bytes()


def test_no_memory_for_a_list_that_is_not_taken(nb):
    # a fine test mesh inside the breakpoints of a few large trial elements: too
    # many close pairs for a list, and none of them is held
    from nihu_amd.mesh import cubed_sphere
    nodes, q = cubed_sphere(64)
    fine, coarse = nb.Mesh(nodes, q), cubed_sphere(2)
    used, far = (nb.Mesh(coarse[0] * 1.3 + move, coarse[1]) for move in (0.0, 100.0))
    for ny in (0, 1):
        operator(nb, fine, used, "galerkin", ny)
        operator(nb, fine, far, "galerkin", ny)      # the same tables, no close pair
        assert used.device_bytes() == far.device_bytes()


def test_close_pairs_of_a_large_mesh(nb, orc):
    # over 2^31 pairs of elements, few of them close: they are listed (the double
    # layer's call before leaves the list as the only thing that the single
    # layer's adds), and the rows are the oracle's
    import torch
    from nihu_amd.mesh import cubed_sphere
    nodes, q = cubed_sphere(63)
    tris = np.ascontiguousarray(np.concatenate([q[:, None, [0, 1, 2]], q[:, None, [0, 2, 3]]], axis=1).reshape(-1, 3))
    assert len(tris) ** 2 > 2 ** 31
    m = nb.Mesh(nodes, tris)
    out = nb.colmajor(m.n_nodes, m.n_nodes, "float32")
    grown = []
    for ny in (1, 0):
        nb.assemble(m, m, out, nb.NB_LAPLACE, 0, ny, accumulate=False, formalism="galerkin_linear")
        torch.cuda.synchronize()
        grown.append(m.device_bytes())
    assert grown[1] > grown[0]
    rows = np.array([0, 1000, m.n_nodes - 1])
    el = np.unique(np.nonzero(np.isin(tris, rows))[0]).astype(np.int32)
    ref = orc.assemble_galerkin(nodes, tris, 0, 0, 0, linear=True, test_elems=el)[rows].real
    got = out[torch.from_numpy(rows).cuda()].cpu().numpy()
    assert np.abs(got - ref).max() < 2e-6 * np.abs(ref).max()


@pytest.mark.parametrize("two", [False, True], ids=["one-mesh", "two-meshes"])
@pytest.mark.parametrize("quads", [False, True], ids=["triangles", "quadrilaterals"])
def test_capture_without_a_list(nb, quads, two):
    # the double layer's call leaves every table that the single layer takes, not
    # its list: a graph captured then holds the pass that needs none
    import torch
    from nihu_amd.mesh import cubed_sphere
    nodes, el = cubed_sphere(5) if quads else sphere()
    m = nb.Mesh(nodes, el)
    t = nb.Mesh(nodes * 1.2, el) if two else m
    operator(nb, t, m, "galerkin_linear", 1)
    out = nb.colmajor(t.n_nodes, m.n_nodes)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        nb.assemble(t, m, out, nb.NB_HELMHOLTZ, 0, 0, 3.0, accumulate=False, formalism="galerkin_linear")
    want = operator(nb, t, m, "galerkin_linear", 0, dtype="complex128")     # with the list
    for _ in range(3):
        out.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        # float32 sums in another order: 2^-24 per addition, some 40 to an entry
        assert (out - want).abs().max() < 2.4e-6 * want.abs().max()


def test_a_captured_list_stays(nb):
    # a graph holds the list's addresses: eighty other test meshes (far away,
    # their lists are empty) do not displace it
    import torch
    m, t = nb.Mesh(*sphere()), nb.Mesh(*sphere(1, 0.3))
    want = operator(nb, t, m, "galerkin_linear")
    out = nb.colmajor(t.n_nodes, m.n_nodes)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        nb.assemble(t, m, out, nb.NB_HELMHOLTZ, 0, 0, 3.0, accumulate=False, formalism="galerkin_linear")
    held = m.device_bytes()
    others = [nb.Mesh(*sphere(0, 50.0 + i)) for i in range(80)]
    for o in others:
        operator(nb, o, m, "galerkin_linear")
    assert m.device_bytes() == held
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert (out - want).abs().max() < 2.4e-6 * want.abs().max()
