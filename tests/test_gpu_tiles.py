"""Sizes at which the launch shapes change or leave remainders: element counts
around a wave, a workgroup and the steps of the trial-column rule, compared
with the FP64 oracle on sampled rows (the first, the last and those at the
edges of a workgroup's 256 rows), every column.

Bars as in the parity tests: 2e-6 of the row's largest entry and 1e-5 relative
Frobenius (FP32 regular pairs)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NIHU = (dict(rule="nihu", near="mean_edge", limit=1.5), dict(rule=0, fixed_degree=0, near_mode=0, near_limit=1.5))
SEVEN = (dict(rule="fixed", degree=5, near="diameter", limit=2.0),
         dict(rule=1, fixed_degree=5, near_mode=1, near_limit=2.0))


@pytest.fixture(scope="module")
def nb():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    from nihu_amd import nbem
    return nbem


def check(got, ref):
    scale = np.abs(ref).max(axis=1, keepdims=True)
    assert (np.abs(got - ref) / scale).max() < 2e-6
    assert np.linalg.norm(got - ref) < 1e-5 * np.linalg.norm(ref)


def surface(n_elem, quads=False):
    """the first n_elem elements of a cube sphere (triangles: its squares cut in two, jittered)"""
    from nihu_amd.mesh import cubed_sphere
    n = int(np.ceil(np.sqrt(n_elem / (6 if quads else 12))))
    nodes, q = cubed_sphere(n)
    if quads:
        return nodes, np.ascontiguousarray(q[:n_elem])
    nodes = nodes * (1.0 + np.random.default_rng(n_elem).uniform(-0.01, 0.01, len(nodes)))[:, None]
    t = np.concatenate([q[:, None, [0, 1, 2]], q[:, None, [0, 2, 3]]], axis=1).reshape(-1, 3)
    return nodes, np.ascontiguousarray(t[:n_elem])


def sample(n):
    return np.unique([r for r in (0, 63, 64, 255, 256, 511, 512, n - 2, n - 1) if 0 <= r < n]).astype(np.int32)


@pytest.mark.parametrize("policy", [NIHU, SEVEN], ids=["nihu", "seven"])
@pytest.mark.parametrize("n_elem", [1, 63, 65, 255, 257, 1999, 3001, 5003, 9001])
def test_burton_miller_triangles(nb, orc, n_elem, policy):
    import torch
    nodes, tris = surface(n_elem)
    m = nb.Mesh(nodes, tris)
    A, B = nb.colmajor(n_elem, n_elem), nb.colmajor(n_elem, n_elem)
    nb.assemble_bm(m, 4.0, A, B, pol=nb.policy(**policy[0]))
    torch.cuda.synchronize()
    rows = sample(n_elem)
    Ar, Br = orc.assemble_bm(nodes, tris, 4.0, pol=orc.policy(**policy[1]), rows=rows)
    check(A[rows].cpu().numpy(), Ar)
    check(B[rows].cpu().numpy(), Br)


@pytest.mark.parametrize("n_elem", [1, 63, 65, 257, 2999, 9001])
def test_burton_miller_quadrilaterals(nb, orc, n_elem):
    import torch
    nodes, quads = surface(n_elem, quads=True)
    m = nb.Mesh(nodes, quads)
    A, B = nb.colmajor(n_elem, n_elem), nb.colmajor(n_elem, n_elem)
    nb.assemble_bm(m, 4.0, A, B)
    torch.cuda.synchronize()
    rows = sample(n_elem)
    Ar, Br = orc.assemble_bm(nodes, quads, 4.0, rows=rows)
    check(A[rows].cpu().numpy(), Ar)
    check(B[rows].cpu().numpy(), Br)


def galerkin(nb, m, t, form, ny, k, pol=None):
    import torch
    out = nb.colmajor(m.dofs(form, "test"), t.dofs(form, "trial"))
    nb.assemble(m, t, out, nb.NB_HELMHOLTZ, 0, ny, k, pol=pol, accumulate=False, formalism=form)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("form", ["galerkin_linear", "galerkin"])
@pytest.mark.parametrize("quads", [False, True], ids=["triangles", "quadrilaterals"])
@pytest.mark.parametrize("n_elem", [1, 2, 63, 65, 129, 701])
def test_galerkin_nihu(nb, orc, n_elem, quads, form):
    # test tiles, trial chunks and the wave-per-pair list with remainders
    nodes, el = surface(n_elem, quads)
    m = nb.Mesh(nodes, el)
    scale = 0.0      # the single layer's at least: the double layer of one flat element is rounding
    for ny in (0, 1):
        ref = orc.assemble_galerkin(nodes, el, 1, 0, ny, k=3.0, linear=form == "galerkin_linear")
        got = galerkin(nb, m, m, form, ny, 3.0)
        scale = max(scale, np.abs(ref).max())
        assert np.abs(got - ref).max() < 2e-6 * scale


@pytest.mark.parametrize("quads", [False, True], ids=["triangles", "quadrilaterals"])
def test_galerkin_mostly_close_pairs(nb, quads):
    # a fine test mesh inside the near breakpoints of a few large trial
    # elements: too many close pairs for a list, so the tiled pass takes every
    # degree; a part of the mesh has few enough and takes the list.  The two
    # evaluate the same points in other orders (points as close as these
    # leave FP32 itself 1e-5 to 1e-4 off the oracle, whatever the pass)
    nodes, el = surface(24300, quads)
    coarse, cel = surface(24 if quads else 12, quads)
    assert len(el) * len(cel) > (len(el) * len(cel) + 2 ** 24) / 64
    t = nb.Mesh(coarse * 1.3, cel)
    whole, part = nb.Mesh(nodes, el), nb.Mesh(nodes, np.ascontiguousarray(el[:2000]))
    for ny in (0, 1):
        check(galerkin(nb, part, t, "galerkin", ny, 2.0), galerkin(nb, whole, t, "galerkin", ny, 2.0)[:2000])


@pytest.mark.parametrize("kind", [("complex64", False), ("complex64", True), ("complex128", False)],
                         ids=["c64", "c64-accumulate", "c128"])
@pytest.mark.parametrize("degree", [4, 2])
@pytest.mark.parametrize("n_elem", [1, 2, 63, 65, 129, 701])
def test_galerkin_fixed_single_layer(nb, orc, n_elem, degree, kind):
    # one mesh, one rule: pairs taken once and mirrored (not into a result that
    # already holds something)
    import torch
    nodes, el = surface(n_elem)
    m = nb.Mesh(nodes, el)
    n = m.n_nodes
    rng = np.random.default_rng(n_elem)
    ref = orc.assemble_galerkin(nodes, el, 1, 0, 0, k=3.0, linear=True, pol=orc.policy(rule=1, fixed_degree=degree))
    out = nb.colmajor(n, n, kind[0])
    old = np.zeros((n, n), dtype=complex)
    if kind[1]:
        old = (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))) * np.abs(ref).max()
        out.copy_(torch.from_numpy(old))
    nb.assemble(m, m, out, nb.NB_HELMHOLTZ, 0, 0, 3.0, pol=nb.policy("fixed", degree=degree), accumulate=kind[1],
                formalism="galerkin_linear")
    torch.cuda.synchronize()
    # an accumulated float32 entry also rounds the old content (up to 5 times the largest entry)
    assert np.abs(out.cpu().numpy() - old - ref).max() < 2e-6 * np.abs(ref).max()


@pytest.mark.parametrize("dtype,fam,k,alpha", [("float32", 0, 0.0, 1.0), ("float32", 0, 0.0, -0.75), ("float64", 0, 0.0, 2.5),
                                               ("complex64", 1, 3.0, 0.8 + 0.25j), ("complex128", 1, 3.0, -0.5j),
                                               ("complex64", 1, complex(3.0, -0.4), 1.0)])
@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("n_elem", [1, 65, 701])
def test_galerkin_fixed_single_layer_outputs(nb, orc, n_elem, pad, dtype, fam, k, alpha):
    # the mirrored pairs in every type of result, with rows to spare below each
    # column (left alone) and a factor; bar as above
    import torch
    nodes, el = surface(n_elem)
    m = nb.Mesh(nodes, el)
    n = m.n_nodes
    ref = orc.assemble_galerkin(nodes, el, fam, 0, 0, k=k, alpha=alpha, linear=True, pol=orc.policy(rule=1, fixed_degree=4))
    full = torch.full((n, n + pad), 7.0, dtype=getattr(torch, dtype), device="cuda")
    out = full.t()[:n]
    nb.assemble(m, m, out, fam, 0, 0, k, alpha=alpha, pol=nb.policy("fixed", degree=4), accumulate=False,
                formalism="galerkin_linear")
    torch.cuda.synchronize()
    assert (full[:, n:] == 7.0).all()
    assert np.abs(out.cpu().numpy() - ref).max() < 2e-6 * np.abs(ref).max()


def test_field_blocks_follow_the_arrays(nb):
    # more field points than one block: the kept blocks give the result of a new
    # mesh, also after the field mesh's node array has changed
    import torch
    from nihu_amd import postproc
    from nihu_amd.mesh import create_slab
    nodes, quads = surface(54, quads=True)
    s = nb.Mesh(nodes, quads)
    corners = np.array([[-2, -2, 2.5], [2, -2, 2.5], [2, 2, 3], [-2, 2, 3]], dtype=float)
    fn, fe = create_slab(corners, 20, 15)
    field = nb.Mesh(fn, fe)
    p = torch.ones(54, dtype=torch.complex128, device="cuda")
    first = postproc.field_pressure(field, s, 2.0, p, 1j * p, block_rows=128)
    again = postproc.field_pressure(field, s, 2.0, p, 1j * p, block_rows=128)
    whole = postproc.field_pressure(field, s, 2.0, p, 1j * p)
    assert torch.equal(first, again)
    assert (first - whole).abs().max() <= 1e-12 * whole.abs().max()
    field.nodes[:, 2] += 0.5
    moved = postproc.field_pressure(field, s, 2.0, p, 1j * p, block_rows=128)
    fresh = postproc.field_pressure(nb.Mesh(field.nodes.copy(), fe), s, 2.0, p, 1j * p, block_rows=128)
    assert torch.equal(moved, fresh)


def test_field_blocks_in_the_byte_count(nb):
    # the kept blocks are in the field mesh's count; of a field of more blocks
    # than are kept none stays, and every way of cutting gives the same values
    import torch
    from nihu_amd import postproc
    from nihu_amd.mesh import create_slab
    nodes, quads = surface(54, quads=True)
    s = nb.Mesh(nodes, quads)
    corners = np.array([[-2, -2, 2.5], [2, -2, 2.5], [2, 2, 3], [-2, 2, 3]], dtype=float)
    field = nb.Mesh(*create_slab(corners, 20, 15))
    p = torch.ones(54, dtype=torch.complex128, device="cuda")
    whole = postproc.field_pressure(field, s, 2.0, p, 1j * p)
    alone = field.device_bytes()
    many = postproc.field_pressure(field, s, 2.0, p, 1j * p, block_rows=8)      # 38 blocks
    assert field.device_bytes() == alone
    few = postproc.field_pressure(field, s, 2.0, p, 1j * p, block_rows=128)
    assert field.device_bytes() >= 2 * alone - 200
    for got in (many, few):
        assert (got - whole).abs().max() <= 1e-12 * whole.abs().max()


@pytest.mark.parametrize("rows,cols,ld", [(1, 5, 1), (257, 3001, 300), (8191, 8193, 8191), (8192, 8192, 8192),
                                          (8195, 8195, 8201)])
def test_product_sizes(nb, rows, cols, ld):
    """Matrix-vector product on both sides of the size from which the matrix
    is read past the caches, with partial steps of eight columns and chunks and a
    padded leading dimension; bound of FP64 sums in any order, cols * 2^-52 times
    sum |a| |x|."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(rows)
    A = torch.randn(cols, ld, dtype=torch.complex64, device="cuda", generator=g).t()[:rows]
    x = torch.randn(cols, dtype=torch.complex128, device="cuda", generator=g)
    y = nb.gemv(A, x)
    ref, mag = torch.zeros_like(y), torch.zeros(rows, dtype=torch.float64, device="cuda")
    for j in range(0, cols, 1024):
        b = A[:, j:j + 1024].to(torch.complex128)
        ref += (b * x[j:j + 1024]).sum(1)
        mag += (b.abs() * x[j:j + 1024].abs()).sum(1)
    assert ((y - ref).abs() <= cols * 2.0 ** -52 * mag).all()


def test_launch_shape_set_and_reset(nb):
    # a fixed column count serialises a small matrix (5 workgroups of 1280
    # columns); 0 gives the rule by the grid's size back, and neither changes the
    # result.  The passes take about 1 ms and 0.02 ms: a factor of 4 is asked for
    import torch
    from nihu_amd.mesh import jittered_icosphere
    nodes, tris = jittered_icosphere(3, seed=0)
    m = nb.Mesh(nodes, tris)

    def run():
        A, B = nb.colmajor(m.n, m.n), nb.colmajor(m.n, m.n)
        nb.assemble_bm(m, 3.0, A, B)
        nb.profile(True)
        nb.profile_read(reset=True)
        for _ in range(5):
            nb.assemble_bm(m, 3.0, A, B)
        ms, launches = nb.profile_read(reset=True)["regular"]
        nb.profile(False)
        torch.cuda.synchronize()
        return A, ms / launches

    try:
        nb.set_launch(tile_cols=4096)
        fixed, slow = run()
        nb.set_launch(tile_cols=0)
        auto, fast = run()
    finally:
        nb.set_launch()
    print("4096 columns %.3f ms, by the grid %.3f ms" % (slow, fast), flush=True)
    assert torch.equal(torch.view_as_real(fixed), torch.view_as_real(auto))
    assert fast < slow / 4
