"""Batch sizes at the edges of the resident-grid launches' split: fewer items
than waves, one item to 64 per wave, exactly the resident lanes, one more
(the first range from the shared counter), and several ranges per wave with a
ragged end.  Every size equals the one-item-per-lane kernels bit for bit."""
import numpy as np
import pytest

from gpu_util import bits, build_tree, dev, host
from xdg_amd import geometry as G
from xdg_amd import philox as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIZES = [1, 63, 65, 1023, 1025, 4097, 65537, 262143, 262144, 262145, 300001, 700001]


@pytest.fixture(scope="module")
def setup():
    from xdg_amd import capi
    ctx = capi.Context(0)
    m = G.nested_spheres(3)
    vols = list(m.volumes)
    trees = [build_tree(ctx, m, v) for v in vols]
    n = max(SIZES)
    pts = P.box_points(71, P.STREAM_POS, n, [-19] * 3, [19] * 3)
    lim = min(ctx.tree_info(t)["o_limit"] for t in trees)
    pts[::997] *= 3.0 * lim / 19.0  # beyond the FP32 boxes' limit
    dirs = P.iso_dirs(71, P.STREAM_DIR, n)
    tpr = np.array([trees[i % 5] for i in range(n)], np.int32)
    tpr[5::1000] = 999  # not a tree
    yield ctx, m, vols, trees, dev(torch, pts), dev(torch, dirs), dev(torch, tpr)
    ctx.close()


def both_forms(ctx, call):
    """The result of the per-item and of the resident kernels."""
    try:
        ctx.set_traversal(persistent=False)
        ref = call()
        ctx.set_traversal(persistent=True)
        return ref, call()
    finally:
        ctx.set_traversal()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", SIZES)
def test_ray_fire_split(setup, n, prec):
    ctx, m, vols, trees, pts, dirs, tpr = setup
    excl = torch.zeros((n, 2), dtype=torch.int32, device="cuda")
    ref, got = both_forms(ctx, lambda: [host(x) for x in ctx.ray_fire(
        0, pts[:n], dirs[:n], tree_per_ray=tpr[:n], excl=excl, precision=prec)])
    assert np.array_equal(bits(got[0]), bits(ref[0]))
    assert np.array_equal(got[1], ref[1]) and np.array_equal(got[2], ref[2])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", SIZES)
def test_find_volume_split(setup, n, prec):
    ctx, m, vols, trees, pts, dirs, tpr = setup
    ref, got = both_forms(ctx, lambda: host(ctx.find_volume(trees, vols, m.ipc, pts[:n], dirs[:n], precision=prec)))
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", SIZES)
def test_point_in_volume_split(setup, n, prec):
    ctx, m, vols, trees, pts, dirs, tpr = setup
    excl = torch.arange(n, dtype=torch.int32, device="cuda").remainder(2000).reshape(n, 1)
    for d, ex in ((dirs[:n], excl), (None, None)):
        ref, got = both_forms(ctx, lambda: host(ctx.point_in_volume(trees[2], pts[:n], d, excl=ex, precision=prec)))
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("n", [1, 3, 65, 4097, 65537, 300001])
def test_closest_split(setup, n):
    """closest on a closed shell with points near, far and (every 101st) close
    to its centre, nearly as far from every triangle."""
    import pyoracle as O
    ctx, m, vols, trees, pts, dirs, tpr = setup
    p = host(pts)[:n].copy()
    p[::101] *= 1e-3
    k = min(n, 4097)
    for v in (0, 1):
        d, f = [host(x) for x in ctx.closest(trees[v], dev(torch, p))]
        rd, rf = O.Tree.from_model(m, vols[v]).closest(p[:k])
        assert np.array_equal(bits(d[:k]), bits(rd)) and np.array_equal(f[:k], rf)
        # the other points: the same as in batches of another split
        for lo in range(k, n, 50000):
            d2, f2 = [host(x) for x in ctx.closest(trees[v], dev(torch, p[lo:lo + 50000]))]
            assert np.array_equal(bits(d[lo:lo + 50000]), bits(d2)) and np.array_equal(f[lo:lo + 50000], f2)


@pytest.mark.parametrize("n", [1, 63, 1025, 65537, 300001])
def test_find_element_split(setup, n):
    """Points inside, on lattice planes and outside the mesh; every batch
    size equals the oracle on its first points and smaller batches beyond."""
    import pyoracle as O
    ctx = setup[0]
    mesh = G.kuhn_cube(7, 0.2, seed=4)
    et = ctx.build_element_tree(mesh.verts, mesh.tets, mesh.adj, mesh.face_order)
    p = P.box_points(73, P.STREAM_POS, n, [-0.1] * 3, [1.1] * 3)
    p[::7] = np.round(p[::7] * 7) / 7
    k = min(n, 20000)
    got = host(ctx.find_element(et, dev(torch, p)))
    om = O.TetMesh(mesh, with_ipc=False)
    assert np.array_equal(got[:k], om.find_element(p[:k]))
    for lo in range(k, n, 50000):
        assert np.array_equal(got[lo:lo + 50000], host(ctx.find_element(et, dev(torch, p[lo:lo + 50000]))))


def test_segments_ending_on_the_boundary(setup):
    """Segments whose ends are clamped onto the mesh's faces, edges and
    corners: some come round the segment loop without moving, up to its cap."""
    import pyoracle as O
    ctx = setup[0]
    mesh = G.kuhn_cube(9, 0.2, seed=4)
    et = ctx.build_element_tree(mesh.verts, mesh.tets, mesh.adj, mesh.face_order)
    bm = mesh.boundary_model()
    ctx.attach_boundary(et, build_tree(ctx, bm, bm.ipc), mesh.bface_elem)
    n = 60000
    p0 = P.box_points(75, P.STREAM_POS, n, [0.0] * 3, [1.0] * 3)
    p1 = np.clip(p0 + P.iso_dirs(75, P.STREAM_DIR, n) * np.geomspace(1e-3, 2.0, n)[:, None], 0.0, 1.0)
    tally = torch.zeros(mesh.tets.shape[0], dtype=torch.int64, device="cuda")
    cnt, hsh = [host(x) for x in ctx.tally_segments(et, dev(torch, p0), dev(torch, p1), tally=tally)]
    rc, rh = O.TetMesh(mesh).segments(p0, p1)
    assert np.array_equal(cnt, rc) and np.array_equal(hsh.view(np.uint64), rh)


@pytest.mark.parametrize("jitter", [0.0, 0.2])
@pytest.mark.parametrize("m", [1, 3, 4, 7])
def test_element_records(setup, m, jitter):
    """Trees of fewer elements than a block, ragged and several blocks of the
    record kernel; without jitter, edges whose ends tie in x and y.  The walks
    use every field of the records and equal the oracle."""
    import pyoracle as O
    ctx = setup[0]
    mesh = G.kuhn_cube(m, jitter, seed=4)
    et = ctx.build_element_tree(mesh.verts, mesh.tets, mesh.adj, mesh.face_order)
    bm = mesh.boundary_model()
    ctx.attach_boundary(et, build_tree(ctx, bm, bm.ipc), mesh.bface_elem)
    n = 3000
    p0 = P.box_points(77, P.STREAM_POS, n, [-0.2] * 3, [1.2] * 3)
    p1 = p0 + P.iso_dirs(77, P.STREAM_DIR, n)
    om = O.TetMesh(mesh)
    assert np.array_equal(host(ctx.find_element(et, dev(torch, p0))), om.find_element(p0))
    cnt, hsh = [host(x) for x in ctx.tally_segments(et, dev(torch, p0), dev(torch, p1))]
    rc, rh = om.segments(p0, p1)
    assert np.array_equal(cnt, rc) and np.array_equal(hsh.view(np.uint64), rh)


def contains(p, v):
    """The reference's containment test (tetrahedron_contain.cpp:11-43) of
    points (n, 3) in tets (n, 4, 3), a zero determinant included."""
    c = [v[:, k + 1] - v[:, 0] for k in range(3)]
    r = p - v[:, 0]
    cross = lambda a, b: np.stack([a[:, (i + 1) % 3] * b[:, (i + 2) % 3] - a[:, (i + 2) % 3] * b[:, (i + 1) % 3]
                                   for i in range(3)], 1)
    rows = [cross(c[1], c[2]), cross(c[2], c[0]), cross(c[0], c[1])]
    det = c[0][:, 0] * rows[0][:, 0] + c[0][:, 1] * rows[0][:, 1] + c[0][:, 2] * rows[0][:, 2]
    tol = 20.0 * 2.220446049250313e-16
    with np.errstate(divide="ignore", invalid="ignore"):
        lam = [b / det[:, None] * r for b in rows]
        lam = [x[:, 0] + x[:, 1] + x[:, 2] for x in lam]
        lam.append(1.0 - (lam[0] + lam[1] + lam[2]))
        return ~np.any([(x < -tol) | (x > 1.0 + tol) for x in lam], axis=0)


def test_flat_elements():
    """Tets of zero volume among ordinary ones: with the reference's division
    by a zero determinant they hold the points of their box for which no
    coordinate comes out infinite."""
    import pyoracle as O
    from xdg_amd import capi
    ctx = capi.Context(0)
    ctx.set_option("leaf_size", 1)  # a flat element is asked about its own box only
    rng = np.random.default_rng(93)
    ref = G.kuhn_cube(5, 0.2, seed=4)
    k = 200  # in lattice planes, whose coordinates are exact
    lo = rng.integers(0, 8, (k, 3)) / 8.0
    ax = rng.integers(0, 3, k)
    flat = lo[:, None] + rng.integers(0, 3, (k, 4, 3)) / 16.0
    flat[np.arange(k), :, ax] = lo[np.arange(k), ax, None]
    tets = np.concatenate([len(ref.verts) + np.arange(4 * k, dtype=np.int32).reshape(k, 4), ref.tets])
    verts = np.concatenate([ref.verts, flat.reshape(-1, 3)])
    adj = np.full(tets.shape, -1, np.int32)
    et = ctx.build_element_tree(verts, tets.astype(np.int32), adj, ref.face_order)
    p = rng.random((20000, 3))
    j = rng.integers(0, k, 10000)
    w = rng.random((10000, 4, 1))
    p[:10000] = (flat[j] * w).sum(1) / w.sum(1)
    p[:3000] = flat[j[:3000], 0] + rng.random((3000, 1)) * (flat[j[:3000], 1] - flat[j[:3000], 0])
    p[3000:4000] = flat[j[3000:4000], 2]
    want = O.TetMesh(ref, with_ipc=False).find_element(p)
    want = np.where(want >= 0, want + k, -1)
    holds = 0
    for e in range(k - 1, -1, -1):
        # its dilated box (tetrahedron_contain.cpp:47-63): points of its plane
        # up to rounding, no other point comes as near
        in_box = ((p >= flat[e].min(0) - 1e-9) & (p <= flat[e].max(0) + 1e-9)).all(1)
        c = in_box & contains(p, np.broadcast_to(flat[e], (len(p), 4, 3)))
        holds += c.sum()
        want = np.where(c, e, want)
    assert holds > 500
    assert np.array_equal(host(ctx.find_element(et, dev(torch, p))), want)
    ctx.close()
