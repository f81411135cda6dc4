"""Trees whose BVH4 could need more stack entries than the 64 a query takes:
primitives in the octants of cubes that halve twenty times, in the radix tree
(one binary level per Morton bit, up to three BVH4 entries for two of them)."""
import numpy as np
import pytest

import pyoracle as O
from gpu_util import bits, dev, host
from xdg_amd import geometry as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SCALES = 20


@pytest.fixture(scope="module")
def ctx():
    from xdg_amd import capi
    c = capi.Context(0)
    c.set_option("build", 0)
    c.set_option("leaf_size", 1)
    yield c
    c.close()


def cells(size):
    """Centres and edge lengths of the eight octants of octants 1..7 of
    [0, size 2^-k]^3."""
    c, s = [], []
    bits3 = np.array([[o >> a & 1 for a in range(3)] for o in range(8)])
    for k in range(SCALES):
        h = size * 2.0 ** -k
        for o in bits3[1:]:
            c.append(h * (0.5 * o + 0.25 * bits3 + 0.125))
            s.append(np.full(8, 0.5 * h))
    return np.concatenate(c), np.concatenate(s)


def points(c, s, n):
    rng = np.random.default_rng(85)
    k = rng.integers(0, len(c), n)
    return c[k] + s[k, None] * rng.uniform(-0.15, 0.15, (n, 3))


CORNERS = 0.1 * np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1], [-1, -1, 1]])


def test_closest_deep_tree(ctx):
    c, s = cells(1e4)
    v9 = (c[:, None] + s[:, None, None] * CORNERS[:3]).reshape(-1, 9)
    n = len(v9)
    face, surf, flip = np.arange(n, dtype=np.int32), np.ones(n, np.int32), np.zeros(n, np.uint8)
    tree = ctx.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(-1, 3), face, surf,
                                  flip, 1e-4)
    info = ctx.tree_info(tree)
    assert info["depth"] <= 64 < info["stack4"]
    pts = points(c, s, 20000)
    pts[::9] += 1e6  # by the binary tree
    d, f = [host(x) for x in ctx.closest(tree, dev(torch, pts))]
    rd, rf = O.Tree(v9, face, surf, flip, 1e-4).closest(pts, brute=True)
    assert np.array_equal(bits(d), bits(rd)) and np.array_equal(f, rf)


def test_element_queries_deep_tree(ctx):
    c, s = cells(1e4)
    verts = (c[:, None] + s[:, None, None] * CORNERS).reshape(-1, 3)
    tets = np.arange(len(verts), dtype=np.int32).reshape(-1, 4)
    det = np.linalg.det(verts[tets[:, 1:]] - verts[tets[:, :1]])
    assert (det > 0).all() or (det < 0).all()
    if det[0] < 0:
        tets = tets[:, [0, 2, 1, 3]].copy()
    ref = G.kuhn_cube(1, 0.0, seed=4)
    mesh = G.TetMesh(verts, tets, np.full(tets.shape, -1, np.int32), ref.face_order, np.zeros((0, 3), np.int32),
                     np.zeros(0, np.int32))
    et = ctx.build_element_tree(mesh.verts, mesh.tets, mesh.adj, mesh.face_order)
    assert 50 < ctx.tree_info(et, element=True)["depth"] <= 64
    om = O.TetMesh(mesh, with_ipc=False)
    pts = points(c, s, 20000)
    rf = om.find_element(pts, brute=True)
    assert (rf >= 0).sum() > 1000 and np.unique(rf).size > 100
    assert np.array_equal(host(ctx.find_element(et, dev(torch, pts))), rf)
    p1 = pts + np.roll(pts, 1, axis=0) * 0.01
    cnt, hsh = [host(x) for x in ctx.tally_segments(et, dev(torch, pts), dev(torch, p1))]
    rc, rh = om.segments(pts, p1)
    assert np.array_equal(cnt, rc) and np.array_equal(hsh.view(np.uint64), rh)
