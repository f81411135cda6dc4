"""Queries captured by a caller's graph, replayed between eager work: those on
a strided share use no scratch of the context, the others were run once at
that size before."""
import numpy as np
import pytest

from gpu_util import build_tree, dev, host
from xdg_amd import geometry as G
from xdg_amd import philox as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def setup():
    from xdg_amd import capi
    ctx = capi.Context(0)
    m = G.nested_spheres(3)
    vols = list(m.volumes)
    trees = [build_tree(ctx, m, v) for v in vols]
    mesh = G.kuhn_cube(5, 0.2, seed=4)
    et = ctx.build_element_tree(mesh.verts, mesh.tets, mesh.adj, mesh.face_order)
    yield ctx, m, vols, trees, et
    ctx.close()


QUERIES = {
    "point_in_volume": lambda c, m, v, t, e, p, d, s: [c.point_in_volume(t[2], p, d, precision=1, stream=s)],
    "closest": lambda c, m, v, t, e, p, d, s: c.closest(t[0], p, stream=s),
    "find_element": lambda c, m, v, t, e, p, d, s: [c.find_element(e, p / 19.0, stream=s)],
    "ray_fire": lambda c, m, v, t, e, p, d, s: c.ray_fire(t[1], p, d, precision=1, stream=s),
    "find_volume": lambda c, m, v, t, e, p, d, s: [c.find_volume(t, v, m.ipc, p, d, precision=1, stream=s)],
}


@pytest.mark.parametrize("n", [700, 70000])
@pytest.mark.parametrize("name", sorted(QUERIES))
def test_replays(setup, name, n):
    pts = P.box_points(95, P.STREAM_POS, n, [-19] * 3, [19] * 3)
    pts[::97] *= 1e4  # beyond the FP32 boxes' limit
    p, d = dev(torch, pts), dev(torch, P.iso_dirs(95, P.STREAM_DIR, n))
    call = lambda s=None: QUERIES[name](*setup, p, d, s)
    ref = [host(x).copy() for x in call()]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = call(torch.cuda.current_stream().cuda_stream)
    for k in range(4):
        for x in out:
            x.fill_(7)
        g.replay()
        torch.cuda.synchronize()
        for x, r in zip(out, ref):
            assert np.array_equal(host(x), r)
        eager = call()
        torch.cuda.synchronize()
        for x, r in zip(eager, ref):
            assert np.array_equal(host(x), r)


def test_overlapping_streams(setup):
    """Scratch-free queries in flight on two streams at once."""
    n = 300000
    sides = []
    for k in range(2):
        pts = P.box_points(97 + k, P.STREAM_POS, n, [-19] * 3, [19] * 3)
        sides.append((dev(torch, pts), dev(torch, P.iso_dirs(97 + k, P.STREAM_DIR, n)), torch.cuda.Stream()))
    names = ("point_in_volume", "closest", "find_element")
    ref = [[[host(x).copy() for x in QUERIES[q](*setup, p, d, None)] for q in names] for p, d, _ in sides]
    torch.cuda.synchronize()
    got = []
    for r in range(3):
        got = [[], []]
        for q in names:
            for k, (p, d, s) in enumerate(sides):
                with torch.cuda.stream(s):
                    got[k].append(QUERIES[q](*setup, p, d, s.cuda_stream))
        torch.cuda.synchronize()
        for k in range(2):
            for a, b in zip(got[k], ref[k]):
                for x, y in zip(a, b):
                    assert np.array_equal(host(x), y)
