"""closest where its FP32 candidate tests are at their limits, against the
oracle's FP64 search bit for bit."""
import numpy as np
import pytest

import pyoracle as O
from gpu_util import bits, dev, host
from xdg_amd import geometry as G
from xdg_amd import philox as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    from xdg_amd import capi
    c = capi.Context(0)
    yield c
    c.close()


def check(ctx, v9, bump, pts, face=None):
    n = len(v9)
    face = np.arange(n, dtype=np.int32) if face is None else face
    surf, flip = np.ones(n, np.int32), np.zeros(n, np.uint8)
    tree = ctx.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(-1, 3), face, surf,
                                  flip, bump)
    d, f = [host(x) for x in ctx.closest(tree, dev(torch, pts))]
    rd, rf = O.Tree(v9, face, surf, flip, bump).closest(pts, brute=True)
    assert np.array_equal(bits(d), bits(rd)) and np.array_equal(f, rf)
    ctx.release_surface_tree(tree)


@pytest.mark.parametrize("radius", [1e-22, 1e-21, 1e-11, 1e-9, 1e-5, 1.0, 1e5, 1e9, 1e10, 1e13])
@pytest.mark.parametrize("subdiv", [1, 3])
def test_closest_scales(ctx, radius, subdiv):
    """Products of four lengths leave FP32's range at both ends, squares its
    normal range at the smallest radii."""
    v, t = G.icosphere(subdiv, radius)
    pts = P.ball_points(81, 0, 2000, 1.5 * radius)
    check(ctx, v[t].reshape(-1, 9), 1e-6 * radius, pts)


def test_closest_thin_triangles(ctx):
    """Triangles of aspects down to 1e-16, whose stored normals are far from
    exact, each twice with the lower face id second: the second must not be
    rejected at the best distance."""
    rng = np.random.default_rng(83)
    n = 4000
    v0, d1 = rng.standard_normal((n, 3)), rng.standard_normal((n, 3)) * 0.05
    off = rng.standard_normal((n, 3)) * 0.05 * 10.0 ** rng.uniform(-16, 0, (n, 1))
    v9 = np.hstack([v0, v0 + d1, v0 + rng.uniform(-0.5, 1.5, (n, 1)) * d1 + off])
    v9 = np.repeat(v9, 2, axis=0)
    b = rng.random((20 * n, 1))
    pts = np.repeat(v0, 20, axis=0) + b * np.repeat(d1, 20, axis=0)
    pts = pts + rng.standard_normal(pts.shape) * 0.05 * 10.0 ** rng.uniform(-3, 0, (20 * n, 1))
    check(ctx, v9, 1e-9, pts, np.arange(2 * n, dtype=np.int32)[::-1].copy())


@pytest.mark.parametrize("ntri,n", [(1, 1), (2, 70), (3, 5000), (20, 300), (20, 40000), (32, (1 << 19) - 1),
                                    (32, 1 << 19), (33, 1 << 19), (256, 9000), (257, 9000), (1280, 300)])
def test_closest_forms(ctx, ntri, n):
    """Trees of a single leaf to several levels, at the edges of the rules
    for one point per lane and for the leading descent: points around, on
    and (every seventh) beyond the FP32 boxes' limit, NaN and infinite ones
    among them."""
    v, t = G.icosphere(3, 5.0)
    rng = np.random.default_rng(ntri)
    v9 = v[t[rng.permutation(len(t))[:ntri]]].reshape(-1, 9)
    k = min(n, 4000)
    pts = P.ball_points(87, 0, k, 8.0)
    pts[::7] *= 10.0 ** rng.uniform(3, 15, (len(pts[::7]), 1))  # the last tie at every face
    pts[1::5] = v9[rng.integers(0, ntri, len(pts[1::5])), :3]
    pts[2::1001] = np.nan
    pts[3::1001, 1] = np.inf
    face = np.arange(ntri, dtype=np.int32)
    surf, flip = np.ones(ntri, np.int32), np.zeros(ntri, np.uint8)
    tree = ctx.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * ntri, dtype=np.int32).reshape(-1, 3), face, surf,
                                  flip, 1e-4)
    p = dev(torch, pts).repeat(-(-n // k), 1)[:n].contiguous()
    d, f = ctx.closest(tree, p)
    rd, rf = O.Tree(v9, face, surf, flip, 1e-4).closest(pts, brute=True)
    for lo in range(0, n, k):
        m = min(k, n - lo)
        assert np.array_equal(bits(host(d[lo:lo + m])), bits(rd[:m])) and np.array_equal(host(f[lo:lo + m]), rf[:m])
    ctx.release_surface_tree(tree)


@pytest.mark.parametrize("shift", [0.0, 3e6])
def test_closest_long_queue(ctx, shift):
    """Waves of 64 points at and near the centre of a sphere of 81 920
    triangles: no box is ever pruned, and the node queue fills until nodes
    are taken one at a time.  shift: the same far beyond the FP32 limit."""
    v, t = G.icosphere(6, 10.0)
    v9 = v[t].reshape(-1, 9)
    n = len(v9)
    face = np.arange(n, dtype=np.int32)
    surf, flip = np.ones(n, np.int32), np.zeros(n, np.uint8)
    tree = ctx.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(-1, 3), face, surf,
                                  flip, 1e-3)
    pts = P.ball_points(91, 0, 64, 1e-9)
    pts[:8] = 0.0
    pts[:, 0] += shift
    d, f = ctx.closest(tree, dev(torch, pts).repeat(2048, 1).contiguous())
    rd, rf = O.Tree(v9, face, surf, flip, 1e-3).closest(pts)
    assert (bits(host(d)).reshape(-1, 64) == bits(rd)).all() and (host(f).reshape(-1, 64) == rf).all()
    ctx.release_surface_tree(tree)
