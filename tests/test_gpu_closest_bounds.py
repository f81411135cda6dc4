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


def check(ctx, v9, bump, pts):
    n = len(v9)
    face = np.arange(n, dtype=np.int32)
    surf, flip = np.ones(n, np.int32), np.zeros(n, np.uint8)
    tree = ctx.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(-1, 3), face, surf,
                                  flip, bump)
    d, f = [host(x) for x in ctx.closest(tree, dev(torch, pts))]
    rd, rf = O.Tree(v9, face, surf, flip, bump).closest(pts, brute=True)
    assert np.array_equal(bits(d), bits(rd)) and np.array_equal(f, rf)
    ctx.release_surface_tree(tree)


@pytest.mark.parametrize("radius", [1e-11, 1e-9, 1e-5, 1.0, 1e5, 1e9, 1e10, 1e13])
@pytest.mark.parametrize("subdiv", [1, 3])
def test_closest_scales(ctx, radius, subdiv):
    """Products of four lengths leave FP32's range at both ends."""
    v, t = G.icosphere(subdiv, radius)
    pts = P.ball_points(81, 0, 2000, 1.5 * radius)
    check(ctx, v[t].reshape(-1, 9), 1e-6 * radius, pts)
