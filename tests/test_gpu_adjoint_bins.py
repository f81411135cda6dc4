"""The binned adjoint (batches of at least 65 536 rays): meshes at the edges of
a bucket of 256 faces, rays crowded on one face (several chunks of a bucket),
a ragged last workgroup, hits without terms, and the largest bucket count
beside the first mesh that falls back to the sorted form."""
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


@pytest.mark.parametrize("ntri,n,crowd", [(1, 65536, 0), (255, 65537, 0), (256, 70000, 0), (257, 65536, 0),
                                          (1280, 100003, 40000), (1048320, 65536, 0), (1048321, 65536, 0)])
def test_binned_adjoint(ctx, ntri, n, crowd):
    m = G.perturbed_sphere(3, 10.0, 0.05)
    reps = -(-ntri // m.tris.shape[0])
    tris = np.ascontiguousarray(np.tile(m.tris, (reps, 1))[:ntri])
    rng = np.random.default_rng(ntri + n)
    face = rng.integers(0, ntri, n).astype(np.int32)
    face[:crowd] = ntri // 2
    b = rng.random((n, 2)) * 0.5
    v = m.verts[tris[face]]
    hit = v[:, 0] + b[:, :1] * (v[:, 1] - v[:, 0]) + b[:, 1:] * (v[:, 2] - v[:, 0])
    org = P.ball_points(9, 0, n, 9.0)
    t = np.linalg.norm(hit - org, axis=1)
    dirs = (hit - org) / t[:, None]
    w = rng.standard_normal(n)
    face[::11] = -1
    t[5::13] = np.inf
    dirs[7::101] = 0.0  # no derivative: n.d = 0
    face[3::503] = ntri + 5
    gv = torch.zeros((m.verts.shape[0], 3), dtype=torch.float64, device="cuda")
    go = torch.empty((n, 3), dtype=torch.float64, device="cuda")
    gd = torch.empty_like(go)
    ctx.ray_distance_adjoint(dev(torch, org), dev(torch, dirs), dev(torch, t), dev(torch, face), dev(torch, w),
                             dev(torch, m.verts), dev(torch, tris), gv, go, gd)
    ov, oo, od = O.adjoint(m.verts, tris, org, dirs, t, face, w)
    assert np.array_equal(bits(host(go)), bits(oo)) and np.array_equal(bits(host(gd)), bits(od))
    # at most n terms of the largest vertex sum's size, each rounded a few times
    assert np.allclose(host(gv), ov, rtol=1e-12, atol=1e-12 * np.abs(ov).max())


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e300, -1e305])
def test_binned_adjoint_extreme_weights(ctx, value):
    """Infinite, NaN and huge dL/dt on a few rays: every vertex component is
    infinite, NaN or finite as the sum of single rays' terms is."""
    m = G.perturbed_sphere(3, 10.0, 0.05)
    n = 70000
    rng = np.random.default_rng(89)
    face = rng.integers(0, len(m.tris), n).astype(np.int32)
    v = m.verts[m.tris[face]]
    b = rng.random((n, 2)) * 0.5
    hit = v[:, 0] + b[:, :1] * (v[:, 1] - v[:, 0]) + b[:, 1:] * (v[:, 2] - v[:, 0])
    org = P.ball_points(9, 0, n, 9.0)
    t = np.linalg.norm(hit - org, axis=1)
    dirs = (hit - org) / t[:, None]
    w = rng.standard_normal(n)
    w[::9001] = value
    gv = torch.zeros((m.verts.shape[0], 3), dtype=torch.float64, device="cuda")
    go = torch.empty((n, 3), dtype=torch.float64, device="cuda")
    gd = torch.empty_like(go)
    ctx.ray_distance_adjoint(dev(torch, org), dev(torch, dirs), dev(torch, t), dev(torch, face), dev(torch, w),
                             dev(torch, m.verts), dev(torch, m.tris), gv, go, gd)
    ov, oo, od = O.adjoint(m.verts, m.tris, org, dirs, t, face, w)
    gv = host(gv)
    assert np.array_equal(host(go), oo, equal_nan=True) and np.array_equal(host(gd), od, equal_nan=True)
    if not np.isfinite(value):
        assert (~np.isfinite(ov)).sum() > 20
    assert np.array_equal(np.isnan(gv), np.isnan(ov)) and np.array_equal(np.isinf(gv), np.isinf(ov))
    inf, fin = np.isinf(ov), np.isfinite(ov)
    assert np.array_equal(gv[inf], ov[inf])
    big = np.zeros(len(gv), bool)
    big[m.tris[face[::9001]]] = True
    for part in (fin & big[:, None], fin & ~big[:, None]):
        scale = np.abs(ov[part]).max(initial=0.0)
        assert np.allclose(gv[part], ov[part], rtol=1e-12, atol=1e-12 * scale)


def test_sorted_form_under_capture():
    """Captured on a context without bins but with ray-order scratch of that
    size: the sorted form, replayed between eager calls."""
    from xdg_amd import capi
    c = capi.Context(0)
    m = G.perturbed_sphere(3, 10.0, 0.05)
    n = 70000
    org, dirs, w = P.ball_points(9, 0, n, 9.0), P.iso_dirs(9, 1, n), P.normals(9, 2, n)
    verts, tris = dev(torch, m.verts), dev(torch, m.tris)
    o, d, dw = dev(torch, org), dev(torch, dirs), dev(torch, w)
    v9, f, s, fl = m.tree_arrays(1)
    tree = c.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * len(f), dtype=np.int32).reshape(-1, 3), f, s, fl,
                                m.bump(1))
    c.set_option("ray_order", 1)
    t, _, face = c.ray_fire(tree, o, d, precision=capi.MIXED)
    gv, go, gd = torch.zeros_like(verts), torch.empty_like(o), torch.empty_like(d)
    ov, oo, od = O.adjoint(m.verts, m.tris, org, dirs, host(t), host(face), w)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gv.zero_()
        c.ray_distance_adjoint(o, d, t, face, dw, verts, tris, gv, go, gd,
                               stream=torch.cuda.current_stream().cuda_stream)
    ev = torch.zeros_like(verts)
    for k in range(4):
        go.fill_(float(k))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bits(host(go)), bits(oo)) and np.array_equal(bits(host(gd)), bits(od))
        assert np.allclose(host(gv), ov, rtol=1e-12, atol=1e-12 * np.abs(ov).max())
        c.ray_fire(tree, o, d, precision=capi.MIXED)  # eager work on the same scratch
        if k:  # binned, in memory of its own
            ev.zero_()
            c.ray_distance_adjoint(o, d, t, face, dw, verts, tris, ev, go, gd)
            assert np.allclose(host(ev), ov, rtol=1e-12, atol=1e-12 * np.abs(ov).max())
        torch.cuda.synchronize()
    c.close()
