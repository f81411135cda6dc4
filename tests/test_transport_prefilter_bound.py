"""The derivation of the transport start stage's FP32 volume prefilter, in
numpy: with its extra slack it never drops a volume that the FP64 slab test of
the same dilated box reaches, and without it it does (boxes from 1e-3 to 1e6
away, near-axis and axis-parallel directions).  The kernel's own code, slots
without hits and coordinates beyond FP32's range are checked by
test_fp32_bounds.py."""
import numpy as np

F = np.float32


def f32_down(x):
    f = x.astype(F)
    return np.where(f.astype(np.float64) > x, np.nextafter(f, F(-np.inf)), f)


def f32_up(x):
    return -f32_down(-x)


def hit_fp64(lo, hi, o, d):
    """may_hit_tree on boxes that carry their slack."""
    a, b = np.zeros(len(o)), np.full(len(o), np.finfo(np.float64).max)
    ok = np.ones(len(o), bool)
    with np.errstate(divide="ignore", invalid="ignore", over="ignore"):
        for k in range(3):
            par = d[:, k] == 0.0
            ok &= ~par | ((o[:, k] >= lo[:, k]) & (o[:, k] <= hi[:, k]))
            inv = 1.0 / np.where(par, 1.0, d[:, k])
            t0, t1 = (lo[:, k] - o[:, k]) * inv, (hi[:, k] - o[:, k]) * inv
            a = np.where(par, a, np.maximum(a, np.minimum(t0, t1)))
            b = np.where(par, b, np.minimum(b, np.maximum(t0, t1)))
    return ok & (a <= b)


def hit_fp32(lo, hi, o, d):
    o = o.astype(F)
    df = d.astype(F)
    small = np.abs(df) <= F(1e-30)
    with np.errstate(over="ignore"):
        inv = F(1.0) / np.where(small, np.copysign(F(1e-30), df), df)
        t0, t1 = (lo - o) * inv, (hi - o) * inv
    a = np.maximum(np.minimum(t0, t1).max(axis=1), F(0.0))
    return a <= np.maximum(t0, t1).min(axis=1)


def test_fp32_prefilter_is_conservative():
    rng = np.random.default_rng(11)
    n = 400_000
    scale = 10.0 ** rng.uniform(-3, 6, (n, 1))
    src_lo = -scale * rng.random((n, 3))
    src_hi = scale * rng.random((n, 3))
    o = src_lo + (src_hi - src_lo) * rng.random((n, 3))
    half = scale * 10.0 ** rng.uniform(-4, 0, (n, 1)) * rng.random((n, 3))
    mid = scale * rng.uniform(-2, 2, (n, 3))
    blo, bhi = f32_down(mid - half).astype(np.float64), f32_up(mid + half).astype(np.float64)
    bump = 1e-3 * rng.random((n, 1))
    ext = np.abs(blo) + np.abs(bhi) + 1.0
    slack = 2.0 * bump + 2.0 ** -30 * ext
    # aim at box corners and edges, where the tests are closest to a miss
    d = np.where(rng.random((n, 3)) < 0.5, blo - slack, bhi + slack) - o
    d[::5] = rng.standard_normal((len(d[::5]), 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[::7, 0] = 0.0
    d[1::7, 1] *= 1e-33
    ref = hit_fp64(blo - slack, bhi + slack, o, d)
    more = slack + 2.0 ** -19 * (ext + np.abs(src_lo) + np.abs(src_hi))
    got = hit_fp32(f32_down(blo - more), f32_up(bhi + more), o, d)
    assert ref.sum() > n // 10
    assert not (ref & ~got).any()
    # without the extra slack some would be dropped
    tight = hit_fp32(f32_down(blo - slack), f32_up(bhi + slack), o, d)
    assert (ref & ~tight).any()
