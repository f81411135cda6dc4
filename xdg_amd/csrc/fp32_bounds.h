// fp32_bounds.h -- FP32 tests that decide which candidates get the FP64
// arithmetic: rounding helpers and conservative bounds.  Host and device, so
// that CPU tests compile the code the kernels run.
#pragma once

#include "xdg_device.h"

namespace xdgd {

__host__ __device__ __forceinline__ float safe_inv_f(float d)
{
  const float eps = 1e-30f;
  return 1.0f / (fabsf(d) > eps ? d : copysignf(eps, d));
}

__host__ __device__ __forceinline__ float f32_up(double x)
{
  float f = (float)x;
  if ((double)f < x) f = nextafterf(f, INFINITY);
  return f;
}
__host__ __device__ __forceinline__ float f32_down_d(double x)
{
  float f = (float)x;
  if ((double)f > x) f = nextafterf(f, -INFINITY);
  return f;
}

// 1/x within two units in the last place; the host's is the correctly rounded
// one
__host__ __device__ __forceinline__ float rcp_approx(float x)
{
#if __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.0f / x;
#endif
}

// Is the triangle certainly farther from p than best?  An FP32 distance to
// its three edges, or to its plane (FP64, stored normal) where p projects
// inside it, against best^2.  With M the sum of squares of p - v0 and two
// edges, every FP32 quantity here is off by at most about 10 x 2^-24 M; a
// projection misjudged as outside lies within 4 x 2^-24 M (squared) of an
// edge whatever the triangle's shape, and the plane is never farther than
// the triangle.  A triangle thinner than 2^-10 of its length goes by its
// edges alone, which are within 2^-20 M (squared) of its interior: FP32 does
// not tell inside from outside there, and the stored normal of a far thinner
// one is off by more than the margin.  The margin is 2^-17 M.  The products of four lengths leave
// FP32's normal range for M above 2^64 or well below 2^-50 (projections are
// then misjudged by more than that): the test rejects nothing there, nor
// where a coordinate is NaN.
// Box distances let about 100 triangles per point pass on a sphere of
// 20 480 (an inclined triangle's box reaches far beyond it) of which a few
// need the FP64 closest point, four times this test's work.
__host__ __device__ __forceinline__ bool closest_beyond(const D3& v0, const D3& v1, const D3& v2, const D3& n,
                                                        const D3& p, float best2)
{
  const D3 d0 = sub(v0, p), d1 = sub(v1, v0), d2 = sub(v2, v0);
  const double plane = n.x * d0.x + n.y * d0.y + n.z * d0.z;
  const float wx = (float)d0.x, wy = (float)d0.y, wz = (float)d0.z;
  const float sx = (float)d1.x, sy = (float)d1.y, sz = (float)d1.z;
  const float tx = (float)d2.x, ty = (float)d2.y, tz = (float)d2.z;
  const float pp = wx * wx + wy * wy + wz * wz;
  const float ss = sx * sx + sy * sy + sz * sz;
  const float tt = tx * tx + ty * ty + tz * tz;
  const float m = pp + ss + tt;
  const float st = sx * tx + sy * ty + sz * tz;
  const float sp = sx * wx + sy * wy + sz * wz;
  const float tp = tx * wx + ty * wy + tz * wz;
  const float s = st * tp - tt * sp, t = st * sp - ss * tp;
  const float pr = ss * tt, det = pr - st * st;
  const bool inside = s >= 0.0f && t >= 0.0f && s + t <= det && det > 0x1p-20f * pr;
  // edges v0v1, v0v2 and v1v2: |w + a e|^2 at the clamped minimum
  const float a = fminf(fmaxf(-sp * rcp_approx(ss), 0.0f), 1.0f);
  const float b = fminf(fmaxf(-tp * rcp_approx(tt), 0.0f), 1.0f);
  const float ee = ss - 2.0f * st + tt, qe = (tp - sp) + (st - ss), qq = pp + 2.0f * sp + ss;
  const float c = fminf(fmaxf(-qe * rcp_approx(ee), 0.0f), 1.0f);
  const float e0 = pp + a * (2.0f * sp + a * ss), e1 = pp + b * (2.0f * tp + b * tt), e2 = qq + c * (2.0f * qe + c * ee);
  const float pl = (float)plane;
  const float lb = inside ? pl * pl : fminf(fminf(e0, e1), e2);
  return m >= 0x1p-50f && m <= 0x1p60f && lb - 0x1p-17f * m > best2;
}

// A point against the BVH4's FP32 boxes.  The boxes were dilated by the
// tree's bump; pm = p - s and pp = p + s with s just below the bump take that
// back, so the distance to a box is that to its vertices' bounds.  pm is
// rounded up and pp down, and the bump loses 2^-40 of the coordinates, more
// than the rounding of a closest point: only relative roundings are left
// (one difference, a square, two sums: 5 x 2^-24), which the factor on the
// limit covers, and the absolute ones of squares below FP32's normal range,
// which the addend covers.  A box whose distance exceeds the limit holds no triangle
// at the best distance or below.
struct ClosestPointF {
  float mx, my, mz, px, py, pz;
};
__host__ __device__ __forceinline__ float closest_limit(double best)
{
  return f32_up(best * best) * (1.0f + 0x1p-21f) + 0x1p-126f;
}
__host__ __device__ __forceinline__ double closest_shrink(double bump, double max_abs)
{
  return bump - 0x1p-40 * (max_abs + bump);
}
__host__ __device__ __forceinline__ ClosestPointF closest_point(const D3& p, double s)
{
  return ClosestPointF{f32_up(p.x - s),     f32_up(p.y - s),     f32_up(p.z - s),
                       f32_down_d(p.x + s), f32_down_d(p.y + s), f32_down_d(p.z + s)};
}
// squared distance to a box of the tree
__host__ __device__ __forceinline__ float closest_box(float lx, float hx, float ly, float hy, float lz, float hz,
                                                     const ClosestPointF& c)
{
  const float ex = fmaxf(fmaxf(lx - c.mx, c.px - hx), 0.0f);
  const float ey = fmaxf(fmaxf(ly - c.my, c.py - hy), 0.0f);
  const float ez = fmaxf(fmaxf(lz - c.mz, c.pz - hz), 0.0f);
  return ex * ex + ey * ey + ez * ez;
}

// Box of a volume for the transport's start stage: the tree's vertex bounds
// dilated as in the FP64 test of a ray against them (twice the bump and a
// relative slack), for an FP32 slab test of rays from the source box
// [src_lo, src_hi]: outward-rounded, with 2^-19 of the largest coordinates on
// either side as further slack.  The test's rounding moves a plane by at most
// 5 x 2^-24 of |plane| + |origin|, so its boxes never miss one that the FP64
// test would reach.  Coordinates near FP32's range or beyond it, whose
// differences it does not hold, give a box that every ray reaches.
__host__ __device__ __forceinline__ void start_box(const float* lo, const float* hi, double bump, const double* src_lo,
                                                  const double* src_hi, float* box)
{
  double most = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double ext = fabs((double)lo[k]) + fabs((double)hi[k]) + 1.0 + fabs(src_lo[k]) + fabs(src_hi[k]);
    const double slack = 2.0 * bump + (0x1p-30 + 0x1p-19) * ext;
    box[k] = f32_down_d((double)lo[k] - slack);
    box[3 + k] = f32_up((double)hi[k] + slack);
    most = fmax(most, ext + slack);
  }
  if (!(most <= 0x1p120))
    for (int k = 0; k < 3; ++k) {
      box[k] = -INFINITY;
      box[3 + k] = INFINITY;
    }
}
// a ray's origin for the slab test, finite
__host__ __device__ __forceinline__ float start_coord(double x)
{
  return fminf(fmaxf((float)x, -0x1.fffffep127f), 0x1.fffffep127f);
}
// The box of a slot that can hold no hit (the implicit complement, an unknown
// or empty tree).  The slab test orders the planes of an axis itself, so an
// inverted box would be reached by every ray; NaN planes leave the exit NaN
// and the comparison false.  (Looking for an inverted box cost a compare per
// box: 17 370 histories among 344 volumes 1.640 -> 1.662 ms.)
__host__ __device__ __forceinline__ void start_box_none(float* box)
{
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    box[k] = NAN;
    box[3 + k] = NAN;
  }
}
// Slab test of such a box (o and inv are finite, so no product of a box with
// planes is NaN; fminf and fmaxf pass over a NaN).  FP64 and a branch per
// axis bound the counting pass by VALU issue: 2^20 histories x 513 boxes 1.17
// -> 0.40 ms.
__host__ __device__ __forceinline__ bool start_box_hit(const float* b, const float3& o, const float3& inv)
{
  const float x0 = (b[0] - o.x) * inv.x, x1 = (b[3] - o.x) * inv.x;
  const float y0 = (b[1] - o.y) * inv.y, y1 = (b[4] - o.y) * inv.y;
  const float z0 = (b[2] - o.z) * inv.z, z1 = (b[5] - o.z) * inv.z;
  const float a = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), 0.0f));
  const float e = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1));
  return a <= e;
}

}  // namespace xdgd
