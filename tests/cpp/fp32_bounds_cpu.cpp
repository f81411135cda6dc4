// CPU checks of the kernels' conservative tests, which decide what gets the
// full FP64 arithmetic (host side of the same functions): fp32_bounds.h, and
// the early rejects of tet_contains.  argv[1] names the check;
// prints "ok" or what failed.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "fp32_bounds.h"

using namespace xdgd;

namespace {

std::mt19937_64 rng(12345);
double uni() { return std::uniform_real_distribution<double>(0.0, 1.0)(rng); }
double nrm() { return std::normal_distribution<double>()(rng); }

typedef long double LD;
struct L3 {
  LD x, y, z;
};
L3 l3(const D3& a) { return L3{a.x, a.y, a.z}; }
L3 operator-(const L3& a, const L3& b) { return L3{a.x - b.x, a.y - b.y, a.z - b.z}; }
LD dotl(const L3& a, const L3& b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
L3 crossl(const L3& a, const L3& b)
{
  return L3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

LD segment_distance(const L3& p, const L3& a, const L3& e)
{
  const L3 w = p - a;
  const LD ee = dotl(e, e);
  LD s = ee > 0 ? dotl(w, e) / ee : 0;
  s = s < 0 ? 0 : (s > 1 ? 1 : s);
  const L3 d{w.x - s * e.x, w.y - s * e.y, w.z - s * e.z};
  return sqrtl(dotl(d, d));
}

// distance of p to the triangle in 80-bit arithmetic
LD distance(const D3& v0, const D3& v1, const D3& v2, const D3& q)
{
  const L3 a = l3(v0), p = l3(q), e0 = l3(v1) - a, e1 = l3(v2) - a, e2 = e1 - e0, w = p - a;
  LD best = fminl(fminl(segment_distance(p, a, e0), segment_distance(p, a, e1)), segment_distance(p, l3(v1), e2));
  const L3 n = crossl(e0, e1);
  const LD nn = dotl(n, n);
  if (nn > 0) {
    const LD u = dotl(crossl(w, e1), n) / nn, v = dotl(crossl(e0, w), n) / nn;
    if (u >= 0 && v >= 0 && u + v <= 1) best = fminl(best, fabsl(dotl(w, n)) / sqrtl(nn));
  }
  return best;
}

// the normal as the tree stores it (face_normal's operations)
D3 normal(const D3& v0, const D3& v1, const D3& v2)
{
  D3 n = cross(sub(v1, v0), sub(v2, v0));
  double len = sqrt(n.x * n.x + n.y * n.y + n.z * n.z);
  len = len < (double)MIN_RCP_INPUT ? (double)MIN_RCP_INPUT : len;
  return D3{n.x / len, n.y / len, n.z / len};
}

D3 rnd(double s) { return D3{s * nrm(), s * nrm(), s * nrm()}; }

// closest_beyond keeps every triangle whose distance is the best one, with
// points near to and far from it, everything scaled by 10^e for e in
// [lo, hi].  thin: aspects down to 1e-16.
int closest_bound(int lo, int hi, bool thin)
{
  long wrong = 0, rejected = 0, total = 0;
  for (int e = lo; e <= hi; ++e) {
    const double scale = std::pow(10.0, e);
    long w = 0;
    for (int k = 0; k < 20000; ++k) {
      const double size = std::pow(10.0, -3.0 * uni());
      const double aspect = thin ? std::pow(10.0, -16.0 * uni()) : 1.0, f = 2.0 * uni() - 0.5;
      const D3 d1 = rnd(size), off = rnd(size * aspect);
      D3 v0 = rnd(k % 2 ? 1.0 : 0.0), v1{v0.x + d1.x, v0.y + d1.y, v0.z + d1.z};
      D3 v2{v0.x + f * d1.x + off.x, v0.y + f * d1.y + off.y, v0.z + f * d1.z + off.z};
      const double b = 1.4 * uni() - 0.2, c = 1.4 * uni() - 0.2, h = size * std::pow(10.0, 1.0 - 4.0 * uni());
      const D3 dn = k % 4 < 2 ? normal(v0, v1, v2) : rnd(1.0);
      D3 p{v0.x + b * (v1.x - v0.x) + c * (v2.x - v0.x) + h * dn.x,
           v0.y + b * (v1.y - v0.y) + c * (v2.y - v0.y) + h * dn.y,
           v0.z + b * (v1.z - v0.z) + c * (v2.z - v0.z) + h * dn.z};
      for (D3* q : {&v0, &v1, &v2, &p}) *q = D3{q->x * scale, q->y * scale, q->z * scale};
      const D3 n = normal(v0, v1, v2);
      const double d = (double)distance(v0, v1, v2, p);
      w += closest_beyond(v0, v1, v2, n, p, f32_up(d * d));
      rejected += closest_beyond(v0, v1, v2, n, p, f32_up(0.49 * d * d));
      ++total;
    }
    if (w) std::printf("scale 1e%d: %ld of 20000 triangles at the best distance rejected\n", e, w);
    wrong += w;
  }
  if (rejected * 4 < 20000) {
    std::printf("only %ld of %ld farther triangles rejected\n", rejected, total);
    ++wrong;
  }
  return wrong != 0;
}

// a box whose vertices' bounds are at the best distance or nearer passes the
// limit, at every scale whose distances' squares FP64 holds exactly enough
int closest_boxes()
{
  long wrong = 0, passed = 0, total = 0;
  for (int e = -44; e <= 18; ++e) {
    const double scale = std::pow(10.0, e);
    long w = 0;
    for (int k = 0; k < 20000; ++k) {
      const double bump = scale * std::pow(10.0, -2.0 - 12.0 * uni());
      double lo[3], hi[3], q[3], ext = 0.0;
      float flo[3], fhi[3];
      for (int j = 0; j < 3; ++j) {
        lo[j] = scale * nrm();
        hi[j] = lo[j] + scale * uni();
        q[j] = scale * 2.0 * nrm();
        ext = std::fmax(ext, std::fmax(std::fabs(lo[j]), std::fabs(hi[j])) + bump);
        flo[j] = f32_down_d(lo[j] - bump);
        fhi[j] = f32_up(hi[j] + bump);
      }
      LD d2 = 0;
      for (int j = 0; j < 3; ++j) {
        const LD x = fmaxl(fmaxl((LD)lo[j] - q[j], (LD)q[j] - hi[j]), 0.0L);
        d2 += x * x;
      }
      const double best = (double)sqrtl(d2);
      const ClosestPointF c = closest_point(D3{q[0], q[1], q[2]}, closest_shrink(bump, ext));
      const float d = closest_box(flo[0], fhi[0], flo[1], fhi[1], flo[2], fhi[2], c);
      w += !(d <= closest_limit(best));
      passed += d <= closest_limit(0.9 * best);
      ++total;
    }
    if (w) std::printf("scale 1e%d: %ld of 20000 boxes at the best distance pruned\n", e, w);
    wrong += w;
  }
  if (passed * 2 > total) {
    std::printf("%ld of %ld farther boxes not pruned\n", passed, total);
    ++wrong;
  }
  return wrong != 0;
}

// the FP64 test of a ray against a box that carries its slack
bool slab64(const double* lo, const double* hi, const double* o, const double* d)
{
  double a = 0.0, b = INFTY;
  for (int k = 0; k < 3; ++k) {
    if (d[k] == 0.0) {
      if (o[k] < lo[k] || o[k] > hi[k]) return false;
      continue;
    }
    const double inv = 1.0 / d[k], t0 = (lo[k] - o[k]) * inv, t1 = (hi[k] - o[k]) * inv;
    a = std::fmax(a, std::fmin(t0, t1));
    b = std::fmin(b, std::fmax(t0, t1));
  }
  return a <= b;
}

// The start stage's boxes: a box that the FP64 test reaches is reached
// (coordinates 10^lo to 10^hi, near-axis and axis-parallel directions, aimed
// at corners and edges, where a miss is nearest), and a slot without hits
// never is.
int start_boxes(double lo_exp, double hi_exp)
{
  long dropped = 0, reached = 0, none = 0;
  const int n = 400000;
  for (int i = 0; i < n; ++i) {
    const double scale = std::pow(10.0, lo_exp + (hi_exp - lo_exp) * uni());
    const double half = scale * std::pow(10.0, -4.0 * uni()), bump = 1e-3 * uni();
    float blo[3], bhi[3], box[6], empty[6];
    double slo[3], shi[3], o[3], d[3], wlo[3], whi[3], len = 0.0;
    for (int k = 0; k < 3; ++k) {
      slo[k] = -scale * uni();
      shi[k] = scale * uni();
      o[k] = slo[k] + (shi[k] - slo[k]) * uni();
      const double mid = scale * (4.0 * uni() - 2.0), h = half * uni();
      blo[k] = f32_down_d(mid - h);
      bhi[k] = f32_up(mid + h);
      const double slack = 2.0 * bump + 0x1p-30 * (std::fabs((double)blo[k]) + std::fabs((double)bhi[k]) + 1.0);
      wlo[k] = blo[k] - slack;
      whi[k] = bhi[k] + slack;
      d[k] = i % 5 == 0 ? nrm() : (uni() < 0.5 ? wlo[k] : whi[k]) - o[k];
    }
    if (i % 7 == 0) d[0] = i % 2 ? 0.0 : -0.0;
    for (int k = 0; k < 3; ++k) len += d[k] / scale * (d[k] / scale);
    for (int k = 0; k < 3; ++k) d[k] /= scale * std::sqrt(len);
    if (i % 7 == 1) d[1] *= 1e-33;
    start_box(blo, bhi, bump, slo, shi, box);
    start_box_none(empty);
    const float3 fo = make_float3(start_coord(o[0]), start_coord(o[1]), start_coord(o[2]));
    const float3 inv = make_float3(safe_inv_f((float)d[0]), safe_inv_f((float)d[1]), safe_inv_f((float)d[2]));
    const bool ref = slab64(wlo, whi, o, d);
    reached += ref;
    dropped += ref && !start_box_hit(box, fo, inv);
    none += start_box_hit(empty, fo, inv);
  }
  if (dropped) std::printf("%ld of %ld reached boxes dropped\n", dropped, reached);
  if (none) std::printf("%ld of %d rays reach a slot without hits\n", none, n);
  if (reached < n / 10) std::printf("only %ld boxes reached\n", reached);
  return dropped || none || reached < n / 10;
}

// tet_contains without its early rejects
bool contains(const D3& p, const D3& v0, const D3& v1, const D3& v2, const D3& v3)
{
  const D3 c0 = sub(v1, v0), c1 = sub(v2, v0), c2 = sub(v3, v0), r = sub(p, v0);
  // rows of the adjugate: the cross products of the columns
  const D3 b[3] = {cross(c1, c2), cross(c2, c0), cross(c0, c1)};
  const double det = c0.x * b[0].x + c0.y * b[0].y + c0.z * b[0].z, hi = 1.0 + PLUCKER_ZERO_TOL;
  double l[4], sum = 0.0;
  for (int k = 0; k < 3; ++k) l[k] = b[k].x / det * r.x + b[k].y / det * r.y + b[k].z / det * r.z;
  sum = l[0] + l[1] + l[2];
  l[3] = 1.0 - sum;
  for (double x : l)
    if (x < -PLUCKER_ZERO_TOL || x > hi) return false;
  return true;
}

// The early rejects change no answer: tets thin to flat, near to and far from
// the origin, points on their faces, edges and vertices and a few ulps off
// them, scales 1e-110 to 1e105.
int containment()
{
  long wrong = 0;
  for (int e = -110; e <= 105; e += 5) {
    const double scale = std::pow(10.0, e);
    long bad = 0, inside = 0;
    for (int i = 0; i < 40000; ++i) {
      const double thin = i % 3 ? 1.0 : std::pow(10.0, -17.0 * uni()), at = i % 2 ? 1.0 : 1e3;
      const D3 o = rnd(at);
      D3 v[4], p{0.0, 0.0, 0.0};
      for (D3& q : v) q = D3{o.x + nrm(), o.y + nrm(), o.z + thin * nrm()};
      double w[4], t = 0.0;
      for (int k = 0; k < 4; ++k) t += w[k] = (i % 7 == k || (i % 7 < 2 && k == 3)) ? 0.0 : uni();
      for (int k = 0; k < 4; ++k)
        p = D3{p.x + w[k] / t * v[k].x, p.y + w[k] / t * v[k].y, p.z + w[k] / t * v[k].z};
      if (i % 11 < 5) p.x *= 1.0 + (i % 11 - 2) * 0x1p-51;
      if (i % 11 == 6) p = v[i % 4];
      for (D3& q : v) q = D3{q.x * scale, q.y * scale, q.z * scale};
      p = D3{p.x * scale, p.y * scale, p.z * scale};
      const bool ref = contains(p, v[0], v[1], v[2], v[3]);
      inside += ref;
      bad += ref != tet_contains(p, v[0], v[1], v[2], v[3]);
    }
    if (bad) std::printf("scale 1e%d: %ld of 40000 answers differ\n", e, bad);
    if (inside < 1000 || inside > 39000) std::printf("scale 1e%d: %ld of 40000 inside\n", e, inside);
    wrong += bad;
  }
  return wrong != 0;
}

}  // namespace

int main(int argc, char** argv)
{
  int rc = 1;
  if (argc == 2 && !std::strcmp(argv[1], "closest")) rc = closest_bound(-24, 24, false);
  if (argc == 2 && !std::strcmp(argv[1], "closest_thin")) rc = closest_bound(-24, 24, true);
  if (argc == 2 && !std::strcmp(argv[1], "closest_boxes")) rc = closest_boxes();
  if (argc == 2 && !std::strcmp(argv[1], "start_boxes")) rc = start_boxes(-3.0, 6.0);
  if (argc == 2 && !std::strcmp(argv[1], "start_boxes_huge")) rc = start_boxes(6.0, 60.0);
  if (argc == 2 && !std::strcmp(argv[1], "containment")) rc = containment();
  if (!rc) std::printf("ok\n");
  return rc;
}
