// adjoint.hip -- reverse-mode derivative of the ray_fire hit distance.
//
// For a ray that hit triangle f = (v0, v1, v2) at distance t, the distance
// is the plane intersection t = n.(v0 - o) / (n.d) with n = e1 x e2,
// e1 = v1 - v0, e2 = v2 - v0 (the Pluecker test of triangle_intersect.cpp
// and plucker.h:64-161 decides which triangle and returns this t).  With
// D = n.d and q = v0 - (o + t d):
//   dt/do = -n / D            dt/dd = -t n / D
//   dt/dv1 = (e2 x q) / D     dt/dv2 = (q x e1) / D
//   dt/dv0 = (n - e2 x q - q x e1) / D
// One lane per ray scales these by dL/dt; vertex gradients are scattered
// with FP64 atomics (so their summation order varies run to run), ray
// gradients are written directly.  Large batches avoid nine atomics per ray:
// the vertex terms of one face are linear in the sums of w and w q over its
// rays (w = dL/dt / D), so the binned form writes these four numbers per ray
// into buckets of 256 faces and sums each bucket in LDS, which leaves nine
// atomics per face and bucket chunk.  The sorted form (meshes with too many
// buckets) orders the rays by hit face (a stable radix sort) and sums each
// wave's run of rays on one face with shuffles.  No counterpart in the
// reference.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.h"

using namespace xdgd;

namespace xdgh {
namespace {

__device__ __forceinline__ D3 ld3(const double* p) { return d3(p[0], p[1], p[2]); }
__device__ __forceinline__ D3 add3(const D3& a, const D3& b) { return d3(a.x + b.x, a.y + b.y, a.z + b.z); }

// The gradient terms of ray i: false for a ray without a usable hit.
struct AdjTerms {
  int32_t i0, i1, i2;
  D3 g0, g1, g2;  // dL/d(v0, v1, v2)
  double w;       // dL/dt / D
  D3 wq;          // w q
};

__device__ __forceinline__ bool adjoint_ray(const AdjointArgs& a, int64_t i, AdjTerms& A)
{
  const int32_t f = a.face[i];
  const double ti = a.t[i];
  bool ok = f >= 0 && f < a.ntri && ti < INFTY;
  int32_t i0 = 0, i1 = 0, i2 = 0;
  D3 v0 = d3(0, 0, 0), e1 = d3(0, 0, 0), e2 = d3(0, 0, 0), nn = d3(0, 0, 0);
  const D3 o = ld3(a.org + 3 * i), d = ld3(a.dir + 3 * i);
  double den = 0.0;
  if (ok) {
    i0 = a.tris[3 * (int64_t)f];
    i1 = a.tris[3 * (int64_t)f + 1];
    i2 = a.tris[3 * (int64_t)f + 2];
    ok = i0 >= 0 && i0 < a.nv && i1 >= 0 && i1 < a.nv && i2 >= 0 && i2 < a.nv;
  }
  if (ok) {
    v0 = ld3(a.verts + 3 * (int64_t)i0);
    e1 = sub(ld3(a.verts + 3 * (int64_t)i1), v0);
    e2 = sub(ld3(a.verts + 3 * (int64_t)i2), v0);
    nn = cross(e1, e2);
    den = dot(nn, d);
    ok = den != 0.0;
  }
  if (!ok) {
    if (a.dldo) a.dldo[3 * i] = a.dldo[3 * i + 1] = a.dldo[3 * i + 2] = 0.0;
    if (a.dldd) a.dldd[3 * i] = a.dldd[3 * i + 1] = a.dldd[3 * i + 2] = 0.0;
    return false;
  }
  const double w = a.dldt[i] / den;
  const D3 q = d3(v0.x - (o.x + ti * d.x), v0.y - (o.y + ti * d.y), v0.z - (o.z + ti * d.z));
  const D3 a1 = cross(e2, q);
  const D3 a2 = cross(q, e1);
  A.i0 = i0;
  A.i1 = i1;
  A.i2 = i2;
  A.w = w;
  A.wq = d3(w * q.x, w * q.y, w * q.z);
  A.g1 = d3(w * a1.x, w * a1.y, w * a1.z);
  A.g2 = d3(w * a2.x, w * a2.y, w * a2.z);
  A.g0 = d3(w * (nn.x - a1.x - a2.x), w * (nn.y - a1.y - a2.y), w * (nn.z - a1.z - a2.z));
  if (a.dldo) {
    a.dldo[3 * i] = -w * nn.x;
    a.dldo[3 * i + 1] = -w * nn.y;
    a.dldo[3 * i + 2] = -w * nn.z;
  }
  if (a.dldd) {
    a.dldd[3 * i] = -w * ti * nn.x;
    a.dldd[3 * i + 1] = -w * ti * nn.y;
    a.dldd[3 * i + 2] = -w * ti * nn.z;
  }
  return true;
}

__device__ __forceinline__ void add_vertex(double* dldv, int32_t v, const D3& g)
{
  double* p = dldv + 3 * (int64_t)v;
  atomicAdd(p + 0, g.x);
  atomicAdd(p + 1, g.y);
  atomicAdd(p + 2, g.z);
}

__global__ void k_adjoint(AdjointArgs a)
{
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  AdjTerms A;
  if (!adjoint_ray(a, i, A) || !a.dldv) return;
  add_vertex(a.dldv, A.i1, A.g1);
  add_vertex(a.dldv, A.i2, A.g2);
  add_vertex(a.dldv, A.i0, A.g0);
}

// sort key: the hit face, or ntri for a ray without one (sorts last)
__global__ void k_adjoint_keys(AdjointArgs a, uint32_t* keys, int32_t* idx)
{
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int32_t f = a.face[i];
  keys[i] = (f >= 0 && f < a.ntri && a.t[i] < INFTY) ? (uint32_t)f : (uint32_t)a.ntri;
  idx[i] = (int32_t)i;
}

__device__ __forceinline__ D3 shfl_down3(const D3& v, int off)
{
  return d3(__shfl_down(v.x, off), __shfl_down(v.y, off), __shfl_down(v.z, off));
}

// rays in face order: lane l sums the terms of lanes l, l+1, ... of its run
// (equal face, contiguous after the sort) in six shuffle steps; the run's
// first lane in the wave adds them.  Every lane of the wave takes part in
// the shuffles (lanes past n carry no terms).
__global__ void k_adjoint_sorted(AdjointArgs a, const int32_t* order)
{
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  AdjTerms A;
  bool ok = false;
  if (j < a.n) ok = adjoint_ray(a, order[j], A);
  const int32_t face = ok ? a.face[order[j]] : -1 - lane;  // a lane without terms is a run of its own
  if (!ok) {
    A.i0 = A.i1 = A.i2 = 0;
    A.g0 = A.g1 = A.g2 = d3(0, 0, 0);
  }
  // runs by the position of their first lane: a hit without terms inside a
  // run splits it in two that share a face
  const int32_t fprev = __shfl_up(face, 1);
  const bool start = lane == 0 || fprev != face;
  const int run = 63 - __clzll((long long)(__ballot(start) & (~0ull >> (63 - lane))));
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const D3 h0 = shfl_down3(A.g0, off), h1 = shfl_down3(A.g1, off), h2 = shfl_down3(A.g2, off);
    const int ro = __shfl_down(run, off);
    if (lane + off < 64 && ro == run) {
      A.g0 = add3(A.g0, h0);
      A.g1 = add3(A.g1, h1);
      A.g2 = add3(A.g2, h2);
    }
  }
  const bool head = ok && start;
  if (head && a.dldv) {
    add_vertex(a.dldv, A.i1, A.g1);
    add_vertex(a.dldv, A.i2, A.g2);
    add_vertex(a.dldv, A.i0, A.g0);
  }
}

// ---- binned form ------------------------------------------------------------
constexpr int ADJ_FACES = 256;      // faces per bucket: 8 KB of sums in LDS
constexpr int ADJ_RAY_BLOCK = 512;  // k_adj_rays: rays per workgroup = ADJ_RAY_BLOCK * ADJ_RAYS
constexpr int ADJ_RAYS = 4;
constexpr int ADJ_CHUNK = 16384;    // k_adj_faces: rays per workgroup at most
// A ray with a larger (or NaN) w or w q adds its own vertex terms: an
// infinite sum of w q would make them NaN where they are infinite one by one,
// and sums of 2^31 smaller ones, times edges of up to 2^190, do not overflow.
constexpr double ADJ_SUM_MAX = 0x1p800;

__device__ __forceinline__ bool adj_hit(const AdjointArgs& a, int64_t i, int32_t& f)
{
  f = a.face[i];
  return f >= 0 && f < a.ntri && a.t[i] < INFTY;
}

__global__ void k_adj_zero(uint32_t* cnt, int nb)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nb) cnt[i] = 0u;
}

// rays per bucket
__global__ __launch_bounds__(256) void k_adj_count(AdjointArgs a, AdjointBins b)
{
  __shared__ uint32_t c[ADJ_BUCKETS_MAX + 1];
  for (int k = threadIdx.x; k < b.nb; k += blockDim.x) c[k] = 0u;
  __syncthreads();
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * blockDim.x) {
    int32_t f;
    if (adj_hit(a, i, f)) atomicAdd(&c[f / ADJ_FACES], 1u);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < b.nb; k += blockDim.x)
    if (c[k]) atomicAdd(b.cnt + k, c[k]);
}

// first slot of each bucket (off), write cursors (cur) and first chunk of
// each bucket (chunk); entry nb of off and chunk holds the totals.  One
// workgroup of 1024 threads, four entries each.
__global__ __launch_bounds__(1024) void k_adj_offsets(AdjointBins b)
{
  constexpr int PER = (ADJ_BUCKETS_MAX + 1) / 1024;
  __shared__ uint32_t wr[16], wc[16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t r[PER], rs = 0, cs = 0;
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x * PER + k;
    r[k] = i < b.nb ? b.cnt[i] : 0u;
    rs += r[k];
    cs += (r[k] + ADJ_CHUNK - 1) / ADJ_CHUNK;
  }
  uint32_t xr = rs, xc = cs;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t yr = __shfl_up(xr, o), yc = __shfl_up(xc, o);
    if (lane >= o) {
      xr += yr;
      xc += yc;
    }
  }
  if (lane == 63) {
    wr[wv] = xr;
    wc[wv] = xc;
  }
  __syncthreads();
  uint32_t er = xr - rs, ec = xc - cs;
  for (int q = 0; q < wv; ++q) {
    er += wr[q];
    ec += wc[q];
  }
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x * PER + k;
    if (i <= b.nb) {
      b.off[i] = er;
      b.chunk[i] = ec;
      if (i < b.nb) b.cur[i] = er;
    }
    er += r[k];
    ec += (r[k] + ADJ_CHUNK - 1) / ADJ_CHUNK;
  }
}

// Ray gradients, and each hit's (w, w q) into its bucket.  A workgroup
// counts its rays per bucket in LDS, reserves one range per bucket and
// writes the entries there.
__global__ __launch_bounds__(ADJ_RAY_BLOCK) void k_adj_rays(AdjointArgs a, AdjointBins b)
{
  __shared__ uint32_t c[ADJ_BUCKETS_MAX + 1];
  for (int k = threadIdx.x; k < b.nb; k += blockDim.x) c[k] = 0u;
  __syncthreads();
  const int64_t base = blockIdx.x * (int64_t)(ADJ_RAY_BLOCK * ADJ_RAYS) + threadIdx.x;
  int32_t face[ADJ_RAYS];
  uint32_t rank[ADJ_RAYS];
  double w[ADJ_RAYS];
  D3 wq[ADJ_RAYS];
#pragma unroll
  for (int k = 0; k < ADJ_RAYS; ++k) {
    const int64_t i = base + (int64_t)k * ADJ_RAY_BLOCK;
    face[k] = -1;
    w[k] = 0.0;
    wq[k] = d3(0, 0, 0);
    if (i < a.n) {
      AdjTerms A;
      if (adjoint_ray(a, i, A)) {
        if (fabs(A.w) <= ADJ_SUM_MAX && fabs(A.wq.x) <= ADJ_SUM_MAX && fabs(A.wq.y) <= ADJ_SUM_MAX &&
            fabs(A.wq.z) <= ADJ_SUM_MAX) {
          w[k] = A.w;
          wq[k] = A.wq;
        } else {
          add_vertex(a.dldv, A.i1, A.g1);
          add_vertex(a.dldv, A.i2, A.g2);
          add_vertex(a.dldv, A.i0, A.g0);
        }
      }
      int32_t f;
      if (adj_hit(a, i, f)) {  // as counted: a hit without terms adds zeros
        face[k] = f;
        rank[k] = atomicAdd(&c[f / ADJ_FACES], 1u);
      }
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < b.nb; k += blockDim.x)
    if (c[k]) c[k] = atomicAdd(b.cur + k, c[k]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ADJ_RAYS; ++k) {
    if (face[k] < 0) continue;
    const uint32_t pos = c[face[k] / ADJ_FACES] + rank[k];
    b.local[pos] = (uint8_t)(face[k] % ADJ_FACES);
    b.terms[pos] = AdjointEntry{w[k], wq[k].x, wq[k].y, wq[k].z};
  }
}

// x into *sum, and the rounding error of that addition into *err (the exact
// error of a floating-point sum: Knuth, TAOCP vol. 2, 4.2.2 theorem B)
__device__ __forceinline__ void add_exact(double* sum, double* err, double x)
{
  const double old = atomicAdd(sum, x);
  const double s = old + x;
  const double bb = s - old;
  atomicAdd(err, (old - (s - bb)) + (x - bb));
}

// Sums of one chunk of a bucket in LDS, then the vertex terms of its faces.
// A face's rays are added one after another, which rounds more often than
// the tree of the sorted form (relative error of dL/dV, 4 M rays on 81 920
// faces: 7.9e-16 against 6.2e-16), so each sum carries its rounding errors
// in a second one: 6.3e-16.
__global__ __launch_bounds__(256) void k_adj_faces(AdjointArgs a, AdjointBins b)
{
  __shared__ double sum[4][ADJ_FACES], err[4][ADJ_FACES];
  const uint32_t item = blockIdx.x;
  if (item >= b.chunk[b.nb]) return;
  int lo = 0, hi = b.nb;  // the bucket: last one whose first chunk is <= item
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (b.chunk[mid] <= item)
      lo = mid;
    else
      hi = mid;
  }
  for (int k = 0; k < 4; ++k) sum[k][threadIdx.x] = err[k][threadIdx.x] = 0.0;
  __syncthreads();
  const uint32_t first = b.off[lo] + (item - b.chunk[lo]) * ADJ_CHUNK;
  const uint32_t last = min(first + (uint32_t)ADJ_CHUNK, b.off[lo + 1]);
  for (uint32_t j = first + threadIdx.x; j < last; j += 256) {
    const int f = b.local[j];
    const AdjointEntry e = b.terms[j];
    add_exact(&sum[0][f], &err[0][f], e.w);
    add_exact(&sum[1][f], &err[1][f], e.x);
    add_exact(&sum[2][f], &err[2][f], e.y);
    add_exact(&sum[3][f], &err[3][f], e.z);
  }
  __syncthreads();
  auto total = [&](int k) { return sum[k][threadIdx.x] + err[k][threadIdx.x]; };
  const int64_t f = (int64_t)lo * ADJ_FACES + threadIdx.x;
  const double w = total(0);
  const D3 q = d3(total(1), total(2), total(3));
  if (f >= a.ntri || (w == 0.0 && q.x == 0.0 && q.y == 0.0 && q.z == 0.0)) return;
  const int32_t i0 = a.tris[3 * f], i1 = a.tris[3 * f + 1], i2 = a.tris[3 * f + 2];
  if (i0 < 0 || i0 >= a.nv || i1 < 0 || i1 >= a.nv || i2 < 0 || i2 >= a.nv) return;
  const D3 v0 = ld3(a.verts + 3 * (int64_t)i0);
  const D3 e1 = sub(ld3(a.verts + 3 * (int64_t)i1), v0), e2 = sub(ld3(a.verts + 3 * (int64_t)i2), v0);
  const D3 nn = cross(e1, e2), g1 = cross(e2, q), g2 = cross(q, e1);
  add_vertex(a.dldv, i1, g1);
  add_vertex(a.dldv, i2, g2);
  add_vertex(a.dldv, i0, d3(w * nn.x - g1.x - g2.x, w * nn.y - g1.y - g2.y, w * nn.z - g1.z - g2.z));
}

}  // namespace

void launch_adjoint(const AdjointArgs& a, int block, hipStream_t s)
{
  if (a.n <= 0) return;
  hipLaunchKernelGGL(k_adjoint, dim3((unsigned)((a.n + block - 1) / block)), dim3(block), 0, s, a);
}

void launch_adjoint_sorted(const AdjointArgs& a, const RayOrderScratch& w, hipStream_t s)
{
  if (a.n <= 0) return;
  const unsigned g = (unsigned)((a.n + 255) / 256);
  hipLaunchKernelGGL(k_adjoint_keys, dim3(g), dim3(256), 0, s, a, w.keys_in, w.idx_in);
  int bits = 1;
  while (bits < 32 && ((int64_t)1 << bits) <= a.ntri) ++bits;
  radix_sort_pairs(w.keys_in, w.idx_in, w.keys_out, w.idx_out, a.n, bits, (uint32_t*)w.temp, s);
  hipLaunchKernelGGL(k_adjoint_sorted, dim3(g), dim3(256), 0, s, a, w.idx_in);
}

int adjoint_buckets(int64_t ntri) { return (int)std::min<int64_t>((ntri + ADJ_FACES - 1) / ADJ_FACES, INT32_MAX); }

size_t adjoint_bins_bytes(int64_t n)
{
  return (size_t)n * (sizeof(AdjointEntry) + 1) + 256 + sizeof(uint32_t) * 4 * (size_t)(ADJ_BUCKETS_MAX + 1);
}

// Bound by the bytes of k_adj_rays: 116 in, 48 of ray gradients and 33 of
// terms per ray.  4 M rays on 81 920 faces, whole call: one atomic set per
// ray 1.6 ms, sorted by face (six radix passes) 1.02 ms, binned 0.40 ms
// (rays 0.25, faces 0.07, count 0.03).
void launch_adjoint_binned(const AdjointArgs& a, void* mem, hipStream_t s)
{
  if (a.n <= 0) return;
  AdjointBins b;
  b.nb = adjoint_buckets(a.ntri);
  b.terms = (AdjointEntry*)mem;
  b.cnt = (uint32_t*)(b.terms + a.n);
  b.cur = b.cnt + ADJ_BUCKETS_MAX + 1;
  b.off = b.cur + ADJ_BUCKETS_MAX + 1;
  b.chunk = b.off + ADJ_BUCKETS_MAX + 1;
  b.local = (uint8_t*)(b.chunk + ADJ_BUCKETS_MAX + 1);
  hipLaunchKernelGGL(k_adj_zero, dim3((unsigned)((b.nb + 255) / 256)), dim3(256), 0, s, b.cnt, b.nb);
  const unsigned gc = (unsigned)std::min<int64_t>((a.n + 2047) / 2048, 1024);
  hipLaunchKernelGGL(k_adj_count, dim3(gc), dim3(256), 0, s, a, b);
  hipLaunchKernelGGL(k_adj_offsets, dim3(1), dim3(1024), 0, s, b);
  const int64_t per = ADJ_RAY_BLOCK * ADJ_RAYS;
  hipLaunchKernelGGL(k_adj_rays, dim3((unsigned)((a.n + per - 1) / per)), dim3(ADJ_RAY_BLOCK), 0, s, a, b);
  // at most one partly filled chunk per bucket
  const unsigned gf = (unsigned)(a.n / ADJ_CHUNK + b.nb);
  hipLaunchKernelGGL(k_adj_faces, dim3(gf), dim3(256), 0, s, a, b);
}

}  // namespace xdgh
