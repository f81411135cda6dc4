// surface_query.hip -- batched surface-tree queries on one MI355X.
//
// Reference semantics (one ray per call there, one ray per lane here):
//   ray_fire         EmbreeRayTracer::ray_fire  src/embree/ray_tracer.cpp:290-326
//                    + TriangleIntersectionFunc src/triangle_intersect.cpp:52-109
//   point_in_volume  ray_tracer.cpp:259-287
//   find_volume      XDG::find_volume src/xdg.cpp:113-128
//   occluded         ray_tracer.cpp:347-370 + TriangleOcclusionFunc
//                    triangle_intersect.cpp:139-161
//   closest          ray_tracer.cpp:328-345 + TriangleClosestFunc
//                    triangle_intersect.cpp:111-137
// The answer of every query is the exact FP64 minimum over all primitives
// passing the reference's culls (the BVH only prunes conservatively), with
// one deterministic tie rule: among bitwise-equal distances the smallest
// face id wins (the reference keeps the last candidate Embree visits).
//
// Traversal: one ray per lane, wave64, over the BVH4 (WIDE, default) or the
// binary LBVH; near child first, others pushed on a per-lane stack in LDS
// laid out [slot][lane] (conflict-free).  PLAIN tests FP64 boxes; MIXED
// tests the outward-rounded FP32 boxes with an FP32 ray and keeps FP64 only
// for the Pluecker test, the distance and the normal/parity decision.  A
// mixed ray whose origin lies beyond the tree's conservative-rounding limit
// is traced with FP64 boxes (for ray_fire: queued to a second pass so that
// the mixed kernel carries no FP64 box state).
#include <algorithm>
#include <cstddef>

#include "fp32_bounds.h"
#include "internal.h"
#include "surface_traverse.h"
#include "xdg_hip.h"

namespace xdgh {

using namespace xdgd;

namespace {

constexpr int MAXK = XDG_HIP_MAX_EXCLUDE;  // exclusion entries per ray (read in place)

constexpr int RF_MIN_LANES = 16;
constexpr int FV_MIN_LANES = 16;
constexpr int PIV_MIN_LANES = 16, PIV_REFILL = 24;

// One ray of ray_fire.  DEFER (mixed only): a ray beyond the FP32-rounding
// limit is queued for the FP64 pass instead of traced here.
template <bool MIXED, bool DEFER, bool WIDE, bool SPEC = false>
__device__ __forceinline__ void ray_fire_one(const RayFireArgs& a, int64_t i, int32_t* stk, int cap)
{
  int32_t tree = a.tree_per_ray ? a.tree_per_ray[i] : a.tree;
  double* tout = a.t_out;
  if (tree < 1 || tree > a.ntrees) {
    tout[i] = INFTY;
    a.surf_out[i] = ID_NONE;
    if (a.face_out) a.face_out[i] = ID_NONE;
    return;
  }
  const SurfTreeDev& T = a.table[tree];
  RayD ray = make_ray(a.org + 3 * i, a.dir + 3 * i);
  if (DEFER && !mixed_safe(T, ray)) {
    const unsigned int j = atomicAdd(a.fb_count, 1u);
    a.fb_list[j] = (int32_t)i;
    return;
  }
  const int32_t* ex = a.excl ? a.excl + (int64_t)a.k * i : nullptr;
  const int k = a.excl ? (a.k < MAXK ? a.k : MAXK) : 0;
  HitState h;
  h.t = a.tmax ? a.tmax[i] : INFTY;
  h.face = INT32_MAX;
  h.surf = ID_NONE;
  h.inside = false;
  if (DEFER)
    trace_f32<RAYFIRE, false, WIDE, SPEC>(T, ray, a.orientation, ex, k, stk, blockDim.x, cap, h);
  else
    trace<RAYFIRE, MIXED, false, WIDE, SPEC>(T, ray, a.orientation, ex, k, stk, blockDim.x, cap, h);
  if (h.surf == ID_NONE) {
    tout[i] = INFTY;
    a.surf_out[i] = ID_NONE;
    if (a.face_out) a.face_out[i] = ID_NONE;
  } else {
    tout[i] = h.t;
    a.surf_out[i] = h.surf;
    if (a.face_out) a.face_out[i] = h.face;
  }
}

template <bool MIXED, bool DEFER, bool WIDE, bool SPEC = false>
__global__ void k_ray_fire(RayFireArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  ray_fire_one<MIXED, DEFER, WIDE, SPEC>(a, a.order ? (int64_t)a.order[i] : i, lds + threadIdx.x, cap);
}

// FP64 pass over the rays the mixed kernel queued (grid-stride; the count is
// read on the device, so no host round trip separates the two passes).
template <bool WIDE>
__global__ void k_ray_fire_deferred(RayFireArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  const unsigned int cnt = *a.fb_count;
  for (unsigned int j = blockIdx.x * blockDim.x + threadIdx.x; j < cnt; j += gridDim.x * blockDim.x)
    ray_fire_one<false, false, WIDE>(a, a.fb_list[j], lds + threadIdx.x, cap);
}

// work counter and deferral count of one launch (either nullable)
__global__ void k_zero_counters(unsigned long long* next, unsigned int* count)
{
  if (next) *next = 0ull;
  if (count) *count = 0u;
}
__global__ void k_zero_u32(unsigned int* p) { *p = 0u; }

__device__ __forceinline__ void write_hit(const RayFireArgs& a, int64_t i, const HitState& h)
{
  if (h.surf == ID_NONE) {
    a.t_out[i] = INFTY;
    a.surf_out[i] = ID_NONE;
    if (a.face_out) a.face_out[i] = ID_NONE;
  } else {
    a.t_out[i] = h.t;
    a.surf_out[i] = h.surf;
    if (a.face_out) a.face_out[i] = h.face;
  }
}

// Persistent ray_fire over the BVH4.  A fixed grid of resident waves works
// through the batch; each lane traces one ray at a time as a state machine,
// and lanes whose ray is done wait until refill_min of their wave are, then
// write their results and start new rays together (the set-up path is long,
// and runs for the whole wave).  MIXED queues far-origin rays for the FP64
// pass (k_ray_fire_deferred).  The loop's control is wave-uniform: a wave
// leaves once its ranges are dry and every lane is done.
//
// What bounds it: VALU issue at about two thirds of the peak and node
// latency, four waves per SIMD (127 VGPRs).  10 M nested-sphere rays:
// 2.89 -> 2.19 ms (4 M with FP64 boxes 2.09 -> 1.8), 1 M sphere rays, FP64,
// 0.456 -> 0.383 ms: ranges per wave instead of one atomic per refill,
// leaving the node loop when few lanes descend, pushes without branches
// (wave instructions 110 -> 88 per ray, active lanes 27 -> 37 %).
// FEW: a far-origin ray is traced with FP64 boxes at once instead.
template <bool MIXED, bool FEW = false>
__device__ __forceinline__ void ray_fire_pt_body(const RayFireArgs& a, unsigned long long* next_ray,
                                                 const ResidentCfg& c, int cap = 0)
{
  extern __shared__ int32_t lds[];
  GuardedStack S(lds + threadIdx.x, blockDim.x);
  const int32_t DONE = CHILD_EMPTY;
  int64_t ri = -1;
  bool have = false;  // ri's result is pending
  TreeView T{nullptr, nullptr, nullptr, nullptr};
  RayD ray{};
  BoxRayF bf{0, 0, 0, 0, 0, 0};
  BoxRayD bd{0, 0, 0, 0, 0, 0};
  HitState h{INFTY, INT32_MAX, ID_NONE, false};
  const int32_t* ex = nullptr;
  const int k = a.excl ? (a.k < MAXK ? a.k : MAXK) : 0;
  float tf = 0.0f;
  PlaneOfs po{0, 0, 0, 0, 0, 0};
  int32_t node = DONE;
  int32_t leaf = DONE;  // a leaf parked while the wave keeps descending
  WaveRange w(a.n, c.lanes_first);
  while (true) {
    const bool done = node == DONE && leaf == DONE;
    const unsigned long long dmask = __ballot(done);
    const int nd = __popcll(dmask);
    if (nd == 64 || (nd >= c.refill && !w.dry)) {
      if (done && have) {
        write_hit(a, ri, h);
        have = false;
      }
      if (w.dry) break;  // nd == 64
      const int64_t slot = w.take(dmask, a.n, c.chunk, c.lanes_first, next_ray);
      if (done && slot < a.n) {
        ri = a.order ? (int64_t)a.order[slot] : slot;
        const int32_t tree = a.tree_per_ray ? a.tree_per_ray[ri] : a.tree;
        h.t = a.tmax ? a.tmax[ri] : INFTY;
        h.face = INT32_MAX;
        h.surf = ID_NONE;
        h.inside = false;
        have = true;
        if (tree >= 1 && tree <= a.ntrees) {
          const SurfTreeDev& TT = a.table[tree];
          ray = make_ray(a.org + 3 * ri, a.dir + 3 * ri);
          if (MIXED && !FEW && !mixed_safe(TT, ray)) {
            const unsigned int j = atomicAdd(a.fb_count, 1u);
            a.fb_list[j] = (int32_t)ri;
            have = false;
          } else if (MIXED && FEW && !mixed_safe(TT, ray)) {
            traverse4<RAYFIRE, false>(TT, ray, a.orientation, a.excl ? a.excl + (int64_t)a.k * ri : nullptr, k, S.base,
                                      S.stride, cap, h);
          } else {
            T.nodes4_d = TT.nodes4_d;
            T.nodes4_f = TT.nodes4_f;
            T.tris = TT.tris;
            T.normals = TT.normals;
            ex = a.excl ? a.excl + (int64_t)a.k * ri : nullptr;
            tf = f32_up(h.t);
            box_ray<MIXED>(ray, bf, bd, po);
            S.reset();
            node = TT.n_prims > 0 ? TT.root4 : DONE;
          }
        }
      }
    }
    descend4<MIXED>(T, S, bf, bd, po, tf, h.t, c.min_lanes, node, leaf);
    if (leaf != DONE) {
      leaf_pairs<RAYFIRE>(T, leaf, ray, a.orientation, ex, k, h);
      leaf = DONE;
      tf = f32_up(h.t);
    }
  }
}

__global__ void k_ray_fire_pt_mixed(RayFireArgs a, unsigned long long* next_ray, ResidentCfg c)
{
  ray_fire_pt_body<true>(a, next_ray, c);
}
// Mixed batches that leave every wave with fewer than 64 rays: no counter, no
// deferral list, and so one launch instead of three (1 000 rays: 41 -> 37
// us a call).  The FP64 boxes' state costs registers, which larger batches
// would pay for in waves per SIMD.
__global__ __launch_bounds__(256) void k_ray_fire_few_mixed(RayFireArgs a, ResidentCfg c, int cap)
{
  ray_fire_pt_body<true, true>(a, nullptr, c, cap);
}
__global__ void k_ray_fire_pt_plain(RayFireArgs a, unsigned long long* next_ray, ResidentCfg c)
{
  ray_fire_pt_body<false>(a, next_ray, c);
}

// Instrumented ray_fire, one ray per lane: the traversal of k_ray_fire (the
// resident grid leaves its node loop earlier and refills lanes, so its wave
// iterations are fewer), plus per-ray work counters summed into
// counters[0..7] = rays, V, F, E, C, N, hits, mixed-fallbacks.
template <bool MIXED, bool WIDE>
__global__ void k_ray_fire_stats(RayFireArgs a, int cap, unsigned long long* counters, int spec)
{
  extern __shared__ int32_t lds[];
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  if (a.order) i = a.order[i];
  int32_t tree = a.tree_per_ray ? a.tree_per_ray[i] : a.tree;
  if (tree < 1 || tree > a.ntrees) return;
  const SurfTreeDev& T = a.table[tree];
  RayD ray = make_ray(a.org + 3 * i, a.dir + 3 * i);
  const int32_t* ex = a.excl ? a.excl + (int64_t)a.k * i : nullptr;
  const int k = a.excl ? (a.k < MAXK ? a.k : MAXK) : 0;
  HitState h;
  h.t = a.tmax ? a.tmax[i] : INFTY;
  h.face = INT32_MAX;
  h.surf = ID_NONE;
  h.inside = false;
  TraceStats st{0, 0, 0, 0, 0, 0, 0};
  if (WIDE && spec)
    trace<RAYFIRE, MIXED, true, WIDE, true>(T, ray, a.orientation, ex, k, lds + threadIdx.x, blockDim.x, cap, h, &st);
  else
    trace<RAYFIRE, MIXED, true, WIDE>(T, ray, a.orientation, ex, k, lds + threadIdx.x, blockDim.x, cap, h, &st);
  atomicAdd(counters + 0, 1ULL);
  atomicAdd(counters + 1, (unsigned long long)st.V);
  atomicAdd(counters + 2, (unsigned long long)st.F);
  atomicAdd(counters + 3, (unsigned long long)st.E);
  atomicAdd(counters + 4, (unsigned long long)st.C);
  atomicAdd(counters + 5, (unsigned long long)st.N);
  if (h.surf != ID_NONE) atomicAdd(counters + 6, 1ULL);
  if (MIXED && !mixed_safe(T, ray)) atomicAdd(counters + 7, 1ULL);
  if (st.WV) atomicAdd(counters + 8, (unsigned long long)st.WV);
  if (st.WF) atomicAdd(counters + 9, (unsigned long long)st.WF);
  // longest ray of the wave (node visits, triangle tests): the iterations a
  // wave needs if lanes never wait for each other between leaves
  const unsigned int mv = wave_max_u24(st.V), mf = wave_max_u24(st.F);
  if (first_active_lane()) {
    atomicAdd(counters + 10, (unsigned long long)mv);
    atomicAdd(counters + 11, (unsigned long long)mf);
  }
}

template <bool MIXED, bool WIDE>
__global__ void k_piv(PivArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  if (a.tree < 1 || a.tree > a.ntrees) {
    a.inside[i] = 0;
    return;
  }
  const SurfTreeDev& T = a.table[a.tree];
  const double* d = a.dir ? a.dir + 3 * i : a.dflt;
  RayD ray = make_ray(a.pts + 3 * i, d);
  const int32_t* ex = a.excl ? a.excl + (int64_t)a.k * i : nullptr;
  const int k = a.excl ? (a.k < MAXK ? a.k : MAXK) : 0;
  HitState h;
  h.t = INFTY;
  h.face = INT32_MAX;
  h.surf = ID_NONE;
  h.inside = false;
  trace<PIV, MIXED, false, WIDE>(T, ray, ORIENT_ANY, ex, k, lds + threadIdx.x, blockDim.x, cap, h);
  a.inside[i] = (h.surf != ID_NONE && h.inside) ? 1 : 0;
}

// Persistent point_in_volume over the BVH4: the per-lane state machine of
// the persistent ray_fire with a strided share per wave, so that a launch
// uses no scratch and may overlap others or be captured.  A point beyond the
// tree's FP32 limit (mixed) is traced with FP64 boxes at once.  Bound by VALU
// issue and node latency; the per-point kernel (k_piv) waited for each wave's
// longest traversal with a quarter of its lanes active.
// 1 M points in the 163 840-triangle shell: FP64 boxes 650 -> 475 us, mixed
// 315 us.
template <bool MIXED>
__device__ __forceinline__ void piv_pt_body(const PivArgs& a, int cap, const ResidentCfg& c)
{
  extern __shared__ int32_t lds[];
  GuardedStack S(lds + threadIdx.x, blockDim.x);
  const int32_t DONE = CHILD_EMPTY;
  int64_t pi = 0;
  bool have = false;  // pi's answer is pending
  const SurfTreeDev& TT = a.table[a.tree];
  const TreeView T{TT.nodes4_d, TT.nodes4_f, TT.tris, TT.normals};
  const int k = a.excl ? (a.k < MAXK ? a.k : MAXK) : 0;
  const int32_t* ex = nullptr;
  RayD ray{};
  BoxRayF bf{0, 0, 0, 0, 0, 0};
  BoxRayD bd{0, 0, 0, 0, 0, 0};
  PlaneOfs po{0, 0, 0, 0, 0, 0};
  HitState h{INFTY, INT32_MAX, ID_NONE, false};
  float tf = INFINITY;
  int32_t node = DONE, leaf = DONE;
  WaveStride w(a.n, c.lanes_first);
  while (true) {
    const bool done = node == DONE && leaf == DONE;
    const unsigned long long dmask = __ballot(done);
    const int nd = __popcll(dmask);
    if (nd == 64 || (nd >= c.refill && !w.dry)) {
      if (done && have) {
        a.inside[pi] = (h.surf != ID_NONE && h.inside) ? 1 : 0;
        have = false;
      }
      if (w.dry) break;  // nd == 64
      const int64_t pos = w.take(dmask, a.n, c.lanes_first);
      if (done && pos < a.n) {
        pi = pos;
        have = true;
        const double* d = a.dir ? a.dir + 3 * pi : a.dflt;
        ray = make_ray(a.pts + 3 * pi, d);
        ex = a.excl ? a.excl + (int64_t)a.k * pi : nullptr;
        h = HitState{INFTY, INT32_MAX, ID_NONE, false};
        if (MIXED && !mixed_safe(TT, ray)) {
          traverse4<PIV, false>(TT, ray, ORIENT_ANY, ex, k, S.base, S.stride, cap, h);
        } else {
          tf = INFINITY;
          box_ray<MIXED>(ray, bf, bd, po);
          S.reset();
          node = TT.n_prims > 0 ? TT.root4 : DONE;
        }
      }
    }
    descend4<MIXED>(T, S, bf, bd, po, tf, h.t, c.min_lanes, node, leaf);
    if (leaf != DONE) {
      leaf_pairs<PIV>(T, leaf, ray, ORIENT_ANY, ex, k, h);
      leaf = DONE;
      tf = f32_up(h.t);
    }
  }
}

__global__ void k_piv_pt_mixed(PivArgs a, int cap, ResidentCfg c) { piv_pt_body<true>(a, cap, c); }
__global__ void k_piv_pt_plain(PivArgs a, int cap, ResidentCfg c) { piv_pt_body<false>(a, cap, c); }

template <bool MIXED, bool WIDE>
__global__ void k_find_volume(FindVolumeArgs a, int cap, int spec)
{
  extern __shared__ int32_t lds[];
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const double* d = a.dir ? a.dir + 3 * i : a.dflt;
  RayD ray = make_ray(a.pts + 3 * i, d);
  int32_t found = a.ipc;
  for (int v = 0; v < a.nvol; ++v) {
    const int32_t vid = a.vol_ids[v];
    const int32_t tree = a.vol_trees[v];
    if (vid == a.ipc || tree < 1 || tree > a.ntrees) continue;
    HitState h;
    h.t = INFTY;
    h.face = INT32_MAX;
    h.surf = ID_NONE;
    h.inside = false;
    if (WIDE && spec)
      trace<PIV, MIXED, false, WIDE, true>(a.table[tree], ray, ORIENT_ANY, nullptr, 0, lds + threadIdx.x, blockDim.x,
                                           cap, h);
    else
      trace<PIV, MIXED, false, WIDE>(a.table[tree], ray, ORIENT_ANY, nullptr, 0, lds + threadIdx.x, blockDim.x, cap,
                                     h);
    if (h.surf != ID_NONE && h.inside) {
      found = vid;
      break;
    }
  }
  a.vol_out[i] = found;
}

__device__ __forceinline__ void find_volume_point(const FindVolumeArgs& a, int64_t i, int32_t* stk, int cap)
{
  const double* d = a.dir ? a.dir + 3 * i : a.dflt;
  RayD ray = make_ray(a.pts + 3 * i, d);
  int32_t found = a.ipc;
  for (int v = 0; v < a.nvol; ++v) {
    const int32_t vid = a.vol_ids[v];
    const int32_t tree = a.vol_trees[v];
    if (vid == a.ipc || tree < 1 || tree > a.ntrees) continue;
    HitState h{INFTY, INT32_MAX, ID_NONE, false};
    trace<PIV, false, false, true>(a.table[tree], ray, ORIENT_ANY, nullptr, 0, stk, blockDim.x, cap, h);
    if (h.surf != ID_NONE && h.inside) {
      found = vid;
      break;
    }
  }
  a.vol_out[i] = found;
}

// FP64 pass over the points the mixed persistent kernel queued
__global__ void k_find_volume_deferred(FindVolumeArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  const unsigned int cnt = *a.fb_count;
  for (unsigned int j = blockIdx.x * blockDim.x + threadIdx.x; j < cnt; j += gridDim.x * blockDim.x)
    find_volume_point(a, a.fb_list[j], lds + threadIdx.x, cap);
}

// Persistent find_volume over the BVH4: a lane holds one point and runs its
// point_in_volume traversals volume after volume (a new traversal on the
// same ray costs only a reset), as a per-lane state machine like the
// persistent ray_fire: lanes whose traversal has ended record the answer or
// start the next volume, and claim new points, together once c.refill of
// the wave are ready, while the other lanes keep descending.  Bound by VALU
// issue like ray_fire.  4 M nested-sphere points, mixed: 3.24 -> 1.92 ms,
// 0.6 ms of it from ranges per wave and cheap refills, the rest from leaving
// the node loop below 16 descending lanes (threshold 1 / 8 / 16 / 24: 2.64 /
// 1.98 / 1.92 / 2.00 ms).
template <bool MIXED>
__device__ __forceinline__ void find_volume_pt_body(const FindVolumeArgs& a, const ResidentCfg& c)
{
  extern __shared__ int32_t lds[];
  GuardedStack S(lds + threadIdx.x, blockDim.x);
  const int32_t DONE = CHILD_EMPTY;
  int64_t pi = 0;
  bool hasp = false;   // the lane holds a point whose volume is not known yet
  bool traced = false; // a point_in_volume traversal of volume v is under way or ended
  int v = 0;
  TreeView T{nullptr, nullptr, nullptr, nullptr};
  RayD ray{};
  BoxRayF bf{0, 0, 0, 0, 0, 0};
  BoxRayD bd{0, 0, 0, 0, 0, 0};
  PlaneOfs po{0, 0, 0, 0, 0, 0};
  HitState h{INFTY, INT32_MAX, ID_NONE, false};
  float tf = INFINITY;
  int32_t node = DONE, leaf = DONE;
  WaveRange w(a.n, c.lanes_first);
  while (true) {
    // lanes whose traversal has ended wait until c.refill of the wave (or
    // all that still have work) have too; then they act together: record or
    // advance to the next volume, claim new points, start traversals
    const bool done = node == DONE && leaf == DONE;
    const bool busy = __ballot(!done) != 0;
    const int ready = __popcll(__ballot(done && (hasp || !w.dry)));
    if (ready == 0 && !busy) break;
    if (ready >= c.refill || !busy) {
      if (done && traced) {
        traced = false;
        if (h.surf != ID_NONE && h.inside) {
          a.vol_out[pi] = a.vol_ids[v];
          hasp = false;
        } else {
          ++v;
        }
      }
      const bool need = done && !hasp;
      const unsigned long long cmask = __ballot(need);
      if (cmask && !w.dry) {
        const int64_t pos = w.take(cmask, a.n, c.chunk, c.lanes_first, a.next);
        if (need && pos < a.n) {
          pi = pos;
          const double* d = a.dir ? a.dir + 3 * pi : a.dflt;
          ray = make_ray(a.pts + 3 * pi, d);
          box_ray<MIXED>(ray, bf, bd, po);
          v = 0;
          hasp = true;
        }
      }
      if (done && hasp) {  // the point's next volume
        while (v < a.nvol && (a.vol_ids[v] == a.ipc || a.vol_trees[v] < 1 || a.vol_trees[v] > a.ntrees)) ++v;
        if (v >= a.nvol) {
          a.vol_out[pi] = a.ipc;
          hasp = false;
        } else {
          const SurfTreeDev& TT = a.table[a.vol_trees[v]];
          if (MIXED && !mixed_safe(TT, ray)) {  // the whole point goes to the FP64 pass
            const unsigned int j = atomicAdd(a.fb_count, 1u);
            a.fb_list[j] = (int32_t)pi;
            hasp = false;
          } else {
            T.nodes4_d = TT.nodes4_d;
            T.nodes4_f = TT.nodes4_f;
            T.tris = TT.tris;
            T.normals = TT.normals;
            h = HitState{INFTY, INT32_MAX, ID_NONE, false};
            tf = INFINITY;
            S.reset();
            node = TT.n_prims > 0 ? TT.root4 : DONE;
            traced = true;
          }
        }
      }
    }
    descend4<MIXED>(T, S, bf, bd, po, tf, h.t, c.min_lanes, node, leaf);
    if (leaf != DONE) {
      const int32_t first = leaf_first(leaf);
      const int32_t cnt = leaf_count(leaf);
      leaf = DONE;
      for (int32_t j = 0; j < cnt; ++j) tri_closest_hit<PIV>(T, first + j, ray, ORIENT_ANY, nullptr, 0, h);
      tf = f32_up(h.t);
    }
  }
}

__global__ void k_find_volume_pt_mixed(FindVolumeArgs a, ResidentCfg c) { find_volume_pt_body<true>(a, c); }
__global__ void k_find_volume_pt_plain(FindVolumeArgs a, ResidentCfg c) { find_volume_pt_body<false>(a, c); }

template <bool MIXED, bool WIDE>
__global__ void k_occluded(OccludedArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  bool hit = false;
  if (a.tree >= 1 && a.tree <= a.ntrees) {
    RayD ray = make_ray(a.org + 3 * i, a.dir + 3 * i);
    HitState h;
    h.t = INFTY;
    h.face = INT32_MAX;
    h.surf = ID_NONE;
    h.inside = false;
    hit = trace<OCCL, MIXED, false, WIDE>(a.table[a.tree], ray, ORIENT_ANY, nullptr, 0, lds + threadIdx.x,
                                          blockDim.x, cap, h);
  }
  a.hit[i] = hit ? 1 : 0;
  if (a.dist) a.dist[i] = hit ? -INFTY : INFTY;
}

// squared distance from p to an FP64 box
__device__ __forceinline__ double box_d2(const double* b, const D3& p)
{
  double ex = fmax(fmax(b[0] - p.x, p.x - b[3]), 0.0);
  double ey = fmax(fmax(b[1] - p.y, p.y - b[4]), 0.0);
  double ez = fmax(fmax(b[2] - p.z, p.z - b[5]), 0.0);
  return ex * ex + ey * ey + ez * ez;
}

// The triangles of one leaf against the best distance and face so far (ties:
// the smaller face).  reject: farther ones by their FP32 bound first.
__device__ __forceinline__ void closest_tri(const SurfTreeDev& T, int32_t first, int32_t cnt, const D3& p, bool reject,
                                            double& best, int32_t& bface)
{
  for (int32_t j = 0; j < cnt; ++j) {
    const auto r = as_global(T.tris + first + j);
    const auto pn = as_global(T.normals + 3 * (int64_t)(first + j));
    const D3 v0 = d3(r->v[0], r->v[1], r->v[2]);
    const D3 v1 = d3(r->v[3], r->v[4], r->v[5]);
    const D3 v2 = d3(r->v[6], r->v[7], r->v[8]);
    if (reject && closest_beyond(v0, v1, v2, d3(pn[0], pn[1], pn[2]), p, f32_up(best * best))) continue;
    const D3 q = closest_on_triangle(v0, v1, v2, p);
    const D3 e = sub(q, p);
    const double dist = sqrt(e.x * e.x + e.y * e.y + e.z * e.z);
    const int32_t face = r->face;
    if (dist < best || (dist == best && face < bface)) {
      best = dist;
      bface = face;
    }
  }
}

// children within the limit, nearest first (others CHILD_EMPTY)
__device__ __forceinline__ void node4_dist(const Node4F* nodes, int32_t node, const ClosestPointF& c, float lim,
                                           float* te, int32_t* ch)
{
  const Node4F* nd = nodes + node;
  const float4 lx = gload_at<float4>(nd, 0u), hx = gload_at<float4>(nd, 16u);
  const float4 ly = gload_at<float4>(nd, 32u), hy = gload_at<float4>(nd, 48u);
  const float4 lz = gload_at<float4>(nd, 64u), hz = gload_at<float4>(nd, 80u);
  const int4 cc = gload_at<int4>(nd, 96u);
  const float lxa[4] = {lx.x, lx.y, lx.z, lx.w}, hxa[4] = {hx.x, hx.y, hx.z, hx.w};
  const float lya[4] = {ly.x, ly.y, ly.z, ly.w}, hya[4] = {hy.x, hy.y, hy.z, hy.w};
  const float lza[4] = {lz.x, lz.y, lz.z, lz.w}, hza[4] = {hz.x, hz.y, hz.z, hz.w};
  const int32_t cca[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float d = closest_box(lxa[i], hxa[i], lya[i], hya[i], lza[i], hza[i], c);
    const bool in = d <= lim && cca[i] != CHILD_EMPTY;
    te[i] = in ? d : INFINITY;
    ch[i] = in ? cca[i] : CHILD_EMPTY;
  }
  cswap(te[0], ch[0], te[1], ch[1]);
  cswap(te[2], ch[2], te[3], ch[3]);
  cswap(te[0], ch[0], te[2], ch[2]);
  cswap(te[1], ch[1], te[3], ch[3]);
  cswap(te[1], ch[1], te[2], ch[2]);
}

// The same in FP64 for a point beyond the FP32 boxes' limit, whose distances
// to them FP32 does not tell apart: the dilated boxes as they are, and a
// factor on the limit for the rounding of a distance far beyond the bump.
// te holds what each distance adds to the least of the four.
__device__ __forceinline__ void node4_dist_far(const Node4D* nodes, int32_t node, const D3& p, double best, float* te,
                                               int32_t* ch)
{
  const auto nd = as_global(nodes + node);
  const double lim = best * best * (1.0 + 0x1p-48);
  double d[4], least = INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const double ex = fmax(fmax(nd->lox[i] - p.x, p.x - nd->hix[i]), 0.0);
    const double ey = fmax(fmax(nd->loy[i] - p.y, p.y - nd->hiy[i]), 0.0);
    const double ez = fmax(fmax(nd->loz[i] - p.z, p.z - nd->hiz[i]), 0.0);
    d[i] = ex * ex + ey * ey + ez * ez;
    ch[i] = d[i] <= lim ? nd->child[i] : CHILD_EMPTY;
    if (ch[i] != CHILD_EMPTY) least = fmin(least, d[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) te[i] = ch[i] != CHILD_EMPTY ? (float)(d[i] - least) : INFINITY;
  cswap(te[0], ch[0], te[1], ch[1]);
  cswap(te[2], ch[2], te[3], ch[3]);
  cswap(te[0], ch[0], te[2], ch[2]);
  cswap(te[1], ch[1], te[3], ch[3]);
  cswap(te[1], ch[1], te[2], ch[2]);
}

// LDS of one wave of k_closest: up to 64 points and the queues they share.
// A queue entry is a child code and a tag: the point's lane, and the upper
// half of the entry's FP32 box distance (a lower bound).
constexpr int CLOSEST_NODES = 1536;  // node queue
constexpr int CLOSEST_STACK_MAX = 192;  // stack bound of any BVH4: three entries for each of 64 levels
static_assert(CLOSEST_NODES >= 64 + 3 * 64 + CLOSEST_STACK_MAX, "a wave's points and one full step fit the queue");
constexpr int CLOSEST_LEAVES = 320;  // leaf queue: below 64, plus one step's 4 x 64
struct ClosestLds {
  double px[64], py[64], pz[64];
  unsigned long long best[64];  // bits of the best distance (non-negative: ordered as integers)
  ClosestPointF c[64];
  float lim[64];
  int32_t face[64];
  int32_t leaf[CLOSEST_LEAVES];
  uint32_t ltag[CLOSEST_LEAVES];
  uint32_t ntag[CLOSEST_NODES];
  int32_t node[CLOSEST_NODES];
};
__device__ __forceinline__ uint32_t closest_tag(int owner, float d)
{
  return (__float_as_uint(d) & 0xffff0000u) | (uint32_t)owner;
}
__device__ __forceinline__ bool closest_live(uint32_t tag, float lim)
{
  return (tag >> 16) <= (__float_as_uint(lim) >> 16);  // non-negative floats order as integers
}
__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Children of one node step into the queues: farther ones first, so that
// the lanes' nearest children are the next taken.
__device__ __forceinline__ void closest_push(ClosestLds& L, int owner, const float* te, const int32_t* ch, int& nn,
                                             int& nl)
{
  const unsigned long long below = (1ull << (threadIdx.x & 63)) - 1ull;
#pragma unroll
  for (int i = 3; i >= 0; --i) {
    const bool node = ch[i] >= 0, leaf = ch[i] < 0 && ch[i] != CHILD_EMPTY;
    const unsigned long long kn = __ballot(node), kl = __ballot(leaf);
    if (node) {
      const int k = nn + __popcll(kn & below);
      L.node[k] = ch[i];
      L.ntag[k] = closest_tag(owner, te[i]);
    }
    if (leaf) {
      const int k = nl + __popcll(kl & below);
      L.leaf[k] = ch[i];
      L.ltag[k] = closest_tag(owner, te[i]);
    }
    nn += __popcll(kn);
    nl += __popcll(kl);
  }
}

// The steps of one batch of points until both queues are empty.  FAR: some
// of them (fars, by lane) are beyond the FP32 boxes' limit; without any, the
// steps carry no FP64 boxes (which cost them 4 to 9 % of their time).
template <bool FAR>
__device__ __forceinline__ void closest_run(ClosestLds& L, const SurfTreeDev& T, unsigned long long fars, bool queued,
                                            int reserve, int nn, int nl)
{
  const int lane = threadIdx.x;
  while (nn + nl > 0) {
    if (nl < 64 && nn > 0) {
      const int m = nn + 3 * 64 + reserve <= CLOSEST_NODES ? (nn < 64 ? nn : 64) : 1;
      float te[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
      int32_t ch[4] = {CHILD_EMPTY, CHILD_EMPTY, CHILD_EMPTY, CHILD_EMPTY};
      int owner = 0;
      if (lane < m) {
        const int k = nn - 1 - lane;
        const uint32_t tag = L.ntag[k];
        owner = (int)(tag & 63u);
        const float lim = L.lim[owner];
        if (FAR && (fars >> owner & 1)) {
          node4_dist_far(T.nodes4_d, L.node[k], d3(L.px[owner], L.py[owner], L.pz[owner]),
                         __longlong_as_double((long long)L.best[owner]), te, ch);
          te[0] = te[1] = te[2] = te[3] = 0.0f;  // entries of far points always live
        } else if (closest_live(tag, lim)) {
          node4_dist(T.nodes4_f, L.node[k], L.c[owner], lim, te, ch);
        }
      }
      nn -= m;
      wave_lds_sync();
      closest_push(L, owner, te, ch, nn, nl);
    } else {
      const int m = nl < 64 ? nl : 64;
      bool cand = false;
      int owner = 0;
      double b = INFTY, b0 = INFTY;
      int32_t f = INT32_MAX;
      if (lane < m) {
        const int k = nl - 1 - lane;
        const uint32_t tag = L.ltag[k];
        owner = (int)(tag & 63u);
        if (closest_live(tag, L.lim[owner])) {
          b = b0 = __longlong_as_double((long long)L.best[owner]);
          f = L.face[owner];
          const int32_t f0 = f, code = L.leaf[k];
          closest_tri(T, leaf_first(code), leaf_count(code), d3(L.px[owner], L.py[owner], L.pz[owner]),
                      !FAR || !(fars >> owner & 1), b, f);
          cand = b < b0 || f != f0;
        }
      }
      nl -= m;
      if (__ballot(cand)) {
        // several lanes may hold one point's leaves: the least distance
        // first, then the smallest face at that distance
        const unsigned long long bits = (unsigned long long)__double_as_longlong(b);
        if (cand) atomicMin(&L.best[owner], bits);
        wave_lds_sync();
        const bool win = cand && L.best[owner] == bits;
        if (win && b < b0) L.face[owner] = INT32_MAX;
        wave_lds_sync();
        if (win) atomicMin(&L.face[owner], f);
        wave_lds_sync();
        if (queued) L.lim[lane] = closest_limit(__longlong_as_double((long long)L.best[lane]));
      }
    }
    wave_lds_sync();
  }
}

// closest over the BVH4, one wave per workgroup.  A wave holds up to 64
// points and works on their descents together: node and leaf entries of all
// points share two LDS queues, and each step takes up to 64 entries of one
// queue, one per lane.  A descent per lane left most lanes idle, since
// points nearly as far from a large part of the surface as from its nearest
// triangle (the centre of a sphere) visit thousands of nodes where others
// visit tens; here the wave's lanes share whatever is left.
//
// Steps take nodes while fewer than 64 leaves wait, else leaves.  While the
// node queue has no room for a full step's pushes (3 x 64 net) above
// `reserve` entries (the BVH4's stack bound), nodes are taken one at a time:
// depth first, at most that many more entries, so it cannot overflow.
//
// lead: each lane first takes its own point's nearest child down to a leaf.
// With that leaf's distance as limit the queues stay short; without one they
// fill with every point's siblings of its first path, and in trees of 80 000
// triangles run the node queue into its one-at-a-time mode (1 M points near
// a sphere of 81 920 triangles 1.35 -> 0.49 ms, 100 003 of them 0.130 ->
// 0.075, 4 000 0.061 -> 0.042).
// 100 003 points in a ball around a sphere of 20 480 triangles: 7.4 -> 0.35 ms
// (a descent per lane on these boxes, the last 16 points of a wave finished
// by all its lanes: 0.73 ms).  Bound by the latency of the steps, two waves
// per SIMD (19 KB of LDS each).
__global__ __launch_bounds__(64) void k_closest(ClosestArgs a, int reserve, int lanes_first, bool lead)
{
  extern __shared__ __align__(16) unsigned char smem[];
  ClosestLds& L = *(ClosestLds*)smem;
  const int lane = threadIdx.x;
  const SurfTreeDev T = a.table[a.tree];
  double ext = 0.0;
  for (int k = 0; k < 3; ++k) ext = fmax(ext, fmax(fabs((double)T.box_lo[k]), fabs((double)T.box_hi[k])));
  const double shrink = closest_shrink(T.bump, ext);
  const double limit = (double)T.o_limit;
  WaveStride w(a.n, lanes_first);
  while (!w.dry) {
    const unsigned long long first = lanes_first < 64 ? (1ull << lanes_first) - 1ull : ~0ull;
    const int64_t pi = w.take(first, a.n, lanes_first);
    const bool have = lane < lanes_first && pi < a.n;
    const bool queued = have && T.n_prims > 0;
    bool far = false;
    if (have) {
      const D3 p = d3(a.pts[3 * pi], a.pts[3 * pi + 1], a.pts[3 * pi + 2]);
      const ClosestPointF c = closest_point(p, shrink);
      far = !(fmax(fmax(fabs(p.x), fabs(p.y)), fabs(p.z)) <= limit);
      double best = INFTY;
      int32_t bface = INT32_MAX;
      int32_t node = lead && queued ? T.root4 : CHILD_EMPTY;
      float te[4];
      int32_t ch[4];
      while (node >= 0 && !far) {
        node4_dist(T.nodes4_f, node, c, INFINITY, te, ch);
        node = ch[0];
      }
      while (node >= 0) {
        node4_dist_far(T.nodes4_d, node, p, best, te, ch);
        node = ch[0];
      }
      if (node != CHILD_EMPTY) closest_tri(T, leaf_first(node), leaf_count(node), p, false, best, bface);
      L.px[lane] = p.x;
      L.py[lane] = p.y;
      L.pz[lane] = p.z;
      L.c[lane] = c;
      L.best[lane] = (unsigned long long)__double_as_longlong(best);
      L.face[lane] = bface;
      L.lim[lane] = closest_limit(best);
    }
    const unsigned long long fars = __ballot(far);
    int nn = 0, nl = 0;  // entries in the node and leaf queues
    {
      const float te[4] = {0.0f, INFINITY, INFINITY, INFINITY};
      const int32_t ch[4] = {queued ? T.root4 : CHILD_EMPTY, CHILD_EMPTY, CHILD_EMPTY, CHILD_EMPTY};
      closest_push(L, lane, te, ch, nn, nl);
    }
    wave_lds_sync();
    if (fars)
      closest_run<true>(L, T, fars, queued, reserve, nn, nl);
    else
      closest_run<false>(L, T, fars, queued, reserve, nn, nl);
    if (have) {
      const int32_t f = L.face[lane];
      a.dist[pi] = f == INT32_MAX ? INFTY : __longlong_as_double((long long)L.best[lane]);
      a.face[pi] = f == INT32_MAX ? ID_NONE : f;
    }
    wave_lds_sync();
  }
}

// Distance and face of one point by the binary tree's FP64 boxes, one point
// per lane: large batches on a tree of a few triangles, whose descents are
// alike (launch_closest).  The limit's factor is node4_dist_far's.
__device__ inline void closest_fp64(const SurfTreeDev& T, const D3& p, int32_t* stk, int stride, int cap, double& best,
                                    int32_t& bface)
{
  int sp = 0;
  int32_t node = T.root;
  while (true) {
    if (node >= 0) {
      const NodeD nd = T.nodes_d[node];
      double d0 = box_d2(nd.b0, p), d1 = box_d2(nd.b1, p);
      double lim = best * best * (1.0 + 0x1p-48);
      bool h0 = d0 <= lim, h1 = d1 <= lim;
      int32_t c0 = nd.c0, c1 = nd.c1;
      if (h0 && h1) {
        if (d1 < d0) {
          int32_t tmp = c0;
          c0 = c1;
          c1 = tmp;
        }
        if (sp < cap) stk[sp++ * stride] = c1;
        node = c0;
      } else if (h0) {
        node = c0;
      } else if (h1) {
        node = c1;
      } else {
        if (sp == 0) break;
        node = stk[--sp * stride];
      }
      continue;
    }
    closest_tri(T, leaf_first(node), leaf_count(node), p, false, best, bface);
    if (sp == 0) break;
    node = stk[--sp * stride];
  }
}

__global__ void k_closest_lane(ClosestArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const SurfTreeDev& T = a.table[a.tree];
  double best = INFTY;
  int32_t bface = INT32_MAX;
  if (T.n_prims > 0)
    closest_fp64(T, d3(a.pts[3 * i], a.pts[3 * i + 1], a.pts[3 * i + 2]), lds + threadIdx.x, blockDim.x, cap, best,
                 bface);
  a.dist[i] = bface == INT32_MAX ? INFTY : best;
  a.face[i] = bface == INT32_MAX ? ID_NONE : bface;
}

inline dim3 grid1(int64_t n, int blk) { return dim3((unsigned)((n + blk - 1) / blk)); }
inline size_t lds_bytes(const LaunchCfg& c) { return sizeof(int32_t) * (size_t)c.stack * c.block; }
inline size_t lds_bytes_guarded(const LaunchCfg& c)
{
  return sizeof(int32_t) * (size_t)(c.stack + GUARDED_STACK_EXTRA) * c.block;
}

#define XDG_DISPATCH2(KERNEL, MIXED, WIDE, ...)                                              \
  do {                                                                                       \
    if (MIXED) {                                                                             \
      if (WIDE)                                                                              \
        hipLaunchKernelGGL((KERNEL<true, true>), __VA_ARGS__);                               \
      else                                                                                   \
        hipLaunchKernelGGL((KERNEL<true, false>), __VA_ARGS__);                              \
    } else {                                                                                 \
      if (WIDE)                                                                              \
        hipLaunchKernelGGL((KERNEL<false, true>), __VA_ARGS__);                              \
      else                                                                                   \
        hipLaunchKernelGGL((KERNEL<false, false>), __VA_ARGS__);                             \
    }                                                                                        \
  } while (0)

}  // namespace

void launch_ray_fire(const RayFireArgs& a, bool mixed, const LaunchCfg& c, hipStream_t s)
{
  if (a.n <= 0) return;
  const dim3 g = grid1(a.n, c.block), b(c.block);
  const size_t sh = lds_bytes(c);
  const bool persist = (c.persistent & (mixed ? 2 : 1)) != 0;
  if (persist && c.wide && a.next_ray && (!mixed || (a.fb_list && a.fb_count))) {
    const size_t shg = lds_bytes_guarded(c);
    const ResidentLaunch L =
        resident_launch(a.n, mixed ? resident_grid(k_ray_fire_pt_mixed, c.block, shg)
                                   : resident_grid(k_ray_fire_pt_plain, c.block, shg), c.block, c.refill, RF_MIN_LANES);
    if (mixed && !L.counted && L.c.lanes_first < 64 && c.block <= 256) {
      hipLaunchKernelGGL(k_ray_fire_few_mixed, dim3(L.grid), b, shg, s, a, L.c, c.stack);
      return;
    }
    if (mixed || L.counted)
      hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(1), 0, s, a.next_ray, mixed ? a.fb_count : nullptr);
    if (mixed) {
      hipLaunchKernelGGL(k_ray_fire_pt_mixed, dim3(L.grid), b, shg, s, a, a.next_ray, L.c);
      const unsigned gd = (unsigned)std::min<int64_t>((a.n + c.block - 1) / c.block, 1024);
      hipLaunchKernelGGL((k_ray_fire_deferred<true>), dim3(gd), b, sh, s, a, c.stack);
    } else {
      hipLaunchKernelGGL(k_ray_fire_pt_plain, dim3(L.grid), b, shg, s, a, a.next_ray, L.c);
    }
    return;
  }
  if (mixed && a.fb_list && a.fb_count) {
    const unsigned gd = (unsigned)std::min<int64_t>((a.n + c.block - 1) / c.block, 1024);
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, s, a.fb_count);
    if (c.wide) {
      if (c.spec)
        hipLaunchKernelGGL((k_ray_fire<true, true, true, true>), g, b, sh, s, a, c.stack);
      else
        hipLaunchKernelGGL((k_ray_fire<true, true, true>), g, b, sh, s, a, c.stack);
      hipLaunchKernelGGL((k_ray_fire_deferred<true>), dim3(gd), b, sh, s, a, c.stack);
    } else {
      hipLaunchKernelGGL((k_ray_fire<true, true, false>), g, b, sh, s, a, c.stack);
      hipLaunchKernelGGL((k_ray_fire_deferred<false>), dim3(gd), b, sh, s, a, c.stack);
    }
  } else if (mixed) {
    if (c.wide)
      hipLaunchKernelGGL((k_ray_fire<true, false, true>), g, b, sh, s, a, c.stack);
    else
      hipLaunchKernelGGL((k_ray_fire<true, false, false>), g, b, sh, s, a, c.stack);
  } else {
    if (c.wide && c.spec)
      hipLaunchKernelGGL((k_ray_fire<false, false, true, true>), g, b, sh, s, a, c.stack);
    else if (c.wide)
      hipLaunchKernelGGL((k_ray_fire<false, false, true>), g, b, sh, s, a, c.stack);
    else
      hipLaunchKernelGGL((k_ray_fire<false, false, false>), g, b, sh, s, a, c.stack);
  }
}

void launch_ray_fire_stats(const RayFireArgs& a, bool mixed, const LaunchCfg& c, unsigned long long* counters,
                           hipStream_t s)
{
  if (a.n <= 0) return;
  XDG_DISPATCH2(k_ray_fire_stats, mixed, c.wide, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack,
                counters, c.spec);
}

void launch_point_in_volume(const PivArgs& a, bool mixed, const LaunchCfg& c, hipStream_t s)
{
  if (a.n <= 0) return;
  if ((c.persistent & 4) && c.wide && a.tree >= 1 && a.tree <= a.ntrees) {
    const size_t sh = lds_bytes_guarded(c);
    const int refill = c.fv_refill ? c.fv_refill : PIV_REFILL;
    const ResidentLaunch L = resident_launch(a.n, mixed ? resident_grid(k_piv_pt_mixed, c.block, sh)
                                                        : resident_grid(k_piv_pt_plain, c.block, sh), c.block, refill,
                                             PIV_MIN_LANES);
    if (mixed)
      hipLaunchKernelGGL(k_piv_pt_mixed, dim3(L.grid), dim3(c.block), sh, s, a, c.stack, L.c);
    else
      hipLaunchKernelGGL(k_piv_pt_plain, dim3(L.grid), dim3(c.block), sh, s, a, c.stack, L.c);
    return;
  }
  XDG_DISPATCH2(k_piv, mixed, c.wide, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack);
}

void launch_find_volume(const FindVolumeArgs& a, bool mixed, const LaunchCfg& c, hipStream_t s)
{
  if (a.n <= 0) return;
  // bit 2 of the persistent mask: the resident grid whose lanes move on to
  // their next volume or point while others still traverse (default), or
  // the per-point kernel that keeps a wave's lanes on the same tree volume
  // after volume but waits for its longest traversal at each.  Refill
  // 8 / 24 / 40 / 56: 1.90 / 1.92 / 2.13 / 3.05 ms mixed (4 M nested-sphere
  // points), 1.56 / 1.55 / 1.58 / 2.07 ms FP64 (2 M)
  const bool persist = (c.persistent & 4) != 0;
  const int refill = c.fv_refill ? c.fv_refill : 24;
  if (persist && c.wide && a.next && (!mixed || (a.fb_list && a.fb_count))) {
    const size_t sh = lds_bytes_guarded(c);
    const dim3 b(c.block);
    const ResidentLaunch L =
        resident_launch(a.n, mixed ? resident_grid(k_find_volume_pt_mixed, c.block, sh)
                                   : resident_grid(k_find_volume_pt_plain, c.block, sh), c.block, refill, FV_MIN_LANES);
    if (mixed || L.counted)
      hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(1), 0, s, a.next, mixed ? a.fb_count : nullptr);
    if (mixed) {
      hipLaunchKernelGGL(k_find_volume_pt_mixed, dim3(L.grid), b, sh, s, a, L.c);
      const unsigned gd = (unsigned)std::min<int64_t>((a.n + c.block - 1) / c.block, 1024);
      hipLaunchKernelGGL(k_find_volume_deferred, dim3(gd), b, lds_bytes(c), s, a, c.stack);
    } else {
      hipLaunchKernelGGL(k_find_volume_pt_plain, dim3(L.grid), b, sh, s, a, L.c);
    }
    return;
  }
  // speculative leaf parking measured faster for the plain kernel only
  // (nested spheres, 10 M points: plain 14.98 -> 14.16 ms, mixed 9.67 -> 9.77 ms)
  XDG_DISPATCH2(k_find_volume, mixed, c.wide, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack,
                mixed ? 0 : c.spec);
}

// check_location_for_overlap (tools/overlap.cpp:9-61): point_in_volume of
// each location, with its own direction and no exclusions, against every
// volume of the list in order (no early exit).  The first max_k volumes
// that contain it are written, and their count.
template <bool MIXED, bool WIDE>
__global__ void k_point_in_volumes(VolumesArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const RayD ray = make_ray(a.pts + 3 * i, a.dir + 3 * i);
  int32_t* ids = a.ids_out + (int64_t)a.max_k * i;
  int cnt = 0;
  for (int v = 0; v < a.nvol; ++v) {
    const int32_t tree = a.vol_trees[v];
    if (tree < 1 || tree > a.ntrees) continue;
    HitState h{INFTY, INT32_MAX, ID_NONE, false};
    trace<PIV, MIXED, false, WIDE>(a.table[tree], ray, ORIENT_ANY, nullptr, 0, lds + threadIdx.x, blockDim.x, cap,
                                   h);
    if (h.surf != ID_NONE && h.inside) {
      if (cnt < a.max_k) ids[cnt] = a.vol_ids[v];
      ++cnt;
    }
  }
  a.count_out[i] = cnt;
}

// check_along_edge (tools/overlap.cpp:229-265): XDG::ray_fire(vol, origin,
// direction, edge length) (EXITING, no exclusions) against each volume of the
// list in order except the ray's two skipped volumes (the parents of the
// edge's surface); the first volume with a hit ends the search.
template <bool MIXED, bool WIDE>
__global__ void k_edge_rays(VolumesArgs a, int cap)
{
  extern __shared__ int32_t lds[];
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const RayD ray = make_ray(a.pts + 3 * i, a.dir + 3 * i);
  const int32_t s0 = a.skip[2 * i], s1 = a.skip[2 * i + 1];
  const double lim = a.len[i];
  double t = INFTY;
  int32_t surf = ID_NONE, vol = ID_NONE;
  for (int v = 0; v < a.nvol; ++v) {
    const int32_t vid = a.vol_ids[v];
    const int32_t tree = a.vol_trees[v];
    if (vid == s0 || vid == s1 || tree < 1 || tree > a.ntrees) continue;
    HitState h{lim, INT32_MAX, ID_NONE, false};
    trace<RAYFIRE, MIXED, false, WIDE>(a.table[tree], ray, ORIENT_EXITING, nullptr, 0, lds + threadIdx.x, blockDim.x,
                                       cap, h);
    if (h.surf != ID_NONE) {
      t = h.t;
      surf = h.surf;
      vol = vid;
      break;
    }
  }
  a.t_out[i] = t;
  a.surf_out[i] = surf;
  a.vol_out[i] = vol;
}

void launch_point_in_volumes(const VolumesArgs& a, bool mixed, const LaunchCfg& c, hipStream_t s)
{
  if (a.n <= 0) return;
  XDG_DISPATCH2(k_point_in_volumes, mixed, c.wide, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack);
}

void launch_edge_rays(const VolumesArgs& a, bool mixed, const LaunchCfg& c, hipStream_t s)
{
  if (a.n <= 0) return;
  XDG_DISPATCH2(k_edge_rays, mixed, c.wide, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack);
}

void launch_occluded(const OccludedArgs& a, bool mixed, const LaunchCfg& c, hipStream_t s)
{
  if (a.n <= 0) return;
  XDG_DISPATCH2(k_occluded, mixed, c.wide, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack);
}

void launch_closest(const ClosestArgs& a, const LaunchCfg& c, const SurfTreeDev& t, hipStream_t s)
{
  if (a.n <= 0) return;
  // 20 triangles, 1 M points (lane / queues): around the sphere 0.190 / 0.20
  // ms, near it 0.135 / 0.18; 100 003: 0.062 / 0.046 and 0.047 / 0.045; 80
  // triangles, 1 M around: 0.51 / 0.28
  if (t.n_prims <= 32 && a.n >= 1 << 19) {
    hipLaunchKernelGGL(k_closest_lane, grid1(a.n, c.block), dim3(c.block), lds_bytes(c), s, a, c.stack);
    return;
  }
  const size_t sh = sizeof(ClosestLds);
  // spread over every resident wave: its lanes are busy however few points
  // it holds
  const int64_t waves = resident_grid(k_closest, 64, sh);
  const int lanes_first = (int)std::min<int64_t>(64, (a.n + waves - 1) / waves);
  const unsigned grid = (unsigned)std::min<int64_t>(waves, (a.n + lanes_first - 1) / lanes_first);
  // the leading descent costs a few waves of a handful of points more than it
  // saves in a tree of a few levels (80 triangles, 4 000 points: 32 us without
  // it, 35 with; 320: 41 and 41; 80 triangles, 20 000 points: 42 and 38)
  const bool lead = t.n_prims > 256 || lanes_first >= 8;
  hipLaunchKernelGGL(k_closest, dim3(grid), dim3(64), sh, s, a, t.stack4, lanes_first, lead);
}

// ---- primitive evaluation (parity checks of the device geometry kernels) --

namespace {

__global__ void k_eval(int kind, int64_t n, const double* __restrict__ in, double* __restrict__ out)
{
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (kind == 0) {  // plucker: v0 v1 v2 o d tmax tmin use ori -> hit, t
    const double* c = in + 19 * i;
    const D3 v0 = d3(c[0], c[1], c[2]), v1 = d3(c[3], c[4], c[5]), v2 = d3(c[6], c[7], c[8]);
    const D3 o = d3(c[9], c[10], c[11]), d = d3(c[12], c[13], c[14]);
    const D3 rb = cross(d, o);
    const int idx = major_axis(d);
    const double oi = pick3(o.x, o.y, o.z, idx), di = pick3(d.x, d.y, d.z, idx);
    double t = 0.0;
    bool hit;
    if (c[17] != 0.0)
      hit = plucker_oriented(v0, v1, v2, d, rb, idx, oi, di, (double)(int)c[18], c[15], c[16], t);
    else
      hit = plucker_any(v0, v1, v2, d, rb, idx, oi, di, c[15], c[16], t);
    out[2 * i] = hit ? 1.0 : 0.0;
    out[2 * i + 1] = hit ? t : 0.0;
  } else if (kind == 1) {  // face normal: 9 -> 3
    const double* c = in + 9 * i;
    const D3 nrm = face_normal(d3(c[0], c[1], c[2]), d3(c[3], c[4], c[5]), d3(c[6], c[7], c[8]));
    out[3 * i] = nrm.x;
    out[3 * i + 1] = nrm.y;
    out[3 * i + 2] = nrm.z;
  } else if (kind == 2) {  // closest point: 12 -> 3
    const double* c = in + 12 * i;
    const D3 q = closest_on_triangle(d3(c[0], c[1], c[2]), d3(c[3], c[4], c[5]), d3(c[6], c[7], c[8]),
                                     d3(c[9], c[10], c[11]));
    out[3 * i] = q.x;
    out[3 * i + 1] = q.y;
    out[3 * i + 2] = q.z;
  } else if (kind == 3) {  // tet containment: p v0 v1 v2 v3 (15) -> 1
    const double* c = in + 15 * i;
    out[i] = tet_contains(d3(c[0], c[1], c[2]), d3(c[3], c[4], c[5]), d3(c[6], c[7], c[8]),
                          d3(c[9], c[10], c[11]), d3(c[12], c[13], c[14]))
                 ? 1.0
                 : 0.0;
  } else if (kind == 4) {  // sqrt (1 -> 1)
    out[i] = sqrt(in[i]);
  } else if (kind == 5) {  // division a / b (2 -> 1)
    out[i] = in[2 * i] / in[2 * i + 1];
  }
}

}  // namespace

void launch_eval(int kind, int64_t n, const double* in, double* out, hipStream_t s)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_eval, grid1(n, 256), dim3(256), 0, s, kind, n, in, out);
}

// ---- build helpers --------------------------------------------------------

namespace {

__global__ void k_tri_boxes(const double* __restrict__ v9, int64_t n, double bump, double* box6)
{
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* v = v9 + 9 * i;
  for (int k = 0; k < 3; ++k) {
    double lo = fmin(fmin(v[k], v[3 + k]), v[6 + k]);
    double hi = fmax(fmax(v[k], v[3 + k]), v[6 + k]);
    box6[6 * i + k] = lo - bump;
    box6[6 * i + 3 + k] = hi + bump;
  }
}

__global__ void k_write_tris(const double* __restrict__ v9, const int32_t* __restrict__ face,
                             const int32_t* __restrict__ surf, const uint8_t* __restrict__ flip,
                             const int32_t* __restrict__ order, int64_t n, TriRec* out)
{
  int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (s >= n) return;
  int64_t p = order[s];
  TriRec r;
  for (int k = 0; k < 9; ++k) r.v[k] = v9[9 * p + k];
  r.face = face[p];
  const unsigned fb = tri_first_bits(d3(r.v[0], r.v[1], r.v[2]), d3(r.v[3], r.v[4], r.v[5]), d3(r.v[6], r.v[7], r.v[8]));
  r.surf2 = (surf[p] << TRI_SURF_SHIFT) | (int32_t)(fb << 1) | (flip[p] ? 1 : 0);
  out[s] = r;
}

// face_normal of every triangle record (mesh_manager_interface.cpp:216-220)
__global__ void k_tri_normals(const TriRec* __restrict__ tris, int64_t n, double* out)
{
  int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (s >= n) return;
  const TriRec& r = tris[s];
  const D3 nrm = face_normal(d3(r.v[0], r.v[1], r.v[2]), d3(r.v[3], r.v[4], r.v[5]), d3(r.v[6], r.v[7], r.v[8]));
  out[3 * s] = nrm.x;
  out[3 * s + 1] = nrm.y;
  out[3 * s + 2] = nrm.z;
}

}  // namespace

void launch_tri_normals(const TriRec* tris, int64_t n, double* out, hipStream_t s)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_tri_normals, grid1(n, 256), dim3(256), 0, s, tris, n, out);
}

void launch_tri_boxes(const double* verts9, int64_t n, double bump, double* box6, hipStream_t s)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_tri_boxes, grid1(n, 256), dim3(256), 0, s, verts9, n, bump, box6);
}

void launch_write_tris(const double* verts9, const int32_t* face, const int32_t* surf, const uint8_t* flip,
                       const int32_t* order, int64_t n, TriRec* out, hipStream_t s)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_write_tris, grid1(n, 256), dim3(256), 0, s, verts9, face, surf, flip, order, n, out);
}

}  // namespace xdgh
