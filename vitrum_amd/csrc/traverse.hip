// traverse.hip -- closest-hit and any-hit TLAS->BLAS traversal for gfx950.
//
// Semantics are those of the reference's traversal, so hit records are
// bit-identical to it:
//   traceTlasClosest / traceTlasAny  packages/shared-bvh/src/wgsl/tlasSceneHitTraversal.wgsl.ts:92-269
//   pt-webgpu instance augmentation  packages/pt-webgpu/src/wgsl/pathTrace/intersection.wgsl.ts:31-152
//   traceMeshBvh                     packages/pt-webgpu/src/wgsl/pathTrace/intersectionCore.wgsl.ts:461-596
//   watertight triangle test         packages/shared-bvh/src/opticalWatertightTriangle.ts:98-220
//   safeInvDir / slab test           packages/shared-bvh/src/wgsl/bvhIntersect.wgsl.ts:86-111,
//                                    intersectionCore.wgsl.ts:24-31
// Every float operation rounds once (built with -ffp-contract=off and
// correctly rounded division and square root).
//
// Design (MI355X):
//  * wide_kernel walks Node128 trees (four child boxes per node); scenes
//    whose Node128 stack bound is too deep or that hold no instance, and the
//    work counters, take trace_kernel.
//  * Node64 BVH2 nodes: the two child boxes sit in the parent, so a node
//    expansion is one 64-byte load and two slab tests.  The traversal order
//    is the reference's left-first depth-first order; a child's entry
//    distance is kept on the stack and re-checked against the current best
//    when it is popped, which is exactly the reference's pop-time cull.
//  * Persistent waves: each wave pulls rays from a global counter.  Lanes that
//    finish are refilled together once enough of the wave is idle: a ballot
//    of idle lanes, one atomicAdd per refill, and a prefix count (mbcnt) to
//    hand out consecutive ray indices.  A launch with fewer rays than 64 per
//    resident wave hands each wave at most its even share, so small batches
//    (late bounces, training paths) occupy every wave slot of every SIMD and
//    the dependent node loads of one wave hide behind the others'.
//  * One combined TLAS+BLAS stack per lane in LDS (entry-major so a wave's
//    accesses at equal depth hit 64 distinct banks), spilling the rare deep
//    entries to a per-thread global area.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "traverse.h"
#include "cwbvh.h"
#include "fast_div.h"

namespace vtk {

constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kEmpty = 0x80000000u;
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kMiss = 0xFFFFFFFFu;
// Deferred per-lane operations of the traversal loop.
constexpr uint32_t kPendNone = 0, kPendLeaf = 1, kPendEnter = 2, kPendExit = 3;

__device__ __forceinline__ float u2f(uint32_t u) { return __uint_as_float(u); }
__device__ __forceinline__ uint32_t f2u(float f) { return __float_as_uint(f); }
__device__ __forceinline__ float safe_max() { return __uint_as_float(0x7F7FFFFDu); }  // 3.402823e38
__device__ __forceinline__ float inf_const() { return __uint_as_float(0x7F7FFFFFu); }  // 3.402823466e38

__device__ __forceinline__ float fabs_(float x) { return __builtin_fabsf(x); }
__device__ __forceinline__ bool finite_(float x) { return __builtin_isfinite(x); }
__device__ __forceinline__ bool nan_(float x) { return __builtin_isnan(x); }
// Math.max: NaN-propagating (the TS mirror's semantics).
__device__ __forceinline__ float jmax(float a, float b) {
  return (nan_(a) || nan_(b)) ? __builtin_nanf("") : (a > b ? a : b);
}
__device__ __forceinline__ float max3abs(float x, float y, float z) {
  return jmax(fabs_(x), jmax(fabs_(y), fabs_(z)));
}
__device__ __forceinline__ float sel3(int k, float x, float y, float z) {
  return k == 0 ? x : (k == 1 ? y : z);
}

// Clang vector types travel in registers through the (rare) out-of-line
// calls below; plain structs would be passed through scratch memory.
typedef float V3 __attribute__((ext_vector_type(3)));
typedef float F4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ V3 v3(float x, float y, float z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 sub(V3 a, V3 b) { return V3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ float dot3(V3 a, V3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }

// ---------------------------------------------------------------------------
// Watertight triangle test (opticalWatertightTriangle.ts:15-220)
// ---------------------------------------------------------------------------

__device__ __forceinline__ float edge_fn(float ax, float ay, float bx, float by) {
  if (ax == bx && ay == by) return 0.0f;
  const bool ordered = ax < bx || (ax == bx && ay < by);
  const float fx = ordered ? ax : bx, fy = ordered ? ay : by;
  const float sx = ordered ? bx : ax, sy = ordered ? by : ay;
  const float canonical = fx * sy - fy * sx;
  return ordered ? canonical : -canonical;
}

__device__ __forceinline__ float ray_param_inl(V3 o, V3 dir, V3 p) {
  const V3 delta = sub(p, o);
  const float ds = max3abs(delta.x, delta.y, delta.z);
  const float rs = max3abs(dir.x, dir.y, dir.z);
  if (!(rs > 0.0f) || !finite_(rs) || !finite_(ds)) return -1.0f;
  if (!(ds > 0.0f)) return 0.0f;
  const V3 d = v3(dir.x / rs, dir.y / rs, dir.z / rs);
  const V3 q = v3(delta.x / ds, delta.y / ds, delta.z / ds);
  const float num = (q.x * d.x + q.y * d.y) + q.z * d.z;
  const float den = (d.x * d.x + d.y * d.y) + d.z * d.z;
  return (num / den) * (ds / rs);
}

__device__ __noinline__ float ray_param(V3 o, V3 dir, V3 p) { return ray_param_inl(o, dir, p); }

__device__ __forceinline__ bool lex_before(V3 a, V3 b) {
  return a.x < b.x || (a.x == b.x && (a.y < b.y || (a.y == b.y && a.z < b.z)));
}

// Returns (t, point) of an edge hit in registers.
__device__ __noinline__ F4 edge_ray_param(V3 o, V3 dir, V3 fi, V3 si, float fpx, float fpy, float spx,
                                          float spy) {
  const bool ordered = lex_before(fi, si);
  const V3 f = ordered ? fi : si, s = ordered ? si : fi;
  const float ax = ordered ? fpx : spx, ay = ordered ? fpy : spy;
  const float bx = ordered ? spx : fpx, by = ordered ? spy : fpy;
  const float ddx = bx - ax, ddy = by - ay;
  float interp;
  if (fabs_(ddx) >= fabs_(ddy)) {
    if (ddx == 0.0f) return F4{-1.0f, 0.0f, 0.0f, 0.0f};
    interp = -ax / ddx;
  } else {
    if (ddy == 0.0f) return F4{-1.0f, 0.0f, 0.0f, 0.0f};
    interp = -ay / ddy;
  }
  const V3 point = v3(f.x + interp * (s.x - f.x), f.y + interp * (s.y - f.y), f.z + interp * (s.z - f.z));
  return F4{ray_param(o, dir, point), point.x, point.y, point.z};
}

struct TriHit {
  float t;
  float u, v;  // bary.y, bary.z
  V3 point;
  bool front;  // side > 0: the ray meets the authored front face
};

// Ray-only part of the watertight test (opticalWatertightTriangle.ts:106-124):
// the dominant axis permutation and shear, computed once per ray per instance.
struct WtRay {
  float ds;          // max |dir| component
  float sx, sy, sz;  // shear constants
  uint32_t perm;     // kx | ky << 2 | kz << 4; 0xFFFFFFFF = invalid direction
};

__device__ __forceinline__ WtRay wt_setup(V3 dir) {
  WtRay w;
  w.ds = max3abs(dir.x, dir.y, dir.z);
  if (!(w.ds > 0.0f) || !finite_(w.ds)) {
    w.perm = 0xFFFFFFFFu;
    w.sx = w.sy = w.sz = 0.0f;
    return w;
  }
  const V3 d = v3(dir.x / w.ds, dir.y / w.ds, dir.z / w.ds);
  int kz = fabs_(d.y) > fabs_(d.x) ? 1 : 0;
  if (fabs_(d.z) > fabs_(sel3(kz, d.x, d.y, d.z))) kz = 2;
  int kx = kz == 2 ? 0 : kz + 1;
  int ky = kx == 2 ? 0 : kx + 1;
  const float dkz = sel3(kz, d.x, d.y, d.z);
  if (dkz < 0.0f) {
    const int t = kx;
    kx = ky;
    ky = t;
  }
  w.sx = sel3(kx, d.x, d.y, d.z) / dkz;
  w.sy = sel3(ky, d.x, d.y, d.z) / dkz;
  w.sz = 1.0f / dkz;
  w.perm = (uint32_t)kx | ((uint32_t)ky << 2) | ((uint32_t)kz << 4);
  return w;
}

// Rare tail of an in-window hit (opticalWatertightTriangle.ts:164-220): the
// authored-normal side test.  Returns 0 for a rejected hit, 1 for the front
// face (side > 0), -1 for the back face.
__device__ __forceinline__ int wt_side_inl(V3 dir, float ds, V3 a, V3 b, V3 c) {
  const V3 e1r = sub(b, a), e2r = sub(c, a);
  const float es = jmax(max3abs(e1r.x, e1r.y, e1r.z), max3abs(e2r.x, e2r.y, e2r.z));
  if (!(es > 0.0f) || !finite_(es)) return 0;
  const V3 s1 = v3(e1r.x / es, e1r.y / es, e1r.z / es);
  const V3 s2 = v3(e2r.x / es, e2r.y / es, e2r.z / es);
  const V3 nr = v3(s1.y * s2.z - s1.z * s2.y, s1.z * s2.x - s1.x * s2.z, s1.x * s2.y - s1.y * s2.x);
  const float ns = max3abs(nr.x, nr.y, nr.z);
  if (!(ns > 0.0f) || !finite_(ns)) return 0;
  const V3 nd = v3(nr.x / ns, nr.y / ns, nr.z / ns);
  const float nl = __builtin_sqrtf((nd.x * nd.x + nd.y * nd.y) + nd.z * nd.z);
  if (!(nl > 0.0f) || !finite_(nl)) return 0;
  const V3 n = v3(nd.x / nl, nd.y / nl, nd.z / nl);
  const V3 d = v3(dir.x / ds, dir.y / ds, dir.z / ds);
  const float side = -((d.x * n.x + d.y * n.y) + d.z * n.z);
  if (side == 0.0f || !finite_(side)) return 0;
  return side > 0.0f ? 1 : -1;
}

__device__ __noinline__ int wt_side(V3 dir, float ds, V3 a, V3 b, V3 c) { return wt_side_inl(dir, ds, a, b, c); }

// Returns true and fills h when the triangle is hit with lo < t < hi (or
// t <= hi when `incl_hi`), where lo = tmin (also the predicate's exclusive
// minimum) and hi the current bound.  Work that can only turn an
// out-of-window hit into a miss is skipped for out-of-window hits, which
// leaves the accepted set unchanged.
__device__ __forceinline__ bool tri_test(V3 o, V3 dir, const WtRay& w, V3 a, V3 b, V3 c, float tmin,
                                         float hi, bool incl_hi, TriHit& h) {
  if (w.perm == 0xFFFFFFFFu || nan_(tmin)) return false;
  const int kx = w.perm & 3, ky = (w.perm >> 2) & 3, kz = w.perm >> 4;
  const V3 pa = sub(a, o), pb = sub(b, o), pc = sub(c, o);
  const float paz = sel3(kz, pa.x, pa.y, pa.z), pbz = sel3(kz, pb.x, pb.y, pb.z),
              pcz = sel3(kz, pc.x, pc.y, pc.z);
  const float apx = sel3(kx, pa.x, pa.y, pa.z) - w.sx * paz, apy = sel3(ky, pa.x, pa.y, pa.z) - w.sy * paz;
  const float bpx = sel3(kx, pb.x, pb.y, pb.z) - w.sx * pbz, bpy = sel3(ky, pb.x, pb.y, pb.z) - w.sy * pbz;
  const float cpx = sel3(kx, pc.x, pc.y, pc.z) - w.sx * pcz, cpy = sel3(ky, pc.x, pc.y, pc.z) - w.sy * pcz;
  const float e0 = edge_fn(bpx, bpy, cpx, cpy);
  const float e1 = edge_fn(cpx, cpy, apx, apy);
  const float e2 = edge_fn(apx, apy, bpx, bpy);
  const float det = (e0 + e1) + e2;
  if (det == 0.0f || !finite_(det)) return false;
  const bool positive = det > 0.0f;
  const float n0 = positive ? e0 : -e0, n1 = positive ? e1 : -e1, n2 = positive ? e2 : -e2;
  if (n0 < 0.0f || n1 < 0.0f || n2 < 0.0f) return false;
  const float scaled_t = (e0 * (paz * w.sz) + e1 * (pbz * w.sz)) + e2 * (pcz * w.sz);
  float t = (scaled_t / det) / w.ds;
  V3 point = v3(0, 0, 0);
  const int zc = (n0 == 0.0f) + (n1 == 0.0f) + (n2 == 0.0f);
  if (zc != 0) {
    if (zc >= 2) {
      if (n0 != 0.0f) point = a, t = ray_param(o, dir, point);
      if (n1 != 0.0f) point = b, t = ray_param(o, dir, point);
      if (n2 != 0.0f) point = c, t = ray_param(o, dir, point);
    } else {
      F4 ep;
      if (n0 == 0.0f)
        ep = edge_ray_param(o, dir, b, c, bpx, bpy, cpx, cpy);
      else if (n1 == 0.0f)
        ep = edge_ray_param(o, dir, c, a, cpx, cpy, apx, apy);
      else
        ep = edge_ray_param(o, dir, a, b, apx, apy, bpx, bpy);
      t = ep.x;
      point = v3(ep.y, ep.z, ep.w);
    }
  }
  const float lo = tmin > 0.0f ? tmin : 0.0f;
  if (!(t > lo) || !finite_(t)) return false;
  if (!(t > tmin && (t < hi || (incl_hi && t == hi)))) return false;  // traversal acceptance window
  // opticalWatertightTriangle.ts:164-219: authored-normal side test, then
  // barycentrics and the canonical hit point.
  const int side = wt_side(dir, w.ds, a, b, c);
  if (side == 0) return false;
  h.front = side > 0;
  h.t = t;
  h.u = e1 / det;
  h.v = e2 / det;
  if (zc == 0) {
    point = v3(a.x + (h.u * (b.x - a.x) + h.v * (c.x - a.x)), a.y + (h.u * (b.y - a.y) + h.v * (c.y - a.y)),
               a.z + (h.u * (b.z - a.z) + h.v * (c.z - a.z)));
  }
  h.point = point;
  return true;
}

// ---------------------------------------------------------------------------
// Slab test, transforms (bvhIntersect.wgsl.ts:86-111; intersectionCore.wgsl.ts:24-83)
// ---------------------------------------------------------------------------

__device__ __forceinline__ float safe_inv(float v) {
  const float m = safe_max();
  if (v == 0.0f) return v >= 0.0f ? m : -m;
  const float r = 1.0f / v;
  return r < -m ? -m : (r > m ? m : r);
}

// Computes tNear and returns the bound-independent part of the test:
// !(tNear > tFar || tFar < tMin).
__device__ __forceinline__ bool slab(V3 o, V3 inv, float mnx, float mny, float mnz, float mxx,
                                     float mxy, float mxz, float tmin, float& tnear) {
  const float t1x = (mnx - o.x) * inv.x, t1y = (mny - o.y) * inv.y, t1z = (mnz - o.z) * inv.z;
  const float t2x = (mxx - o.x) * inv.x, t2y = (mxy - o.y) * inv.y, t2z = (mxz - o.z) * inv.z;
  const float tn = fmaxf(fmaxf(fminf(t1x, t2x), fminf(t1y, t2y)), fminf(t1z, t2z));
  const float tf = fminf(fminf(fmaxf(t1x, t2x), fmaxf(t1y, t2y)), fmaxf(t1z, t2z));
  tnear = tn;
  return !(tn > tf || tf < tmin);
}

__device__ __forceinline__ V3 xform_point(float4 c0, float4 c1, float4 c2, float4 c3, V3 p) {
  const float rx = ((c0.x * p.x + c1.x * p.y) + c2.x * p.z) + c3.x;
  const float ry = ((c0.y * p.x + c1.y * p.y) + c2.y * p.z) + c3.y;
  const float rz = ((c0.z * p.x + c1.z * p.y) + c2.z * p.z) + c3.z;
  const float rw = ((c0.w * p.x + c1.w * p.y) + c2.w * p.z) + c3.w;
  const float s = fmaxf(fmaxf(fabs_(rx), fabs_(ry)), fmaxf(fabs_(rz), fabs_(rw)));
  if (!(s > 0.0f) || s > safe_max()) return v3(0, 0, 0);
  const float qx = rx / s, qy = ry / s, qz = rz / s, qw = rw / s;
  if (qw == 0.0f) return v3(0, 0, 0);
  const V3 q = v3(qx / qw, qy / qw, qz / qw);
  if (nan_(q.x) || nan_(q.y) || nan_(q.z) || fabs_(q.x) > safe_max() || fabs_(q.y) > safe_max() ||
      fabs_(q.z) > safe_max())
    return v3(0, 0, 0);
  return q;
}

__device__ __forceinline__ V3 safe_normalize(V3 v) {
  const float s = fmaxf(fabs_(v.x), fmaxf(fabs_(v.y), fabs_(v.z)));
  if (!(s > 0.0f) || s > safe_max()) return v3(0, 1, 0);
  const V3 q = v3(v.x / s, v.y / s, v.z / s);
  const float len = __builtin_sqrtf((q.x * q.x + q.y * q.y) + q.z * q.z);
  return v3(q.x / len, q.y / len, q.z / len);
}

__device__ __forceinline__ V3 xform_dir(float4 c0, float4 c1, float4 c2, V3 d) {
  return safe_normalize(v3((c0.x * d.x + c1.x * d.y) + c2.x * d.z, (c0.y * d.x + c1.y * d.y) + c2.y * d.z,
                           (c0.z * d.x + c1.z * d.y) + c2.z * d.z));
}

// ---------------------------------------------------------------------------
// Persistent traversal kernel
// ---------------------------------------------------------------------------

// Single-step persistent loop: each iteration a lane pops (with the
// reference's pop-time cull), expands one Node64 (two child boxes), tests
// one leaf's triangles or enters / leaves one instance.
//
// Child order.  The reference visits the left child first.  With
// near_first = 1 (closest hit only) the child with the smaller entry distance
// is visited first inside each BLAS, and equal triangle distances are
// resolved as the reference's order resolves them (the lower reordered index
// wins); instances are still visited in the reference's TLAS order, because
// with coplanar geometry in different instances the reference's choice
// depends on that order through the rounding of the instance transforms.
// near_first = 2 also orders the TLAS by distance.  The reference's choice
// between instances depends on its order only through near-ties: an
// instance's local search is bounded by the best world distance found so far,
// mapped into the instance's space, and where two instances' hits lie within
// the rounding of that mapping the earlier-visited one can exclude the other.
// So in this mode every world bound is widened by a margin (2^-13 of the
// distance plus the origin's magnitude, far above the transforms' rounding),
// which keeps every hit near the current best visible, and a lane that sees
// two instances' hits within that margin of each other walks its ray again in
// the reference's TLAS order.  Without such a near-tie the minimum world
// distance is what any order finds, so the hit records equal the reference's.
// Node culling stays `tNear > bound` (equal distances are still visited).  The
// counting variant always uses the reference order, so its work counts are
// the reference's.
template <bool ANY, bool COUNT, bool MULTI, uint32_t BLOCK, uint32_t LDS_DEPTH>
// Register budget: four waves per SIMD (128 VGPRs; with the 20-entry LDS
// stack, 8 blocks of 128 fit a CU), which beats three waves without spills.
__global__ __launch_bounds__(BLOCK, 4) void trace_kernel(TraceParams p) {
  // Per-lane stack: LDS_DEPTH entries in LDS (entry-major, so a wave's
  // accesses at equal depth touch 64 distinct banks), deeper entries in a
  // per-thread global spill area.  The shared array is indexed directly so the
  // compiler emits ds_* instructions, and the spill area is accessed as 64-bit
  // words, a different type, so the two branches cannot be merged into one
  // generic (flat) access with the latency of global memory.
  __shared__ uint2 lds_stack[LDS_DEPTH * BLOCK];
  const uint32_t tid = threadIdx.x;
  const size_t spill_stride = (size_t)gridDim.x * BLOCK, gtid = (size_t)blockIdx.x * BLOCK + threadIdx.x;
  unsigned long long* __restrict__ spill = reinterpret_cast<unsigned long long*>(p.spill);
  auto stk_store = [&](uint32_t i, uint2 v) {
    if (i < LDS_DEPTH)
      lds_stack[i * BLOCK + tid] = v;
    else
      spill[(i - LDS_DEPTH) * spill_stride + gtid] = (unsigned long long)v.x | ((unsigned long long)v.y << 32);
  };
  auto stk_load = [&](uint32_t i) -> uint2 {
    if (i < LDS_DEPTH) return lds_stack[i * BLOCK + tid];
    const unsigned long long w = spill[(i - LDS_DEPTH) * spill_stride + gtid];
    return make_uint2((uint32_t)w, (uint32_t)(w >> 32));
  };
  // Scene of the current ray: the launch's scene, or (batched) the one whose
  // ray range holds the ray, looked up when the lane takes a new ray.
  const float4* __restrict__ blas = p.scene.blas_nodes;
  const float4* __restrict__ tlas = p.scene.tlas_nodes;
  const float4* __restrict__ tris = p.scene.tris;
  const float4* __restrict__ insts = p.scene.instances;
  uint32_t tlas_root = p.scene.tlas_root, tlas_count = p.scene.tlas_node_count;
  const uint32_t lane = __lane_id();
  const uint64_t lane_below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const bool near = !ANY && !COUNT && p.near_first != 0u;        // inside BLASes
  const bool near_tlas = !ANY && !COUNT && p.near_first == 2u;  // also across instances

  const uint32_t n_rays = p.n_ptr ? *p.n_ptr : p.n;
  const uint32_t n_waves = gridDim.x * (BLOCK / 64u);
  const uint32_t take_cap = max(1u, min(64u, n_rays / n_waves + (n_rays % n_waves != 0u)));
  bool active = false;
  uint32_t ray_idx = 0;
  // World ray and best hit.
  V3 ro{}, rd{}, rinv{};
  float tmin = 0, tmax = 0, best = 0, bu = 0, bv = 0;
  V3 bpos{};
  uint32_t bprim = 0, binst = kMiss;
  bool bfront = false;  // the best hit is on the front face (world orientation)
  // near_first = 2: the lane walks in the reference's TLAS order (after a
  // near-tie), a near-tie was seen, and the magnitude of the ray origin.
  bool ref_order = false, recheck = false;
  float rscale = 0.0f;
  // Instance-local state.
  V3 lo{}, ld{}, linv{}, lpos{};
  WtRay lw{};
  bool lw_ready = false;
  float ltmin = 0, lbest = 0, lu = 0, lv = 0;
  uint32_t lprim = 0, inst_id = 0;
  bool lhit = false, lfront = false;
  bool lmirror = false;  // the instance's local-to-world map reverses orientation
  uint32_t slot = 0, slot_end = 0, enter_slot = 0;
  uint32_t level = 0, cur = kNone, sp = 0, blas_base = 0;
  uint32_t pend = 0;  // pending deferred operation (kPend*)
  uint32_t c_blas = 0, c_tri = 0, c_tlas = 0, c_inst = 0;

  // The world-space bound of the TLAS walk: the best distance, widened by the
  // near-tie margin while the lane orders the TLAS by distance.
  auto world_bound = [&]() -> float {
    if (ANY) return tmax;
    if (near_tlas && !ref_order && binst != kMiss) return best + (best + rscale) * 0x1p-13f;
    return best;
  };

  auto enter_instance = [&](uint32_t s) {
    const float4* ir = insts + 9 * (size_t)s;
    const float4 c0 = ir[0], c1 = ir[1], c2 = ir[2], c3 = ir[3];
    const uint4 meta = *reinterpret_cast<const uint4*>(ir + 8);
    lo = xform_point(c0, c1, c2, c3, ro);
    ld = xform_dir(c0, c1, c2, rd);
    linv = v3(safe_inv(ld.x), safe_inv(ld.y), safe_inv(ld.z));
    lw_ready = false;  // the watertight set-up waits for the first leaf
    const V3 start = v3(ro.x + rd.x * tmin, ro.y + rd.y * tmin, ro.z + rd.z * tmin);
    ltmin = fmaxf(dot3(sub(xform_point(c0, c1, c2, c3, start), lo), ld), 0.0f);
    // Closest: localTMax starts at INFINITY; any-hit: at the ray's tMax
    // (tlasSceneHitTraversal.wgsl.ts:103-108 and :168-173).
    const float bound = world_bound();
    float ltmax = ANY ? tmax : inf_const();
    if (bound < inf_const() * 0.5f) {
      const V3 end = v3(ro.x + rd.x * bound, ro.y + rd.y * bound, ro.z + rd.z * bound);
      ltmax = fmaxf(dot3(sub(xform_point(c0, c1, c2, c3, end), lo), ld), ltmin);
    }
    lbest = ltmax;
    lhit = false;
    lfront = false;
    lmirror = meta.w != 0u;
    inst_id = meta.y;
    level = 1;
    blas_base = sp;
    cur = meta.x;
    if (COUNT) ++c_inst;
  };

  auto finalize_instance = [&]() {
    if (!ANY && lhit && lbest > ltmin) {
      const float4* ir = insts + 9 * (size_t)slot + 4;
      const V3 w = xform_point(ir[0], ir[1], ir[2], ir[3], lpos);
      const float wd = dot3(sub(w, ro), rd);
      if (near_tlas && !ref_order && binst != kMiss && fabsf(wd - best) <= (best + rscale) * 0x1p-13f)
        recheck = true;
      if (wd > tmin && wd < best) {
        best = wd;
        bpos = w;
        bprim = lprim;
        binst = inst_id;
        bu = lu;
        bv = lv;
        bfront = lfront != lmirror;
      }
    }
  };

  auto finish = [&](bool occluded) {
    if (ANY) {
      p.occluded[ray_idx] = occluded ? 1u : 0u;
    } else {
      const bool hit = binst != kMiss;
      uint32_t* h = p.hits + 5 * (size_t)ray_idx;
      h[0] = hit ? bprim : kMiss;
      h[1] = hit ? binst : kMiss;
      h[2] = hit ? f2u(best) : 0x7F800000u;
      h[3] = hit ? f2u(bu) : 0u;
      h[4] = hit ? f2u(bv) : 0u;
      if (p.hit_pos) {
        float* hp = p.hit_pos + 3 * (size_t)ray_idx;
        hp[0] = bpos.x;
        hp[1] = bpos.y;
        hp[2] = bpos.z;
      }
    }
    if (COUNT) p.counts[ray_idx] = make_uint4(c_blas, c_tri, c_tlas, c_inst);
    active = false;
  };

  auto push = [&](uint32_t ref, float tn) {
    if (sp >= kStackCapacity) {
      atomicOr(p.error, kErrorStack);
      return false;
    }
    stk_store(sp++, make_uint2(ref, f2u(tn)));
    return true;
  };

  // Once a refill hands out indices past the last ray the supply is gone for
  // good; the wave then only finishes its active lanes (no further atomics on
  // the shared counter, which every finishing wave would otherwise hit).
  // The first fill is static -- wave w takes rays [w * take_cap, (w + 1) *
  // take_cap) -- so a launch starts without every wave hitting the shared
  // counter at once (and an empty launch touches it not at all); the counter
  // hands out the rays after that range.
  bool exhausted = false, first_fill = true;
  const uint32_t wave_id = blockIdx.x * (BLOCK / 64u) + threadIdx.x / 64u;
  const uint32_t static_end = n_waves * take_cap;
  for (;;) {
    // ---- wave-level refill: ballot idle lanes, one atomic, prefix ranks ----
    const uint64_t idle = __ballot(!active);
    const uint32_t n_idle = (uint32_t)__popcll(idle);
    if (!exhausted && (n_idle >= p.refill_min || idle == __ballot(1))) {
      const uint32_t take = min(n_idle, take_cap);
      uint32_t base = 0;
      if (first_fill) {
        base = wave_id * take_cap;  // every lane is idle: take == take_cap
      } else {
        if (lane == 0) base = static_end + atomicAdd(p.counter, take);
        base = __shfl(base, 0);
      }
      first_fill = false;
      exhausted = base + take >= n_rays;
      const uint32_t rank = (uint32_t)__popcll(idle & lane_below);
      if (!active && rank < take) {
        const uint32_t idx = base + rank;
        if (idx < n_rays) {
          ray_idx = idx;
          if (MULTI) {
            uint32_t lo_s = 0, hi_s = p.scene_count;
            while (lo_s + 1u < hi_s) {
              const uint32_t mid = (lo_s + hi_s) >> 1;
              if (p.scene_offsets[mid] <= idx) lo_s = mid; else hi_s = mid;
            }
            const DeviceScene& S = p.scenes[lo_s];
            blas = S.blas_nodes;
            tlas = S.tlas_nodes;
            tris = S.tris;
            insts = S.instances;
            tlas_root = S.tlas_root;
            tlas_count = S.tlas_node_count;
          }
          const float4 a = p.rays[2 * (size_t)idx], b = p.rays[2 * (size_t)idx + 1];
          ro = v3(a.x, a.y, a.z);
          tmin = a.w;
          rd = v3(b.x, b.y, b.z);
          tmax = b.w;
          rinv = v3(safe_inv(rd.x), safe_inv(rd.y), safe_inv(rd.z));
          rscale = fmaxf(fabs_(ro.x), fmaxf(fabs_(ro.y), fabs_(ro.z)));
          ref_order = false;
          recheck = false;
          best = tmax;
          binst = kMiss;
          bprim = 0;
          bu = bv = 0;
          level = 0;
          sp = 0;
          pend = kPendNone;
          cur = tlas_count ? tlas_root : kNone;
          if (COUNT) c_blas = c_tri = c_tlas = c_inst = 0;
          active = true;
          if (cur == kNone) finish(false);  // no TLAS: fail closed
        }
      }
    }
    if (!__any(active)) {
      // A scene without instances closes its rays in the refill: the wave is
      // done only when the supply is.
      if (exhausted) break;
      continue;
    }

    for (uint32_t step = 0; step < p.steps; ++step) {
      // ---- deferred expensive work, shared by the lanes that need it ----
      // A lane whose next operation is an instance exit (merge of the local
      // hit), an instance entry (ray transform) or a BLAS leaf (triangle
      // tests) waits until `defer_min` lanes of the wave -- or half of its
      // active lanes, when fewer are left -- need the same operation, or
      // until no lane has cheap node work left; each lane still performs
      // exactly its own sequence of operations.
      const uint64_t m_exit = __ballot(active && pend == kPendExit);
      const uint64_t m_enter = __ballot(active && pend == kPendEnter);
      const uint64_t m_leaf = __ballot(active && pend == kPendLeaf);
      const uint64_t m_cheap = __ballot(active && pend == kPendNone);
      if ((m_exit | m_enter | m_leaf | m_cheap) == 0ull) break;
      const bool all = m_cheap == 0ull;
      const uint32_t n_act = (uint32_t)__popcll(m_exit | m_enter | m_leaf | m_cheap);
      const uint32_t dm = min(p.defer_min, (n_act + 1u) >> 1);
      if (m_exit && (all || (uint32_t)__popcll(m_exit) >= dm) && active && pend == kPendExit) {
        finalize_instance();
        level = 0;
        if (++slot < slot_end) {
          enter_slot = slot;
          pend = kPendEnter;
        } else {
          pend = kPendNone;
        }
      }
      if (m_enter && (all || (uint32_t)__popcll(m_enter) >= dm) && active && pend == kPendEnter) {
        slot = enter_slot;
        enter_instance(slot);
        pend = kPendNone;
      }
      if (m_leaf && (all || (uint32_t)__popcll(m_leaf) >= dm)) {
        const bool mine = active && pend == kPendLeaf;
        uint32_t cnt = 0, tfirst = 0;
        if (mine) {
          cnt = (cur >> 27) & 15u;
          tfirst = cur & 0x07FFFFFFu;
          cur = kNone;
          pend = kPendNone;
          if (!lw_ready) {
            lw = wt_setup(ld);
            lw_ready = true;
          }
        }
        if (COUNT) {
          // Work counting: each lane tests its own leaf, one triangle at a time.
          for (uint32_t i = 0; i < cnt; ++i) {
            const uint32_t t = tfirst + i;
            const float4* tr = tris + 3 * (size_t)t;
            const float4 w0 = tr[0], w1 = tr[1], w2 = tr[2];
            ++c_tri;
            TriHit h;
            if (tri_test(lo, ld, lw, v3(w0.x, w0.y, w0.z), v3(w0.w, w1.x, w1.y), v3(w1.z, w1.w, w2.x), ltmin,
                         lbest, near && lhit, h)) {
              if (h.t == lbest && lhit && !(t < lprim)) continue;  // equal t: lower index wins
              lhit = true;
              lbest = h.t;
              lprim = t;
              lu = h.u;
              lv = h.v;
              lpos = h.point;
              lfront = h.front;
            }
          }
        } else {
          // The leaves' (ray, triangle) pairs are spread over all 64 lanes,
          // 64 pairs per round: pair q belongs to the lane whose exclusive
          // prefix of triangle counts is the largest one <= q.  Every pair is
          // tested against its ray's state at the start of the round, then
          // each ray keeps the lexicographic minimum (t, triangle index) of
          // its pairs -- exactly what testing them one after another gives
          // (a later triangle replaces the best only with a smaller t or, at
          // equal t, a lower index), so the hit records are unchanged.
          uint32_t excl = 0, total = 0;
#pragma unroll
          for (uint32_t b = 0; b < 4; ++b) {  // counts are below 16: one ballot per bit
            const uint64_t m = __ballot((cnt >> b) & 1u);
            excl += (uint32_t)__popcll(m & lane_below) << b;
            total += (uint32_t)__popcll(m) << b;
          }
          const uint32_t incl = excl + cnt;
          bool occl = false;
          for (uint32_t base = 0; base < total; base += 64u) {
            const uint32_t q = base + lane;
            const bool work = q < total;
            // owner: the lowest lane whose inclusive prefix exceeds q
            uint32_t o_lo = 0, o_hi = 63;
#pragma unroll
            for (uint32_t it = 0; it < 6; ++it) {
              const uint32_t mid = (o_lo + o_hi) >> 1;
              if ((uint32_t)__shfl((int)incl, (int)mid) > q) o_hi = mid; else o_lo = mid + 1u;
            }
            const int o = (int)min(o_lo, 63u);
            const uint32_t o_first = (uint32_t)__shfl((int)tfirst, o), o_excl = (uint32_t)__shfl((int)excl, o);
            const V3 wo = v3(__shfl(lo.x, o), __shfl(lo.y, o), __shfl(lo.z, o));
            const V3 wd = v3(__shfl(ld.x, o), __shfl(ld.y, o), __shfl(ld.z, o));
            WtRay ww;
            ww.ds = __shfl(lw.ds, o);
            ww.sx = __shfl(lw.sx, o);
            ww.sy = __shfl(lw.sy, o);
            ww.sz = __shfl(lw.sz, o);
            ww.perm = (uint32_t)__shfl((int)lw.perm, o);
            const float w_tmin = __shfl(ltmin, o), w_hi = __shfl(lbest, o);
            const bool w_incl = __shfl((int)(near && lhit), o) != 0;
            const bool w_mirror = __shfl((int)lmirror, o) != 0;
            uint32_t kt = 0xFFFFFFFFu, ki = 0xFFFFFFFFu, kl = lane;
            TriHit h;
            h.t = h.u = h.v = 0.0f;
            h.point = v3(0, 0, 0);
            h.front = false;
            // A batched launch can hold rays of different scenes in one wave:
            // the pair's triangle is in its owner's scene.
            const float4* otris = tris;
            if (MULTI) {
              const uint64_t tp = (uint64_t)(uintptr_t)tris;
              const uint32_t p_lo = (uint32_t)__shfl((int)(uint32_t)tp, o);
              const uint32_t p_hi = (uint32_t)__shfl((int)(uint32_t)(tp >> 32), o);
              otris = reinterpret_cast<const float4*>((uintptr_t)(((uint64_t)p_hi << 32) | p_lo));
            }
            if (work) {
              const uint32_t t = o_first + (q - o_excl);
              const float4* tr = otris + 3 * (size_t)t;
              const float4 w0 = tr[0], w1 = tr[1], w2 = tr[2];
              // Any hit through the path tracer's wrappers (traceAny /
              // traceSurfaceVisibility): a back face of a single-sided
              // material does not block.
              if (tri_test(wo, wd, ww, v3(w0.x, w0.y, w0.z), v3(w0.w, w1.x, w1.y), v3(w1.z, w1.w, w2.x), w_tmin,
                           w_hi, w_incl, h) &&
                  (!ANY || !p.sided || h.front != w_mirror || !(w2.y > 0.5f))) {
                kt = f2u(h.t);  // t > 0: the bit patterns order as the values
                ki = t;
              }
            }
            // Segmented minimum over each owner's run of lanes (at most 15).
#pragma unroll
            for (uint32_t d = 1; d < 16; d <<= 1) {
              const uint32_t ot = (uint32_t)__shfl_down((int)kt, d), oi = (uint32_t)__shfl_down((int)ki, d);
              const uint32_t ol = (uint32_t)__shfl_down((int)kl, d);
              const int oo = __shfl_down(o, d);
              if (lane + d < 64u && oo == o && (ot < kt || (ot == kt && oi < ki))) {
                kt = ot;
                ki = oi;
                kl = ol;
              }
            }
            // Each ray reads its run's minimum (its run in this round starts at
            // lane max(excl, base) - base) and the winner's hit data.
            const bool here = mine && cnt > 0u && excl < base + 64u && incl > base;
            const int src = (int)((max(excl, base) - base) & 63u);
            const uint32_t rt = (uint32_t)__shfl((int)kt, src), ri = (uint32_t)__shfl((int)ki, src);
            const int rl = __shfl((int)kl, src);
            const float ru = __shfl(h.u, rl), rv = __shfl(h.v, rl);
            const V3 rp = v3(__shfl(h.point.x, rl), __shfl(h.point.y, rl), __shfl(h.point.z, rl));
            const bool rf = __shfl((int)h.front, rl) != 0;
            if (here && rt != 0xFFFFFFFFu) {
              if (ANY) {
                occl = true;
              } else {
                const float t = u2f(rt);
                if (!lhit || t < lbest || (t == lbest && ri < lprim)) {
                  lhit = true;
                  lbest = t;
                  lprim = ri;
                  lu = ru;
                  lv = rv;
                  lpos = rp;
                  lfront = rf;
                }
              }
            }
          }
          if (ANY && occl) finish(true);
        }
      }
      if (!active || pend != kPendNone) continue;
      // ---- cheap work: pop with the reference's pop-time cull, expand ----
      if (cur == kNone) {
        for (;;) {
          if (level == 1) {
            if (sp > blas_base) {
              const uint2 e = stk_load(--sp);
              if (!(u2f(e.y) > lbest)) {
                cur = e.x;
                break;
              }
              continue;
            }
            pend = kPendExit;  // BLAS exhausted
            break;
          }
          if (sp > 0) {
            const uint2 e = stk_load(--sp);
            if (!(u2f(e.y) > world_bound())) {
              cur = e.x;
              break;
            }
            continue;
          }
          if (recheck) {
            // A near-tie between instances: walk the ray again, from its
            // original interval, in the reference's TLAS order.
            const float4 a = p.rays[2 * (size_t)ray_idx], b = p.rays[2 * (size_t)ray_idx + 1];
            tmin = a.w;
            tmax = b.w;
            best = tmax;
            binst = kMiss;
            bprim = 0;
            bu = bv = 0.0f;
            level = 0;
            sp = 0;
            ref_order = true;
            recheck = false;
            cur = tlas_root;
            break;
          }
          // traceClosest (intersection.wgsl.ts:462-490): a back-face hit on a
          // single-sided material is not a surface; the trace starts again
          // with its distance as the exclusive lower bound, and ends as a
          // miss once that bound stops advancing or reaches tMax.
          if (!ANY && p.sided && binst != kMiss && !bfront && tris[3 * (size_t)bprim + 2].y > 0.5f) {
            if (best > tmin && best < tmax) {
              tmin = best;
              best = tmax;
              binst = kMiss;
              bprim = 0;
              bu = bv = 0.0f;
              level = 0;
              sp = 0;
              cur = tlas_root;
              break;
            }
            binst = kMiss;
          }
          finish(false);
          break;
        }
        if (!active || pend != kPendNone) continue;
      }
      if ((cur & kLeafBit) == 0) {
        // ---- interior: one Node64 load, two child boxes ----
        const float4* nd = (level ? blas : tlas) + 4 * (size_t)cur;
        const float4 q0 = nd[0], q1 = nd[1], q2 = nd[2], q3 = nd[3];
        const uint32_t ref_l = f2u(q3.x), ref_r = f2u(q3.y);
        const V3 o = level ? lo : ro;
        const V3 inv = level ? linv : rinv;
        const float tm = level ? ltmin : tmin;
        const float bound = level ? lbest : world_bound();
        float tn_l, tn_r;
        const bool pass_l = ref_l != kEmpty && slab(o, inv, q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, tm, tn_l);
        const bool pass_r = ref_r != kEmpty && slab(o, inv, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, tm, tn_r);
        if (COUNT) {
          const uint32_t tested = (ref_l != kEmpty) + (ref_r != kEmpty);
          if (level) c_blas += tested; else c_tlas += tested;
        }
        const bool take_l = pass_l && !(tn_l > bound), take_r = pass_r && !(tn_r > bound);
        if (take_l && take_r) {
          const bool right_first = (level ? near : (near_tlas && !ref_order)) && tn_r < tn_l;
          if (!push(right_first ? ref_l : ref_r, right_first ? tn_l : tn_r)) {
            finish(false);
            continue;
          }
          cur = right_first ? ref_r : ref_l;
        } else {
          cur = take_l ? ref_l : (take_r ? ref_r : kNone);
        }
      }
      // A leaf reached by the pop or the expansion becomes pending work.
      if (cur != kNone && (cur & kLeafBit)) {
        if (level == 0) {
          enter_slot = cur & 0x07FFFFFFu;
          slot_end = enter_slot + ((cur >> 27) & 15u);
          cur = kNone;
          pend = enter_slot < slot_end ? kPendEnter : kPendNone;
        } else {
          pend = kPendLeaf;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Operations with a shared denominator (fast_div.h)
// ---------------------------------------------------------------------------

using vtd::div_by;
using vtd::div_den;
using vtd::div_key;
using vtd::kDivNum;
using vtd::recip_of;

__device__ __forceinline__ V3 div_by(V3 a, float b, float y) {
  return v3(div_by(a.x, b, y), div_by(a.y, b, y), div_by(a.z, b, y));
}
__device__ __forceinline__ uint32_t div_key(V3 a) { return min(min(div_key(a.x), div_key(a.y)), div_key(a.z)); }

// xform_point, safe_normalize and safe_inv with the shared-denominator
// division; the general forms answer every operand outside its range.
__device__ __forceinline__ V3 xform_point_fast(float4 c0, float4 c1, float4 c2, float4 c3, V3 p) {
  const V3 r = v3(((c0.x * p.x + c1.x * p.y) + c2.x * p.z) + c3.x, ((c0.y * p.x + c1.y * p.y) + c2.y * p.z) + c3.y,
                  ((c0.z * p.x + c1.z * p.y) + c2.z * p.z) + c3.z);
  const float rw = ((c0.w * p.x + c1.w * p.y) + c2.w * p.z) + c3.w;
  const float s = fmaxf(fmaxf(fabs_(r.x), fabs_(r.y)), fmaxf(fabs_(r.z), fabs_(rw)));
  const float ys = recip_of(s);
  const float qw = div_by(rw, s, ys);
  const float sum = (r.x + r.y) + (r.z + rw);  // NaN when any of the four is
  if (__builtin_expect(!(div_den(s) && div_den(qw) && sum == sum && min(div_key(r), div_key(rw)) >= kDivNum), 0))
    return xform_point(c0, c1, c2, c3, p);
  return div_by(div_by(r, s, ys), qw, recip_of(qw));
}

__device__ __forceinline__ V3 xform_dir_fast(float4 c0, float4 c1, float4 c2, V3 d) {
  const V3 v = v3((c0.x * d.x + c1.x * d.y) + c2.x * d.z, (c0.y * d.x + c1.y * d.y) + c2.y * d.z,
                  (c0.z * d.x + c1.z * d.y) + c2.z * d.z);
  const float s = fmaxf(fabs_(v.x), fmaxf(fabs_(v.y), fabs_(v.z)));
  if (__builtin_expect(!(div_den(s) && div_key(v) >= kDivNum), 0)) return safe_normalize(v);
  const V3 q = div_by(v, s, recip_of(s));
  const float len = __builtin_sqrtf((q.x * q.x + q.y * q.y) + q.z * q.z);  // in [1, sqrt 3]
  return div_by(q, len, recip_of(len));
}

__device__ __forceinline__ V3 safe_inv3(V3 v) {
  if (__builtin_expect(!(div_den(v.x) && div_den(v.y) && div_den(v.z)), 0))
    return v3(safe_inv(v.x), safe_inv(v.y), safe_inv(v.z));
  return v3(div_by(1.0f, v.x, recip_of(v.x)), div_by(1.0f, v.y, recip_of(v.y)), div_by(1.0f, v.z, recip_of(v.z)));
}

// The watertight test of one (ray, triangle) pair, as tri_test: the same
// operations in the same order, with the divisions by the determinant and
// by the edge and normal scales shared, and the rare zero-edge cases inline.
__device__ __forceinline__ bool pair_test(V3 o, V3 dir, const WtRay& w, V3 a, V3 b, V3 c, float tmin, float hi,
                                          bool incl_hi, TriHit& h) {
  const int kx = w.perm & 3, ky = (w.perm >> 2) & 3, kz = (w.perm >> 4) & 3;
  const V3 pa = sub(a, o), pb = sub(b, o), pc = sub(c, o);
  const float paz = sel3(kz, pa.x, pa.y, pa.z), pbz = sel3(kz, pb.x, pb.y, pb.z), pcz = sel3(kz, pc.x, pc.y, pc.z);
  const float apx = sel3(kx, pa.x, pa.y, pa.z) - w.sx * paz, apy = sel3(ky, pa.x, pa.y, pa.z) - w.sy * paz;
  const float bpx = sel3(kx, pb.x, pb.y, pb.z) - w.sx * pbz, bpy = sel3(ky, pb.x, pb.y, pb.z) - w.sy * pbz;
  const float cpx = sel3(kx, pc.x, pc.y, pc.z) - w.sx * pcz, cpy = sel3(ky, pc.x, pc.y, pc.z) - w.sy * pcz;
  const float e0 = edge_fn(bpx, bpy, cpx, cpy);
  const float e1 = edge_fn(cpx, cpy, apx, apy);
  const float e2 = edge_fn(apx, apy, bpx, bpy);
  const float det = (e0 + e1) + e2;
  if (w.perm == 0xFFFFFFFFu || nan_(tmin) || det == 0.0f || !finite_(det)) return false;
  const bool positive = det > 0.0f;
  const float n0 = positive ? e0 : -e0, n1 = positive ? e1 : -e1, n2 = positive ? e2 : -e2;
  if (n0 < 0.0f || n1 < 0.0f || n2 < 0.0f) return false;
  const float scaled_t = (e0 * (paz * w.sz) + e1 * (pbz * w.sz)) + e2 * (pcz * w.sz);
  const int zc = (n0 == 0.0f) + (n1 == 0.0f) + (n2 == 0.0f);
  float t;
  V3 point = v3(0, 0, 0);
  if (__builtin_expect(zc != 0, 0)) {
    // On an edge or a vertex (opticalWatertightTriangle.ts:120-160): the
    // canonical point of the shared edge, or the vertex itself.
    bool ok = true;
    if (zc >= 2) {
      if (n0 != 0.0f) point = a;
      if (n1 != 0.0f) point = b;
      if (n2 != 0.0f) point = c;
    } else {
      const bool on0 = n0 == 0.0f, on1 = n1 == 0.0f;
      const V3 fi = on0 ? b : (on1 ? c : a), si = on0 ? c : (on1 ? a : b);
      const float fx = on0 ? bpx : (on1 ? cpx : apx), fy = on0 ? bpy : (on1 ? cpy : apy);
      const float gx = on0 ? cpx : (on1 ? apx : bpx), gy = on0 ? cpy : (on1 ? apy : bpy);
      const bool ordered = lex_before(fi, si);
      const V3 f = ordered ? fi : si, s = ordered ? si : fi;
      const float ax = ordered ? fx : gx, ay = ordered ? fy : gy;
      const float ddx = (ordered ? gx : fx) - ax, ddy = (ordered ? gy : fy) - ay;
      const bool use_x = fabs_(ddx) >= fabs_(ddy);
      const float num = use_x ? -ax : -ay, den = use_x ? ddx : ddy;
      ok = den != 0.0f;
      const float q = num / (ok ? den : 1.0f);
      point = ok ? v3(f.x + q * (s.x - f.x), f.y + q * (s.y - f.y), f.z + q * (s.z - f.z)) : point;
    }
    t = ok ? ray_param_inl(o, dir, point) : -1.0f;
  }
  const float yd = recip_of(det);
  const bool fast = div_den(det * 0x1p20f) && div_den(w.ds) && fabs_(scaled_t) < 0x1p40f &&
                    min(min(div_key(scaled_t), div_key(e1)), div_key(e2)) >= kDivNum;
  if (zc == 0) {
    if (__builtin_expect(fast, 1)) {
      const float t1 = div_by(scaled_t, det, yd);
      t = div_key(t1) >= kDivNum ? div_by(t1, w.ds, recip_of(w.ds)) : t1 / w.ds;
    } else {
      t = (scaled_t / det) / w.ds;
    }
  }
  const float lo = tmin > 0.0f ? tmin : 0.0f;
  if (!(t > lo) || !finite_(t)) return false;
  if (!(t > tmin && (t < hi || (incl_hi && t == hi)))) return false;
  // The authored-normal side test (opticalWatertightTriangle.ts:164-219).
  const V3 e1r = sub(b, a), e2r = sub(c, a);
  const float es = fmaxf(fmaxf(fmaxf(fabs_(e1r.x), fabs_(e1r.y)), fmaxf(fabs_(e1r.z), fabs_(e2r.x))),
                         fmaxf(fabs_(e2r.y), fabs_(e2r.z)));
  int side;
  // Only the sign of the authored normal along the ray counts.  The reference
  // normalises both; its rounding and that of this product together stay below
  // 2^-17 es^2 ds (90 half-ulps of terms at most that large), so a larger
  // product has the sign already.  Slivers and grazing rays take the long way.
  const V3 nr = v3(e1r.y * e2r.z - e1r.z * e2r.y, e1r.z * e2r.x - e1r.x * e2r.z, e1r.x * e2r.y - e1r.y * e2r.x);
  const float along = (dir.x * nr.x + dir.y * nr.y) + dir.z * nr.z;
  if (__builtin_expect(div_den(es) && div_den(w.ds) && fabs_(along) > ((es * es) * w.ds) * 0x1p-17f, 1))
    side = along > 0.0f ? -1 : 1;
  else
    side = wt_side_inl(dir, w.ds, a, b, c);
  if (side == 0) return false;
  h.front = side > 0;
  h.t = t;
  h.u = fast ? div_by(e1, det, yd) : e1 / det;
  h.v = fast ? div_by(e2, det, yd) : e2 / det;
  h.point = zc == 0 ? v3(a.x + (h.u * (b.x - a.x) + h.v * (c.x - a.x)), a.y + (h.u * (b.y - a.y) + h.v * (c.y - a.y)),
                         a.z + (h.u * (b.z - a.z) + h.v * (c.z - a.z)))
                    : point;
  return true;
}

// A 16-byte load through a pointer to global memory.  Of a pointer that comes
// out of memory the compiler does not know that, and a flat load also waits
// for LDS.
typedef float f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 load4(const float4* p) {
  const f4 v = *(const __attribute__((address_space(1))) f4*)p;
  return make_float4(v.x, v.y, v.z, v.w);
}

// ---------------------------------------------------------------------------
// Persistent traversal of the Node128 trees
// ---------------------------------------------------------------------------

// The walk of trace_kernel over the 4-wide trees: the same boxes, triangles,
// tests and acceptance rules, so the same hit records.
//
// What bounds it is VALU issue (a wave's lanes diverge) and, at the end of a
// launch, the serial chain of its longest rays.  Three things follow.
//
// One current ray.  Origin, reciprocal direction, lower bound, cull bound and
// node array are those of the level a lane walks; an instance exit reloads
// the world ray from memory instead of keeping both in registers (and nothing
// selects between them in each step).  A ray's record is written when an
// instance improves it, so its prim, u, v and position take no registers.
//
// Divisions share their denominators (div_by).
//
// Lanes without a ray help.  Once a wave has no rays left to fetch, an idle
// lane takes the bottom entry of a busy lane's BLAS stack -- the largest
// subtree it has not begun -- with a copy of its local ray, and walks it as
// if it were its own.  The lane that entered the instance (the owner) waits
// at the instance's exit until all its helpers are done and takes the
// smallest (t, triangle) over them.  The group shares its best distance
// through LDS.  Any-hit answers do not depend on the order of a walk.  A
// closest hit does in two rare cases, and a group that meets one of them
// walks the instance again, its owner alone in the usual order:
//  * Two hits within a margin of each other (2^-13 of the distance and the
//    origin's magnitude, as between instances): which of them the pop-time
//    cull lets through depends on the order.
//  * A hit nearer than its own triangle's box by more than the margin.  The
//    watertight distance is a weighted mean of the three vertices' depths
//    along the ray's dominant axis; at a grazing angle (determinant near
//    zero) the weights are inexact and it can fall anywhere between them,
//    and whether such a triangle is tested depends on the order.
// To see every such hit a group culls more cautiously than a lone lane:
// against its best distance plus the margin, and by each box's near plane on
// the dominant axis, which no distance of a triangle inside can undercut
// (less 2^-20 of the slab for rounding); entries pushed before the lane
// joined a group carry the usual entry distance and are culled by the bound
// it had then, as the lone walk would have culled them.  Where neither case is
// met, the nearest triangle is tested and kept in any order.
//
// Long rays are neighbours (those along a wall, say), and a wave that holds
// many of them outlasts the launch.  So where one fill covers the queue a
// wave's rays are taken n_waves apart, and the last kTailRays per wave of a
// longer queue are handed out transposed, 64 places apart; the rest goes out
// in order, for its coherence.  With tails of 0, 64, 128 and 512 rays: the
// 16-scene batch 1.98, 1.74, 1.73 and 1.83 ms, four 1080p frames of the box
// 35.8, 34.7, 33.6 and 33.8 ms, shadow rays in the box 1.08 (0) and 0.59 ms
// (128); the 1M-triangle scene, whose nodes fit no cache, 0.950, 0.956, 0.967
// and 1.095 ms.  The 256 x 256 frame below: 2.73 -> 2.13 ms.
// Any hits among small meshes have no long rays, and lose the coherence for
// nothing: below 1,024 triangles an instance their queues end in order.  Any
// hits of 1024 x 1024 primary rays and of shadow rays, transposed and in
// order: 8,192 boxes of 12 triangles 558 -> 483 and 584 -> 511 us, the box at
// 256 triangles an instance 244 -> 227 and 248 -> 232, at 512 251 -> 234 and
// 292 -> 304, at 1,024 272 -> 257 and 385 -> 439, at 4,096 311 -> 291 and
// 875 -> 1,060 us.
//
// Measured against the same walk without these three (trace_kernel over
// Node128): 1,677,721 rays of the 1M-triangle scene 1.27 -> 0.97 ms;
// 419,430 rays of the 32,768-triangle box, one launch after another on three
// streams, 0.356 -> 0.165 ms and alone 0.99 -> 0.37 ms (its longest ray takes
// 322 steps, most rays under 60); a 256 x 256 path-traced frame of that box
// (17 launches of at most 65,536 rays) 7.6 -> 2.13 ms.  The care that makes a
// group's closest hit independent of its order costs 0.08 ms of the first; in
// one step loop for both phases instead of two it is 0.04 ms slower.
constexpr uint32_t kIdle = 0, kNode = 1, kLeaf = 2, kEnter = 3, kExit = 4, kDone = 5;  // what a lane does next
constexpr uint32_t kfHit = 1u;         // the record holds a hit
constexpr uint32_t kfReject = 2u;      // ... on the back face of a single-sided material
constexpr uint32_t kfRefOrder = 4u;    // walking the TLAS in the reference's order
constexpr uint32_t kfRecheck = 8u;     // two instances' hits came within the margin
constexpr uint32_t kfLevel = 16u;      // inside an instance
constexpr uint32_t kfMirror = 32u;     // ... whose local-to-world map reverses orientation
constexpr uint32_t kfLHit = 128u;      // local hit, and its two bits
constexpr uint32_t kfLFront = 256u;
constexpr uint32_t kfLSingle = 512u;
constexpr uint32_t kfSplit = 1024u;    // in a group: an owner with helpers, or a helper
constexpr uint32_t kfHelper = 2048u;
constexpr uint32_t kfTie = 4096u;      // the group met a hit whose fate depends on the order
constexpr uint32_t kfAlone = 8192u;    // no helpers in this instance (walked again because of kfTie)
constexpr uint32_t kfLocal = kfLevel | kfMirror | kfLHit | kfLFront | kfLSingle | kfSplit | kfTie;
constexpr uint32_t kHelpSteps = 4;     // steps between two rounds of taking work
constexpr uint32_t kTailRays = 128;    // per wave, of a queue's end
constexpr uint32_t kTailMesh = 1024;   // triangles an instance, for any hits

// Orders a wave's LDS accesses of different lanes (they execute in program
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <bool ANY, bool MULTI>
// Four waves per SIMD: 128 VGPRs, and 8 blocks of 128 fit a CU's LDS.
__global__ __launch_bounds__(kTraceBlock, 4) void wide_kernel(TraceParams p) {
  constexpr uint32_t B = kTraceBlock, D = kWideLdsDepth;
  // Stack entries (child ref, entry distance), entry-major, deeper ones in a
  // per-thread global area; per wave: the pair table of a leaf operation
  // (also the donors' lanes), the groups' best distances and helper counts.
  __shared__ uint2 stack[D * B];
  __shared__ uint32_t table[B], group_best[B], helpers[B];
  const uint32_t tid = threadIdx.x, lane = __lane_id(), wbase = tid & ~63u;
  const size_t spill_stride = (size_t)gridDim.x * B, gtid = (size_t)blockIdx.x * B + tid;
  unsigned long long* __restrict__ spill = reinterpret_cast<unsigned long long*>(p.spill);
  const uint64_t lane_below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const bool near = !ANY && p.near_first != 0u;
  const bool near_tlas = !ANY && p.near_first == 2u;
  helpers[tid] = 0u;

  const uint32_t n_rays = p.n_ptr ? *p.n_ptr : p.n;
  const uint32_t n_waves = gridDim.x * (B / 64u);
  const uint32_t take_cap = max(1u, min(64u, n_rays / n_waves + (n_rays % n_waves != 0u)));
  const uint32_t wave_id = blockIdx.x * (B / 64u) + tid / 64u;
  const uint32_t static_end = n_waves * take_cap;
  // The order in which rays are handed out (see above): `far` apart where one
  // fill covers them all, and the last `tail` of a longer queue transposed.
  const bool one_fill = static_end >= n_rays;
  const uint32_t far = take_cap < 64u ? n_waves : 1u;
  const bool in_order = ANY && !MULTI && p.scene.tri_count / kTailMesh < p.scene.inst_count;
  const uint32_t tail = one_fill || in_order ? 0u : min(n_waves * kTailRays, n_rays - static_end) & ~63u;
  const uint32_t tail_begin = n_rays - tail;

  uint32_t mode = kIdle, fl = 0, ray_idx = 0, sid = 0;
  // The current level's ray: origin, reciprocal direction, lower bound, cull
  // bound and nodes.  World: `best` (any hit: tMax) and the lower bound.
  V3 o{}, inv{};
  float tlow = 0, cullb = 0, best = 0, wlow = 0;
  const float4* nodes = nullptr;
  // Local: direction, watertight set-up, best hit, the bound it entered with.
  V3 ld{}, lpos{};
  WtRay lw{};
  float lbest = 0, lcap = 0, cull0 = 0, lu = 0, lv = 0;
  uint32_t lprim = 0, slot = 0, slot_end = 0, own = lane;
  // Stack: next entry, the level's first, the TLAS part's end, and the end of
  // the entries pushed before joining a group (culled by `cull0`).
  uint32_t cur = kNone, sp = 0, base = 0, tsp = 0, mark = 0;

  auto scene_of = [&]() -> const DeviceScene& { return MULTI ? p.scenes[sid] : p.scene; };
  auto margin = [&](float t) { return (t + max(fabs_(o.x), max(fabs_(o.y), fabs_(o.z)))) * 0x1p-13f; };
  // The TLAS walk's bound (o is the world origin), widened by the near-tie
  // margin while the lane orders the TLAS by distance.
  auto world_bound = [&]() -> float {
    if (!ANY && near_tlas && (fl & (kfHit | kfRefOrder)) == kfHit) return best + margin(best);
    return best;
  };
  auto stk_load = [&](uint32_t i) -> uint2 {
    if (i < D) return stack[i * B + tid];
    const unsigned long long w = spill[(i - D) * spill_stride + gtid];
    return make_uint2((uint32_t)w, (uint32_t)(w >> 32));
  };
  auto finish = [&](bool occluded) {
    if (ANY) {
      p.occluded[ray_idx] = occluded ? 1u : 0u;
    } else if (!(fl & kfHit)) {
      uint32_t* h = p.hits + 5 * (size_t)ray_idx;
      h[0] = h[1] = kMiss;
      h[2] = 0x7F800000u;
      h[3] = h[4] = 0u;
      if (p.hit_pos) {
        float* hp = p.hit_pos + 3 * (size_t)ray_idx;
        hp[0] = hp[1] = hp[2] = 0.0f;
      }
    }
    mode = kIdle;
  };
  // From the TLAS root with the interval (wlow, best); o and inv are the world ray's.
  auto restart = [&]() {
    fl &= ~(kfHit | kfReject);
    tlow = wlow;
    cullb = best;
    sp = base = 0;
    cur = MULTI ? p.scenes[sid].tlas4_root : p.scene.tlas4_root;
    mode = kNode;
  };
  // A lane's subtree or interval is done: the next entry that its bound keeps.
  auto pop = [&](auto helping) {
    constexpr bool GROUP = !ANY && decltype(helping)::value;
    for (;;) {
      if (sp > base) {
        const uint2 e = stk_load(--sp);
        const bool before = GROUP && (fl & kfSplit) && sp < mark;
        if (GROUP) mark = before ? sp : mark;
        if (u2f(e.y) > (before ? cull0 : cullb)) continue;
        cur = e.x;
        return;
      }
      if (fl & kfLevel) {
        mode = (fl & kfHelper) ? kDone : kExit;
        return;
      }
      if (!ANY && (fl & kfRecheck)) {
        // A near-tie between instances: walk the ray again, from its
        // original interval, in the reference's TLAS order.
        wlow = p.rays[2 * (size_t)ray_idx].w;
        best = p.rays[2 * (size_t)ray_idx + 1].w;
        fl = (fl & ~kfRecheck) | kfRefOrder;
        restart();
        return;
      }
      // traceClosest (intersection.wgsl.ts:462-490): a back-face hit on a
      // single-sided material is not a surface; the trace starts again
      // with its distance as the exclusive lower bound, and ends as a
      // miss once that bound stops advancing or reaches tMax.
      if (!ANY && (fl & kfReject)) {
        const float tmax = p.rays[2 * (size_t)ray_idx + 1].w;
        if (best > wlow && best < tmax) {
          wlow = best;
          best = tmax;
          restart();
          return;
        }
        fl &= ~kfHit;
      }
      finish(false);
      return;
    }
  };

  // One step of a lane with an interior node: its four children.
  auto expand = [&](auto helping) {
    constexpr bool GROUP = !ANY && decltype(helping)::value;
    // one Node128: four child boxes tested axis by axis
    static_assert(kWideKids == 4, "the expansion below is written for 4-wide nodes");
    const float4* nd = nodes + (size_t)kWideNodeFloat4s * cur;
    float4 a = load4(nd), b = load4(nd + 3);
    float n0, n1, n2, n3, f0, f1, f2, f3;
    {
      const float p0 = (a.x - o.x) * inv.x, q0 = (b.x - o.x) * inv.x;
      const float p1 = (a.y - o.x) * inv.x, q1 = (b.y - o.x) * inv.x;
      const float p2 = (a.z - o.x) * inv.x, q2 = (b.z - o.x) * inv.x;
      const float p3 = (a.w - o.x) * inv.x, q3 = (b.w - o.x) * inv.x;
      n0 = fminf(p0, q0), f0 = fmaxf(p0, q0);
      n1 = fminf(p1, q1), f1 = fmaxf(p1, q1);
      n2 = fminf(p2, q2), f2 = fmaxf(p2, q2);
      n3 = fminf(p3, q3), f3 = fmaxf(p3, q3);
    }
    a = load4(nd + 1), b = load4(nd + 4);
    {
      const float p0 = (a.x - o.y) * inv.y, q0 = (b.x - o.y) * inv.y;
      const float p1 = (a.y - o.y) * inv.y, q1 = (b.y - o.y) * inv.y;
      const float p2 = (a.z - o.y) * inv.y, q2 = (b.z - o.y) * inv.y;
      const float p3 = (a.w - o.y) * inv.y, q3 = (b.w - o.y) * inv.y;
      n0 = fmaxf(n0, fminf(p0, q0)), f0 = fminf(f0, fmaxf(p0, q0));
      n1 = fmaxf(n1, fminf(p1, q1)), f1 = fminf(f1, fmaxf(p1, q1));
      n2 = fmaxf(n2, fminf(p2, q2)), f2 = fminf(f2, fmaxf(p2, q2));
      n3 = fmaxf(n3, fminf(p3, q3)), f3 = fminf(f3, fmaxf(p3, q3));
    }
    a = load4(nd + 2), b = load4(nd + 5);
    {
      const float p0 = (a.x - o.z) * inv.z, q0 = (b.x - o.z) * inv.z;
      const float p1 = (a.y - o.z) * inv.z, q1 = (b.y - o.z) * inv.z;
      const float p2 = (a.z - o.z) * inv.z, q2 = (b.z - o.z) * inv.z;
      const float p3 = (a.w - o.z) * inv.z, q3 = (b.w - o.z) * inv.z;
      n0 = fmaxf(n0, fminf(p0, q0)), f0 = fminf(f0, fmaxf(p0, q0));
      n1 = fmaxf(n1, fminf(p1, q1)), f1 = fminf(f1, fmaxf(p1, q1));
      n2 = fmaxf(n2, fminf(p2, q2)), f2 = fminf(f2, fmaxf(p2, q2));
      n3 = fmaxf(n3, fminf(p3, q3)), f3 = fminf(f3, fmaxf(p3, q3));
    }
    const float4 rf = load4(nd + 6);
    const uint4 r = make_uint4(f2u(rf.x), f2u(rf.y), f2u(rf.z), f2u(rf.w));
    // What the bound culls and the stack keeps: the entry distance, in a
    // group the near plane on the dominant axis.
    float g0 = n0, g1 = n1, g2 = n2, g3 = n3;
    if (GROUP && (fl & kfSplit)) {
      const int kz = (int)min((lw.perm >> 4) & 3u, 2u);
      const float4 lo_k = load4(nd + kz), hi_k = load4(nd + 3 + kz);
      const float ok = sel3(kz, o.x, o.y, o.z), ik = sel3(kz, inv.x, inv.y, inv.z);
      auto near_plane = [&](float mn, float mx) {
        const float p = (mn - ok) * ik, q = (mx - ok) * ik;
        return fminf(p, q) - fmaxf(fabs_(p), fabs_(q)) * 0x1p-20f;
      };
      g0 = near_plane(lo_k.x, hi_k.x);
      g1 = near_plane(lo_k.y, hi_k.y);
      g2 = near_plane(lo_k.z, hi_k.z);
      g3 = near_plane(lo_k.w, hi_k.w);
    }
    // The slab test of each child: !(tNear > tFar || tFar < tMin), then
    // the bound (the pop-time cull re-checks it against the best hit).
    const bool k0 = r.x != kEmpty && !(n0 > f0 || f0 < tlow) && !(g0 > cullb);
    const bool k1 = r.y != kEmpty && !(n1 > f1 || f1 < tlow) && !(g1 > cullb);
    const bool k2 = r.z != kEmpty && !(n2 > f2 || f2 < tlow) && !(g2 > cullb);
    const bool k3 = r.w != kEmpty && !(n3 > f3 || f3 < tlow) && !(g3 > cullb);
    // Visit first: the nearest passing child (inside BLASes with
    // near_first, lowest slot on equal distances), else the first passing
    // slot, which is the reference's depth-first order.  The others are
    // pushed so that they pop in slot order.
    uint32_t first = k0 ? 0u : (k1 ? 1u : (k2 ? 2u : (k3 ? 3u : 4u)));
    float bt = k0 ? n0 : (k1 ? n1 : (k2 ? n2 : n3));
    const bool by_distance = (fl & kfLevel) ? near : (near_tlas && !(fl & kfRefOrder));
    const bool c1 = k1 && by_distance && n1 < bt;
    bt = c1 ? n1 : bt;
    first = c1 ? 1u : first;
    const bool c2 = k2 && by_distance && n2 < bt;
    bt = c2 ? n2 : bt;
    first = c2 ? 2u : first;
    first = (k3 && by_distance && n3 < bt) ? 3u : first;
    const bool u3 = k3 && first != 3u, u2 = k2 && first != 2u, u1 = k1 && first != 1u, u0 = k0 && first != 0u;
    if (__builtin_expect(sp + 4u <= D, 1)) {
      // without branches: each entry is written at the top, which moves
      // past it only when its child is kept
      stack[sp * B + tid] = make_uint2(r.w, f2u(g3));
      sp += u3 ? 1u : 0u;
      stack[sp * B + tid] = make_uint2(r.z, f2u(g2));
      sp += u2 ? 1u : 0u;
      stack[sp * B + tid] = make_uint2(r.y, f2u(g1));
      sp += u1 ? 1u : 0u;
      stack[sp * B + tid] = make_uint2(r.x, f2u(g0));
      sp += u0 ? 1u : 0u;
    } else {
      for (uint32_t c = 4; c-- > 0;) {
        const bool use = c == 3 ? u3 : (c == 2 ? u2 : (c == 1 ? u1 : u0));
        if (!use) continue;
        const uint32_t ref = c == 3 ? r.w : (c == 2 ? r.z : (c == 1 ? r.y : r.x));
        const float tn = c == 3 ? g3 : (c == 2 ? g2 : (c == 1 ? g1 : g0));
        if (sp < D) {
          stack[sp * B + tid] = make_uint2(ref, f2u(tn));
        } else if (sp < kStackCapacity) {
          spill[(sp - D) * spill_stride + gtid] = (unsigned long long)ref | ((unsigned long long)f2u(tn) << 32);
        } else {
          atomicOr(p.error, kErrorStack);  // the host's bound rules this out
          continue;
        }
        ++sp;
      }
    }
    cur = first == 0u ? r.x : (first == 1u ? r.y : (first == 2u ? r.z : (first == 3u ? r.w : kNone)));
  };

  // `n_steps` steps of the wave: deferred work, then a node each.  Built twice:
  // without anything about groups for the time the wave still fetches rays,
  // and with it (`helping`) for the time after.
  auto run = [&](auto helping, uint32_t n_steps) {
    constexpr bool HELP = decltype(helping)::value, GROUP = !ANY && HELP;
    for (uint32_t step = 0; step < n_steps; ++step) {
      if (HELP) {
        // ---- helpers that are done ----
        uint64_t done = __ballot(mode == kDone);
        if (done) {
          uint64_t found = __ballot(mode == kDone && (fl & (kfLHit | kfTie)));
          if (mode == kDone) {
            atomicSub(&helpers[wbase + own], 1u);
            mode = kIdle;
          }
          while (found) {
            const int h = __ffsll((unsigned long long)found) - 1;
            found &= found - 1ull;
            const uint32_t ho = (uint32_t)__builtin_amdgcn_readlane((int)own, h);
            if (ANY) {
              // occluded: the owner is done, and so is every lane of its group
              const bool mine = lane == ho && mode != kIdle && own == lane;
              if (mine) finish(true);
              if ((fl & kfHelper) && own == ho) mode = kIdle;
              found &= __ballot(!((fl & kfHelper) && own == ho));
              if (lane == ho) helpers[tid] = 0u;
            } else {
              const uint32_t hf = (uint32_t)__builtin_amdgcn_readlane((int)fl, h);
              const float ht = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(lbest), h));
              const uint32_t hprim = (uint32_t)__builtin_amdgcn_readlane((int)lprim, h);
              const float hu = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(lu), h));
              const float hv = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(lv), h));
              const V3 hp = v3(u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(lpos.x), h)),
                               u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(lpos.y), h)),
                               u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(lpos.z), h)));
              if (lane == ho) {
                fl |= hf & kfTie;
                if (hf & kfLHit) {
                  if ((fl & kfLHit) && fabs_(ht - lbest) <= margin(fminf(ht, lbest))) fl |= kfTie;
                  if (!(fl & kfLHit) || ht < lbest) {
                    fl = (fl & ~(kfLFront | kfLSingle)) | kfLHit | (hf & (kfLFront | kfLSingle));
                    lbest = ht;
                    lprim = hprim;
                    lu = hu;
                    lv = hv;
                    lpos = hp;
                    cullb = fminf(lcap, ht + margin(ht));
                  }
                }
              }
            }
          }
        }
      }
      // ---- deferred work, shared by the lanes that need it (see trace_kernel) ----
      const uint64_t m_pend = __ballot(mode >= kLeaf && mode <= kExit);
      const uint64_t m_cheap = __ballot(mode == kNode);
      if ((m_pend | m_cheap) == 0ull) break;
      const uint32_t dm = min(p.defer_min, ((uint32_t)__popcll(m_pend | m_cheap) + 1u) >> 1);
      if (m_cheap == 0ull || (uint32_t)__popcll(m_pend) >= dm) {
        const bool all = m_cheap == 0ull;
        const bool at_exit = mode == kExit && !(HELP && (fl & kfSplit) && helpers[tid] != 0u);
        const uint64_t m_exit = __ballot(at_exit);
        const uint64_t m_enter = __ballot(mode == kEnter);
        const uint64_t m_leaf = __ballot(mode == kLeaf);
        if (HELP && all && (m_exit | m_enter | m_leaf) == 0ull) {
          // Only owners that wait, and no helper to wait for: cannot happen.
          // Report it and end the wave rather than wait for ever.
          if (lane == 0) atomicOr(p.error, kErrorGroup);
          mode = kIdle;
          break;
        }
        if (m_exit && (all || (uint32_t)__popcll(m_exit) >= dm) && at_exit) {
          mode = kNode;
          cur = kNone;
          sp = tsp;
          base = 0;
          // (a hit within the margin of the bound the walk entered with is
          // the same kind of tie)
          if (GROUP && (fl & kfSplit) && (fl & kfLHit) && lcap - lbest <= margin(lbest)) fl |= kfTie;
          if (GROUP && (fl & kfTie)) {
            // this instance again, alone
            fl = (fl & ~kfLocal) | kfAlone;
            mode = kEnter;
          } else {
            const DeviceScene& S = scene_of();
            const float4 a = p.rays[2 * (size_t)ray_idx], b = p.rays[2 * (size_t)ray_idx + 1];
            const V3 rd = v3(b.x, b.y, b.z);
            const bool hit = !ANY && (fl & kfLHit) && lbest > tlow;
            o = v3(a.x, a.y, a.z);
            inv = safe_inv3(rd);
            nodes = S.tlas4_nodes;
            if (hit) {
              const float4* ir = S.instances + 9 * (size_t)slot + 4;
              const float4 c0 = ir[0], c1 = ir[1], c2 = ir[2], c3 = ir[3];
              const uint32_t inst = reinterpret_cast<const uint4*>(ir + 4)->y;
              const V3 w = xform_point_fast(c0, c1, c2, c3, lpos);
              const float wd = dot3(sub(w, o), rd);
              if (near_tlas && (fl & (kfHit | kfRefOrder)) == kfHit && fabsf(wd - best) <= margin(best)) fl |= kfRecheck;
              if (wd > wlow && wd < best) {
                const bool front = ((fl & kfLFront) != 0u) != ((fl & kfMirror) != 0u);
                best = wd;
                fl = (fl & ~kfReject) | kfHit | (p.sided && !front && (fl & kfLSingle) ? kfReject : 0u);
                uint32_t* h = p.hits + 5 * (size_t)ray_idx;
                h[0] = lprim;
                h[1] = inst;
                h[2] = f2u(wd);
                h[3] = f2u(lu);
                h[4] = f2u(lv);
                if (p.hit_pos) {
                  float* hp = p.hit_pos + 3 * (size_t)ray_idx;
                  hp[0] = w.x;
                  hp[1] = w.y;
                  hp[2] = w.z;
                }
              }
            }
            fl &= ~(kfLocal | kfAlone);
            tlow = wlow;
            cullb = world_bound();
            if (++slot < slot_end) mode = kEnter;
          }
        }
        if (m_enter && (all || (uint32_t)__popcll(m_enter) >= dm) && mode == kEnter) {
          const DeviceScene& S = scene_of();
          const float4* ir = S.instances + 9 * (size_t)slot;
          const float4 a = p.rays[2 * (size_t)ray_idx], b = p.rays[2 * (size_t)ray_idx + 1];
          const float4 c0 = ir[0], c1 = ir[1], c2 = ir[2], c3 = ir[3];
          const uint4 meta = *reinterpret_cast<const uint4*>(ir + 8);
          const V3 ro = v3(a.x, a.y, a.z), rd = v3(b.x, b.y, b.z);
          o = ro;
          const float bound = ANY ? best : world_bound();
          const V3 lo = xform_point_fast(c0, c1, c2, c3, ro);
          ld = xform_dir_fast(c0, c1, c2, rd);
          const V3 start = v3(ro.x + rd.x * wlow, ro.y + rd.y * wlow, ro.z + rd.z * wlow);
          tlow = fmaxf(dot3(sub(xform_point_fast(c0, c1, c2, c3, start), lo), ld), 0.0f);
          // Closest: localTMax starts at INFINITY; any-hit: at the ray's tMax
          // (tlasSceneHitTraversal.wgsl.ts:103-108 and :168-173).
          lcap = ANY ? best : inf_const();
          if (bound < inf_const() * 0.5f) {
            const V3 end = v3(ro.x + rd.x * bound, ro.y + rd.y * bound, ro.z + rd.z * bound);
            lcap = fmaxf(dot3(sub(xform_point_fast(c0, c1, c2, c3, end), lo), ld), tlow);
          }
          o = lo;
          inv = safe_inv3(ld);
          lw = wt_setup(ld);
          lbest = cullb = lcap;
          fl = (fl & ~kfLocal) | kfLevel | (meta.w != 0u ? kfMirror : 0u);
          nodes = S.blas4_nodes;
          tsp = base = sp;
          cur = meta.z;
          mode = kNode;
        }
        if (m_leaf && (all || (uint32_t)__popcll(m_leaf) >= dm)) {
          // The leaves' (ray, triangle) pairs are spread over all 64 lanes,
          // 64 pairs a round; every pair is tested against its ray's state at
          // the start of the round, then each ray keeps the smallest
          // (t, triangle index) of its pairs -- what testing them one after
          // another gives.
          const bool mine = mode == kLeaf;
          uint32_t cnt = 0;
          const uint32_t tfirst = cur & 0x07FFFFFFu;
          if (mine) {
            cnt = (cur >> 27) & 15u;
            cur = kNone;
            mode = kNode;
          }
          uint32_t excl = 0, total = 0;
#pragma unroll
          for (uint32_t b = 0; b < 4; ++b) {  // counts are below 16: one ballot per bit
            const uint64_t m = __ballot((cnt >> b) & 1u);
            excl += (uint32_t)__popcll(m & lane_below) << b;
            total += (uint32_t)__popcll(m) << b;
          }
          bool occl = false;
          for (uint32_t first = 0; first < total; first += 64u) {
            uint32_t most = 0;  // the largest count
            for (; __ballot(most < cnt) != 0ull; ++most) {
              const uint32_t q = excl + most - first;
              if (most < cnt && q < 64u) table[wbase + q] = lane | (most << 8);
            }
            wave_sync();
            const bool work = first + lane < total;
            const uint32_t entry = work ? table[wbase + lane] : lane;
            wave_sync();
            const int ol = (int)(entry & 63u);
            const uint32_t tri = (uint32_t)__shfl((int)tfirst, ol) + (entry >> 8);
            const V3 wo = v3(__shfl(o.x, ol), __shfl(o.y, ol), __shfl(o.z, ol));
            const V3 wd = v3(__shfl(ld.x, ol), __shfl(ld.y, ol), __shfl(ld.z, ol));
            WtRay ww;
            ww.ds = __shfl(lw.ds, ol);
            ww.sx = __shfl(lw.sx, ol);
            ww.sy = __shfl(lw.sy, ol);
            ww.sz = __shfl(lw.sz, ol);
            ww.perm = (uint32_t)__shfl((int)lw.perm, ol);
            const float w_low = __shfl(tlow, ol);
            // An owner or helper accepts up to its cull bound (its best plus
            // the margin); otherwise hits below the best, or at it.
            const float w_hi = __shfl(GROUP && (fl & kfSplit) ? cullb : lbest, ol);
            const uint32_t w_fl = (uint32_t)__shfl((int)fl, ol);
            const float4* otris = p.scene.tris;
            if (MULTI) otris = p.scenes[(uint32_t)__shfl((int)sid, ol)].tris;
            TriHit h;
            h.t = h.u = h.v = 0.0f;
            h.point = v3(0, 0, 0);
            h.front = false;
            bool hit = false;
            float single = 0.0f;
            if (work) {
              const float4* tr = otris + 3 * (size_t)tri;
              const float4 w0 = load4(tr), w1 = load4(tr + 1), w2 = load4(tr + 2);
              single = w2.y;
              hit = pair_test(wo, wd, ww, v3(w0.x, w0.y, w0.z), v3(w0.w, w1.x, w1.y), v3(w1.z, w1.w, w2.x), w_low, w_hi,
                              near && (w_fl & (GROUP ? kfLHit | kfSplit : kfLHit)) == kfLHit, h);
              // Any hit through the path tracer's wrappers: a back face of a
              // single-sided material does not block.
              if (ANY && hit && p.sided && h.front == ((w_fl & kfMirror) != 0u) && single > 0.5f) hit = false;
            }
            const uint64_t hits = __ballot(hit);
            if (hits == 0ull) continue;
            uint64_t early = 0ull;  // hits nearer than their own triangle's box
            if (GROUP && __any((fl & kfSplit) != 0u)) {
              const V3 wi = v3(__shfl(inv.x, ol), __shfl(inv.y, ol), __shfl(inv.z, ol));
              bool e = false;
              if (hit) {
                const float4* tr = otris + 3 * (size_t)tri;
                const float4 w0 = load4(tr), w1 = load4(tr + 1), w2 = load4(tr + 2);
                float tn;
                (void)slab(wo, wi, fminf(w0.x, fminf(w0.w, w1.z)), fminf(w0.y, fminf(w1.x, w1.w)),
                           fminf(w0.z, fminf(w1.y, w2.x)), fmaxf(w0.x, fmaxf(w0.w, w1.z)),
                           fmaxf(w0.y, fmaxf(w1.x, w1.w)), fmaxf(w0.z, fmaxf(w1.y, w2.x)), w_low, tn);
                const float m = (h.t + max(fabs_(wo.x), max(fabs_(wo.y), fabs_(wo.z)))) * 0x1p-13f;
                e = !(h.t >= tn - m);
              }
              early = __ballot(e);
            }
            // Each ray's run of lanes in this round: [lo, hi).
            const uint32_t lo = min(max(excl, first) - first, 64u), hi = min(max(excl + cnt, first) - first, 64u);
            const uint64_t run = (hi > lo) ? ((~0ull >> (64u - (hi - lo))) << lo) & hits : 0ull;
            if (ANY) {
              occl = occl || run != 0ull;
              continue;
            }
            float rt = __builtin_inff();
            uint32_t rl = lane, ri = 0;
            for (uint32_t i = 0; i < most; ++i) {
              const uint32_t q = excl + i - first;
              const float t = __shfl(h.t, (int)(q & 63u));
              if (i < cnt && q < 64u && ((hits >> (q & 63u)) & 1ull) && t < rt) {
                rt = t;
                rl = q;
                ri = tfirst + i;
              }
            }
            const uint32_t bits = (h.front ? kfLFront : 0u) | (single > 0.5f ? kfLSingle : 0u);
            const float ru = __shfl(h.u, (int)rl), rv = __shfl(h.v, (int)rl);
            const V3 rp = v3(__shfl(h.point.x, (int)rl), __shfl(h.point.y, (int)rl), __shfl(h.point.z, (int)rl));
            const uint32_t rb = (uint32_t)__shfl((int)bits, (int)rl);
            if (run != 0ull) {
              if (GROUP && (fl & kfSplit)) {
                // two hits in one leaf, or one within the margin of the best
                if ((run & (run - 1ull)) != 0ull || (run & early) != 0ull) fl |= kfTie;
                if ((fl & kfLHit) && fabs_(rt - lbest) <= margin(fminf(rt, lbest))) fl |= kfTie;
              }
              if (!(fl & kfLHit) || rt < lbest || (rt == lbest && ri < lprim)) {
                fl = (fl & ~(kfLFront | kfLSingle)) | kfLHit | rb;
                lbest = rt;
                lprim = ri;
                lu = ru;
                lv = rv;
                lpos = rp;
                cullb = GROUP && (fl & kfSplit) ? fminf(cullb, fminf(lcap, rt + margin(rt))) : rt;
              }
            }
          }
          if (ANY && occl) {
            // A group's lanes end together, at the owner.
            if (HELP && (fl & kfHelper)) {
              fl |= kfLHit;
              mode = kDone;
            } else {
              finish(true);
            }
          }
          if (ANY && HELP) {
            // helpers of owners that have just finished
            const uint64_t busy = __ballot(mode != kIdle);
            if ((fl & kfHelper) && mode != kIdle && !((busy >> own) & 1ull)) mode = kIdle;
            if (mode == kIdle) helpers[tid] = 0u;
          }
        }
      }
      // ---- cheap work: pop with the reference's pop-time cull, expand ----
      if (mode != kNode) continue;
      if (cur == kNone) pop(helping);
      if (mode == kNode && !(cur & kLeafBit)) expand(helping);
      // A leaf reached by the pop or the expansion becomes pending work.
      if (mode == kNode && cur != kNone && (cur & kLeafBit)) {
        mode = kLeaf;
        if (!(fl & kfLevel)) {
          slot = cur & 0x07FFFFFFu;
          slot_end = slot + ((cur >> 27) & 15u);
          cur = kNone;
          mode = slot < slot_end ? kEnter : kNode;
        }
      }
    }
  };

  // The first fill is static, later ones go through the shared counter (see
  // trace_kernel); `exhausted`: no more rays for this wave.
  bool exhausted = false, first_fill = true;
  for (;;) {
    const uint64_t idle = __ballot(mode == kIdle);
    const uint32_t n_idle = (uint32_t)__popcll(idle);
    if (!exhausted) {
      if (n_idle >= p.refill_min || n_idle == 64u) {
        const uint32_t take = min(n_idle, take_cap);
        uint32_t first = far == 1u ? wave_id * take_cap : wave_id, step = far;
        if (!first_fill) {
          if (lane == 0) first = static_end + atomicAdd(p.counter, take);
          first = (uint32_t)__shfl((int)first, 0);
          step = 1u;
        }
        exhausted = first_fill ? one_fill : first + take >= n_rays;
        first_fill = false;
        const uint32_t rank = (uint32_t)__popcll(idle & lane_below);
        uint32_t idx = first + rank * step;
        if (tail != 0u && idx >= tail_begin && idx < n_rays) {
          const uint32_t q = idx - tail_begin;
          idx = tail_begin + (q & 63u) * (tail >> 6) + (q >> 6);
        }
        if (mode == kIdle && rank < take && idx < n_rays) {
          ray_idx = idx;
          if (MULTI) {
            uint32_t lo_s = 0, hi_s = p.scene_count;
            while (lo_s + 1u < hi_s) {
              const uint32_t mid = (lo_s + hi_s) >> 1;
              if (p.scene_offsets[mid] <= idx) lo_s = mid; else hi_s = mid;
            }
            sid = lo_s;
          }
          const float4 a = p.rays[2 * (size_t)idx], b = p.rays[2 * (size_t)idx + 1];
          const DeviceScene& S = scene_of();
          nodes = S.tlas4_nodes;
          o = v3(a.x, a.y, a.z);
          inv = safe_inv3(v3(b.x, b.y, b.z));
          wlow = a.w;
          best = b.w;
          fl = 0;
          own = lane;
          restart();
        }
      }
    } else if (idle != 0ull && n_idle != 64u) {
      // ---- share the groups' bounds, then hand out work ----
      if (mode == kIdle) fl = 0;
      if (!ANY && (fl & kfSplit)) {
        if (fl & kfLHit) atomicMin(&group_best[wbase + own], f2u(lbest));  // t > 0: ordered as integers
      }
      wave_sync();
      if (!ANY && (fl & kfSplit)) {
        const float g = u2f(group_best[wbase + own]);
        cullb = fminf(cullb, g + margin(g));
      }
      const bool donor = (fl & (kfLevel | kfAlone)) == kfLevel && (mode == kNode || mode == kLeaf) && sp > base && base < D;
      const uint64_t donors = __ballot(donor);
      if (donors != 0ull) {
        // The r-th idle lane takes entry r / n_donors of donor r % n_donors.
        const uint32_t n_don = (uint32_t)__popcll(donors), rank_d = (uint32_t)__popcll(donors & lane_below);
        const uint32_t share = donor && n_idle > rank_d ? (n_idle - rank_d - 1u) / n_don + 1u : 0u;
        if (share != 0u && !(fl & kfSplit)) {
          fl |= kfSplit;
          mark = sp;
          cull0 = cullb;
          if (!ANY) group_best[tid] = (fl & kfLHit) ? f2u(lbest) : 0x7F7FFFFFu;
          if (!ANY && (fl & kfLHit)) cullb = fminf(lcap, lbest + margin(lbest));
        }
        const uint32_t avail = donor ? min(sp, D) - base : 0u;
        if (donor) table[wbase + rank_d] = lane;
        wave_sync();
        const uint32_t r = (uint32_t)__popcll(idle & lane_below), k = r / n_don;
        const int d = mode == kIdle ? (int)table[wbase + (r - k * n_don)] : (int)lane;
        wave_sync();
        const uint32_t d_avail = (uint32_t)__shfl((int)avail, d);
        const bool got = mode == kIdle && k < d_avail;
        const uint32_t at = (uint32_t)__shfl((int)base, d) + k;
        const uint32_t d_own = (uint32_t)__shfl((int)own, d), d_fl = (uint32_t)__shfl((int)fl, d);
        const V3 d_o = v3(__shfl(o.x, d), __shfl(o.y, d), __shfl(o.z, d));
        const V3 d_inv = v3(__shfl(inv.x, d), __shfl(inv.y, d), __shfl(inv.z, d));
        const V3 d_ld = v3(__shfl(ld.x, d), __shfl(ld.y, d), __shfl(ld.z, d));
        const float d_low = __shfl(tlow, d), d_cull = __shfl(cullb, d), d_cap = __shfl(lcap, d);
        const float d_cull0 = __shfl(cull0, d);
        const uint32_t d_mark = (uint32_t)__shfl((int)mark, d);
        const uint32_t d_sid = MULTI ? (uint32_t)__shfl((int)sid, d) : 0u;
        WtRay d_lw;
        d_lw.ds = __shfl(lw.ds, d);
        d_lw.sx = __shfl(lw.sx, d);
        d_lw.sy = __shfl(lw.sy, d);
        d_lw.sz = __shfl(lw.sz, d);
        d_lw.perm = (uint32_t)__shfl((int)lw.perm, d);
        if (donor) base += min(avail, share);
        wave_sync();
        if (got) {
          const uint2 e = stack[at * B + wbase + (uint32_t)d];
          own = d_own;
          lw = d_lw;
          o = d_o;
          inv = d_inv;
          ld = d_ld;
          tlow = d_low;
          cullb = d_cull;
          lcap = d_cap;
          sid = d_sid;
          nodes = scene_of().blas4_nodes;
          fl = kfHelper | kfSplit | kfLevel | (d_fl & kfMirror);
          lbest = d_cap;
          sp = base = tsp = mark = 0;
          cur = u2f(e.y) > (!ANY && at < d_mark ? d_cull0 : cullb) ? kNone : e.x;
          mode = (cur != kNone && (cur & kLeafBit)) ? kLeaf : kNode;
          atomicAdd(&helpers[wbase + own], 1u);
        }
      }
    }
    if (!__any(mode != kIdle)) {
      if (exhausted) break;
      continue;
    }

    if (exhausted)
      run(std::true_type{}, kHelpSteps);
    else
      run(std::false_type{}, p.steps);
  }
}

__global__ void zero_u32_kernel(uint32_t* p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

__global__ void copy16_kernel(uint4* __restrict__ dst, const uint4* __restrict__ src, size_t n16) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

__global__ void fp32_selftest_kernel(const float* a, const float* b, float* q, float* r, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    q[i] = a[i] / b[i];
    r[i] = __builtin_sqrtf(a[i]);
  }
}

}  // namespace vtk

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------

namespace vtk {

// The Node128 kernel when every scene has those trees (p.wide), else the
// Node64 kernel.
template <bool ANY, bool MULTI>
static hipError_t launch_one(const TraceParams& p, uint32_t grid, hipStream_t s) {
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, p.counter, 1u);
  if (p.wide)
    hipLaunchKernelGGL((wide_kernel<ANY, MULTI>), dim3(grid), dim3(kTraceBlock), 0, s, p);
  else
    hipLaunchKernelGGL((trace_kernel<ANY, false, MULTI, kTraceBlock, kLdsDepth>), dim3(grid), dim3(kTraceBlock), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_trace_batch(const TraceParams& p, uint32_t grid, hipStream_t s) {
  return launch_one<false, true>(p, grid, s);
}

hipError_t launch_trace_batch_any(const TraceParams& p, uint32_t grid, hipStream_t s) {
  return launch_one<true, true>(p, grid, s);
}

hipError_t launch_trace(const TraceParams& p, bool any, bool count, uint32_t grid, hipStream_t s) {
  if (count) {
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, p.counter, 1u);
    hipLaunchKernelGGL((trace_kernel<false, true, false, kTraceBlock, kLdsDepth>), dim3(grid), dim3(kTraceBlock), 0, s, p);
    return hipGetLastError();
  }
  return any ? launch_one<true, false>(p, grid, s) : launch_one<false, false>(p, grid, s);
}

// The smallest of the two kernels' resident blocks per CU.
template <bool ANY, bool MULTI>
static hipError_t occupancy_of(int* out) {
  int a = 0, b = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &a, trace_kernel<ANY, false, MULTI, kTraceBlock, kLdsDepth>, kTraceBlock, 0);
  if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, wide_kernel<ANY, MULTI>, kTraceBlock, 0);
  *out = a < b ? a : b;
  return e;
}

hipError_t trace_occupancy_batch(int* blocks_per_cu) { return occupancy_of<false, true>(blocks_per_cu); }

// The counting variant (measurement only) is left out: its extra blocks
// simply start as others retire.
hipError_t trace_occupancy(bool any, int* blocks_per_cu) {
  return any ? occupancy_of<true, false>(blocks_per_cu) : occupancy_of<false, false>(blocks_per_cu);
}

hipError_t launch_zero(uint32_t* p, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(zero_u32_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_copy16(uint4* dst, const uint4* src, size_t n16, hipStream_t s) {
  if (n16 == 0) return hipSuccess;
  const size_t want = (n16 + 255) / 256;
  const uint32_t blocks = (uint32_t)(want < 8192 ? want : 8192);
  hipLaunchKernelGGL(copy16_kernel, dim3(blocks), dim3(256), 0, s, dst, src, n16);
  return hipGetLastError();
}

hipError_t launch_fp32_selftest(const float* a, const float* b, float* q, float* r, uint32_t n,
                                hipStream_t s) {
  hipLaunchKernelGGL(fp32_selftest_kernel, dim3((n + 255) / 256), dim3(256), 0, s, a, b, q, r, n);
  return hipGetLastError();
}

}  // namespace vtk

// ---------------------------------------------------------------------------
// cwbvh-closest mode: pt-webgpu's opt-in wide traversal
// (pathTrace/intersection.wgsl.ts:576-838).  One ray per lane over the
// reference-layout TLAS; each BLAS is walked in its 8-wide compressed tree
// (cwbvhIntersect.wgsl.ts:197-336) with the Moller-Trumbore core
// (bvhIntersect.wgsl.ts:160-238); the proposed hit is accepted only when the
// watertight test reproduces its distance bit for bit, and a disagreement, an
// invalid wide layout or a stack overflow answers that BLAS with the binary
// traversal (intersectionCore.wgsl.ts:461-596).  Any-hit rays never use it.
// ---------------------------------------------------------------------------

namespace vtw {

using vtk::F4;
using vtk::TriHit;
using vtk::V3;
using vtk::WtRay;

constexpr uint32_t kWideStack = 64;  // cwbvhIntersect.wgsl.ts stack depth
constexpr uint32_t kBinStack = 60;   // strides.ts:110
constexpr uint32_t kTlasStack = 64;  // strides.ts:112
constexpr uint32_t kLeafMask = 0xFFFF0000u;

// The WGSL select-based min / max (NaN compares false).
__device__ __forceinline__ float max2(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ float min2(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float cw_inf() { return 3.402823e38f; }

__device__ __forceinline__ float decode(uint32_t q, float mn, float mx) {
  if (!(mx > mn)) return mn;
  if (q == 0) return mn;
  if (q >= 65535u) return mx;
  const float t = (float)q / 65535.0f;
  return mn * (1.0f - t) + mx * t;
}

__device__ __forceinline__ bool bounds_valid(V3 mn, V3 mx) {
  const float m = cw_inf();
  return mn.x <= mx.x && mn.y <= mx.y && mn.z <= mx.z && vtk::fabs_(mn.x) <= m && vtk::fabs_(mn.y) <= m &&
         vtk::fabs_(mn.z) <= m && vtk::fabs_(mx.x) <= m && vtk::fabs_(mx.y) <= m && vtk::fabs_(mx.z) <= m;
}

__device__ __forceinline__ bool aabb_entry(V3 o, V3 inv, V3 bmn, V3 bmx, float tmax) {
  const float t0x = (bmn.x - o.x) * inv.x, t0y = (bmn.y - o.y) * inv.y, t0z = (bmn.z - o.z) * inv.z;
  const float t1x = (bmx.x - o.x) * inv.x, t1y = (bmx.y - o.y) * inv.y, t1z = (bmx.z - o.z) * inv.z;
  const float tn = max2(max2(min2(t0x, t1x), min2(t0y, t1y)), min2(t0z, t1z));
  const float tf = min2(min2(max2(t0x, t1x), max2(t0y, t1y)), max2(t0z, t1z));
  return !(tn > tf || tf < 0.0f || tn > tmax);
}

__device__ __forceinline__ V3 cross3(V3 a, V3 b) {
  return vtk::v3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ V3 scale_div(V3 a, float s) { return vtk::v3(a.x / s, a.y / s, a.z / s); }

// mollerTrumboreCore: equilibrated edges and direction, angular determinant
// rejection at 1e-7, barycentric tolerance 1e-6.  Returns t, or -1 for a miss.
__device__ __noinline__ float mt_core(V3 o, V3 dir, V3 a, V3 b, V3 c, float tmin) {
  using vtk::dot3;
  using vtk::fabs_;
  using vtk::nan_;
  const V3 e1r = vtk::sub(b, a), e2r = vtk::sub(c, a);
  const float es = max2(max2(max2(fabs_(e1r.x), fabs_(e1r.y)), fabs_(e1r.z)),
                        max2(max2(fabs_(e2r.x), fabs_(e2r.y)), fabs_(e2r.z)));
  const float ds = max2(fabs_(dir.x), max2(fabs_(dir.y), fabs_(dir.z)));
  if (!(es > 0.0f) || es > cw_inf() || !(ds > 0.0f) || ds > cw_inf()) return -1.0f;
  const V3 e1 = scale_div(e1r, es), e2 = scale_div(e2r, es), dn = scale_div(dir, ds);
  const V3 ao = scale_div(vtk::sub(o, a), es);
  const V3 n = cross3(e1, e2);
  const float ns = max2(fabs_(n.x), max2(fabs_(n.y), fabs_(n.z)));
  if (!(ns > 0.0f) || ns > cw_inf()) return -1.0f;
  const V3 nd = scale_div(n, ns);
  const float nl = __builtin_sqrtf(dot3(nd, nd));
  const float dl = __builtin_sqrtf(dot3(dn, dn));
  const V3 rd = scale_div(dn, dl);
  const float det = -dot3(dn, n);
  const V3 nn = scale_div(nd, nl);
  const float ang = fabs_(dot3(rd, nn));
  if (!(ang > 1e-7f) || det == 0.0f) return -1.0f;
  const float inv_det = 1.0f / det;
  const V3 dao = cross3(ao, dn);
  const float u = dot3(e2, dao) * inv_det;
  const float v = -dot3(e1, dao) * inv_det;
  const float st = dot3(ao, n) * inv_det;
  const float t = (st * es) / ds;
  const float w = (1.0f - u) - v;
  if (nan_(u) || nan_(v) || nan_(w) || nan_(t) || fabs_(u) > cw_inf() || fabs_(v) > cw_inf() ||
      fabs_(w) > cw_inf() || fabs_(t) > cw_inf() || u < -1e-6f || v < -1e-6f || w < -1e-6f ||
      t < max2(tmin, 0.0f))
    return -1.0f;
  return t;
}

__device__ __forceinline__ V3 vload(const Scene& s, uint32_t i) {
  const float4 p = s.positions[i];
  return vtk::v3(p.x, p.y, p.z);
}

struct LocalHit {
  bool hit;
  float t;
  V3 pos;
  uint32_t tri;
  float u, v;
  bool front;  // local front face (the watertight test's side)
};

// traceMeshBvh over the reference node layout (8 words per node), left child
// first, closest hit.
__device__ __noinline__ LocalHit mesh_binary(const Scene& s, V3 o, V3 d, V3 inv, const WtRay& w, float tmin,
                                             float tmax, uint32_t root) {
  LocalHit h{false, tmax, vtk::v3(0, 0, 0), 0u, 0.0f, 0.0f, false};
  if (s.bvh_node_count == 0 || root >= s.bvh_node_count) return h;
  uint32_t stack[kBinStack];
  uint32_t sp = 0;
  stack[sp++] = root;
  while (sp > 0) {
    const uint32_t ni = stack[--sp];
    if (ni >= s.bvh_node_count) continue;
    const uint4* nd = reinterpret_cast<const uint4*>(s.bvh_nodes + 8 * (size_t)ni);
    const uint4 lo = nd[0], hi = nd[1];
    float tn;
    if (!vtk::slab(o, inv, vtk::u2f(lo.x), vtk::u2f(lo.y), vtk::u2f(lo.z), vtk::u2f(lo.w), vtk::u2f(hi.x),
                   vtk::u2f(hi.y), tmin, tn) ||
        tn > h.t)
      continue;
    if ((hi.w & kLeafMask) == kLeafMask) {
      const uint32_t count = hi.w & 0xFFFFu, start = hi.z;
      for (uint32_t i = 0; i < count; ++i) {
        const uint32_t t = start + i;
        if (t >= s.tri_count) continue;
        const uint4 ix = s.indices[t];
        if (ix.x >= s.vertex_count || ix.y >= s.vertex_count || ix.z >= s.vertex_count) continue;
        TriHit th;
        if (vtk::tri_test(o, d, w, vload(s, ix.x), vload(s, ix.y), vload(s, ix.z), tmin, h.t, false, th)) {
          h.hit = true;
          h.t = th.t;
          h.pos = th.point;
          h.tri = t;
          h.u = th.u;
          h.v = th.v;
          h.front = th.front;
        }
      }
    } else {
      if (sp + 2 > kBinStack) return h;
      stack[sp++] = ni + hi.z;
      stack[sp++] = ni + 1;
    }
  }
  return h;
}

// Wide walk.  status: 0 complete, 1 stack overflow, 2 invalid layout.
struct WideHit {
  uint32_t status;
  bool hit;
  float t;
  uint32_t tri;
};

__device__ __noinline__ WideHit wide_walk(const Scene& s, V3 o, V3 d, V3 inv, float tmin, float tmax,
                                          uint32_t root) {
  WideHit best{0u, false, tmax, 0u};
  const uint32_t nc = s.wide_count;
  if (nc == 0) return best;
  if (root >= nc) {
    best.status = 2;
    return best;
  }
  uint32_t stack[kWideStack];
  uint32_t sp = 0;
  stack[sp++] = root;
  while (sp > 0) {
    const uint32_t node = stack[--sp];
    if (node >= nc) {
      best.status = 2;
      return best;
    }
    const uint32_t count = s.child_count[node];
    if (count > kKids) {
      best.status = 2;
      return best;
    }
    const float* pb = s.node_bounds + 6 * (size_t)node;
    const V3 pmn = vtk::v3(pb[0], pb[1], pb[2]), pmx = vtk::v3(pb[3], pb[4], pb[5]);
    if (!bounds_valid(pmn, pmx)) {
      best.status = 2;
      return best;
    }
    for (uint32_t slot = 0; slot < count; ++slot) {
      const size_t k = ((size_t)node * kKids + slot) * 3;
      const uint32_t kind = s.child_meta[k], ref = s.child_meta[k + 1], cnt = s.child_meta[k + 2];
      if (kind == 0) {
        best.status = 2;
        return best;
      }
      const uint32_t q0 = s.child_bounds[k], q1 = s.child_bounds[k + 1], q2 = s.child_bounds[k + 2];
      const V3 bmn = vtk::v3(decode(q0 & 0xFFFFu, pmn.x, pmx.x), decode(q0 >> 16, pmn.y, pmx.y),
                             decode(q1 & 0xFFFFu, pmn.z, pmx.z));
      const V3 bmx = vtk::v3(decode(q1 >> 16, pmn.x, pmx.x), decode(q2 & 0xFFFFu, pmn.y, pmx.y),
                             decode(q2 >> 16, pmn.z, pmx.z));
      if (!bounds_valid(bmn, bmx)) {
        best.status = 2;
        return best;
      }
      if (!aabb_entry(o, inv, bmn, bmx, best.t)) continue;
      if (kind == 1) {
        if (ref >= nc) {
          best.status = 2;
          return best;
        }
        if (sp >= kWideStack) {
          best.status = 1;
          return best;
        }
        stack[sp++] = ref;
      } else if (kind == 2) {
        if (cnt == 0 || ref > s.tri_count || cnt > s.tri_count - ref) {
          best.status = 2;
          return best;
        }
        for (uint32_t i = 0; i < cnt; ++i) {
          const uint32_t tri = ref + i;
          const uint4 ix = s.indices[tri];
          if (ix.x >= s.vertex_count || ix.y >= s.vertex_count || ix.z >= s.vertex_count) {
            best.status = 2;
            return best;
          }
          const float t = mt_core(o, d, vload(s, ix.x), vload(s, ix.y), vload(s, ix.z), tmin);
          if (t >= 0.0f && t > tmin && t < best.t) {
            best.hit = true;
            best.t = t;
            best.tri = tri;
          }
        }
      } else {
        best.status = 2;
        return best;
      }
    }
  }
  return best;
}

// traceMeshCwbvhClosest.
__device__ __forceinline__ LocalHit mesh_cwbvh(const Scene& s, V3 o, V3 d, V3 inv, const WtRay& w, float tmin,
                                               float tmax, uint32_t wide_root, uint32_t binary_root) {
  if (s.wide_count == 0 || wide_root >= s.wide_count) return mesh_binary(s, o, d, inv, w, tmin, tmax, binary_root);
  const WideHit c = wide_walk(s, o, d, inv, tmin, tmax, wide_root);
  if (c.status != 0) return mesh_binary(s, o, d, inv, w, tmin, tmax, binary_root);
  LocalHit h{false, tmax, vtk::v3(0, 0, 0), 0u, 0.0f, 0.0f, false};
  if (!c.hit || c.t <= tmin || c.t >= tmax) return h;
  if (c.tri >= s.tri_count) return mesh_binary(s, o, d, inv, w, tmin, tmax, binary_root);
  const uint4 ix = s.indices[c.tri];
  TriHit e;
  if (!vtk::tri_test(o, d, w, vload(s, ix.x), vload(s, ix.y), vload(s, ix.z), tmin, vtk::inf_const(), true, e) ||
      vtk::f2u(e.t) != vtk::f2u(c.t))
    return mesh_binary(s, o, d, inv, w, tmin, tmax, binary_root);
  h.hit = true;
  h.t = c.t;
  h.pos = e.point;
  h.tri = c.tri;
  h.u = e.u;
  h.v = e.v;
  h.front = e.front;
  return h;
}

__device__ __forceinline__ void load_cols(const float* m, float4& c0, float4& c1, float4& c2, float4& c3) {
  const float4* q = reinterpret_cast<const float4*>(m);
  c0 = q[0];
  c1 = q[1];
  c2 = q[2];
  c3 = q[3];
}

struct WorldHit {
  float t;
  uint32_t prim, inst;
  float u, v;
  V3 pos;
  bool front;  // world front face (flipped by an orientation-reversing instance)
};

// One instance of traceTlasClosestCwbvh / tlasInstanceClosest: the local ray,
// its [ltmin, ltmax] window, the BLAS walk and the world-distance acceptance.
__device__ __forceinline__ void instance_closest(const Scene& s, uint32_t inst, bool wide, V3 ro, V3 rd,
                                                 float tmin, WorldHit& b) {
  if (inst >= s.inst_count) return;
  float4 c0, c1, c2, c3;
  load_cols(s.w2l + 16 * (size_t)inst, c0, c1, c2, c3);
  const V3 lo = vtk::xform_point(c0, c1, c2, c3, ro);
  const V3 ld = vtk::xform_dir(c0, c1, c2, rd);
  const V3 linv = vtk::v3(vtk::safe_inv(ld.x), vtk::safe_inv(ld.y), vtk::safe_inv(ld.z));
  const V3 sp = vtk::v3(ro.x + rd.x * tmin, ro.y + rd.y * tmin, ro.z + rd.z * tmin);
  const float ltmin = max2(vtk::dot3(vtk::sub(vtk::xform_point(c0, c1, c2, c3, sp), lo), ld), 0.0f);
  float ltmax = vtk::inf_const();
  if (b.t < vtk::inf_const() * 0.5f) {
    const V3 ep = vtk::v3(ro.x + rd.x * b.t, ro.y + rd.y * b.t, ro.z + rd.z * b.t);
    ltmax = max2(vtk::dot3(vtk::sub(vtk::xform_point(c0, c1, c2, c3, ep), lo), ld), ltmin);
  }
  const WtRay w = vtk::wt_setup(ld);
  const LocalHit lh = wide ? mesh_cwbvh(s, lo, ld, linv, w, ltmin, ltmax, s.wide_roots[inst], s.blas_roots[inst])
                           : mesh_binary(s, lo, ld, linv, w, ltmin, ltmax, s.blas_roots[inst]);
  if (!lh.hit || !(lh.t > ltmin)) return;
  load_cols(s.l2w + 16 * (size_t)inst, c0, c1, c2, c3);
  const V3 wpos = vtk::xform_point(c0, c1, c2, c3, lh.pos);
  const float wd = vtk::dot3(vtk::sub(wpos, ro), rd);
  // intersection.wgsl.ts:811 rejects with `<=` / `>=` (a NaN distance is kept),
  // unlike tlasInstanceClosest's `>` / `<` acceptance.
  if (wide && (wd <= tmin || wd >= b.t)) return;
  if (!wide && !(wd > tmin && wd < b.t)) return;
  b.t = wd;
  b.prim = lh.tri;
  b.inst = inst;
  b.u = lh.u;
  b.v = lh.v;
  b.pos = wpos;
  b.front = lh.front != (s.inst_reversed[inst] != 0);
}

__global__ __launch_bounds__(128) void trace_cwbvh_kernel(Params p) {
  const Scene& s = p.s;
  // With a device count, p.n is the capacity of the ray and hit buffers.
  const uint32_t n = p.n_ptr ? min(*p.n_ptr, p.n) : p.n;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float4 ra = p.rays[2 * (size_t)i], rb = p.rays[2 * (size_t)i + 1];
    const V3 ro = vtk::v3(ra.x, ra.y, ra.z), rd = vtk::v3(rb.x, rb.y, rb.z);
    const float tmax = rb.w;
    const V3 rinv = vtk::v3(vtk::safe_inv(rd.x), vtk::safe_inv(rd.y), vtk::safe_inv(rd.z));
    WorldHit b;
    // traceClosest (intersection.wgsl.ts:462-490) with p.sided: a back-face
    // hit on a single-sided material is skipped by tracing again from its
    // distance (exclusive); a bound that stops advancing or reaches tMax
    // ends the ray as a miss.
    float tmin = ra.w;
    for (;;) {
      // Mode 0: wide BLAS walks; 1: binary BLAS walks (a TLAS stack overflow in
      // mode 0 restarts here, as traceTlasClosestCwbvh falls back to
      // traceTlasClosest); 2: every instance in permutation order
      // (tlasClosestFallback, on a TLAS stack overflow in mode 1).
      uint32_t mode = (s.tlas_node_count == 0 || s.inst_index_count == 0) ? 3u : 0u;
      for (;;) {
        b.t = tmax;
        b.prim = 0;
        b.inst = vtk::kMiss;
        b.u = b.v = 0.0f;
        b.pos = vtk::v3(0, 0, 0);
        b.front = false;
        if (mode == 3) break;  // no TLAS: fail closed
        if (mode == 2) {
          for (uint32_t pi = 0; pi < s.inst_index_count; ++pi)
            instance_closest(s, s.inst_indices[pi], false, ro, rd, tmin, b);
          break;
        }
        uint32_t stack[kTlasStack];
        uint32_t sp = 0;
        stack[sp++] = 0;
        bool overflow = false;
        while (sp > 0 && !overflow) {
          const uint32_t ni = stack[--sp];
          if (ni >= s.tlas_node_count) continue;
          const uint4* nd = reinterpret_cast<const uint4*>(s.tlas_nodes + 8 * (size_t)ni);
          const uint4 lo = nd[0], hi = nd[1];
          float tn;
          if (!vtk::slab(ro, rinv, vtk::u2f(lo.x), vtk::u2f(lo.y), vtk::u2f(lo.z), vtk::u2f(lo.w),
                         vtk::u2f(hi.x), vtk::u2f(hi.y), tmin, tn) ||
              tn > b.t)
            continue;
          if ((hi.w & kLeafMask) == kLeafMask) {
            const uint32_t count = hi.w & 0xFFFFu, start = hi.z;
            for (uint32_t k = 0; k < count; ++k) {
              const uint32_t pi = start + k;
              if (pi >= s.inst_index_count) continue;
              instance_closest(s, s.inst_indices[pi], mode == 0, ro, rd, tmin, b);
            }
          } else if (sp + 2 <= kTlasStack) {
            stack[sp++] = ni + hi.z;
            stack[sp++] = ni + 1;
          } else {
            overflow = true;
          }
        }
        if (!overflow) break;
        ++mode;
      }
      if (!p.sided || b.inst == vtk::kMiss || b.front || b.prim >= s.tri_count || !s.single_sided[b.prim]) break;
      if (!(b.t > tmin) || !(b.t < tmax)) {
        b.inst = vtk::kMiss;
        break;
      }
      tmin = b.t;
    }
    const bool hit = b.inst != vtk::kMiss;
    uint32_t* h = p.hits + 5 * (size_t)i;
    h[0] = hit ? b.prim : vtk::kMiss;
    h[1] = hit ? b.inst : vtk::kMiss;
    h[2] = hit ? vtk::f2u(b.t) : 0x7F800000u;
    h[3] = hit ? vtk::f2u(b.u) : 0u;
    h[4] = hit ? vtk::f2u(b.v) : 0u;
    if (p.hit_pos) {
      float* hp = p.hit_pos + 3 * (size_t)i;
      hp[0] = b.pos.x;
      hp[1] = b.pos.y;
      hp[2] = b.pos.z;
    }
  }
}

hipError_t launch_trace(const Params& p, uint32_t grid, hipStream_t s) {
  if (grid == 0) return hipSuccess;
  hipLaunchKernelGGL(trace_cwbvh_kernel, dim3(grid), dim3(128), 0, s, p);
  return hipGetLastError();
}

}  // namespace vtw
