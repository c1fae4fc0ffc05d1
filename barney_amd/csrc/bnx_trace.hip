// bnx_trace.hip -- two-level closest-hit / any-hit traversal on gfx950.
//
// Replaces TraceInterface::traceRay (rtcore/cuda/TraceInterface.h:24-139,
// CPU: rtcore/cpu/Device.cpp:112-201) together with the trace kernel of
// kernels/traceRays.dev.cu:26-54.
//
// Design (wave64):
//   * as many waves as fit (five per SIMD: the walk's 96 registers, of which
//     the plain and the ray-array kernels spill none and the extended ones 19
//     to 23; seven with 19 to 39 spilled took 34.2 ms where five take 26.4,
//     secondary rays of 37.5M primitives, 1920x1080, 8 spp) share a
//     generation's rays out in chunks (Claims) and take new rays as walks
//     end, so short walks do not idle behind the wave's longest; many rays in
//     a world of few primitives go one to a thread instead (few_prims);
//   * a wave runs one kind of step a trip, the one most of its lanes are at
//     (a node, a leaf, into or out of an instance), so that it does not pay
//     for every kind on every trip.  Bound by VALU issue where it has rays
//     for all waves; the 128-byte nodes and 48-byte triangles come from L2
//     and beyond.  One ray a thread until its walk ended, either kind of step
//     per trip: the same frame's traces 48.3 ms, a batch of 60001 rays 170 us
//     (112 now), a million any-hit rays 580 us (303);
//   * nearest-child-first traversal of a 4-wide BVH (collapsed from the
//     binary build) over 128-byte nodes: the four child boxes in one fetch
//     (seven 16-byte loads, near and far planes told apart by their offsets, not
//     by compares), entry distances ordered by a sorting network;
//   * short stack: a 16-entry ring per lane in LDS laid out [entry][lane]
//     (bank-conflict free), spilling its oldest entries to a per-lane
//     private array when deeper;
//   * two levels: a TLAS leaf pushes a LEAVE marker and switches the ray to
//     object space (enterBlas, rtcore/cuda/TraceInterface.h:107-122);
//   * primitive programs are a closed type switch (triangles / spheres)
//     instead of SBT function pointers (rtcore/cuda/Geom.h:21-36);
//   * ties in t go to the lower (instance, geometry, primitive) ID, and a
//     box whose entry distance equals the current best is still visited;
//   * the extended kernels (EXT) add the cylinder leaf test and the
//     renderer's cut plane, which rejects surface hits on its negative side
//     in every trace (OptixGlobals::hitOnInvisibleSide, render/
//     OptixGlobals.h:36-45); worlds without cylinders traced without a cut
//     plane keep the plain kernels and their register allocation.
#include "bnx_claims.h"
#include "bnx_internal.h"
#include "bnx_render.h"

#include <algorithm>

namespace bnx {
namespace {

constexpr int TB = 256;        // threads per block
// waves per SIMD the queue-trace kernels are compiled for (register budget:
// 512 / waves VGPRs); the walks are latency bound, so more resident waves
// hide more of each dependent node fetch
#ifndef BNX_TRACE_WAVES
#define BNX_TRACE_WAVES 5
#endif
// traversal stack: the top SH entries per lane in an LDS ring (SH a power
// of two: 8, 16 or 32, chosen per device; 16 by default), the rest spilled
// to a private array, STACK_CAP entries in all whatever SH is
constexpr int STACK_CAP = 192;
constexpr int API_SHORT = 16;  // the ray-array entry point's ring
// Chunks a wave of a frame's trace, where there are as many rays: pixels next
// to each other differ by what they see.  (An array's rays are dealt without:
// a million random any-hit rays, 314 us so and 345 in chunks of 128.)
constexpr int BALANCE = 2;
constexpr int TAKE = 16;       // idle lanes that make a wave take new rays

struct HitRec {
  float t, u, v;
  int prim, geom, inst;
};

BNX_D bool id_less(int i0, int g0, int p0, int i1, int g1, int p1)
{
  if (i0 != i1) return i0 < i1;
  if (g0 != g1) return g0 < g1;
  return p0 < p1;
}

BNX_D bool accept_t(float t, const HitRec &b, int inst, int geom, int prim)
{
  if (t < b.t) return true;
  if (t > b.t) return false;
  return b.prim < 0 ? false : id_less(inst, geom, prim, b.inst, b.geom, b.prim);
}

// The cut plane (nx, ny, nz, w; off when w <= -1e28) and the ray's world
// frame (its queue record: origin at rorg, direction at rdir).  Every
// surface program of the reference rejects a hit at t whose world position
// org + t dir lies on the plane's negative side (OptixGlobals::
// hitOnInvisibleSide, render/OptixGlobals.h:36-45; Triangles.dev.cu:39,
// Spheres.dev.cu:170, Cylinders.dev.cu:258).  t is the same in the object
// frame of an instance, whose transform is affine.
//
// Stochastic opacity (EXT kernels): a triangle of a geometry whose alpha can
// be below 1 (GeomDev::translucent) is kept as a candidate only with
// probability alpha (Triangles.dev.cu:120-133).  Its draw is taken from a
// copy of the ray's RNG state advanced by the bits of the candidate's
// object-space position, so each candidate's fate depends on the ray and the
// candidate alone and the closest kept candidate is the same in any
// traversal order (the reference advances the ray's own state, in its
// traversal order).  rng null: every surface is opaque (the ray-array entry
// point).  The closest candidate the opacity test rejected goes to rej: the
// ID channels report the closest candidate whatever its opacity
// (Triangles.dev.cu:45-60).
struct Cut {
  float4 plane;
  const float4 *rorg, *rdir;
  const uint64_t *rng;
  const SceneDev *S;
  int geom_base;          // the walk's instance: its first geometry-table entry
  bool translucent;       // its BLAS holds a translucent geometry
  HitRec *rej;
};
BNX_D Cut no_cut()
{
  return Cut{make_float4(0.f, 0.f, 0.f, -1e30f), nullptr, nullptr, nullptr, nullptr, 0, false, nullptr};
}

// whether the candidate (triangle prim of geometry G at barycentrics u, v,
// rtc instance inst) survives its opacity draw
BNX_D bool opacity_keeps(const SceneDev &S, const GeomDev &G, int inst, int prim, float u, float v, uint64_t seed)
{
  const int *ix = G.indices + 3 * prim;
  const v3 v0 = ld3(G.vertices + 3 * ix[0]), v1 = ld3(G.vertices + 3 * ix[1]), v2 = ld3(G.vertices + 3 * ix[2]);
  const v3 osP = (((1.f - u) - v) * v0 + u * v1) + v * v2;
  const InstDev &I = S.insts[inst];
  const v3 P = I.identity ? osP : xfm_point_rows(I.o2w, osP);
  const float4 base = material_color(S, G, inst, prim, tri_corners(ix, prim, u, v), make_float4(0.f, 0.f, 0.f, 1.f),
                                     P, osP);
  const float alpha = material_alpha(G, base);
  if (alpha < 1.f) {
    rng_next_h(seed, (uint64_t)__float_as_uint(osP.x));
    rng_next_h(seed, (uint64_t)__float_as_uint(osP.y));
    rng_next_h(seed, (uint64_t)__float_as_uint(osP.z));
    Random2 rng(seed, 290374u);
    if (rng() > alpha) return false;
  }
  return true;
}
template <bool EXT> BNX_D bool cut_rejects(const Cut &c, float t)
{
  if (!EXT || c.plane.w <= -1e28f) return false;
  const v3 o = xyz(*c.rorg);
  const v3 d = fix_dir(xyz(*c.rdir));
  const v3 P = o + t * d;
  return dot(v3{c.plane.x, c.plane.y, c.plane.z}, P) + c.plane.w < 0.f;
}

// barney's triangle test (rtcore/hiprt/TraceInterface.h:38-76) on a BVH-
// ordered record (v0|prim, e1|geom, e2); acceptance under the tie rule.
// Evaluated without early exits: the reference's returns (a ray parallel to
// the plane, t behind tmin, a degenerate projection, a point outside the
// triangle) become one acceptance test after the three divisions, which
// keeps a wave's lanes together through the test and lets the three record
// loads issue at once (the values of every accepted hit are the same
// operations as the reference's, in the same order)
template <bool EXT>
BNX_D bool tri_test(float4 A, float4 B, float4 C, v3 o, v3 d, float tmin, HitRec &best, int inst, const Cut &cut)
{
  const v3 v0 = xyz(A), e1 = xyz(B), e2 = xyz(C);
  const int prim = __float_as_int(A.w), geom = __float_as_int(B.w);
  const v3 N = cross(e1, e2);
  const float dn = dot(d, N);
  const float t = -dot(o - v0, N) / dn;
  const v3 P = (o - v0) + t * d;
  const bool px = fabsf(N.x) >= fmx(fabsf(N.y), fabsf(N.z));
  const bool pz = !px && !(fabsf(N.y) > fabsf(N.z));
  const float e1u = px ? e1.y : e1.x, e2u = px ? e2.y : e2.x, Pu = px ? P.y : P.x;
  const float e1v = pz ? e1.y : e1.z, e2v = pz ? e2.y : e2.z, Pv = pz ? P.y : P.z;
  const float den = e1u * e2v - e1v * e2u;
  const float u = (Pu * e2v - Pv * e2u) / den;
  const float v = (e1u * Pv - e1v * Pu) / den;
  const bool in = !(fabsf(dn) < 1e-12f) & !(t <= tmin) & !(den == 0.f) & !(u < 0.f) & !(v < 0.f) & !((u + v) >= 1.f);
  if (!in || !accept_t(t, best, inst, geom, prim)) return false;
  if (cut_rejects<EXT>(cut, t)) return false;
  if (EXT && cut.translucent && cut.rng) {
    const GeomDev &G = cut.S->geoms[cut.geom_base + geom];
    if (G.translucent && !opacity_keeps(*cut.S, G, inst, prim, u, v, *cut.rng)) {
      HitRec &r = *cut.rej;
      if (t < r.t || (t == r.t && (r.prim < 0 || id_less(inst, geom, prim, r.inst, r.geom, r.prim))))
        r = HitRec{t, u, v, prim, geom, inst};
      return false;
    }
  }
  best = HitRec{t, u, v, prim, geom, inst};
  return true;
}

// SpheresPrograms::intersect (Spheres.dev.cu:114-166), "move the origin"
template <bool EXT>
BNX_D bool sphere_test(float4 S, const int2 *ref, v3 o, v3 d, float tmin, HitRec &best, int inst, const Cut &cut)
{
  v3 center = xyz(S);
  float radius = S.w;
  float t_move = fmx(0.f, length(center - o) - 3.f * radius);
  v3 om = o + t_move * d;
  float tmin_l = fmx(0.f, tmin - t_move);
  v3 oc = om - center;
  float a = dot(d, d);
  float b = dot(oc, d);
  float c = dot(oc, oc) - radius * radius;
  float disc = b * b - a * c;
  if (disc < 0.f) return false;
  float sq = sqrtf(disc);
  float r1 = (-b - sq) / a;
  float r2 = (-b + sq) / a;
  float cand;
  if (r1 > tmin_l) cand = r1;
  else if (r2 > tmin_l) cand = r2;
  else return false;
  float t = cand + t_move;
  if (t > best.t) return false;
  int2 r = *ref;
  if (!accept_t(t, best, inst, r.x, r.y)) return false;
  if (cut_rejects<EXT>(cut, t)) return false;
  best = HitRec{t, cand, 0.f, r.y, r.x, inst};
  return true;
}

// The user geometries with two records per primitive: cylinders
// (CylindersPrograms::intersect, native/geometry/Cylinders.dev.cu:107-260,
// records (v0, radius), (v1, 0)), capsules (CapsulesPrograms::intersect,
// Capsules.dev.cu:154-300, records (v0, r0), (v1, r1)) and cones
// (ConesPrograms::intersect, Cones.dev.cu:60-266, records (p0, ra),
// (p1, rb)).  The reference intersects them against the ray's closest hit
// so far; capsules and cones take only candidates strictly nearer, so they
// are given a bound just above it and a candidate at exactly the closest
// distance reaches the tie rule (the nearest candidate below the bound does
// not depend on the bound).  u keeps the hit distance for the shading.
BNX_D float tie_bound(float t) { return t * 1.0001f; }

// whether a capsule candidate at t survives its opacity draw (Capsules.dev.
// cu:266-280): the material's alpha from the hit attributes, the draw from
// Random(ray seed, hash(rtc instance, geometry, primitive)) taken on a copy
// of the ray's state, so that the candidate's fate depends on the ray and
// the candidate alone
BNX_D bool capsule_keeps(const SceneDev &S, const GeomDev &G, int inst, int geom, int prim, float4 A, float4 B, v3 o,
                         v3 d, float t, uint64_t seed)
{
  PairHit h;
  capsule_hit(S.insts[inst], A, B, o, d, t, h);
  const float4 base = material_color(S, G, inst, prim, pair_corners(G, prim, h.lerp), make_float4(0.f, 0.f, 0.f, 1.f),
                                     h.P, h.osP);
  const float alpha = material_alpha(G, base);
  if (alpha < 1.f) {
    const uint64_t hv = fnv3((uint32_t)inst, (uint32_t)geom, (uint32_t)prim);
    rng_next_h(seed, hv ? hv : 290374ull);
    const float r = (float)(rng_next(seed) & 0x00FFFFFFu) * (1.f / (float)0x01000000);
    if (r > alpha) return false;
  }
  return true;
}

BNX_D bool pair_test(int type, const float4 *rec, const int2 *ref, v3 o, v3 d, float tmin, HitRec &best, int inst,
                     const Cut &cut)
{
  const float4 A = rec[0], B = rec[1];
  float t;
  bool h;
  if (type == BLAS_CYLINDERS) h = cyl_intersect(o, d, xyz(A), xyz(B), A.w, tmin, best.t, t, nullptr);
  else if (type == BLAS_CAPSULES) h = capsule_intersect(o, d, A, B, tie_bound(best.t), t, nullptr, nullptr);
  else h = cone_intersect(o, d, A, B, tmin, tie_bound(best.t), t, nullptr, nullptr);
  if (!h) return false;
  const int2 r = *ref;
  if (!accept_t(t, best, inst, r.x, r.y)) return false;
  if (type == BLAS_CAPSULES && cut.translucent && cut.rng) {
    const GeomDev &G = cut.S->geoms[cut.geom_base + r.x];
    if (G.translucent && !capsule_keeps(*cut.S, G, inst, r.x, r.y, A, B, o, d, t, *cut.rng)) return false;
  }
  if (cut_rejects<true>(cut, t)) return false;
  best = HitRec{t, t, 0.f, r.y, r.x, inst};
  return true;
}

struct Counts {
  uint32_t nodes, tris, spheres;
};

// the BLAS a ray is in
struct Blas {
  const Node4 BNX_G *nodes;
  const float4 BNX_G *prims;
  const int2 BNX_G *refs;
  int type, inst, geom_base;
  bool translucent;
};

// the tests of a leaf (at most 4 primitives): whether one was accepted.  The
// records are fetched two triangles or four spheres at a time, ahead of the
// tests.
template <bool EXT>
BNX_D bool leaf_test(uint32_t code, const Blas &b, v3 o, v3 d, float tmin, HitRec &best, const Cut &cut, Counts &cnt)
{
  const uint32_t first = (code & ~LEAF_BIT) >> 3;
  const int count = (int)(code & 7u);
  bool found = false;
  if (b.type == BLAS_TRIANGLES) {
    cnt.tris += count;
    for (int k = 0; k < count; k += 2) {
      const float4 BNX_G *r = b.prims + 3 * (size_t)(first + k);
      const float4 BNX_G *s = b.prims + 3 * (size_t)(first + min(k + 1, count - 1));
      const float4 A = r[0], B = r[1], C = r[2], D = s[0], E = s[1], F = s[2];
      found |= tri_test<EXT>(A, B, C, o, d, tmin, best, b.inst, cut);
      if (k + 1 < count) found |= tri_test<EXT>(D, E, F, o, d, tmin, best, b.inst, cut);
    }
    return found;
  }
  cnt.spheres += count;
  if (!EXT || b.type == BLAS_SPHERES) {
    float4 s[4];
#pragma unroll
    for (int k = 0; k < 4; k++) s[k] = b.prims[first + min(k, count - 1)];
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (k < count)
        found |= sphere_test<EXT>(s[k], (const int2 *)b.refs + first + k, o, d, tmin, best, b.inst, cut);
  } else {
    for (int k = 0; k < count; k++)
      found |= pair_test(b.type, (const float4 *)b.prims + 2 * (first + k), (const int2 *)b.refs + first + k, o, d,
                         tmin, best, b.inst, cut);
  }
  return found;
}

// The ray in the world frame, read again from its record (origin at rorg,
// direction at rdir) when a walk leaves an instance, rather than held in
// registers for the whole walk: the walks are short of registers, and a
// ray changes frame only on entering and leaving an instance.
BNX_D void world_ray(const float4 *rorg, const float4 *rdir, v3 &o, v3 &d, v3 &inv)
{
  o = xyz(*rorg);
  d = fix_dir(xyz(*rdir));
  inv = v3{1.f / d.x, 1.f / d.y, 1.f / d.z};
}

// the ray in an instance's object frame
BNX_D void instance_ray(const float4 w2o[3], const float4 *rorg, const float4 *rdir, v3 &o, v3 &d, v3 &inv)
{
  o = xfm_point_rows(w2o, xyz(*rorg));
  d = fix_dir(xfm_vector_rows(w2o, fix_dir(xyz(*rdir))));
  inv = v3{1.f / d.x, 1.f / d.y, 1.f / d.z};
}

// into the instance of TLAS leaf entry e: its BLAS, and, if it moves the ray
// (XF), the ray in its frame.  false: the ray is not finite there (the
// instance's transform flattens it, and has no inverse) and hits nothing.
template <bool XF>
BNX_D bool enter_instance(const EnterDev BNX_G *e, const float4 *rorg, const float4 *rdir, Blas &b, v3 &o, v3 &d,
                          v3 &inv)
{
  const EnterDev E = *e;
  b = Blas{E.nodes, E.prims, E.refs, E.type, E.inst, E.geom_base, E.translucent != 0};
  if (!XF || E.identity) return true;
  instance_ray(E.w2o, rorg, rdir, o, d, inv);
  return finite(o) && finite(d);
}

// entry distance of child k of a 4-wide node, +inf when the ray misses it.
// Branch-free, so the six box vectors of a node are loaded together up front
// (a short-circuit on the child code let the compiler sink each child's box
// loads behind the code load, doubling the dependent fetches per node).
// Rays are finite, |inv| <= 1e6 (|d| >= 1e-6 after fix_dir) and empty slots
// hold inverted infinite boxes, so no slab distance is NaN and fminf/fmaxf
// give the same values as compares.
BNX_D float child_entry(v3 o, v3 inv, float lx, float hx, float ly, float hy, float lz, float hz, uint32_t code,
                        float tmin, float tmax)
{
  const float t0x = (lx - o.x) * inv.x, t1x = (hx - o.x) * inv.x;
  const float t0y = (ly - o.y) * inv.y, t1y = (hy - o.y) * inv.y;
  const float t0z = (lz - o.z) * inv.z, t1z = (hz - o.z) * inv.z;
  const float tn = fmaxf(fmaxf(fmaxf(tmin, fminf(t0x, t1x)), fminf(t0y, t1y)), fminf(t0z, t1z));
  const float tf = fminf(fminf(fminf(tmax, fmaxf(t0x, t1x)), fmaxf(t0y, t1y)), fmaxf(t0z, t1z));
  const bool h = (tn <= tf * 1.00001f) & (code != EMPTY4);
  return h ? tn : __builtin_huge_valf();
}


BNX_D void cswap(float &ta, uint32_t &ca, float &tb, uint32_t &cb)
{
  const bool s = tb < ta;
  const float t = s ? tb : ta;
  const uint32_t c = s ? cb : ca;
  tb = s ? ta : tb;
  cb = s ? ca : cb;
  ta = t;
  ca = c;
}

// the near and the far plane of a node's axis lie 16 bytes apart; a ray that
// runs down an axis has them the other way round.  `near`: byte offsets of
// the near planes, per ray
struct Octant {
  uint32_t x, y, z;
};
BNX_D Octant octant_of(v3 d)
{
  return Octant{d.x < 0.f ? 16u : 0u, d.y < 0.f ? 48u : 32u, d.z < 0.f ? 80u : 64u};
}

// entry distance of a child whose near and far planes are known, +inf when
// the ray misses it.  |inv| <= 1e6 (|d| >= 1e-6 after fix_dir), so the
// distances are those of the slab test with its minima and maxima taken:
// (plane - o) * inv is monotone in the plane.  An empty slot's planes are
// inverted infinities: its entry lies behind its exit for every finite ray,
// and a ray that is not finite never comes here.
BNX_D float slab_entry(v3 o, v3 inv, float nx, float fx, float ny, float fy, float nz, float fz, float tmin, float tmax)
{
  const float tn = fmaxf(fmaxf(fmaxf(tmin, (nx - o.x) * inv.x), (ny - o.y) * inv.y), (nz - o.z) * inv.z);
  const float tf = fminf(fminf(fminf(tmax, (fx - o.x) * inv.x), (fy - o.y) * inv.y), (fz - o.z) * inv.z);
  return tn <= tf * 1.00001f ? tn : __builtin_huge_valf();
}

// The walk of a wave.  Every lane walks its own ray (one node, or one leaf,
// or into or out of an instance at a time, nearest child first) and the wave
// runs, trip by trip, the kind of step that most of its lanes are at; lanes
// whose rays have ended store their hits and take the next rays of the
// wave's share together, once `take` of them are free.  A ray's own steps do
// not depend on its wave.
//
// SRC: where rays come from and hits go (queue, ray array).  XF: some
// instance transforms the ray; without it the frame never changes, so the
// ray is not set up again.  EXT: see k_trace_static.
template <int SH, bool EXT, bool XF, typename SRC>
BNX_D void walk_rays(Claims &pr, const SceneDev &S, const SRC &src, int take, uint32_t *ring, Counts &cnt)
{
  const int lane = lane_id();
  // stack: entries [low, sp) in the lane's ring, those below spilled.  Four
  // move at a time, so that a node's pushes need no test of their own.
  uint32_t *const lds = ring + lane;
  uint32_t deep[STACK_CAP];
  int sp = 0, low = 0;
  auto slot = [&](int i) -> uint32_t & { return lds[(i & (SH - 1)) * 64]; };
  auto room = [&]() {
    if (sp - low > SH - 4) {
      for (int k = 0; k < 4; k++) deep[low + k] = slot(low + k);
      low += 4;
    }
  };
  uint32_t cur = EMPTY4;              // EMPTY4: no ray, or one that has ended
  auto pop = [&]() {
    if (sp == low && sp > 0) {
      low -= 4;
      for (int k = 0; k < 4; k++) slot(low + k) = deep[low + k];
    }
    const uint32_t v = slot(sp - 1);
    cur = sp > 0 ? v : EMPTY4;
    sp = max(sp - 1, 0);
  };
  int ray = -1;
  bool any_hit = false, in_blas = false;
  float tmin = 0.f;
  v3 o{0.f, 0.f, 0.f}, d{1.f, 1.f, 1.f}, inv{1.f, 1.f, 1.f};
  Octant oct{0, 32, 64};
  HitRec best{0.f, 0.f, 0.f, -1, -1, -1}, rej{0.f, 0.f, 0.f, -1, -1, -1};
  const Node4 BNX_G *nodes = S.tlas_nodes;
  Blas blas{};
  // every node is entered at most once per ray: the walks, and so the loop,
  // end
  for (;;) {
    const uint64_t idle = __ballot(cur == EMPTY4);
    const int n_idle = __popcll(idle);
    if (n_idle >= take && !pr.dry) {
      if (cur == EMPTY4 && ray >= 0) src.store(S, ray, best, rej);
      bool on;
      const int i = pr.claim(n_idle, __popcll(idle & lanemask_lt()), on);
      if (cur == EMPTY4) {
        ray = -1;
        if (on) {
          ray = i;
          float tmax;
          src.load(i, o, d, tmin, tmax, any_hit);
          d = fix_dir(d);
          inv = v3{1.f / d.x, 1.f / d.y, 1.f / d.z};
          oct = octant_of(d);
          best = HitRec{tmax, 0.f, 0.f, -1, -1, -1};
          if (EXT) rej = HitRec{__builtin_huge_valf(), 0.f, 0.f, -1, -1, -1};
          nodes = S.tlas_nodes;
          in_blas = false;
          sp = low = 0;
          // a ray that is not finite would pass every slab test, those of
          // unused child slots too, and no hit could come of it
          cur = S.num_insts > 0 && finite(o) && finite(d) ? 0 : EMPTY4;
        }
      }
      continue;
    }
    if (n_idle == 64) break;
    const int n_node = __popcll(__ballot(cur < EMPTY4));
    const int n_leaf = __popcll(__ballot(in_blas && (cur & LEAF_BIT) != 0));
    const int n_turn = 64 - n_idle - n_node - n_leaf;
    if (n_node >= n_leaf && n_node >= n_turn) {
      // ------------------------------------------------ 4-wide inner node
      if (cur < EMPTY4) {
        cnt.nodes++;
        const char BNX_G *np = (const char BNX_G *)(nodes + cur);
        auto plane = [&](uint32_t off) -> float4 { return *(const float4 BNX_G *)(np + off); };
        const float4 nx = plane(oct.x), fx = plane(oct.x ^ 16u), ny = plane(oct.y), fy = plane(oct.y ^ 16u),
                     nz = plane(oct.z), fz = plane(oct.z ^ 16u);
        const uint4 ch = *(const uint4 BNX_G *)(np + 96);
        float t0 = slab_entry(o, inv, nx.x, fx.x, ny.x, fy.x, nz.x, fz.x, tmin, best.t);
        float t1 = slab_entry(o, inv, nx.y, fx.y, ny.y, fy.y, nz.y, fz.y, tmin, best.t);
        float t2 = slab_entry(o, inv, nx.z, fx.z, ny.z, fy.z, nz.z, fz.z, tmin, best.t);
        float t3 = slab_entry(o, inv, nx.w, fx.w, ny.w, fy.w, nz.w, fz.w, tmin, best.t);
        uint32_t c0 = ch.x, c1 = ch.y, c2 = ch.z, c3 = ch.w;
        // nearest first: a 4-element sorting network on the entry distances
        cswap(t0, c0, t1, c1);
        cswap(t2, c2, t3, c3);
        cswap(t0, c0, t2, c2);
        cswap(t1, c1, t3, c3);
        cswap(t1, c1, t2, c2);
        const float INF = __builtin_huge_valf();
        room();
        slot(sp) = c3;
        sp += t3 < INF ? 1 : 0;
        slot(sp) = c2;
        sp += t2 < INF ? 1 : 0;
        slot(sp) = c1;
        sp += t1 < INF ? 1 : 0;
        cur = c0;
        if (!(t0 < INF)) pop();
      }
    } else if (n_leaf >= n_turn) {
      // ------------------------------------------------------------ leaf
      if (in_blas && (cur & LEAF_BIT) != 0) {
        const Cut cut = EXT ? src.cut(S, ray, blas.geom_base, blas.translucent, &rej) : no_cut();
        const bool found = leaf_test<EXT>(cur, blas, o, d, tmin, best, cut, cnt);
        if (any_hit && found) cur = EMPTY4;
        else pop();
      }
    } else if (cur == LEAVE_BLAS) {
      // ------------------------------------------- out of an instance, ...
      in_blas = false;
      if (XF) {
        world_ray(src.org(ray), src.dir(ray), o, d, inv);
        oct = octant_of(d);
      }
      nodes = S.tlas_nodes;
      pop();
    } else if (!in_blas && (cur & LEAF_BIT) != 0) {
      // ------------------------------------ ... or a TLAS leaf: into its own
      const uint32_t entry = (cur & ~LEAF_BIT) >> 3;
      cur = LEAVE_BLAS;
      if (enter_instance<XF>(S.enter + entry, src.org(ray), src.dir(ray), blas, o, d, inv)) {
        if (XF) oct = octant_of(d);
        room();
        slot(sp++) = LEAVE_BLAS;
        nodes = blas.nodes;
        cur = 0;
      }
      in_blas = true;
    }
  }
  if (ray >= 0) src.store(S, ray, best, rej);
}

// The walk of a ray in speculative while-while order (Aila and Laine,
// "Understanding the Efficiency of Ray Traversal on GPUs", HPG 2009): a
// lane that reaches a primitive leaf sets it aside and keeps stepping inner
// nodes from its stack while other lanes of the wave still step nodes, until
// every lane with a node to step already holds a leaf (or none has a node);
// then the lanes test their leaves together.  Each trip of the wave thus
// serves either node steps or leaf tests for most of its lanes, where the
// plain walk pays for both whenever its lanes are split between them.  A
// node is culled against the best hit known when it is stepped, so a lane
// may step nodes that a hit in its pending leaf would have culled; the hit
// returned is the same (equal t resolves by ID).  cur == EMPTY4: the stack
// is exhausted.
template <int SH, bool EXT, bool XF>
BNX_D HitRec traverse_spec(const SceneDev &S, const float4 *rorg, const float4 *rdir, float tmin, float tmax,
                           bool any_hit, uint32_t *lds, Counts &cnt, float4 cut_plane, const uint64_t *rng,
                           HitRec &rej)
{
  Cut cut{cut_plane, rorg, rdir, rng, &S, 0, false, &rej};
  uint32_t deep[STACK_CAP - SH];
  int sp = 0;
  auto push = [&](uint32_t v) {
    const int s = sp & (SH - 1);
    if (sp >= SH) deep[sp - SH] = lds[s * TB];
    lds[s * TB] = v;
    sp++;
  };
  auto pop = [&]() -> uint32_t {
    if (sp == 0) return EMPTY4;
    sp--;
    const int s = sp & (SH - 1);
    const uint32_t v = lds[s * TB];
    if (sp >= SH) lds[s * TB] = deep[sp - SH];
    return v;
  };
  HitRec best{tmax, 0.f, 0.f, -1, -1, -1};
  v3 o, d, inv;
  world_ray(rorg, rdir, o, d, inv);
  const Node4 BNX_G *nodes = S.tlas_nodes;
  Blas blas{};
  bool in_blas = false;
  uint32_t cur = finite(o) && finite(d) ? 0 : EMPTY4;
  uint32_t leaf = 0;             // primitive leaf set aside (leaf codes carry LEAF_BIT)
  uint32_t nvis = 0;
  // every node is entered at most once per ray; the cap only bounds the
  // loops if the structure were corrupted
  uint32_t trips = 0;
  while (trips < (1u << 28)) {
    // ------------------------------------------------------- node phase
    for (;; trips++) {
      if (leaf == 0 && in_blas && (cur & LEAF_BIT)) {
        leaf = cur;
        cur = pop();
      }
      const bool step = cur < EMPTY4;
      if (!__any(step && leaf == 0) || trips >= (1u << 28)) break;
      if (step) {
        const float4 *np = (const float4 *)(nodes + cur);
        const float4 lx = np[0], hx = np[1], ly = np[2], hy = np[3], lz = np[4], hz = np[5];
        const uint4 ch = ((const uint4 *)np)[6];
        nvis++;
        float t0 = child_entry(o, inv, lx.x, hx.x, ly.x, hy.x, lz.x, hz.x, ch.x, tmin, best.t);
        float t1 = child_entry(o, inv, lx.y, hx.y, ly.y, hy.y, lz.y, hz.y, ch.y, tmin, best.t);
        float t2 = child_entry(o, inv, lx.z, hx.z, ly.z, hy.z, lz.z, hz.z, ch.z, tmin, best.t);
        float t3 = child_entry(o, inv, lx.w, hx.w, ly.w, hy.w, lz.w, hz.w, ch.w, tmin, best.t);
        uint32_t c0 = ch.x, c1 = ch.y, c2 = ch.z, c3 = ch.w;
        cswap(t0, c0, t1, c1);
        cswap(t2, c2, t3, c3);
        cswap(t0, c0, t2, c2);
        cswap(t1, c1, t3, c3);
        cswap(t1, c1, t2, c2);
        const float INF = __builtin_huge_valf();
        if (t0 < INF) {
          if (t3 < INF) push(c3);
          if (t2 < INF) push(c2);
          if (t1 < INF) push(c1);
          cur = c0;
        } else {
          cur = pop();
        }
      }
    }
    // ------------------------------------------------------- leaf phase
    bool found = false;
    if (leaf != 0) {
      found = leaf_test<EXT>(leaf, blas, o, d, tmin, best, cut, cnt);
      leaf = 0;
    } else if ((cur & LEAF_BIT) && !in_blas) {
      // a TLAS leaf (the node phase sets every BLAS leaf aside): enter its
      // instance
      const bool in = enter_instance<XF>(S.enter + ((cur & ~LEAF_BIT) >> 3), rorg, rdir, blas, o, d, inv);
      if (EXT) {
        cut.geom_base = blas.geom_base;
        cut.translucent = blas.translucent;
      }
      if (in) push(LEAVE_BLAS);
      in_blas = true;
      nodes = blas.nodes;
      cur = in ? 0 : LEAVE_BLAS;
    } else if (cur == LEAVE_BLAS) {
      in_blas = false;
      if (XF) world_ray(rorg, rdir, o, d, inv);
      nodes = S.tlas_nodes;
      cur = pop();
    }
    if ((any_hit && found) || (cur == EMPTY4 && leaf == 0)) break;
    trips++;
  }
  cnt.nodes += nvis;
  return best;
}

// Into how many chunks a launch is cut at least.  Half as many as waves: full
// waves before all waves (20k triangles, 512x512, 1 spp: 406 us in three
// launches, and 552 with a chunk for each; 60001 rays: 111 and 135).  The
// extended kernels run a leaf step once for each kind of primitive in the
// wave, and a wave with 64 long rays is one that the launch waits for: twice
// as many as waves (27 instances each of cylinders, capsules and cones,
// 641x363, 4 spp: 3.3 ms, and 4.7 with half as many).
BNX_D int least_chunks(bool ext) { return ext ? 2 * (int)gridDim.x : (int)gridDim.x / 2; }

// rays and hits of the ray-array entry point
struct ArraySource {
  const bnx_ray *rays;
  bnx_hit *hits;
  bool any;
  BNX_D const float4 *org(int i) const { return (const float4 *)(rays + i); }
  BNX_D const float4 *dir(int i) const { return (const float4 *)(rays + i) + 1; }
  BNX_D void load(int i, v3 &o, v3 &d, float &tmin, float &tmax, bool &any_hit) const
  {
    const float4 r0 = *org(i), r1 = *dir(i);
    o = xyz(r0);
    d = xyz(r1);
    tmin = r0.w;
    tmax = r1.w;
    any_hit = any;
  }
  BNX_D Cut cut(const SceneDev &, int, int, bool, HitRec *) const { return no_cut(); }
  BNX_D void store(const SceneDev &S, int i, const HitRec &h, const HitRec &) const
  {
    bnx_hit out;
    out.t = h.t;
    out.u = h.prim >= 0 ? h.u : 0.f;
    out.v = h.prim >= 0 ? h.v : 0.f;
    out.prim_id = h.prim;
    if (h.prim >= 0) {
      const InstDev &I = *(const InstDev *)(S.insts + h.inst);
      out.geom_id = h.geom;
      out.inst = h.inst;
      out.user_inst_id = I.user_id;
      out.obj_id = S.geoms[I.geom_base + h.geom].user_id;
    } else {
      out.geom_id = out.inst = out.user_inst_id = out.obj_id = -1;
    }
    hits[i] = out;
  }
};

template <bool EXT, bool XF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(BNX_TRACE_WAVES))) void k_trace_api(
    SceneDev S, const bnx_ray *rays, int n, bnx_hit *hits, uint32_t flags, int *claims, int least)
{
  __shared__ uint32_t ring[API_SHORT * 64];
  Claims cl;
  cl.begin(n, claims, least, EXT ? BALANCE * (int)gridDim.x : 0);
  Counts cnt{0, 0, 0};
  const ArraySource src{rays, hits, (flags & BNX_TRACE_ANY) != 0};
  walk_rays<API_SHORT, EXT, XF>(cl, S, src, TAKE, ring, cnt);
}

// A translucent candidate the opacity test rejected lies in front of the
// ray's hit: for a primary ray of a request's first sample the trace writes
// the ID channels from it (as the reference's any-hit program writes them
// before the opacity test, Triangles.dev.cu:45-60) and flags the ray so that
// shade leaves them.
BNX_D void translucent_ids(const SlotDev &P, const TraceQueue &q, int i, float4 d, const HitRec &rej)
{
  const uint4 ps = q.ps[i];
  const uint32_t f = __float_as_uint(d.w);
  if ((ps.y >> 24) != 0 || (f & FLAG_SHADOW) || P.accum_base + flag_sample(f) != 0) return;
  const int pixel = (int)ps.z;
  const InstDev &I = P.scene.insts[rej.inst];
  P.fb.prim[pixel] = rej.prim;
  P.fb.inst[pixel] = I.user_id;
  P.fb.obj[pixel] = P.scene.geoms[I.geom_base + rej.geom].user_id;
  q.dir[i].w = __uint_as_float(f | FLAG_IDS);
}

// one ray per thread over the generation's segments (256-thread block map);
// each block lies inside one request's segment, so the request's scene
// pointers are block-uniform.  counters: statistics array (STAT_NODES,
// STAT_TRIS, STAT_SPHERES)
template <int SH, bool EXT, bool XF>
BNX_D void trace_spec(const SlotDev *__restrict__ slots, const SegView &sv, const TraceQueue &q,
                      unsigned long long *counters, uint32_t *ring)
{
  uint32_t *lds = ring + threadIdx.x;
  Counts cnt{0, 0, 0};
  int i;
  bool valid;
  const Segment sg = segment_of<TB>(sv, i, valid);
  const SceneDev S = slots[sg.slot].scene;
  const float4 cut_plane = EXT ? slot_cut_plane(slots[sg.slot]) : no_cut().plane;
  if (valid) {
    float4 o = q.org[i];
    float4 d = q.dir[i];
    const bool shadow = (__float_as_uint(d.w) & FLAG_SHADOW) != 0;
    HitRec h{o.w, 0.f, 0.f, -1, -1, -1};
    HitRec rej{__builtin_huge_valf(), 0.f, 0.f, -1, -1, -1};
    if (S.num_insts > 0)
      h = traverse_spec<SH, EXT, XF>(S, q.org + i, q.dir + i, 0.f, o.w, shadow, lds, cnt, cut_plane, q.rng + i, rej);
    if (h.prim >= 0) q.org[i].w = h.t;
    q.hit[i] = make_int4(h.prim, h.geom, h.inst, __float_as_int(h.u));
    q.hit_v[i] = h.v;
    if (EXT && rej.prim >= 0 && rej.t < h.t) translucent_ids(slots[sg.slot], q, i, d, rej);
  }
  uint32_t a = wave_sum(cnt.nodes), b = wave_sum(cnt.tris), c = wave_sum(cnt.spheres);
  if (lane_id() == 0) {
    stat_add(counters, STAT_NODES, a);
    stat_add(counters, STAT_TRIS, b);
    stat_add(counters, STAT_SPHERES, c);
  }
}

// the rays of a request's segment
struct QueueSource {
  const TraceQueue &q;
  const SlotDev &P;
  float4 plane;
  BNX_D const float4 *org(int i) const { return q.org + i; }
  BNX_D const float4 *dir(int i) const { return q.dir + i; }
  BNX_D void load(int i, v3 &o, v3 &d, float &tmin, float &tmax, bool &any_hit) const
  {
    const float4 ro = q.org[i], rd = q.dir[i];
    o = xyz(ro);
    d = xyz(rd);
    tmin = 0.f;
    tmax = ro.w;
    any_hit = (__float_as_uint(rd.w) & FLAG_SHADOW) != 0;
  }
  BNX_D Cut cut(const SceneDev &S, int i, int geom_base, bool translucent, HitRec *rej) const
  {
    return Cut{plane, q.org + i, q.dir + i, q.rng + i, &S, geom_base, translucent, rej};
  }
  BNX_D void store(const SceneDev &, int i, const HitRec &h, const HitRec &rej) const
  {
    if (h.prim >= 0) q.org[i].w = h.t;
    q.hit[i] = make_int4(h.prim, h.geom, h.inst, __float_as_int(h.u));
    q.hit_v[i] = h.v;
    if (rej.prim >= 0 && rej.t < h.t) translucent_ids(P, q, i, q.dir[i], rej);
  }
};

// a wave's share of the generation, segment by segment (each one request's,
// so the scene's pointers are wave-uniform)
template <int SH, bool EXT, bool XF>
BNX_D void trace_waves(const SlotDev *__restrict__ slots, const SegView &sv, int nsegs, const TraceQueue &q,
                       unsigned long long *counters, uint32_t *ring)
{
  Claims cl;
  cl.begin(sv, nsegs, CLAIMS_TRACE, least_chunks(EXT), BALANCE * (int)gridDim.x);
  Counts cnt{0, 0, 0};
  while (cl.chunk >= 0) {
    const Segment sg = cl.open();
    const SlotDev &P = slots[sg.slot];
    const SceneDev S = uniform_load((const SceneDev BNX_G *)&P.scene);
    cl.refill();
    const QueueSource src{q, P, EXT ? slot_cut_plane(P) : no_cut().plane};
    walk_rays<SH, EXT, XF>(cl, S, src, sg.refill < 64 ? sg.refill : TAKE, ring, cnt);
  }
  const uint32_t a = wave_sum(cnt.nodes), b = wave_sum(cnt.tris), c = wave_sum(cnt.spheres);
  if (lane_id() == 0) {
    stat_add(counters, STAT_NODES, a);
    stat_add(counters, STAT_TRIS, b);
    stat_add(counters, STAT_SPHERES, c);
  }
}

// The trace of a generation.  SPEC: one ray per thread in blocks of TB, the
// speculative walk; otherwise waves that share the rays out.  EXT: the leaf
// test knows cylinder BLASes and the cut plane of each request.  The kernels
// without it serve worlds of triangles and spheres traced without a cut
// plane; the launcher takes the _ext kernels while any built world holds
// cylinders or a request in the launch has a cut plane.
template <int SH, bool SPEC, bool EXT, bool XF>
BNX_D void trace_queue(const SlotDev *__restrict__ slots, const SegView &sv, int nsegs, const TraceQueue &q,
                       unsigned long long *counters, uint32_t *ring)
{
  if constexpr (SPEC) trace_spec<SH, EXT, XF>(slots, sv, q, counters, ring);
  else trace_waves<SH, EXT, XF>(slots, sv, nsegs, q, counters, ring);
}
constexpr int trace_block(bool spec) { return spec ? TB : 64; }

template <int SH, bool SPEC, bool XF>
__global__ __launch_bounds__(trace_block(SPEC)) __attribute__((amdgpu_waves_per_eu(BNX_TRACE_WAVES))) void
k_trace_static(const SlotDev *__restrict__ slots, SegView sv, int nsegs, TraceQueue q, unsigned long long *counters)
{
  __shared__ uint32_t ring[SH * trace_block(SPEC)];
  trace_queue<SH, SPEC, false, XF>(slots, sv, nsegs, q, counters, ring);
}

template <int SH, bool SPEC, bool XF>
__global__ __launch_bounds__(trace_block(SPEC)) __attribute__((amdgpu_waves_per_eu(BNX_TRACE_WAVES))) void
k_trace_static_ext(const SlotDev *__restrict__ slots, SegView sv, int nsegs, TraceQueue q,
                   unsigned long long *counters)
{
  __shared__ uint32_t ring[SH * trace_block(SPEC)];
  trace_queue<SH, SPEC, true, XF>(slots, sv, nsegs, q, counters, ring);
}

using TraceKernel = void (*)(const SlotDev *, SegView, int, TraceQueue, unsigned long long *);
template <int SH, bool SPEC, bool XF> TraceKernel trace_kernel(bool ext)
{
  return ext ? k_trace_static_ext<SH, SPEC, XF> : k_trace_static<SH, SPEC, XF>;
}
template <int SH> TraceKernel trace_kernel(bool spec, bool ext, bool xf)
{
  if (spec) return xf ? trace_kernel<SH, true, true>(ext) : trace_kernel<SH, true, false>(ext);
  return xf ? trace_kernel<SH, false, true>(ext) : trace_kernel<SH, false, false>(ext);
}

// waves of a launch over n rays: as many as are resident at once, in whole
// rounds of the claim groups, and no more than there are chunks of 16 rays
int trace_waves_for(const Device *dev, int fit, long long blocks256)
{
  const long long waves = std::min<long long>((long long)fit * dev->num_cus, 16 * blocks256);
  return (int)std::max<long long>(CLAIM_GROUPS, waves / CLAIM_GROUPS * CLAIM_GROUPS);
}
template <typename K> int resident(K kernel, int &fit)
{
  if (fit == 0) {
    BNX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, (const void *)kernel, 64, 0));
    fit = std::max(1, fit);
  }
  return BNX_OK;
}

} // namespace

int trace_stack_capacity() { return STACK_CAP; }

int launch_trace_api(Group *g, const bnx_ray *d_rays, int n, bnx_hit *d_hits, uint32_t flags)
{
  Device *dev = g->dev;
  if (n <= 0) return BNX_OK;
  const bool ext = g->has_cyl, xf = g->has_xf;
  const auto kernel = ext ? (xf ? k_trace_api<true, true> : k_trace_api<true, false>)
                          : (xf ? k_trace_api<false, true> : k_trace_api<false, false>);
  int &fit = dev->trace_fit[12 + 2 * (ext ? 1 : 0) + (xf ? 1 : 0)];
  int rc = resident(kernel, fit);
  if (rc != BNX_OK) return rc;
  const std::lock_guard<std::mutex> one(dev->api_mutex);
  if ((rc = launch_claims_clear(dev, dev->api_claims.as<int>())) != BNX_OK) return rc;
  // Half as many chunks as waves, see least_chunks; the extended kernel's rays
  // go 16 to a wave only where there are not enough for half of the resident
  // waves at 32, and large arrays in two chunks a wave: capsules, cones and
  // cylinders, 207 of them, 113354 rays, 123 us in 64s, 133 in 32s and 198 in
  // 16s; 960 and 27 instances, 16397 rays, 464 in 16s and 524 in 32s; 2500,
  // 700000 rays, 710 in 64s and 852 in 256s.
  const int waves = trace_waves_for(dev, fit, ((long long)n + 255) / 256);
  const int least = ext ? std::min(waves, fit * dev->num_cus / 2) : waves / 2;
  kernel<<<waves, 64, 0, dev->stream>>>(
      g->scene, d_rays, n, d_hits, flags, dev->api_claims.as<int>(), least);
  BNX_HIP(hipGetLastError());
  return BNX_OK;
}

int launch_trace_queue(Device *dev, const SlotDev *slots, const SegView &sv, int nsegs, int blocks256, bool cut,
                       bool few, const TraceQueue &q, unsigned long long *counters)
{
  if (blocks256 <= 0) return BNX_OK;
  const int sh = dev->trace_stack_lds;
  const bool ext = ext_kernels(dev, cut), xf = dev->xf_worlds > 0;
  const bool spec = dev->trace_walk == 1 || (few && !ext);
  const TraceKernel kernel = sh == 8    ? trace_kernel<8>(spec, ext, xf)
                             : sh == 32 ? trace_kernel<32>(spec, ext, xf)
                                        : trace_kernel<16>(spec, ext, xf);
  if (spec) {
    kernel<<<blocks256, TB, 0, dev->stream>>>(slots, sv, nsegs, q, counters);
  } else {
    int &fit = dev->trace_fit[4 * (sh == 8 ? 0 : sh == 32 ? 2 : 1) + 2 * (ext ? 1 : 0) + (xf ? 1 : 0)];
    const int rc = resident(kernel, fit);
    if (rc != BNX_OK) return rc;
    kernel<<<trace_waves_for(dev, std::min(fit, 4 * dev->trace_blocks_per_cu), blocks256), 64, 0, dev->stream>>>(slots, sv, nsegs, q, counters);
  }
  BNX_HIP(hipGetLastError());
  return BNX_OK;
}

} // namespace bnx
