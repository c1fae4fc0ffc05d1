// bnx_march.hip -- the volume and isosurface march on gfx950: macrocell DDA
// with delta (or ratio) tracking through volumes, and root finding on
// isosurfaces, over structured, tetrahedral and mixed-cell fields.
//
// Replaces MCVolumeAccel::isProg (volume/MCAccelerator.h:550-689) and
// MCIsoSurfaceAccel::isProg (:325-548) with dda3 (volume/DDA.h:60-201),
// Woodcock::sampleRange (volume/Volume.h:154-203) and the samplers
// (StructuredData.h:101-112, UMeshCuBQLSampler.h:46-62).
//
// A ray's march is a nest of loops of data-dependent length (macrocells,
// tentative collisions or sub-steps, the cells a point query tests).  Run as
// nested loops, one ray per lane, a wave waits at every level for its slowest
// lane.  Where samples are cheap and rays run side by side that costs least
// (k_volume_rays, structured fields).  Elsewhere each lane is a small state
// machine whose state says which step its ray takes next (Mode): every trip a
// wave counts the lanes waiting for each group of steps and takes one that
// enough of them wait for.  Rays are set up 64 at a time, all lanes at work,
// and wait in LDS (those that miss the field never leave the set-up); lanes
// whose rays have ended take them from there.  A macrocell and the first
// collision in it are one group, so that a lane passes through both in a
// trip.  Every ray draws the same random numbers and takes the same steps in
// the same order in either form, so results do not change.
//
// One launch serves one program: isosurface k, or volume k, of every request
// (isosurfaces first), clipped to the closest hit so far, which the launches
// hand on in the queue.  A block is one wave: its field's parameters are
// wave-uniform and sit in scalar registers.
#include "bnx_claims.h"
#include "bnx_internal.h"
#include "bnx_render.h"
#include "bnx_volume.h"

#include <algorithm>

namespace bnx {
namespace {

// lanes waiting for a step that make a wave take it (a wave with no fuller
// group takes the fullest): the cheaper the step, the sooner.  A structured
// field is sampled when three in eight of the lanes that have a ray wait for
// it; a fixed 24 lanes made waves with few rays walk on to their slowest lane.
constexpr int BALANCE = 4;       // chunks a wave, where there are as many rays
constexpr int TAKE = 8;          // a new ray, already set up
constexpr int SEED_AT = 4;       // a tet mesh's seed
constexpr int CELL_AT = 12;      // a macrocell, where point queries are most of the work
constexpr int NODE_AT = 10;      // a depth-first query
constexpr int SIDES_AT = 24;     // the sides of a macrocell's sub-steps (isosurfaces; 16 to 32 within 1%)

// what a lane's ray waits for
enum Mode {
  M_IDLE = 0,     // a ray
  M_CELL,         // the next macrocell
  M_DRAW,         // the next tentative collision (volumes)
  M_SAMPLE,       // the field at its point (structured; tets: the seed of its point)
  M_WALK,         // a tet walk's next tet
  M_VALUE,        // to use the value that its point query gave
  M_NODE,         // an element-BVH node or leaf
  M_TEST,         // the Newton inversion of a cell
};

// dda3's state (volume/DDA.h:60-201): the walk over the macrocells of v along
// a ray in macrocell-grid space, from max(0, grid entry) to the grid exit.
// step[k]: the ray's length of a cell along axis k, negative where it walks
// down; left[k]: cells between the current one and the grid's end.
struct Dda {
  float next[3], step[3];
  float ray_t0, begin, tmax;
  int left[3], cell;
  bool over;
};

BNX_D bool dda_init(const VolumeDev &v, v3 org, v3 dir, float dda_tmax, Dda &D)
{
  const v3 dorg = v3{(org.x - v.mc_origin[0]) * v.mc_rcp_spacing[0], (org.y - v.mc_origin[1]) * v.mc_rcp_spacing[1],
                     (org.z - v.mc_origin[2]) * v.mc_rcp_spacing[2]};
  const v3 ddir = v3{dir.x * v.mc_rcp_spacing[0], dir.y * v.mc_rcp_spacing[1], dir.z * v.mc_rcp_spacing[2]};
  const float fs[3] = {(float)v.mc[0], (float)v.mc[1], (float)v.mc[2]};
  const float o3[3] = {dorg.x, dorg.y, dorg.z}, d3[3] = {ddir.x, ddir.y, ddir.z};
  float rcp[3], tn[3], tf[3];
  bool outside = false;
  for (int k = 0; k < 3; k++) {
    rcp[k] = v.rn ? rcp_rn(d3[k]) : 1.f / d3[k];
    const float a = (0.f - o3[k]) * rcp[k];
    const float b = (fs[k] - o3[k]) * rcp[k];
    tn[k] = fmn(a, b);
    tf[k] = fmx(a, b);
    if (d3[k] == 0.f) {
      outside |= o3[k] < 0.f || o3[k] > fs[k];
      tn[k] = -INFINITY;
      tf[k] = INFINITY;
    }
  }
  if (outside) return false;
  const float ray_t0 = fmx(0.f, fmx(fmx(tn[0], tn[1]), tn[2]));
  const float ray_t1 = fmn(dda_tmax, fmn(fmn(tf[0], tf[1]), tf[2]));
  if (ray_t0 > ray_t1) return false;
  int c[3];
  for (int k = 0; k < 3; k++) {
    const float oiv = o3[k] + ray_t0 * d3[k];
    const float fc = fmx(0.f, fmn(fs[k] - 1.f, floorf(oiv)));
    const float fe = d3[k] > 0.f ? fc + 1.f : fc;
    D.step[k] = d3[k] > 0.f ? fabsf(rcp[k]) : -fabsf(rcp[k]);
    D.next[k] = (d3[k] == 0.f) ? INFINITY : fabsf(fe - oiv) * fabsf(rcp[k]);
    c[k] = (int)fc;
    D.left[k] = d3[k] > 0.f ? v.mc[k] - 1 - c[k] : c[k];
  }
  D.cell = c[0] + v.mc[0] * (c[1] + v.mc[1] * c[2]);
  D.ray_t0 = ray_t0;
  D.begin = 0.f;
  D.tmax = dda_tmax;
  D.over = false;
  return true;
}

// the current cell (index, range [c0, c1]); the walk moves on to the next.
// An axis steps when its next crossing is the closest; a NaN crossing never
// steps, which ends the walk.
BNX_D int dda_cell(const VolumeDev &v, Dda &D, float &c0, float &c1)
{
  const float t = fmn(fmn(D.next[0], D.next[1]), D.next[2]);
  c0 = D.ray_t0 + D.begin;
  c1 = D.ray_t0 + fmn(t, D.tmax);
  const int cell = D.cell;
  D.begin = t;
  const int stride[3] = {1, v.mc[0], v.mc[0] * v.mc[1]};
  bool moved = false;
  for (int k = 0; k < 3; k++) {
    const bool s = D.next[k] == t;
    moved |= s;
    D.over |= s && D.left[k] == 0;
    D.next[k] = s ? D.next[k] + fabsf(D.step[k]) : D.next[k];
    D.left[k] -= s ? 1 : 0;
    D.cell += s ? (D.step[k] > 0.f ? stride[k] : -stride[k]) : 0;
  }
  D.over |= !moved;
  return cell;
}

// The depth-first query over an element BVH of mixed cells (UMeshCuBQLSampler
// ::sample, umesh/mc/UMeshCuBQLSampler.h:46-62): the first cell, child 0
// first and leaf cells in order, that contains P; a step at a time.  code:
// the node or leaf to look at; sp, deep, ring: its stack (the ring's rows 64
// apart); leaf, cand: the leaf being tested, its cells still to test (bits
// 0-3) and all its types (2 bits each from 4 on).
enum { CELLS_NODE, CELLS_TEST, CELLS_NONE, CELLS_FOUND };

BNX_D int cells_pop(uint32_t &code, int &sp, uint32_t *deep, uint32_t *ring)
{
  if (sp == 0) return CELLS_NONE;
  sp--;
  const int s = 64 * (sp & (PQ_SHORT - 1));
  code = ring[s];
  if (sp >= PQ_SHORT) ring[s] = deep[sp - PQ_SHORT];
  return CELLS_NODE;
}

// a node (one fetch of its four boxes) or a leaf, which keeps the cells whose
// filter box holds P
BNX_D int cells_node(const VolumeDev &v, v3 P, uint32_t &code, int &sp, uint32_t *deep, uint32_t *ring, int &leaf,
                     uint32_t &cand)
{
  auto push = [&](uint32_t c) {
    const int s = 64 * (sp & (PQ_SHORT - 1));
    if (sp >= PQ_SHORT) deep[sp - PQ_SHORT] = ring[s];
    ring[s] = c;
    sp++;
  };
  uint32_t to = EMPTY4;
  if (!(code & LEAF_BIT)) {
    const float4 BNX_G *np = (const float4 BNX_G *)(v.ebvh4 + code);
    const float4 lx = np[0], hx = np[1], ly = np[2], hy = np[3], lz = np[4], hz = np[5];
    const uint4 ch = ((const uint4 BNX_G *)np)[6];
    // an unused child's box is inverted and holds nothing
    const bool h0 = box_holds(lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, P);
    const bool h1 = box_holds(lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, P);
    const bool h2 = box_holds(lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, P);
    const bool h3 = box_holds(lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, P);
    to = h3 ? ch.w : to;
    if (h2 && to != EMPTY4) push(to);
    to = h2 ? ch.z : to;
    if (h1 && to != EMPTY4) push(to);
    to = h1 ? ch.y : to;
    if (h0 && to != EMPTY4) push(to);
    to = h0 ? ch.x : to;
  } else {
    leaf = (int)((code & ~LEAF_BIT) >> 3);
    const int count = (int)(code & 7u);
    cand = 0;
    float4 lo[4], hi[4];
#pragma unroll
    for (int x = 0; x < 4; x++) {
      const size_t c = 2 * (size_t)(leaf + min(x, count - 1));
      lo[x] = v.ucellbox[c];
      hi[x] = v.ucellbox[c + 1];
    }
#pragma unroll
    for (int x = 0; x < 4; x++) {
      const bool in = x < count && box_holds(lo[x].x, lo[x].y, lo[x].z, hi[x].x, hi[x].y, hi[x].z, P);
      cand |= (in ? 1u << x : 0u) | ((uint32_t)__float_as_int(lo[x].w) << (4 + 2 * x));
    }
    if (cand & 15u) return CELLS_TEST;
  }
  if (to == EMPTY4) return cells_pop(code, sp, deep, ring);
  code = to;
  return CELLS_NODE;
}

// the type of the next cell to test
BNX_D int cells_want(uint32_t cand) { return (int)(cand >> (4 + 2 * max(__ffs(cand & 15u) - 1, 0))) & 3; }

// the cell type most of the lanes that are `on` wait for
BNX_D int cells_type(bool on, uint32_t cand)
{
  const int want = cells_want(cand);
  int type = 0, best = 0;
  for (int y = 0; y < 4; y++) {
    const int c = __popcll(__ballot(on && want == y));
    type = c > best ? y : type;
    best = max(c, best);
  }
  return type;
}

// the next cell of the leaf, which is of this type
BNX_D int cells_test(const VolumeDev &v, v3 P, int type, uint32_t &code, int &sp, uint32_t *deep, uint32_t *ring,
                     int leaf, uint32_t &cand, float &value)
{
  if (cell_value(v, type, leaf + __ffs(cand & 15u) - 1, P, value)) {
    sp = 0;
    return CELLS_FOUND;
  }
  cand &= cand - 1u;
  if (cand & 15u) return CELLS_TEST;
  value = __builtin_nanf("");
  return cells_pop(code, sp, deep, ring);
}

constexpr int READY = 16;     // words of a ray set up in LDS

// LDS written by this wave is read back by this wave: keep the order
BNX_D void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// the segments of this launch's program, one after the other: fn(slot,
// fresh) works through the claims of one.  No trace has run when fresh_launch
// is set: a request's first program then finds no hit records, and a request
// without programs gets its misses here, from the launches with k == 0.
template <typename F>
BNX_D void each_segment(Claims &cl, const SlotDev *__restrict__ slots, const RayQueue &q, int k, bool fresh_launch,
                        bool iso, F &&fn)
{
  while (cl.chunk >= 0) {
    const Segment sg = cl.open();
    const SlotDev &SL = slots[sg.slot];
    const int niso = SL.num_isos, nvol = SL.num_vols;
    const bool fresh = fresh_launch && k == 0 && (iso || niso == 0);
    if (k < (iso ? niso : nvol)) {
      cl.refill();
      if (fn(SL, fresh)) continue;
    }
    // not this launch's: past its chunks
    const int lane = lane_id();
    while (!cl.dry) {
      if (fresh && niso + nvol == 0)
        for (int i = cl.next + lane; i < cl.stop; i += 64) q.hit[cl.base + i] = make_int4(-1, -1, -1, 0);
      cl.next = cl.stop;
      cl.refill();
    }
  }
}

// The volume march (of structured fields, the scattered generations of large
// frames: k_volume_rays has the others).  FIELD: the kind of field this kernel
// serves (FIELD_KIND_*).  Bound by the gathers of the samples (structured: the eight
// corners of a cell in two loads of its corner copy; tets: a 128-byte record)
// and by how many lanes a trip keeps at work.  With nested loops, one ray a
// lane, a quarter to a third of the lanes were: 256^3 volume, 1024^2, 16 spp:
// 3.65 ms a pass then, 1.92 so.
template <int FIELD> struct March {
  static constexpr bool TETS = FIELD == FIELD_KIND_TETS, CELLS = FIELD == FIELD_KIND_CELLS;
  static constexpr bool QUERY = TETS || CELLS;

  // false: the field is another kernel's
  static BNX_D bool run(Claims &pr, const SlotDev &SL, const RayQueue &q, int k, bool fresh, unsigned long long *stats,
                        uint32_t *ready, uint32_t *ring)
  {
    const VolumeDev v = uniform_load(SL.vols + k);
    if (v.field != FIELD) return false;
    const int lane = lane_id();
    const uint64_t child_hash = fnv3((uint32_t)v.rtc_inst, 0u, 0u);
    const bool ratio_on = (SL.rr.flags & BNX_RENDER_RATIO_TRACKING) != 0;
    const bool last_vol = k + 1 == SL.num_vols;

    int pending = 0;                    // rays set up in LDS
    // ------------------------------------------------ per-lane state
    int mode = M_IDLE, ray = 0;
    v3 o{0.f, 0.f, 0.f}, d{1.f, 1.f, 1.f}, P{0.f, 0.f, 0.f};
    float tmax = 0.f;                   // the closest hit so far
    Dda D{};
    uint64_t rs = 0;
    float maj = 0.f, t = 0.f, upper = 0.f, T = 1.f;
    bool ratio = false;
    float rmaj = 0.f;                   // rcp_rn(maj), 0 where the draws divide by maj
    // point query: the tet being tested, the one that held the last point,
    // the walk's steps and whether it started from the seed; the value found
    int cur = 0, last = -1, walk = 0;
    bool seeded = false;
    float value = 0.f;
    // depth-first query over the element BVH (cells)
    uint32_t deep[CELLS ? PQ_DEEP4 : 1];
    uint32_t code = 0;
    int sp = 0, leaf = 0;               // the leaf being looked at
    uint32_t cand = 0;                  // its cells still to test (bits 0-3) and all its types (2 bits each from 4 on)
    uint32_t n_samples = 0, n_cells = 0, n_nodes = 0, n_tests = 0;

    auto rnd = [&]() -> float { return (float)(rng_next(rs) & 0x00FFFFFFu) * (1.f / (float)0x01000000); };
    // ask for the field at P
    auto query = [&]() {
      if (CELLS) {
        code = 0;                       // the root: the stack is empty between queries
        mode = M_NODE;
      } else if (TETS && last >= 0) {
        cur = last;
        walk = 0;
        seeded = false;
        mode = M_WALK;
      } else {
        mode = M_SAMPLE;
      }
    };
    // a ray with ratio-tracking estimate T leaves without a hit: a shadow
    // ray's hit_v carries the estimate to the next volume
    auto leave = [&](int i, float est) {
      if (!last_vol) q.hit_v[i] = est;
      else if (est < 1.f) q.ps[i].w = __float_as_uint(__uint_as_float(q.ps[i].w) * est);
    };
    auto miss = [&]() {
      if (ratio) leave(ray, T);
      mode = M_IDLE;
    };
    auto hit = [&](float at, v3 c) {
      q.org[ray].w = at;
      q.hit[ray] = make_int4(0, VOLUME_GEOM_BASE + k, v.rtc_inst, 0);
      q.vcol[ray] = make_float4(c.x, c.y, c.z, 0.f);
      mode = M_IDLE;
    };
    // Woodcock::sampleRange (volume/Volume.h:168-203), or ratio tracking
    // (Novak, Selle and Jarosz, "Residual Ratio Tracking for Estimating
    // Attenuation in Participating Media", SIGGRAPH Asia 2014, section 3)
    // for shadow rays of requests that ask for it: the estimate takes the
    // null-collision probability instead of ending the ray with it
    auto consume = [&]() {
      const float f = value;
      n_samples++;
      const float4 s = isnan(f) ? make_float4(0.f, 0.f, 0.f, 0.f) : tf_map(v, f, rmaj > 0.f);
      mode = M_DRAW;
      if (ratio) {
        T *= fmx(0.f, 1.f - bnx_num::over_majorant(s.w, maj, rmaj));
        if (T == 0.f) hit(tmax, v3{0.f, 0.f, 0.f});
      } else if (s.w >= rnd() * maj) {
        hit(t, v3{s.x, s.y, s.z});
      }
    };

    // a wave's rays all end: each takes a bounded walk over the macrocells,
    // and in each cell as many steps as the reference's loop takes
    for (;;) {
      const uint64_t idle = __ballot(mode == M_IDLE);
      const int n_idle = __popcll(idle);
      if (pending == 0 && !pr.dry && n_idle >= TAKE) {
        // ------------------------------------------- set up the next rays
        bool on;
        const int i = pr.claim(64, lane, on);
        bool in = false, rt = false;
        float nt = 1.f, r0 = 0.f, r1 = 0.f;
        uint64_t child = 0;
        Dda N{};
        if (on) {
          const float4 qo = q.org[i], qd = q.dir[i];
          const bool shadow = (__float_as_uint(qd.w) & FLAG_SHADOW) != 0;
          int prim = -1;
          if (fresh) q.hit[i] = make_int4(-1, -1, -1, 0);
          else prim = q.hit[i].x;
          if (!(shadow && prim >= 0)) {          // an occluded shadow ray is done
            const v3 no = xyz(qo), nd = fix_dir(xyz(qd));
            r1 = qo.w;
            rt = ratio_on && shadow;
            if (rt && k > 0) nt = q.hit_v[i];
            in = clip_bounds(v, no, nd, r0, r1);
            if (in) {
              // the ray's RNG child for this program (barney-common.h:59-61);
              // isosurfaces draw from it only for opacity < 1, never here
              uint64_t parent = q.rng[i];
              child = parent;
              rng_next(parent);
              rng_next_h(child, child_hash);
              q.rng[i] = parent;
              in = dda_init(v, no, nd, r1, N);
            }
            if (!in && rt) leave(i, nt);
          }
        }
        const uint64_t m = __ballot(in);
        pending = __popcll(m);
        if (in) {
          uint32_t *w = ready + __popcll(m & lanemask_lt());
          auto put = [&](int x, uint32_t y) { w[64 * x] = y; };
          put(0, (uint32_t)i);
          put(1, (uint32_t)child);
          put(2, (uint32_t)(child >> 32));
          put(3, __float_as_uint(nt));
          for (int a = 0; a < 3; a++) {
            put(4 + a, __float_as_uint(N.next[a]));
            put(7 + a, __float_as_uint(N.step[a]));
            put(10 + a, (uint32_t)N.left[a]);
          }
          put(13, __float_as_uint(N.ray_t0));
          put(14, __float_as_uint(N.tmax));
          put(15, (uint32_t)N.cell);
        }
        wave_sync();
        continue;
      }
      if (pending > 0 && n_idle >= min(TAKE, pending)) {
        // ------------------------------------------------- take new rays
        const int rank = __popcll(idle & lanemask_lt());
        const int left = max(0, pending - n_idle);
        if (mode == M_IDLE && rank < pending) {
          const uint32_t *w = ready + (pending - 1 - rank);
          auto get = [&](int x) -> uint32_t { return w[64 * x]; };
          ray = (int)get(0);
          const float4 qo = q.org[ray], qd = q.dir[ray];
          rs = (uint64_t)get(1) | ((uint64_t)get(2) << 32);
          T = __uint_as_float(get(3));
          for (int a = 0; a < 3; a++) {
            D.next[a] = __uint_as_float(get(4 + a));
            D.step[a] = __uint_as_float(get(7 + a));
            D.left[a] = (int)get(10 + a);
          }
          D.ray_t0 = __uint_as_float(get(13));
          D.tmax = __uint_as_float(get(14));
          D.cell = (int)get(15);
          D.begin = 0.f;
          D.over = false;
          o = xyz(qo);
          d = fix_dir(xyz(qd));
          tmax = qo.w;
          ratio = ratio_on && (__float_as_uint(qd.w) & FLAG_SHADOW) != 0;
          last = -1;
          mode = M_CELL;
        }
        pending = left;
        continue;
      }
      // ------------------------------------------------ choose a group
      const int n_samp = CELLS ? 0 : __popcll(__ballot(mode == M_SAMPLE));
      const int n_walk = TETS ? __popcll(__ballot(mode == M_WALK || mode == M_VALUE))
                              : (CELLS ? __popcll(__ballot(mode == M_VALUE)) : 0);
      const int n_node = QUERY ? __popcll(__ballot(mode == M_NODE)) : 0;
      const int n_test = CELLS ? __popcll(__ballot(mode == M_TEST)) : 0;
      const int n_cell = 64 - n_idle - n_samp - n_walk - n_node - n_test;
      if (n_idle == 64) break;
      enum { G_CELL, G_SAMPLE, G_WALK, G_NODE, G_TEST } group = G_CELL;
      if (!QUERY) {
        group = n_samp * 8 >= 3 * (64 - n_idle) ? G_SAMPLE : G_CELL;
      } else {
        const int most = max(max(max(n_cell, n_samp), max(n_walk, n_node)), n_test);
        if (TETS && n_samp >= SEED_AT) group = G_SAMPLE;
        else if (n_cell >= CELL_AT) group = G_CELL;
        else if (TETS && n_node >= NODE_AT) group = G_NODE;
        else if (TETS && n_walk > 0) group = G_WALK;
        else group = most == n_node ? G_NODE : most == n_test ? G_TEST : most == n_walk ? G_WALK
                   : most == n_samp && !CELLS ? G_SAMPLE : G_CELL;
      }
      if (QUERY && group == G_WALK) {
        if (mode == M_VALUE) consume();
        // Walk toward P: test the tet, else cross the face P lies furthest
        // behind, up to TET_WALK_STEPS times from the last point's tet and
        // then from the seed; a tet is taken only when it holds P with
        // margin, so that the value is the depth-first query's (see
        // planes_interior).
        if (TETS && mode == M_WALK) {
          n_tests++;
          const TetPlanes r = tet_planes(v.utetv + TET_REC * (size_t)cur, P);
          if (planes_interior(r)) {
            last = cur;
            value = tet_value(r);
            mode = M_VALUE;
          } else {
            const int next = walk_next(r);
            if (walk == TET_WALK_STEPS || !(r.sum > 0.f) || next < 0) {
              mode = seeded ? M_NODE : M_SAMPLE;
            } else {
              cur = next;
              walk++;
            }
          }
        }
      } else if (group == G_CELL) {
        if (mode == M_CELL) {
          if (D.over) {
            miss();
          } else {
            float c0, c1;
            const int ci = dda_cell(v, D, c0, c1);
            n_cells++;
            maj = v.majorants[ci];
            if (maj != 0.f) {
              upper = fmn(c1, tmax);
              t = c0;
              rmaj = v.rn && bnx_num::short_majorant(maj) ? rcp_rn(maj) : 0.f;
              mode = M_DRAW;
            }
          }
        }
        if (mode == M_DRAW) {
          const float r = rnd();
          const float s = -fast_log(1.f - r);
          t += bnx_num::over_majorant(s, maj, rmaj);
          if (!(t < upper)) {           // also where a NaN in the transfer function made t one
            mode = M_CELL;
          } else {
            P = o + t * d;
            query();
          }
        }
      } else if (!CELLS && group == G_SAMPLE) {
        if (mode == M_SAMPLE) {
          if (!TETS) {
            value = structured_sample(v, P);
            consume();
          } else {
            const int seed = v.ufine ? __float_as_int(v.ufine[seed_cell(v, P)].x) : -1;
            cur = seed;
            walk = 0;
            seeded = true;
            mode = seed >= 0 ? M_WALK : M_NODE;
          }
        }
      } else if (TETS) {
        // what no walk settled: the depth-first query, whole (a few queries
        // in a hundred)
        if (mode == M_NODE) {
          QueryCtx cx{nullptr, 0, 0};
          const int s = umesh_dfs<0>(v, P, cx, value);
          if (s >= 0) last = s;
          n_nodes += cx.unodes;
          n_tests += cx.utets;
          mode = M_VALUE;
        }
      } else if (CELLS && group == G_NODE) {
        if (mode == M_NODE) {
          n_nodes++;
          const int r = cells_node(v, P, code, sp, deep, ring + lane, leaf, cand);
          if (r == CELLS_TEST) mode = M_TEST;
          if (r == CELLS_NONE) {
            value = __builtin_nanf("");
            mode = M_VALUE;
          }
        }
      } else if (CELLS) {
        // the inversions of one cell type, the one most lanes wait for
        const int type = cells_type(mode == M_TEST, cand);
        if (mode == M_TEST && cells_want(cand) == type) {
          n_tests++;
          const int r = cells_test(v, P, type, code, sp, deep, ring + lane, leaf, cand, value);
          mode = r == CELLS_TEST ? M_TEST : r == CELLS_NODE ? M_NODE : M_VALUE;
        }
      }
    }
    const uint32_t s = wave_sum(n_samples), c = wave_sum(n_cells);
    const uint32_t un = wave_sum(n_nodes), ut = wave_sum(n_tests);
    if (lane == 0) {
      stat_add(stats, STAT_SAMPLES, s);
      stat_add(stats, STAT_CELLS, c);
      if (QUERY) {
        stat_add(stats, STAT_UNODES, un);
        stat_add(stats, STAT_UTETS, ut);
      }
    }
    return true;
  }
};

// The isosurface march (MCIsoSurfaceAccel::isProg, volume/MCAccelerator.h:
// 325-548): a walk over the field's macrocells; in every cell whose value
// range holds the iso value, ten linear sub-steps with a sample at each end;
// the first crossing found before tmax ends the walk, and six samples around
// it give the gradient by central differences.  A crossing whose
// interpolation is NaN (both ends exactly at the iso value) is ignored.
//
// The samples of a cell are known before any is taken, so every lane plays
// two parts: it owns a ray, whose walk posts a cell's samples (or the
// gradient's) in LDS, and it works on samples, whosever they are.  A ray's
// samples are then queried side by side instead of one after the other,
// which shortens the longest rays' chains, and lanes are short of work only
// when the whole wave is.  A sub-step's sample is queried only where the fine
// grid's value range at its point holds the iso value: otherwise its side is
// known, and an interval between two samples of one side has no crossing; a
// sample of known side is queried after all when the one next to it turns
// out to lie on the other.  The owner looks all sides of a cell up itself,
// eleven loads in flight at once, and posts what is left: most cells end
// there, and dealing their samples out for a look at the grid each cost more
// than the queries that remain (8^3 cubes of five tets, 1920x1080, 2 spp: 11.0
// ms with that, 7.8 so; 160^3: 12.7 and 11.3).
//
// Bound by the records that the queries read (about 1.8 requests beyond the
// L1 for each tet tested), so what helps is to ask for fewer samples: 20.5M
// tets, 1024^2, 4 spp, isosurface and volume: 24.2 ms a pass as nested loops,
// 16.7 with the samples dealt out, 13.5 with sides from the fine grid, 12.3
// with the owners' look, 10.8 without spills; 14^3 mixed cells, 320x240, 2 spp:
// 41.6, 8.2, 6.6, 6.0.  It still writes 4.5 GB a generation of 16M rays, some
// ten times its results: parts of the queue's lines, and the stack of the
// depth-first queries (its last 8 entries in LDS: 10.5 ms, and 10.5).
enum Owner { O_IDLE = 0, O_CELL, O_SIDES, O_WAIT };
enum Worker { W_FREE = 0, W_WALK, W_NODE, W_TEST };

constexpr int ISO_SUBS = 10, ISO_GRADS = 7, ISO_SLOTS = ISO_SUBS + 1;
constexpr int ISO_ITEMS = 1024;  // ring of posted samples: at most ISO_SLOTS per lane
static_assert(64 * ISO_SLOTS <= ISO_ITEMS, "sample ring");
constexpr uint32_t ALL_SLOTS = (1u << ISO_SLOTS) - 1u;
constexpr int ITEM_GRADIENT = 1 << 10;
struct IsoShared {
  float ray[6][64];              // origin, direction
  float t0[64], t1[64];          // the cell's range, or twice the crossing
  float value[ISO_SLOTS][64];
  int open[64];                  // samples not yet taken
  uint32_t side[64];             // slots that hold a side (an infinity) for a value
  uint16_t item[ISO_ITEMS];      // owner | slot << 6 | ITEM_GRADIENT
};

template <int FIELD> struct IsoMarch {
  static constexpr bool TETS = FIELD == FIELD_KIND_TETS, CELLS = FIELD == FIELD_KIND_CELLS;

  // false: the field is another kernel's
  static BNX_D bool run(Claims &pr, const SlotDev &SL, const RayQueue &q, int k, bool fresh, unsigned long long *stats,
                        IsoShared &L, uint32_t *ring)
  {
    const IsoDev I = uniform_load(SL.isos + k);
    const VolumeDev &v = I.field;
    if (v.field != FIELD) return false;
    const float iso = I.iso;
    const int rtc_inst = I.rtc_inst;
    const int lane = lane_id();
    const v3 bs = v3{v.hi[0] - v.lo[0], v.hi[1] - v.lo[1], v.hi[2] - v.lo[2]};
    const float delta = length(bs) * .1f / (float)(v.mc[0] + v.mc[1] + v.mc[2]);
    // the owner's ray
    int own = O_IDLE, ray = 0;
    float tmax = 0.f, last_t = 0.f, last_f = 0.f, t_hit = 0.f;
    uint32_t last_side = 0;
    bool gradient = false;
    Dda D{};
    // the worker's sample
    int work = W_FREE, owner = 0, slot = 0, cur = 0, walk = 0;
    v3 P{0.f, 0.f, 0.f};
    uint32_t deep[CELLS ? PQ_DEEP4 : 1];
    uint32_t code = 0, cand = 0;
    int sp = 0, leaf = 0;
    int head = 0, tail = 0;             // of the ring; wave-uniform
    uint32_t n_cells = 0, n_nodes = 0, n_tests = 0;

    auto place = [&](int a, float t) { return v3{L.ray[0][a] + t * L.ray[3][a], L.ray[1][a] + t * L.ray[4][a],
                                                 L.ray[2][a] + t * L.ray[5][a]}; };
    // where sub-step i of a cell lies; i / 10 is the rounded product but for
    // 9, which the division's correction gives
    auto at = [&](int i, float t0, float t1) {
      const float fi = div_rn((float)i, 10.f, .1f);
      return (1.f - fi) * t0 + fi * t1;
    };
    auto deliver = [&](float f) {
      L.value[slot][owner] = f;
      atomicAdd(&L.open[owner], -1);
      work = W_FREE;
    };
    // post the samples of this lane's ray whose bits are set in `which`; all
    // lanes call this together
    auto post = [&](uint32_t which, int kind) {
      const int n = __popc(which);
      int off = n;
      for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(off, d, 64);
        if (lane >= d) off += y;
      }
      const int total = __builtin_amdgcn_readlane(off, 63);
      off += tail - n;
      if (n > 0) {
        L.open[lane] = n;
        own = O_WAIT;
      }
      for (; which; which &= which - 1u)
        L.item[off++ & (ISO_ITEMS - 1)] = (uint16_t)(lane | ((__ffs(which) - 1) << 6) | kind);
      tail += total;
    };

    L.open[lane] = 0;
    // a wave ends: each ray takes a bounded walk over the macrocells and
    // posts a bounded number of samples, and a sample's query is bounded by
    // the mesh
    for (;;) {
      const uint64_t idle = __ballot(own == O_IDLE);
      const int n_idle = __popcll(idle);
      wave_sync();
      const bool done = own == O_WAIT && L.open[lane] == 0;
      const int n_done = __popcll(__ballot(done)), n_cell = __popcll(__ballot(own == O_CELL));
      const int n_sides = __popcll(__ballot(own == O_SIDES));
      const uint64_t free = __ballot(work == W_FREE);
      const int n_free = __popcll(free), items = tail - head;
      const bool starved = n_free == 64 && items == 0;
      if (!pr.dry && (n_idle >= 16 || (starved && n_idle > 0 && n_done + n_cell + n_sides < 16))) {
        // ---------------------------------------------------- new rays
        bool on;
        const int i = pr.claim(n_idle, __popcll(idle & lanemask_lt()), on);
        if (own == O_IDLE && on) {
          ray = i;
          const float4 qo = q.org[i], qd = q.dir[i];
          const bool shadow = (__float_as_uint(qd.w) & FLAG_SHADOW) != 0;
          int prim = -1;
          if (fresh) q.hit[i] = make_int4(-1, -1, -1, 0);
          else prim = q.hit[i].x;
          if (!(shadow && prim >= 0)) {          // an occluded shadow ray is done
            const v3 o = xyz(qo), d = fix_dir(xyz(qd));
            tmax = qo.w;
            float r0 = 0.f, r1 = tmax;
            if (clip_bounds(v, o, d, r0, r1)) {
              // the program's RNG child (barney-common.h:59-61) is drawn from
              // only for opacity < 1, never here; the parent moves on
              uint64_t parent = q.rng[i];
              rng_next(parent);
              q.rng[i] = parent;
              if (dda_init(v, o, d, r1, D)) {
                L.ray[0][lane] = o.x; L.ray[1][lane] = o.y; L.ray[2][lane] = o.z;
                L.ray[3][lane] = d.x; L.ray[4][lane] = d.y; L.ray[5][lane] = d.z;
                last_t = __builtin_nanf("");
                gradient = false;
                own = O_CELL;
              }
            }
          }
        }
        continue;
      }
      if (n_idle == 64) break;
      if (n_done >= 16 || (starved && n_done >= max(n_cell, n_sides) && n_done > 0)) {
        // ------------------------------------------- use the values taken
        uint32_t which = 0;
        int kind = 0;
        if (done && !gradient) {
          const float t0 = L.t0[lane], t1 = L.t1[lane];
          const uint32_t side = L.side[lane];
          float f0 = L.value[0][lane], a0 = t0;
          own = O_CELL;
          for (int i = 1; i <= ISO_SUBS; i++) {
            const float f1 = L.value[i][lane], a1 = at(i, t0, t1);
            const float lo = fmn(f0, f1), hi = fmx(f0, f1);
            if (which == 0 && !gradient && !isnan(f0) && !isnan(f1) && iso >= lo && iso <= hi) {
              which = side & (3u << (i - 1));      // sides to make values of before this interval is settled
              float x = (iso - f0) / (f1 - f0);
              x = (1.f - x) * a0 + x * a1;
              if (which == 0 && x < tmax) {
                gradient = true;
                t_hit = x;
              }
            }
            f0 = f1;
            a0 = a1;
          }
          if (which) {
            L.side[lane] = side & ~which;
          } else if (gradient) {
            which = (1u << ISO_GRADS) - 1u;
            kind = ITEM_GRADIENT;
            L.t0[lane] = t_hit;
          } else {
            last_t = a0;
            last_f = f0;
            last_side = (side >> ISO_SUBS) & 1u;
          }
        } else if (done) {
          // central differences, one-sided next to a point outside the field
          const float fP = L.value[0][lane];
          float g[3];
          for (int a = 0; a < 3; a++) {
            float f0 = L.value[1 + 2 * a][lane], f1 = L.value[2 + 2 * a][lane], w = 2.f;
            if (isnan(f0)) { w -= 1.f; f0 = fP; }
            if (isnan(f1)) { w -= 1.f; f1 = fP; }
            g[a] = w == 0.f ? 0.f : (f1 - f0) / w;
          }
          v3 n = v3{g[0], g[1], g[2]};
          if (n == splat(0.f)) n = -normalize(v3{L.ray[3][lane], L.ray[4][lane], L.ray[5][lane]});
          n = normalize(n);
          q.org[ray].w = t_hit;
          q.hit[ray] = make_int4(0, ISO_GEOM_BASE + k, rtc_inst, 0);
          q.vcol[ray] = make_float4(n.x, n.y, n.z, 0.f);
          own = O_IDLE;
        }
        post(which, kind);
        continue;
      }
      if (n_sides >= SIDES_AT || (starved && n_sides > 0 && n_sides >= n_cell)) {
        // --------------------------- sides of a macrocell's sub-steps, ...
        uint32_t which = 0;
        if (own == O_SIDES) {
          const float t0 = L.t0[lane], t1 = L.t1[lane];
          // a cell that begins where the last one's sub-steps ended knows its
          // first value
          uint32_t side = 0, over = 0, under = 0, open = ALL_SLOTS;
          if (last_t == t0) {
            L.value[0][lane] = last_f;
            side = last_side;
            over = last_f > iso || isnan(last_f) ? 1u : 0u;
            under = last_f < iso || isnan(last_f) ? 1u : 0u;
            open &= ~1u;
          }
          if (v.ufine) {
            float2 g[ISO_SLOTS];
#pragma unroll
            for (int i = 0; i < ISO_SLOTS; i++) {
              const v3 Q = place(lane, i == 0 ? t0 : at(i, t0, t1));
              const float BNX_G *r = (const float BNX_G *)(v.ufine + seed_cell(v, Q));
              g[i] = make_float2(r[1], r[2]);
            }
#pragma unroll
            for (int i = 0; i < ISO_SLOTS; i++) {
              const uint32_t bit = open & (1u << i);
              if (bit != 0 && (g[i].x > iso || g[i].y < iso)) {
                L.value[i][lane] = g[i].x > iso ? INFINITY : -INFINITY;
                over |= g[i].x > iso ? bit : 0u;
                under |= g[i].x > iso ? 0u : bit;
                side |= bit;
                open &= ~bit;
              }
            }
          }
          if (over == ALL_SLOTS || under == ALL_SLOTS) {
            // no crossing
            own = O_CELL;
            last_t = at(ISO_SUBS, t0, t1);
            last_f = L.value[ISO_SUBS][lane];
            last_side = 1;
          } else {
            L.side[lane] = side;
            own = O_WAIT;
            which = open;
          }
        }
        post(which, 0);
        continue;
      }
      if (n_cell >= 16 || (starved && n_cell > 0)) {
        // --------------------------------------- ... next macrocells, ...
        if (own == O_CELL) {
          if (D.over) {
            own = O_IDLE;
          } else {
            float c0, c1;
            const int ci = dda_cell(v, D, c0, c1);
            n_cells++;
            if (c0 < fmn(c1, tmax)) {
              const float2 vr = v.ranges[ci];
              if (iso >= vr.x && iso <= vr.y) {
                L.t0[lane] = c0;
                L.t1[lane] = c1;
                own = O_SIDES;
              }
            }
          }
        }
        continue;
      }
      if (items > 0 && (n_free >= 16 || n_free == 64)) {
        // ------------------------------------------------- take samples
        const int rank = __popcll(free & lanemask_lt());
        if (work == W_FREE && rank < items) {
          const uint32_t it = L.item[(head + rank) & (ISO_ITEMS - 1)];
          owner = (int)(it & 63u);
          slot = (int)(it >> 6) & 15;
          const float t0 = L.t0[owner];
          if (it & ITEM_GRADIENT) {
            // the crossing, then -delta and +delta along each axis
            const float s = (slot & 1) ? -delta : +delta;
            P = place(owner, t0);
            if (slot > 0)
              P = P + v3{slot <= 2 ? s : 0.f, slot == 3 || slot == 4 ? s : 0.f, slot >= 5 ? s : 0.f};
          } else {
            P = place(owner, slot == 0 ? t0 : at(slot, t0, L.t1[owner]));
          }
          if (!TETS && !CELLS) {
            deliver(structured_sample(v, P));
          } else {
            if (CELLS) {
              code = 0;
              sp = 0;
              work = W_NODE;
            } else {
              cur = v.ufine ? __float_as_int(v.ufine[seed_cell(v, P)].x) : -1;
              walk = 0;
              work = cur >= 0 ? W_WALK : W_NODE;
            }
          }
        }
        head += min(items, n_free);
        continue;
      }
      // ----------------------------------------------------- point queries
      if (TETS) {
        const int n_node = __popcll(__ballot(work == W_NODE));
        if (n_node >= 12 || n_node + n_free == 64) {
          if (work == W_NODE) {
            QueryCtx cx{nullptr, 0, 0};
            float f;
            (void)umesh_dfs<0>(v, P, cx, f);
            n_nodes += cx.unodes;
            n_tests += cx.utets;
            deliver(f);
          }
        } else if (work == W_WALK) {
          n_tests++;
          const TetPlanes r = tet_planes(v.utetv + TET_REC * (size_t)cur, P);
          if (planes_interior(r)) {
            deliver(tet_value(r));
          } else {
            const int next = walk_next(r);
            if (walk == TET_WALK_STEPS || !(r.sum > 0.f) || next < 0) {
              work = W_NODE;
            } else {
              cur = next;
              walk++;
            }
          }
        }
      }
      if (CELLS) {
        const int n_node = __popcll(__ballot(work == W_NODE)), n_test = 64 - n_free - n_node;
        if (n_node >= n_test) {
          if (work == W_NODE) {
            const int r = cells_node(v, P, code, sp, deep, ring + lane, leaf, cand);
            n_nodes++;
            if (r == CELLS_NONE) deliver(__builtin_nanf(""));
            else if (r == CELLS_TEST) work = W_TEST;
          }
        } else {
          const int type = cells_type(work == W_TEST, cand);
          float f = 0.f;
          if (work == W_TEST && cells_want(cand) == type) {
            n_tests++;
            const int r = cells_test(v, P, type, code, sp, deep, ring + lane, leaf, cand, f);
            if (r != CELLS_TEST) {
              if (r == CELLS_NODE) work = W_NODE;
              else deliver(f);
            }
          }
        }
      }
    }
    const uint32_t c = wave_sum(n_cells), un = wave_sum(n_nodes), ut = wave_sum(n_tests);
    if (lane == 0) {
      stat_add(stats, STAT_CELLS, c);
      stat_add(stats, STAT_UNODES, un);
      stat_add(stats, STAT_UTETS, ut);
    }
    return true;
  }
};

// Waves per SIMD each kernel is compiled for: as many as their registers
// allow without spills.  At five, the tet kernels spilled 15 and 31 and the
// structured isosurface 5, stored and loaded again in every trip (20.5M tets,
// 1024x1024, 4 spp: 12.3 ms a pass, 10.8 at four; 8^3 cubes of five tets,
// 1920x1080, 2 spp: 7.8 and 7.2).  What scratch the tet kernels have left is
// the stack of their few depth-first queries.
constexpr int march_waves(int field) { return field == FIELD_KIND_CELLS ? 3 : field == FIELD_KIND_TETS ? 4 : 5; }
constexpr int iso_waves(int field) { return field == FIELD_KIND_CELLS ? 3 : 4; }

template <int FIELD>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(march_waves(FIELD)))) void k_volume_march(
    const SlotDev *__restrict__ slots, SegView sv, RayQueue q, int k, int nsegs, int program, int fresh,
    unsigned long long *stats, Stamp stamp)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) stamp_write(stamp);
  __shared__ uint32_t ready[READY * 64];
  __shared__ uint32_t ring[FIELD == FIELD_KIND_CELLS ? PQ_SHORT * 64 : 1];
  Claims cl;
  cl.begin(sv, nsegs, program, (int)gridDim.x, BALANCE * (int)gridDim.x);
  each_segment(cl, slots, q, k, fresh != 0, false, [&](const SlotDev &SL, bool f) -> bool {
    return March<FIELD>::run(cl, SL, q, k, f, stats, ready, ring);
  });
}

template <int FIELD>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(iso_waves(FIELD)))) void k_iso_march(
    const SlotDev *__restrict__ slots, SegView sv, RayQueue q, int k, int nsegs, int program, int fresh,
    unsigned long long *stats, Stamp stamp)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) stamp_write(stamp);
  __shared__ IsoShared L;
  __shared__ uint32_t ring[FIELD == FIELD_KIND_CELLS ? PQ_SHORT * 64 : 1];
  Claims cl;
  cl.begin(sv, nsegs, program, (int)gridDim.x, BALANCE * (int)gridDim.x);
  each_segment(cl, slots, q, k, fresh != 0, true, [&](const SlotDev &SL, bool f) -> bool {
    return IsoMarch<FIELD>::run(cl, SL, q, k, f, stats, L, ring);
  });
}

// The volume march of structured fields with one ray a lane from its begin to
// its end, as nested loops.  What a lane waits for here are others' macrocells
// and samples, but a step costs no vote and no state, a wave begins and ends
// by itself, and the corner copy has made a sample one fetch: this is faster
// than March in all launches but those of many rays that do not run side by
// side (launch_volume_march).  A wave takes 64 rays, or 32 or 16 where the
// launch would not fill half of the chip's waves: their loops end sooner.
// March against this, us a frame: edits of 24^3, 128x96, 251 and 239; 48^3,
// 205x492, 440 and 336; 200^3, 900x700, 655 and 520; frames of 64^3, 640x480, 2
// spp, 505 and 365; 30^3, 1920x1080, 1250 and 1060; 256^3, 1024x1024, 4 spp, 1189
// and 1148.  Six waves per SIMD (four and five within 1%, eight 6% slower).
constexpr int RAYS_WAVES = 6;
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RAYS_WAVES))) void k_volume_rays(
    const SlotDev *__restrict__ slots, SegView sv, RayQueue q, int k, int nsegs, int least, int fresh_launch,
    unsigned long long *stats, Stamp stamp)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) stamp_write(stamp);
  // the generation's 256-ray blocks, each cut into 4, 8 or 16 waves' shares
  // until there are `least` waves; the grid is as large as that can get
  const Segment z = uniform_load((const Segment BNX_G *)(sv.segs + nsegs - 1));
  const int blocks = z.block256 + (z.count + 255) / 256;
  int shift = 2;
  while (shift < 4 && (blocks << shift) < least) shift++;
  const int blk = (int)blockIdx.x >> shift, per = 256 >> shift;
  if (blk >= blocks) return;
  const Segment sg =
      uniform_load((const Segment BNX_G *)(sv.segs + __builtin_amdgcn_readfirstlane(sv.blk256[blk])));
  const int local = (blk - sg.block256) * 256 + ((int)blockIdx.x - (blk << shift)) * per + (int)threadIdx.x;
  const int i = sg.begin + local;
  const SlotDev &SL = slots[sg.slot];
  const bool fresh = fresh_launch != 0 && k == 0 && SL.num_isos == 0;
  const bool valid = (int)threadIdx.x < per && local < sg.count;
  if (k >= SL.num_vols) {
    if (fresh && SL.num_vols == 0 && valid) q.hit[i] = make_int4(-1, -1, -1, 0);
    return;
  }
  const VolumeDev v = uniform_load(SL.vols + k);
  if (v.field != FIELD_KIND_STRUCTURED) return;
  const bool last_vol = k + 1 == SL.num_vols, ratio_on = (SL.rr.flags & BNX_RENDER_RATIO_TRACKING) != 0;
  uint32_t n_samples = 0, n_cells = 0;
  if (valid) {
    const float4 qo = q.org[i], qd = q.dir[i];
    const bool shadow = (__float_as_uint(qd.w) & FLAG_SHADOW) != 0;
    int prim = -1;
    if (fresh) q.hit[i] = make_int4(-1, -1, -1, 0);
    else prim = q.hit[i].x;
    const v3 o = xyz(qo), d = fix_dir(xyz(qd));
    const float tmax = qo.w;
    const bool ratio = ratio_on && shadow, done = shadow && prim >= 0;   // an occluded shadow ray is done
    float T = ratio && !done && k > 0 ? q.hit_v[i] : 1.f, at = 0.f, r0 = 0.f, r1 = tmax;
    v3 c{0.f, 0.f, 0.f};
    bool in = false, hit = false;
    uint64_t rs = 0;
    Dda D{};
    if (!done && clip_bounds(v, o, d, r0, r1)) {
      uint64_t parent = q.rng[i];
      rs = parent;
      rng_next(parent);
      rng_next_h(rs, fnv3((uint32_t)v.rtc_inst, 0u, 0u));
      q.rng[i] = parent;
      in = dda_init(v, o, d, r1, D);
    }
    auto rnd = [&]() -> float { return (float)(rng_next(rs) & 0x00FFFFFFu) * (1.f / (float)0x01000000); };
    while (in && !D.over && !hit) {
      float c0, c1;
      const int ci = dda_cell(v, D, c0, c1);
      n_cells++;
      const float maj = v.majorants[ci];
      if (maj == 0.f) continue;
      const float upper = fmn(c1, tmax), rmaj = v.rn && bnx_num::short_majorant(maj) ? rcp_rn(maj) : 0.f;
      float t = c0;
      while (!hit) {
        const float r = rnd();
        const float s = -fast_log(1.f - r);
        t += bnx_num::over_majorant(s, maj, rmaj);
        if (!(t < upper)) break;
        const float f = structured_sample(v, o + t * d);
        n_samples++;
        const float4 m = isnan(f) ? make_float4(0.f, 0.f, 0.f, 0.f) : tf_map(v, f, rmaj > 0.f);
        if (ratio) {
          T *= fmx(0.f, 1.f - bnx_num::over_majorant(m.w, maj, rmaj));
          hit = T == 0.f;
          at = tmax;
        } else if (m.w >= rnd() * maj) {
          hit = true;
          at = t;
          c = v3{m.x, m.y, m.z};
        }
      }
    }
    if (hit) {
      q.org[i].w = at;
      q.hit[i] = make_int4(0, VOLUME_GEOM_BASE + k, v.rtc_inst, 0);
      q.vcol[i] = make_float4(c.x, c.y, c.z, 0.f);
    } else if (ratio && !done) {
      if (!last_vol) q.hit_v[i] = T;
      else if (T < 1.f) q.ps[i].w = __float_as_uint(__uint_as_float(q.ps[i].w) * T);
    }
  }
  const uint32_t a = wave_sum(n_samples), b = wave_sum(n_cells);
  if (lane_id() == 0) {
    stat_add(stats, STAT_SAMPLES, a);
    stat_add(stats, STAT_CELLS, b);
  }
}

using MarchKernel = void (*)(const SlotDev *, SegView, RayQueue, int, int, int, int, unsigned long long *, Stamp);
const MarchKernel KERNELS[2][FIELD_KINDS] = {
    {k_volume_march<FIELD_KIND_STRUCTURED>, k_volume_march<FIELD_KIND_TETS>, k_volume_march<FIELD_KIND_CELLS>},
    {k_iso_march<FIELD_KIND_STRUCTURED>, k_iso_march<FIELD_KIND_TETS>, k_iso_march<FIELD_KIND_CELLS>}};

} // namespace

int launch_volume_march(Device *dev, const SlotDev *slots, const SegView &sv, int nsegs, int blocks256,
                        const RayQueue &q, bool surfaces, bool scattered, const MarchKind &kind,
                        unsigned long long *stats, const Stamp &stamp)
{
  if (blocks256 <= 0 || nsegs <= 0) return BNX_OK;
  int launch = 0;
  for (int p = 0; p < kind.isos + kind.vols; p++) {
    const bool iso = p < kind.isos;
    const int k = iso ? p : p - kind.isos;
    for (int f = 0; f < FIELD_KINDS; f++) {
      if (!(kind.fields & (1 << f))) continue;
      if (!iso && f == FIELD_KIND_STRUCTURED && (!scattered || blocks256 < SCATTERED_BLOCKS)) {
        // half of the resident waves; a grid of fewer than that many shares
        // is cut again, into less than twice as many
        const int least = 2 * RAYS_WAVES * dev->num_cus;
        k_volume_rays<<<std::max(4 * blocks256, std::min(16 * blocks256, 2 * least)), 64, 0, dev->stream>>>(
            slots, sv, q, k, nsegs, least, surfaces ? 0 : 1, stats, launch == 0 ? stamp : Stamp{});
        launch++;
        continue;
      }
      const MarchKernel kernel = KERNELS[iso ? 1 : 0][f];
      // as many waves as are resident at once, in whole rounds of the groups,
      // and no more than there are chunks of 16 rays
      int &fit = dev->march_fit[(iso ? FIELD_KINDS : 0) + f];
      if (fit == 0) {
        BNX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, (const void *)kernel, 64, 0));
        fit = std::max(1, fit);
      }
      const int waves = std::min(fit * dev->num_cus, 16 * blocks256) / CLAIM_GROUPS * CLAIM_GROUPS;
      // the block maps' kernel clears the counters of the first launches
      const int slot = launch % MARCH_PROGRAMS;
      if (launch >= MARCH_PROGRAMS) {
        const int rc = launch_claims_clear(dev, sv.claims + slot * CLAIM_GROUPS * CLAIM_STRIDE);
        if (rc != BNX_OK) return rc;
      }
      kernel<<<std::max(CLAIM_GROUPS, waves), 64, 0, dev->stream>>>(slots, sv, q, k, nsegs, slot, surfaces ? 0 : 1,
                                                                    stats, launch == 0 ? stamp : Stamp{});
      launch++;
    }
  }
  BNX_HIP(hipGetLastError());
  return BNX_OK;
}

} // namespace bnx
