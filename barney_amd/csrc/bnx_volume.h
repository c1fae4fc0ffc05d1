// bnx_volume.h -- volume and isosurface device data (structured and
// tetrahedral fields) and the per-ray march.
#pragma once

#include "bnx_internal.h"
#include "bnx_render.h"

namespace bnx {

// hit-record geometry index of a volume event: VOLUME_GEOM_BASE + volume
// slot; of an isosurface hit: ISO_GEOM_BASE + isosurface slot
constexpr int VOLUME_GEOM_BASE = 0x40000000;
constexpr int ISO_GEOM_BASE = 0x60000000;

// kinds of field; each has march kernels of its own
enum { FIELD_KIND_STRUCTURED = 0, FIELD_KIND_TETS = 1, FIELD_KIND_CELLS = 2, FIELD_KINDS = 3 };

// element-BVH point-query stack: a ring of PQ_SHORT entries per thread in
// LDS ([entry][thread]) spilling to private entries: PQ_DEEP for the binary
// walk, whose stack holds at most one entry per level (a mesh whose element
// BVH is deeper is rejected at creation), PQ_DEEP4 for the 4-wide walk, whose
// stack holds at most three for two levels
constexpr int PQ_SHORT = 16;
constexpr int PQ_DEEP = 48;
constexpr int PQ_DEEP4 = 96;
static_assert(PQ_SHORT + PQ_DEEP4 >= 3 * (PQ_SHORT + PQ_DEEP) / 2, "4-wide point-query stack");

// the float4 words of a tet record (VolumeDev::utetv), 128 bytes apart
constexpr int TET_REC = 8;

struct VolumeDev {
  int field;                  // FIELD_KIND_*
  // structured (StructuredData, volume/StructuredData.h:30-74)
  const float BNX_G *scalars;   // dims[0]*dims[1]*dims[2], x fastest
  // the eight corners of every cell side by side (two float4 a cell, cells x
  // fastest; null: read the layouts below): a sample is one 32-byte fetch
  // where the linear array takes four rows, and a CU's outstanding fetches
  // are what bounds the march
  const float4 BNX_G *corners;
  // the same values in bricks of B^3 cells (B = 1 << brick_shift) with a
  // one-texel apron: (B+1)^3 texels per brick, x fastest inside a brick,
  // bricks x fastest; every trilinear footprint lies inside the brick of
  // its lower corner (null: sample the linear array)
  const float BNX_G *bricks;
  int brick_shift;
  int nbricks[3];
  int dims[3];
  int ncells[3];
  float origin[3];
  float rcp_spacing[3];       // 1/gridSpacing (host float division)
  // tets (UMeshField, umesh/common/UMeshField.h:52-116): per tet, in
  // element-BVH slot order, one 128-byte line (TET_REC float4): words 0-3
  // the normals of the faces opposite vertices 0-3, as the plane test
  // crosses them, each with the tet across that face (int bits, or TET_HULL
  // or TET_OPEN) in w; words 4 and 5 vertices 0 and 1 with their scalars; word
  // 6 the scalars of vertices 2 and 3.  A tet test or a walk step is one
  // dependent fetch and 26 operations on the planes, where crossing the
  // edges again took 92.
  const float4 BNX_G *utetv;
  // meshes with other cells than tets: per slot the cell's vertices
  // (position, scalar; 8 float4, the cell's own first) and its filter box
  // (lo with the cell type CELL_* in w, hi)
  const float4 BNX_G *ucells;
  const float4 BNX_G *ucellbox;
  const Node BNX_G *ebvh;       // element BVH (tets)
  const Node4 BNX_G *ebvh4;     // its 4-wide form (other cells)
  // fine grid over an unstructured field's bounds (null: none), 16 bytes a
  // cell: the tet slot that holds its centre (int bits; -1: none), where a
  // point query with no nearby previous tet starts its walk, and the least
  // and the largest value that the field takes in it (FINE_SLACK included)
  const float4 BNX_G *ufine;
  int seed_dims[3];
  float seed_origin[3];
  float seed_rcp[3];          // cells per unit length (host float division)
  // both
  float lo[3], hi[3];         // world bounds
  int mc[3];
  int cells_per_mc;
  float mc_origin[3];
  float mc_rcp_spacing[3];    // 1 / macrocell spacing (host float division)
  const float2 BNX_G *ranges;   // macrocell value ranges (lo, hi)
  const float BNX_G *majorants;
  const float4 BNX_G *tf;
  int ntf;
  float dom0, dom1, base_density;
  float rcp_span;             // 1 / (dom1 - dom0) (host float division)
  int rn;                     // spacings, domain and densities lie where rcp_rn and div_rn are exact; a
                              // cell's majorant has to as well (short_majorant)
  int rtc_inst;               // rtc instance index (seeds the march RNG)
  int user_inst;
  int user_id;
};

// IsoSurface::DD (geometry/IsoSurface.h:31-42) with its field and an
// opaque matte material
struct IsoDev {
  VolumeDev field;
  float iso;
  float color[3];
  int rtc_inst;
  int user_inst;
  int user_id;
};

struct VolumeList {
  const VolumeDev BNX_G *vols;  // device array
  int count;
};

struct Volume {
  Device *dev;
  uint64_t version = 0;         // bumped whenever dd changes
  bool grid_rn = false;         // the macrocell spacings' part of VolumeDev::rn
  VolumeDev dd{};
  DevMem scalars, corners, bricks, ranges, majorants, tf;
  DevMem ufine, utetv, ucells, ucellbox;
  Bvh ebvh;                     // element BVH (cells)
};

struct IsoSurface {
  Device *dev;
  Volume *field;
  float iso;
  float color[3];
  int user_id;
};

int volume_build(Volume *v);
// the structured field's bricked copy (VolumeDev::bricks) with bricks of
// 2^shift cells; shift 0 keeps the linear layout only
int volume_brick(Volume *v, int shift);
// the structured field's cell-corner copy (VolumeDev::corners), where the
// field is finite and the copy takes no more than an eighth of the device's
// free memory
int volume_corners(Volume *v);
// cells: element BVH, macrocell ranges (rasterTet<5> for tets, the cell's
// box for the others), majorants.  tets4: the host copy of the cells'
// vertex indices 0..3 (num_cells x int4), ext4 of 4..7 and types the cell
// types (CELL_*; both null when every cell is a tet), verts4 of the vertices
int volume_build_umesh(Volume *v, const int4 *tets4, const int4 *ext4, const uint8_t *types, int num_cells,
                       const float4 *verts4, int num_verts);
int volume_rebuild_majorants(Volume *v);
// upload the world's volume and isosurface tables (if changed) and return them
int world_volumes(World *w, VolumeList &vl);
int world_isos(World *w, const struct IsoDev BNX_G *&isos, int &count);
// what a batch's rays have to be marched through: the kinds of field in use
// (1 << FIELD_KIND_*), and the most isosurfaces and volumes of a request
struct MarchKind {
  int fields = 0, isos = 0, vols = 0;
  void merge(const MarchKind &o)
  {
    fields |= o.fields;
    isos = isos > o.isos ? isos : o.isos;
    vols = vols > o.vols ? vols : o.vols;
  }
};
// From this many 256-ray blocks on, rays that scattering has spread (and
// the shadow rays among them) keep more lanes at work in March: 256^3,
// 1024x1024, 16 spp, two such generations of 3 to 4 million: 2.97 ms a frame
// with March, 3.17 without.  At half as many rays both take the same time.
constexpr int SCATTERED_BLOCKS = 8192;
// march every ray of the generation's nsegs segments (at most blocks256
// blocks of 256 rays) through its request's isosurfaces and volumes; surfaces: false when the
// trace kernel did not run, so the hit records are not written yet; scattered:
// no primary rays are among them
int launch_volume_march(Device *dev, const SlotDev *d_slots, const SegView &sv, int nsegs, int blocks256,
                        const RayQueue &q, bool surfaces, bool scattered, const MarchKind &kind,
                        unsigned long long *stats, const Stamp &stamp = {});

// ---------------------------------------------------------------- device

// CPU texture LINEAR/CLAMP addressing (rtcore/cpu/Texture.cpp:324-336)
BNX_D void lerp_coord(int N, float tc, int &i0, int &i1, float &f)
{
  if (tc - .5f <= 0.f) { i0 = i1 = 0; f = 0.f; return; }
  if (tc - .5f >= (float)(N - 1)) { i0 = i1 = N - 1; f = 0.f; return; }
  f = (tc - .5f) - (float)(int)(tc - .5f);
  i0 = (int)(tc - .5f);
  i1 = i0 + 1;
}

BNX_D float lerp_l(float f, float a, float b) { return (1.f - f) * a + f * b; }

// a point query's stack and work counters (nodes and tets tested)
struct QueryCtx {
  uint32_t *ring;             // &ring[0][thread]
  uint32_t unodes, utets;
};

// StructuredDataSampler::DD::sample (volume/StructuredData.h:101-112)
BNX_D float structured_sample(const VolumeDev &v, v3 P)
{
  float rx = (P.x - v.origin[0]) * v.rcp_spacing[0];
  float ry = (P.y - v.origin[1]) * v.rcp_spacing[1];
  float rz = (P.z - v.origin[2]) * v.rcp_spacing[2];
  if (rx < 0.f || ry < 0.f || rz < 0.f) return __builtin_nanf("");
  if (rx >= (float)v.ncells[0] || ry >= (float)v.ncells[1] || rz >= (float)v.ncells[2]) return __builtin_nanf("");
  int x0, x1, y0, y1, z0, z1;
  float fx, fy, fz;
  lerp_coord(v.dims[0], rx + .5f, x0, x1, fx);
  lerp_coord(v.dims[1], ry + .5f, y0, y1, fy);
  lerp_coord(v.dims[2], rz + .5f, z0, z1, fz);
  if (v.corners) {
    // a clamped upper coordinate is its cell's far corner: the same value for
    // finite fields, and only those have this layout
    if (x0 == v.ncells[0]) { x0--; fx = 1.f; }
    if (y0 == v.ncells[1]) { y0--; fy = 1.f; }
    if (z0 == v.ncells[2]) { z0--; fz = 1.f; }
    const float4 BNX_G *c = v.corners + 2 * ((size_t)x0 + (size_t)v.ncells[0] * ((size_t)y0 + (size_t)v.ncells[1] * z0));
    const float4 a = c[0], b = c[1];
    const float c0 = lerp_l(fy, lerp_l(fx, a.x, a.y), lerp_l(fx, a.z, a.w));
    const float c1 = lerp_l(fy, lerp_l(fx, b.x, b.y), lerp_l(fx, b.z, b.w));
    return lerp_l(fz, c0, c1);
  }
  const float BNX_G *b00, *b01, *b10, *b11;
  if (v.bricks) {
    // the brick of the lower corner holds the whole footprint (apron)
    const int sh = v.brick_shift, E = (1 << sh) + 1;
    const int bx = min(x0 >> sh, v.nbricks[0] - 1), by = min(y0 >> sh, v.nbricks[1] - 1),
              bz = min(z0 >> sh, v.nbricks[2] - 1);
    const float BNX_G *br =
        v.bricks + (uint32_t)((bz * v.nbricks[1] + by) * v.nbricks[0] + bx) * (uint32_t)(E * E * E);
    const int lx = x0 - (bx << sh), ly0 = y0 - (by << sh), ly1 = y1 - (by << sh), lz0 = z0 - (bz << sh),
              lz1 = z1 - (bz << sh);
    b00 = br + (ly0 + E * lz0) * E - (bx << sh);
    b01 = br + (ly1 + E * lz0) * E - (bx << sh);
    b10 = br + (ly0 + E * lz1) * E - (bx << sh);
    b11 = br + (ly1 + E * lz1) * E - (bx << sh);
    (void)lx;
  } else {
    const size_t Nx = (size_t)v.dims[0], NxNy = (size_t)v.dims[0] * (size_t)v.dims[1];
    const float BNX_G *sc = v.scalars;
    b00 = sc + (size_t)y0 * Nx + (size_t)z0 * NxNy;
    b01 = sc + (size_t)y1 * Nx + (size_t)z0 * NxNy;
    b10 = sc + (size_t)y0 * Nx + (size_t)z1 * NxNy;
    b11 = sc + (size_t)y1 * Nx + (size_t)z1 * NxNy;
  }
  float v00 = lerp_l(fx, b00[x0], b00[x1]);
  float v01 = lerp_l(fx, b01[x0], b01[x1]);
  float v10 = lerp_l(fx, b10[x0], b10[x1]);
  float v11 = lerp_l(fx, b11[x0], b11[x1]);
  float v0 = lerp_l(fy, v00, v01);
  float v1 = lerp_l(fy, v10, v11);
  return lerp_l(fz, v0, v1);
}

// evalToImplicitPlane (umesh/common/UMeshField.h:365-371)
BNX_D float implicit_plane(v3 P, float4 a, float4 b, float4 c)
{
  const v3 N = cross(xyz(b) - xyz(a), xyz(c) - xyz(a));
  return dot(P - xyz(a), N);
}

// The four plane values of P against a tet (t[k]: against the face opposite
// vertex k, not negative inside; UMeshField::DD::tetScalar, umesh/common/
// UMeshField.h:391-436), with the vertices' scalars and the tets across the
// faces
struct TetPlanes {
  float t[4], s[4];
  int nb[4];
  float sum;
};
BNX_D TetPlanes tet_planes(const float4 BNX_G *rec, v3 P)
{
  const float4 n0 = rec[0], n1 = rec[1], n2 = rec[2], n3 = rec[3], a = rec[4], b = rec[5];
  const float2 c = *(const float2 BNX_G *)(rec + 6);
  TetPlanes r;
  const v3 pa = P - xyz(a), pb = P - xyz(b);
  r.t[3] = dot(pa, xyz(n3));
  r.t[2] = dot(pa, xyz(n2));
  r.t[1] = dot(pa, xyz(n1));
  r.t[0] = dot(pb, xyz(n0));
  r.sum = ((r.t[0] + r.t[1]) + r.t[2]) + r.t[3];
  r.s[0] = a.w;
  r.s[1] = b.w;
  r.s[2] = c.x;
  r.s[3] = c.y;
  r.nb[0] = __float_as_int(n0.w);
  r.nb[1] = __float_as_int(n1.w);
  r.nb[2] = __float_as_int(n2.w);
  r.nb[3] = __float_as_int(n3.w);
  return r;
}
BNX_D float tet_value(const TetPlanes &r)
{
  return (1.f / r.sum) * (((r.t[0] * r.s[0] + r.t[1] * r.s[1]) + r.t[2] * r.s[2]) + r.t[3] * r.s[3]);
}
// No other tet's test can accept P, so that its value is the one the
// depth-first query would return, bit for bit: every normalized barycentric
// coordinate lies above 1e-4 (in a mesh of non-overlapping tets), or is not
// negative against a face that lies in a plane of the mesh's bounding box
// (TET_HULL), beyond which there are no tets.
constexpr int TET_HULL = -1, TET_OPEN = -2;   // across a face: the box's outside; no tet known
BNX_D bool planes_interior(const TetPlanes &r)
{
  const float m = 1e-4f * r.sum;
  bool in = true;
  for (int k = 0; k < 4; k++) in &= r.t[k] > m || (r.nb[k] == TET_HULL && r.t[k] >= 0.f && m > 0.f);
  return in;
}
constexpr int TET_WALK_STEPS = 6;
// the tet across the face that P lies furthest behind
BNX_D int walk_next(const TetPlanes &r)
{
  float far = r.t[0];
  int next = r.nb[0];
  for (int x = 1; x < 4; x++) {
    const bool less = r.t[x] < far;
    far = less ? r.t[x] : far;
    next = less ? r.nb[x] : next;
  }
  return next;
}

// tetScalar on a tet given by its vertices (position, scalar)
BNX_D bool tet_scalar(const float4 BNX_G *vert, v3 P, float &out)
{
  const float4 v0 = vert[0], v1 = vert[1], v2 = vert[2], v3v = vert[3];
  const float t3 = implicit_plane(P, v0, v1, v2);
  if (t3 < 0.f) return false;
  const float t2 = implicit_plane(P, v0, v3v, v1);
  if (t2 < 0.f) return false;
  const float t1 = implicit_plane(P, v0, v2, v3v);
  if (t1 < 0.f) return false;
  const float t0 = implicit_plane(P, v1, v3v, v2);
  if (t0 < 0.f) return false;
  const float scale = 1.f / (((t0 + t1) + t2) + t3);
  out = scale * (((t0 * v0.w + t1 * v1.w) + t2 * v2.w) + t3 * v3v.w);
  return true;
}

// ------------------------------------------------------ isoparametric cells
// Pyramids, prisms and hexahedra (UMeshField::DD::eltScalar and pyrScalar /
// prismScalar / hexScalar, umesh/common/UMeshField.h:372-389, 438-495, with
// the Newton inversions of ElementIntersection.h:77-476): the cell maps
// parametric (r, s, t) to x(r, s, t) = sum_i N_i X_i over its vertices X_i
// in VTK order.  P is mapped back by Newton's method from (.5, .5, .5): at
// most 10 steps, each solving J d = x - P by Cramer's rule; converged when
// every |d_k| < 1e-4; abandoned when |det J| falls below the cell's
// tolerance or a coordinate leaves [-1e6, 1e6].  P is inside when the
// coordinates lie in the parameter domain, widened by 1e-6; the value is
// sum_i N_i f_i with the N_i of the last step's starting point.
enum { CELL_TET = 0, CELL_HEX = 1, CELL_PRISM = 2, CELL_PYR = 3 };
constexpr float CELL_IN_LO = 0.f - 1e-6f, CELL_IN_HI = 1.f + 1e-6f;

template <int TYPE> struct CellShape;
// trilinear on the unit cube
template <> struct CellShape<CELL_HEX> {
  static constexpr int N = 8;
  BNX_D static void eval(float r, float s, float t, float *w, float *dr, float *ds, float *dt)
  {
    const float rm = 1.f - r, sm = 1.f - s, tm = 1.f - t;
    w[0] = rm * sm * tm; w[1] = r * sm * tm; w[2] = r * s * tm; w[3] = rm * s * tm;
    w[4] = rm * sm * t;  w[5] = r * sm * t;  w[6] = r * s * t;  w[7] = rm * s * t;
    dr[0] = -sm * tm; dr[1] = sm * tm; dr[2] = s * tm; dr[3] = -s * tm;
    dr[4] = -sm * t;  dr[5] = sm * t;  dr[6] = s * t;  dr[7] = -s * t;
    ds[0] = -rm * tm; ds[1] = -r * tm; ds[2] = r * tm; ds[3] = rm * tm;
    ds[4] = -rm * t;  ds[5] = -r * t;  ds[6] = r * t;  ds[7] = rm * t;
    dt[0] = -rm * sm; dt[1] = -r * sm; dt[2] = -r * s; dt[3] = -rm * s;
    dt[4] = rm * sm;  dt[5] = r * sm;  dt[6] = r * s;  dt[7] = rm * s;
  }
  BNX_D static bool inside(float r, float s, float t)
  {
    return r >= CELL_IN_LO && r <= CELL_IN_HI && s >= CELL_IN_LO && s <= CELL_IN_HI && t >= CELL_IN_LO &&
           t <= CELL_IN_HI;
  }
};
// linear triangle (r, s) times linear t
template <> struct CellShape<CELL_PRISM> {
  static constexpr int N = 6;
  BNX_D static void eval(float r, float s, float t, float *w, float *dr, float *ds, float *dt)
  {
    w[0] = (1.f - r - s) * (1.f - t); w[1] = r * (1.f - t); w[2] = s * (1.f - t);
    w[3] = (1.f - r - s) * t;         w[4] = r * t;         w[5] = s * t;
    dr[0] = -1.f + t; dr[1] = 1.f - t; dr[2] = 0.f; dr[3] = -t; dr[4] = t;   dr[5] = 0.f;
    ds[0] = -1.f + t; ds[1] = 0.f;     ds[2] = 1.f - t; ds[3] = -t; ds[4] = 0.f; ds[5] = t;
    dt[0] = -1.f + r + s; dt[1] = -r; dt[2] = -s; dt[3] = 1.f - r - s; dt[4] = r; dt[5] = s;
  }
  BNX_D static bool inside(float r, float s, float t)
  {
    return r >= CELL_IN_LO && r <= CELL_IN_HI && s >= CELL_IN_LO && s <= CELL_IN_HI && t >= CELL_IN_LO &&
           t <= CELL_IN_HI && r + s <= CELL_IN_HI;
  }
};
// bilinear base quad collapsing linearly in t onto the apex (vertex 4)
template <> struct CellShape<CELL_PYR> {
  static constexpr int N = 5;
  BNX_D static void eval(float r, float s, float t, float *w, float *dr, float *ds, float *dt)
  {
    const float rm = 1.f - r, sm = 1.f - s, tm = 1.f - t;
    w[0] = rm * sm * tm; w[1] = r * sm * tm; w[2] = r * s * tm; w[3] = rm * s * tm; w[4] = t;
    dr[0] = -(s - 1.f) * (t - 1.f); dr[1] = (s - 1.f) * (t - 1.f); dr[2] = s - s * t; dr[3] = s * (t - 1.f);
    dr[4] = 0.f;
    ds[0] = -(r - 1.f) * (t - 1.f); ds[1] = r * (t - 1.f); ds[2] = r - r * t; ds[3] = (r - 1.f) * (t - 1.f);
    ds[4] = 0.f;
    dt[0] = -(r - 1.f) * (s - 1.f); dt[1] = r * (s - 1.f); dt[2] = -r * s; dt[3] = (r - 1.f) * s; dt[4] = 1.f;
  }
  BNX_D static bool inside(float r, float s, float t) { return CellShape<CELL_HEX>::inside(r, s, t); }
};

// det [a b c] (columns) = a . (b x c)
BNX_D float det3(v3 a, v3 b, v3 c) { return dot(a, cross(b, c)); }

template <int TYPE> BNX_D bool cell_invert(const float4 *V, v3 P, float tol, float &value)
{
  using C = CellShape<TYPE>;
  float r = .5f, s = .5f, t = .5f;
  float w[C::N], dr[C::N], ds[C::N], dt[C::N];
  bool converged = false;
  for (int it = 0; it < 10 && !converged; it++) {
    C::eval(r, s, t, w, dr, ds, dt);
    v3 f{0.f, 0.f, 0.f}, cr{0.f, 0.f, 0.f}, cs{0.f, 0.f, 0.f}, ct{0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < C::N; i++) {
      const v3 X = xyz(V[i]);
      f = f + X * w[i];
      cr = cr + X * dr[i];
      cs = cs + X * ds[i];
      ct = ct + X * dt[i];
    }
    f = f - P;
    const float d = det3(cr, cs, ct);
    if (fabsf(d) < tol) return false;
    // both sides of each quotient in sixteenths (DET_SCALE)
    const float den = d * bnx_num::DET_SCALE, y = rcp_rn(den);
    const float d0 = div_rn(det3(f, cs, ct) * bnx_num::DET_SCALE, den, y);
    const float d1 = div_rn(det3(cr, f, ct) * bnx_num::DET_SCALE, den, y);
    const float d2 = div_rn(det3(cr, cs, f) * bnx_num::DET_SCALE, den, y);
    r = r - d0;
    s = s - d1;
    t = t - d2;
    if (fabsf(d0) < 1e-4f && fabsf(d1) < 1e-4f && fabsf(d2) < 1e-4f) converged = true;
    else if (fabsf(r) > 1e6f || fabsf(s) > 1e6f || fabsf(t) > 1e6f) return false;
  }
  if (!converged || !C::inside(r, s, t)) return false;
  float val = 0.f;
#pragma unroll
  for (int i = 0; i < C::N; i++) val += w[i] * V[i].w;
  value = val;
  return true;
}

// the value of the cell in `slot` at P; false when P is not in it
BNX_D bool cell_value(const VolumeDev &v, int type, int slot, v3 P, float &value)
{
  const float4 BNX_G *rec = v.ucells + 8 * (size_t)slot;
  if (type == CELL_TET) return tet_scalar(rec, P, value);
  float4 V[8];
  for (int i = 0; i < 5; i++) V[i] = rec[i];
  if (type == CELL_PYR) return cell_invert<CELL_PYR>(V, P, 1e-6f, value);
  V[5] = rec[5];
  if (type == CELL_PRISM) return cell_invert<CELL_PRISM>(V, P, 1e-6f, value);
  V[6] = rec[6];
  V[7] = rec[7];
  // hexahedra: the determinant tolerance scales with the cell's size
  v3 lo = xyz(V[0]), hi = lo;
  for (int i = 1; i < 8; i++) {
    lo = v3{fmn(lo.x, V[i].x), fmn(lo.y, V[i].y), fmn(lo.z, V[i].z)};
    hi = v3{fmx(hi.x, V[i].x), fmx(hi.y, V[i].y), fmx(hi.z, V[i].z)};
  }
  return cell_invert<CELL_HEX>(V, P, 1e-10f * length(hi - lo), value);
}

// closed box test, branch-free (bitwise and) so that a node's loads are
// issued together rather than behind each other
BNX_D bool box_holds(float lx, float ly, float lz, float hx, float hy, float hz, v3 P)
{
  return (lx <= P.x) & (P.x <= hx) & (ly <= P.y) & (P.y <= hy) & (lz <= P.z) & (P.z <= hz);
}

// UMeshCuBQLSampler::sample (umesh/mc/UMeshCuBQLSampler.h:46-62) over a tet
// mesh: the first tet, depth first through the element BVH, that contains P;
// its slot (-1: none, the value is then NaN).  STRIDE: threads that share
// the ring's rows; 0: the whole stack is private (in kernels that come here
// for a few queries in a hundred, whose LDS is better spent on waves).
template <int STRIDE> BNX_D int umesh_dfs(const VolumeDev &v, v3 P, QueryCtx &cx, float &value)
{
  constexpr int RING = STRIDE > 0 ? PQ_SHORT : 0;
  uint32_t deep[PQ_SHORT + PQ_DEEP - RING];
  int sp = 0;
  uint32_t cur = 0;
  while (true) {
    if (!(cur & LEAF_BIT)) {
      const float4 BNX_G *np = (const float4 BNX_G *)(v.ebvh + cur);
      const float4 a = np[0], b = np[1], c = np[2];
      const int4 r = ((const int4 BNX_G *)np)[3];
      cx.unodes++;
      const bool h0 = (r.z >= 0) & box_holds(a.x, a.y, a.z, a.w, b.x, b.y, P);
      const bool h1 = (r.w >= 0) & box_holds(b.z, b.w, c.x, c.y, c.z, c.w, P);
      if (h0 && h1) {
        // push child 1
        if (RING > 0) {
          const int s = sp & (RING - 1);
          if (sp >= RING) deep[sp - RING] = cx.ring[s * STRIDE];
          cx.ring[s * STRIDE] = enc_child(r.y, r.w);
        } else {
          deep[sp] = enc_child(r.y, r.w);
        }
        sp++;
        cur = enc_child(r.x, r.z);
        continue;
      }
      if (h0) { cur = enc_child(r.x, r.z); continue; }
      if (h1) { cur = enc_child(r.y, r.w); continue; }
    } else {
      const int first = (int)((cur & ~LEAF_BIT) >> 3);
      const int count = (int)(cur & 7u);
      for (int k = 0; k < count; k++) {
        cx.utets++;
        const TetPlanes r = tet_planes(v.utetv + TET_REC * (size_t)(first + k), P);
        if (!(r.t[3] < 0.f || r.t[2] < 0.f || r.t[1] < 0.f || r.t[0] < 0.f)) {
          value = tet_value(r);
          return first + k;
        }
      }
    }
    if (sp == 0) {
      value = __builtin_nanf("");
      return -1;
    }
    sp--;
    if (RING > 0) {
      const int s = sp & (RING - 1);
      cur = cx.ring[s * STRIDE];
      if (sp >= RING) cx.ring[s * STRIDE] = deep[sp - RING];
    } else {
      cur = deep[sp];
    }
  }
}

// the fine-grid cell of P (clamped to the grid)
BNX_D int seed_cell(const VolumeDev &v, v3 P)
{
  const float p3[3] = {P.x, P.y, P.z};
  int c[3];
  for (int k = 0; k < 3; k++) {
    const float x = fminf(fmaxf((p3[k] - v.seed_origin[k]) * v.seed_rcp[k], 0.f), (float)(v.seed_dims[k] - 1));
    c[k] = (int)x;
  }
  return (c[2] * v.seed_dims[1] + c[1]) * v.seed_dims[0] + c[0];
}

// TransferFunction::DD::map (volume/TransferFunction.h:67-87).  rn: v.rn,
// and the macrocell's majorant is none of the tiny ones.  There a scalar so
// close to the domain's begin that its short quotient may be off in the last
// bit has a density below any product of the majorant with a draw but 0.
BNX_D float4 tf_map(const VolumeDev &v, float s, bool rn)
{
  const int N = v.ntf;
  const float span = v.dom1 - v.dom0, x = s - v.dom0;
  float f = x * v.rcp_span;
  // far above the domain (infinite scalars too) the quotient need not be exact
  if (!rn) f = x / span;
  else if (f < 2.f) f = div_rn(x, span, v.rcp_span);
  f = fmn(fmx(f, 0.f), 1.f);
  f *= (float)(N - 1);
  int idx = (int)f;
  idx = idx < 0 ? 0 : (idx > N - 2 ? N - 2 : idx);
  f -= (float)idx;
  const float4 BNX_G *tf = v.tf;
  float4 a = tf[idx], b = tf[idx + 1];
  float4 r;
  r.x = (1.f - f) * a.x + f * b.x;
  r.y = (1.f - f) * a.y + f * b.y;
  r.z = (1.f - f) * a.z + f * b.z;
  r.w = (1.f - f) * a.w + f * b.w;
  r.w *= v.base_density;
  return r;
}

// TransferFunction::DD::majorant (volume/TransferFunction.h:89-117)
BNX_D float tf_majorant(const VolumeDev &v, float lo, float hi)
{
  if (lo > hi) return 0.f;
  const int N = v.ntf;
  const float span = v.dom1 - v.dom0;
  float f_lo = (lo - v.dom0) / span;
  float f_hi = (hi - v.dom0) / span;
  f_lo = fmn(fmx(f_lo, 0.f), 1.f);
  f_hi = fmn(fmx(f_hi, 0.f), 1.f);
  f_lo *= (float)(N - 1);
  f_hi *= (float)(N - 1);
  int i_lo = (int)f_lo, i_hi = (int)f_hi;
  i_lo = i_lo < 0 ? 0 : (i_lo > N - 2 ? N - 2 : i_lo);
  i_hi = i_hi < 0 ? 0 : (i_hi > N - 2 ? N - 2 : i_hi);
  f_lo -= (float)i_lo;
  f_hi -= (float)i_hi;
  const float4 BNX_G *tf = v.tf;
  float l_lo = (1.f - f_lo) * tf[i_lo].w + f_lo * tf[i_lo + 1].w;
  float l_hi = (1.f - f_hi) * tf[i_hi].w + f_hi * tf[i_hi + 1].w;
  float m = 0.f;
  m = fmx(m, l_lo);
  m = fmx(m, l_hi);
  for (int i = i_lo + 1; i <= i_hi; i++) m = fmx(m, tf[i].w);
  return m * v.base_density;
}

// fastLog (volume/Volume.h:154-165) of f in [2^-24, 1]
BNX_D float fast_log(float f)
{
  f = div_rn(f - 1.f, f + 1.f, rcp_rn(f + 1.f));
  float f2 = f * f;
  float s = f;
  f *= f2;
  s += (1.f / 3.f) * f;
  f *= f2;
  s += (1.f / 5.f) * f;
  return s + s;
}

// boxTest (render/Ray.h:169-181): clip [r0, r1] to the field's bounds
BNX_D bool clip_bounds(const VolumeDev &v, v3 org, v3 dir, float &r0, float &r1)
{
  const v3 rd = v3{rcp_rn(dir.x), rcp_rn(dir.y), rcp_rn(dir.z)};   // dir is fixed: no component below 1e-6
  float tl[3] = {(v.lo[0] - org.x) * rd.x, (v.lo[1] - org.y) * rd.y, (v.lo[2] - org.z) * rd.z};
  float th[3] = {(v.hi[0] - org.x) * rd.x, (v.hi[1] - org.y) * rd.y, (v.hi[2] - org.z) * rd.z};
  float nr = fmx(fmx(fmn(tl[0], th[0]), fmn(tl[1], th[1])), fmn(tl[2], th[2]));
  float fr = fmn(fmn(fmx(tl[0], th[0]), fmx(tl[1], th[1])), fmx(tl[2], th[2]));
  r0 = fmx(r0, nr);
  r1 = fmn(r1, fr);
  return r0 <= r1;
}

} // namespace bnx
