// bnx_volume.hip -- volumes on gfx950: structured and unstructured fields,
// macrocell value ranges and majorants.
//
// Replaces MCVolumeAccel's build (volume/MCAccelerator.h:155-195) over
// StructuredDataSampler and UMeshCuBQLSampler, StructuredData_computeMCs
// (volume/StructuredData.cu:30-62), umeshRasterCells (umesh/common/
// UMeshField.cu:28-161) and mapMCs (volume/MCGrid.cu:96-113).
//
// Structured fields are filtered in software on the raw float grid (hardware
// texture filtering uses 8-bit fixed-point weights); a 256^3 field is 64 MiB
// and stays resident in the 256 MiB Infinity Cache.  Unstructured fields keep
// each cell's vertices (position, scalar) together in element-BVH slot order.
// The march itself is in bnx_march.hip.
#include "bnx_internal.h"
#include "bnx_render.h"
#include "bnx_volume.h"

#include <cmath>

#include <hipcub/hipcub.hpp>

namespace bnx {
namespace {

inline int nblk(long n, int b) { return (int)((n + b - 1) / b); }

// StructuredData_computeMCs: min/max over the (cpm+1)^3 vertices of a macrocell
__global__ void k_mc_ranges(VolumeDev v, float2 *ranges)
{
  int tid = blockIdx.x * blockDim.x + threadIdx.x;
  int n = v.mc[0] * v.mc[1] * v.mc[2];
  if (tid >= n) return;
  int mx = tid % v.mc[0], my = (tid / v.mc[0]) % v.mc[1], mz = tid / (v.mc[0] * v.mc[1]);
  const int c = v.cells_per_mc;
  float lo = INFINITY, hi = -INFINITY;
  for (int iz = 0; iz <= c; iz++) {
    int sz = mz * c + iz;
    if (sz >= v.dims[2]) continue;
    for (int iy = 0; iy <= c; iy++) {
      int sy = my * c + iy;
      if (sy >= v.dims[1]) continue;
      const float *row = v.scalars + (size_t)v.dims[0] * ((size_t)sy + (size_t)v.dims[1] * sz);
      for (int ix = 0; ix <= c; ix++) {
        int sx = mx * c + ix;
        if (sx >= v.dims[0]) continue;
        float f = row[sx];
        lo = fmn(lo, f);
        hi = fmx(hi, f);
      }
    }
  }
  ranges[tid] = make_float2(lo, hi);
}

// mapMCs + TransferFunction::DD::majorant
__global__ void k_majorants(VolumeDev v, const float2 *ranges, float *maj)
{
  int tid = blockIdx.x * blockDim.x + threadIdx.x;
  int n = v.mc[0] * v.mc[1] * v.mc[2];
  if (tid >= n) return;
  float2 r = ranges[tid];
  maj[tid] = tf_majorant(v, r.x, r.y);
}

// ------------------------------------------------------------------ cells
BNX_D int cell_nverts(int type) { return type == CELL_HEX ? 8 : (type == CELL_PRISM ? 6 : (type == CELL_PYR ? 5 : 4)); }

// the vertices (position, scalar) of cell c: k < cell_nverts
BNX_D float4 cell_vertex(const int4 *tets, const int4 *ext, const float4 *verts, int c, int k)
{
  const int4 q = k < 4 ? tets[c] : ext[c];
  const int j = k & 3;
  return verts[j == 0 ? q.x : (j == 1 ? q.y : (j == 2 ? q.z : q.w))];
}

// cellBounds (UMeshField.h:270-345): box of the cell's vertices, position
// in xyz and scalar range in w
BNX_D void cell_box(const int4 *tets, const int4 *ext, const uint8_t *types, const float4 *verts, int c, float4 &lo,
                    float4 &hi)
{
  const int nv = types ? cell_nverts(types[c]) : 4;
  lo = make_float4(INFINITY, INFINITY, INFINITY, INFINITY);
  hi = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
  for (int k = 0; k < nv; k++) {
    const float4 p = cell_vertex(tets, ext, verts, c, k);
    lo = make_float4(fmn(lo.x, p.x), fmn(lo.y, p.y), fmn(lo.z, p.z), fmn(lo.w, p.w));
    hi = make_float4(fmx(hi.x, p.x), fmx(hi.y, p.y), fmx(hi.z, p.z), fmx(hi.w, p.w));
  }
}

// world-space box and index of every cell (element-BVH build input); ext and types
// null: every cell is a tet
__global__ void k_cell_boxes(const int4 *tets, const int4 *ext, const uint8_t *types, const float4 *verts, int n,
                             float4 *lo, float4 *hi)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  float4 l, h;
  cell_box(tets, ext, types, verts, t, l, h);
  lo[t] = make_float4(l.x, l.y, l.z, __int_as_float(t));
  hi[t] = make_float4(h.x, h.y, h.z, 0.f);
}

// tets in element-BVH slot order
__global__ void k_tet_sort(const int4 *tets, const int *order, int n, int4 *out)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) out[s] = tets[order[s]];
}

// the 128-byte tet records (VolumeDev::utetv) in slot order; lo, hi: the
// mesh's bounds
__global__ void k_tet_pack(const int4 *tets, const float4 *verts, const int4 *nbr, int n, v3 lo, v3 hi, float4 *rec)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int4 t = tets[s], b = nbr[s];
  const float4 v0 = verts[t.x], v1 = verts[t.y], v2 = verts[t.z], w = verts[t.w];
  float4 *r = rec + TET_REC * (size_t)s;
  auto face = [&](float4 a, float4 p, float4 q, int nb) {
    if (nb < 0) {
      auto on = [&](float x, float y, float z, float l, float h) { return x == y && y == z && (x == l || x == h); };
      nb = on(a.x, p.x, q.x, lo.x, hi.x) || on(a.y, p.y, q.y, lo.y, hi.y) || on(a.z, p.z, q.z, lo.z, hi.z) ? TET_HULL
                                                                                                    : TET_OPEN;
    }
    const v3 N = cross(xyz(p) - xyz(a), xyz(q) - xyz(a));
    return make_float4(N.x, N.y, N.z, __int_as_float(nb));
  };
  r[0] = face(v1, w, v2, b.x);
  r[1] = face(v0, v2, w, b.y);
  r[2] = face(v0, w, v1, b.z);
  r[3] = face(v0, v1, v2, b.w);
  r[4] = v0;
  r[5] = v1;
  r[6] = make_float4(v2.w, w.w, 0.f, 0.f);
}

// Cells in element-BVH slot order: 128 bytes of vertices, and the filter box
// that a point query tests before a cell's Newton inversion.  A point that
// the inversion accepts lies in the hull of the cell's vertices but for the
// domain's margin (1e-6), the last Newton step (below 1e-4 of the cell in
// each parameter) and the rounding of coordinates: a twentieth of the
// cell's extent and 1e-5 of the coordinates hold all of that many times
// over.  A tet's own test accepts what its planes accept, however thin the
// tet: its box is open.
__global__ void k_cell_pack(const int4 *tets, const int4 *ext, const uint8_t *types, const float4 *verts,
                            const int *order, int n, float4 *rec, float4 *box)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int c = order[s], type = types[c], nv = cell_nverts(type);
  float4 *r = rec + 8 * (size_t)s;
  for (int k = 0; k < 8; k++) r[k] = cell_vertex(tets, ext, verts, c, k < nv ? k : 0);
  float4 lo, hi;
  cell_box(tets, ext, types, verts, c, lo, hi);
  float m = INFINITY;
  if (type != CELL_TET) {
    const float size = fmx(fmx(hi.x - lo.x, hi.y - lo.y), hi.z - lo.z);
    const float far = fmx(fmx(fmx(fabsf(lo.x), fabsf(hi.x)), fmx(fabsf(lo.y), fabsf(hi.y))),
                          fmx(fabsf(lo.z), fabsf(hi.z)));
    m = .05f * size + 1e-5f * far;
  }
  box[2 * (size_t)s] = make_float4(lo.x - m, lo.y - m, lo.z - m, __int_as_float(type));
  box[2 * (size_t)s + 1] = make_float4(hi.x + m, hi.y + m, hi.z + m, 0.f);
}

__global__ void k_fill_ranges(int *lo, int *hi, int n)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  lo[c] = f2o(INFINITY);
  hi[c] = f2o(-INFINITY);
}

__global__ void k_finish_ranges(const int *lo, const int *hi, int n, float2 *ranges)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) ranges[c] = make_float2(o2f(lo[c]), o2f(hi[c]));
}

BNX_D float4 mid4(float4 a, float4 b)
{
  return make_float4(0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z), 0.5f * (a.w + b.w));
}
BNX_D float len3(float4 a, float4 b) { return length(xyz(b) - xyz(a)); }

// macrocell min/max of one cell: a per-thread cache of the last cell, since
// the 32 pieces of a tet mostly fall into the same cell; flushed with
// ordered-int atomics (exact float min/max in any order)
struct RangeCache {
  int cell = -1;
  float lo = INFINITY, hi = -INFINITY;
  BNX_D void flush(int *rlo, int *rhi)
  {
    if (cell < 0) return;
    atomicMin(rlo + cell, f2o(lo));
    atomicMax(rhi + cell, f2o(hi));
  }
  BNX_D void add(int c, float l, float h, int *rlo, int *rhi)
  {
    if (c != cell) {
      flush(rlo, rhi);
      cell = c;
      lo = l;
      hi = h;
    } else {
      lo = fmn(lo, l);
      hi = fmx(hi, h);
    }
  }
};

// umeshRasterCells + rasterTet<5> (UMeshField.cu:28-161): each tet is split
// 5 times on its longest edge (ties: ab, ac, ad, bc, bd, cd in that order);
// the box of each of the 32 pieces is rasterized with rasterBox
// (volume/MCGrid.cuh:95-122), which skips boxes flat in any dimension.
// Piece p is reached by taking child (p >> (4 - level)) & 1 at every level.
// Other cells rasterize their own box (the three-argument rasterBox,
// MCGrid.cuh:66-93, which skips only inverted boxes).
BNX_D void raster_cell_box(const VolumeDev &v, float4 l, float4 h, RangeCache &cache, int *rlo, int *rhi)
{
  if (l.x > h.x || l.y > h.y || l.z > h.z) return;
  int lo[3], hi[3];
  const float bl[3] = {l.x, l.y, l.z}, bh[3] = {h.x, h.y, h.z};
  for (int k = 0; k < 3; k++) {
    lo[k] = (int)((bl[k] - v.mc_origin[k]) * v.mc_rcp_spacing[k]);
    hi[k] = (int)((bh[k] - v.mc_origin[k]) * v.mc_rcp_spacing[k]);
    lo[k] = min(max(lo[k], 0), v.mc[k] - 1);
    hi[k] = min(max(hi[k], 0), v.mc[k] - 1);
  }
  for (int iz = lo[2]; iz <= hi[2]; iz++)
    for (int iy = lo[1]; iy <= hi[1]; iy++)
      for (int ix = lo[0]; ix <= hi[0]; ix++) cache.add(ix + v.mc[0] * (iy + v.mc[1] * iz), l.w, h.w, rlo, rhi);
}

__global__ void k_umesh_raster(const int4 *tets, const int4 *ext, const uint8_t *types, const float4 *verts, int n,
                               VolumeDev v, int *rlo, int *rhi)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  if (types && types[t] != CELL_TET) {
    RangeCache cache;
    float4 l, h;
    cell_box(tets, ext, types, verts, t, l, h);
    raster_cell_box(v, l, h, cache, rlo, rhi);
    cache.flush(rlo, rhi);
    return;
  }
  const int4 q = tets[t];
  const float4 A = verts[q.x], B = verts[q.y], Cc = verts[q.z], D = verts[q.w];
  RangeCache cache;
  for (int p = 0; p < 32; p++) {
    float4 a = A, b = B, c = Cc, d = D;
    for (int level = 0; level < 5; level++) {
      const float lab = len3(a, b), lac = len3(a, c), lad = len3(a, d);
      const float lbc = len3(b, c), lbd = len3(b, d), lcd = len3(c, d);
      const float maxLen = fmx(fmx(fmx(fmx(fmx(lab, lac), lad), lbc), lbd), lcd);
      float4 oa, ob, oc, od0, od1;
      if (lab >= maxLen) { oa = mid4(a, b); ob = c; oc = d; od0 = a; od1 = b; }
      else if (lac >= maxLen) { oa = mid4(a, c); ob = b; oc = d; od0 = a; od1 = c; }
      else if (lad >= maxLen) { oa = mid4(a, d); ob = b; oc = c; od0 = a; od1 = d; }
      else if (lbc >= maxLen) { oa = mid4(b, c); ob = a; oc = d; od0 = b; od1 = c; }
      else if (lbd >= maxLen) { oa = mid4(b, d); ob = a; oc = c; od0 = b; od1 = d; }
      else { oa = mid4(c, d); ob = a; oc = b; od0 = c; od1 = d; }
      a = oa;
      b = ob;
      c = oc;
      d = ((p >> (4 - level)) & 1) ? od1 : od0;
    }
    const float lx = fmn(fmn(fmn(a.x, b.x), c.x), d.x), hx = fmx(fmx(fmx(a.x, b.x), c.x), d.x);
    const float ly = fmn(fmn(fmn(a.y, b.y), c.y), d.y), hy = fmx(fmx(fmx(a.y, b.y), c.y), d.y);
    const float lz = fmn(fmn(fmn(a.z, b.z), c.z), d.z), hz = fmx(fmx(fmx(a.z, b.z), c.z), d.z);
    const float lw = fmn(fmn(fmn(a.w, b.w), c.w), d.w), hw = fmx(fmx(fmx(a.w, b.w), c.w), d.w);
    if (lx >= hx || ly >= hy || lz >= hz) continue;
    int lo[3], hi[3];
    const float bl[3] = {lx, ly, lz}, bh[3] = {hx, hy, hz};
    for (int k = 0; k < 3; k++) {
      lo[k] = (int)((bl[k] - v.mc_origin[k]) * v.mc_rcp_spacing[k]);
      hi[k] = (int)((bh[k] - v.mc_origin[k]) * v.mc_rcp_spacing[k]);
      lo[k] = min(max(lo[k], 0), v.mc[k] - 1);
      hi[k] = min(max(hi[k], 0), v.mc[k] - 1);
    }
    for (int iz = lo[2]; iz <= hi[2]; iz++)
      for (int iy = lo[1]; iy <= hi[1]; iy++)
        for (int ix = lo[0]; ix <= hi[0]; ix++)
          cache.add(ix + v.mc[0] * (iy + v.mc[1] * iz), lw, hw, rlo, rhi);
  }
  cache.flush(rlo, rhi);
}

// one thread per brick texel: the texel of the linear field at the brick's
// cell origin + (lx, ly, lz), clamped to the field (apron texels past the
// last vertex repeat it; no footprint reads them)
__global__ void k_brick(const float *src, int nx, int ny, int nz, int shift, int nbx, int nby, long long total,
                        float *dst)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int E = (1 << shift) + 1, E3 = E * E * E;
  const long long b = i / E3;
  const int t = (int)(i - b * E3);
  const int lx = t % E, ly = (t / E) % E, lz = t / (E * E);
  const int bx = (int)(b % nbx), by = (int)((b / nbx) % nby), bz = (int)(b / ((long long)nbx * nby));
  const int x = min((bx << shift) + lx, nx - 1), y = min((by << shift) + ly, ny - 1),
            z = min((bz << shift) + lz, nz - 1);
  dst[i] = src[(size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z)];
}

// one thread per cell: its eight corners; *bad is raised for a value that is
// not finite
__global__ void k_corners(const float *src, int nx, int ny, int cx, int cy, long long ncells, float4 *dst, int *bad)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncells) return;
  const int x = (int)(i % cx), y = (int)((i / cx) % cy), z = (int)(i / ((long long)cx * cy));
  const float *p = src + (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z);
  const size_t sy = nx, sz = (size_t)nx * ny;
  const float4 a = make_float4(p[0], p[1], p[sy], p[sy + 1]);
  const float4 b = make_float4(p[sz], p[sz + 1], p[sz + sy], p[sz + sy + 1]);
  dst[2 * i] = a;
  dst[2 * i + 1] = b;
  const float m = fabsf(a.x) + fabsf(a.y) + fabsf(a.z) + fabsf(a.w) + fabsf(b.x) + fabsf(b.y) + fabsf(b.z) + fabsf(b.w);
  if (!(m < INFINITY)) *bad = 1;
}

} // namespace

int volume_corners(Volume *v)
{
  VolumeDev &d = v->dd;
  hipStream_t st = v->dev->stream;
  d.corners = nullptr;
  const long long n = (long long)d.ncells[0] * d.ncells[1] * d.ncells[2];
  const size_t bytes = 2 * sizeof(float4) * (size_t)n;
  size_t free_bytes = 0, total = 0;
  BNX_HIP(hipMemGetInfo(&free_bytes, &total));
  if (bytes > free_bytes / 8 || n >= (1LL << 31)) return BNX_OK;
  DevMem bad;
  BNX_HIP(bad.ensure(sizeof(int)));
  if (v->corners.ensure(bytes) != hipSuccess) {
    (void)hipGetLastError();            // no room: the linear layout serves
    return BNX_OK;
  }
  BNX_HIP(hipMemsetAsync(bad.ptr, 0, sizeof(int), st));
  k_corners<<<nblk(n, 256), 256, 0, st>>>(v->scalars.as<float>(), d.dims[0], d.dims[1], d.ncells[0], d.ncells[1], n,
                                          v->corners.as<float4>(), bad.as<int>());
  BNX_HIP(hipGetLastError());
  int h = 0;
  BNX_HIP(hipMemcpyAsync(&h, bad.ptr, sizeof(int), hipMemcpyDeviceToHost, st));
  BNX_HIP(hipStreamSynchronize(st));
  if (h) v->corners.release();
  else BNX_SET(d.corners, v->corners.ptr);
  v->version++;
  return BNX_OK;
}

int volume_brick(Volume *v, int shift)
{
  VolumeDev &d = v->dd;
  if (shift <= 0) {
    v->bricks.release();
    d.bricks = nullptr;
    d.brick_shift = 0;
    return BNX_OK;
  }
  const int B = 1 << shift, E = B + 1;
  for (int k = 0; k < 3; k++) d.nbricks[k] = (d.ncells[k] + B - 1) / B;
  const long long total = (long long)d.nbricks[0] * d.nbricks[1] * d.nbricks[2] * E * E * E;
  BNX_CHECK(total < (1LL << 31), BNX_ERR_UNSUPPORTED, "structured field too large for the bricked layout");
  BNX_HIP(v->bricks.ensure(sizeof(float) * (size_t)total));
  k_brick<<<nblk(total, 256), 256, 0, v->dev->stream>>>(v->scalars.as<float>(), d.dims[0], d.dims[1], d.dims[2],
                                                        shift, d.nbricks[0], d.nbricks[1], total,
                                                        v->bricks.as<float>());
  BNX_HIP(hipGetLastError());
  BNX_SET(d.bricks, v->bricks.ptr);
  d.brick_shift = shift;
  v->version++;
  return BNX_OK;
}

int volume_build(Volume *v)
{
  Device *dev = v->dev;
  VolumeDev &d = v->dd;
  const size_t nmc = (size_t)d.mc[0] * d.mc[1] * d.mc[2];
  BNX_HIP(v->ranges.ensure(sizeof(float2) * nmc));
  BNX_HIP(v->majorants.ensure(sizeof(float) * nmc));
  BNX_SET(d.majorants, v->majorants.ptr);
  BNX_SET(d.ranges, v->ranges.ptr);
  k_mc_ranges<<<nblk((long)nmc, 64), 64, 0, dev->stream>>>(d, v->ranges.as<float2>());
  k_majorants<<<nblk((long)nmc, 256), 256, 0, dev->stream>>>(d, v->ranges.as<float2>(), v->majorants.as<float>());
  BNX_HIP(hipStreamSynchronize(dev->stream));
  BNX_HIP(hipGetLastError());
  return BNX_OK;
}

// ------------------------------------------------- tet face adjacency
// Face k of a tet is the one opposite its vertex k.  Every face gets a
// 64-bit hash of its sorted vertex triple; after sorting the hashes, a run of
// exactly two faces with the same triple is a shared face.  Hash collisions
// and non-manifold faces leave the neighbour at -1 (the walk then falls back
// to the depth-first query), so the table only ever names true neighbours.
__device__ uint64_t mix64(uint64_t x)
{
  x ^= x >> 30;
  x *= 0xbf58476d1ce4e5b9ull;
  x ^= x >> 27;
  x *= 0x94d049bb133111ebull;
  x ^= x >> 31;
  return x;
}

__device__ int3 face_of(const int4 t, int k)
{
  int a, b, c;
  if (k == 0) { a = t.y; b = t.z; c = t.w; }
  else if (k == 1) { a = t.x; b = t.z; c = t.w; }
  else if (k == 2) { a = t.x; b = t.y; c = t.w; }
  else { a = t.x; b = t.y; c = t.z; }
  // sort the triple
  if (a > b) { int x = a; a = b; b = x; }
  if (b > c) { int x = b; b = c; c = x; }
  if (a > b) { int x = a; a = b; b = x; }
  return make_int3(a, b, c);
}

__global__ void k_face_keys(const int4 *tets, int ntet, uint64_t *keys, int *vals, int4 *nbr)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ntet) return;
  const int4 t = tets[i];
  for (int k = 0; k < 4; k++) {
    const int3 f = face_of(t, k);
    keys[4 * (size_t)i + k] =
        mix64(((uint64_t)(uint32_t)f.x << 32 | (uint32_t)f.y) ^ mix64((uint64_t)(uint32_t)f.z + 0x9e3779b97f4a7c15ull));
    vals[4 * (size_t)i + k] = 4 * i + k;
  }
  nbr[i] = make_int4(-1, -1, -1, -1);
}

__global__ void k_face_match(const int4 *tets, const uint64_t *keys, const int *vals, long long nf, int4 *nbr)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i + 1 >= nf) return;
  if (keys[i] != keys[i + 1]) return;
  if (i > 0 && keys[i - 1] == keys[i]) return;         // not the first of its run
  if (i + 2 < nf && keys[i + 2] == keys[i]) return;    // a run of more than two
  const int fa = vals[i], fb = vals[i + 1];
  const int ta = fa >> 2, ka = fa & 3, tb = fb >> 2, kb = fb & 3;
  const int3 A = face_of(tets[ta], ka), B = face_of(tets[tb], kb);
  if (A.x != B.x || A.y != B.y || A.z != B.z || ta == tb) return;
  ((int *)nbr)[4 * (size_t)ta + ka] = tb;
  ((int *)nbr)[4 * (size_t)tb + kb] = ta;
}

int build_tet_neighbors(Device *dev, const int4 *tets, int ntet, DevMem &nbr)
{
  hipStream_t st = dev->stream;
  const size_t nf = 4 * (size_t)ntet;
  DevMem keys, keys2, vals, vals2, tmp;
  BNX_HIP(nbr.ensure(sizeof(int4) * (size_t)(ntet > 0 ? ntet : 1)));
  if (ntet == 0) return BNX_OK;
  BNX_HIP(keys.ensure(sizeof(uint64_t) * nf));
  BNX_HIP(keys2.ensure(sizeof(uint64_t) * nf));
  BNX_HIP(vals.ensure(sizeof(int) * nf));
  BNX_HIP(vals2.ensure(sizeof(int) * nf));
  k_face_keys<<<nblk(ntet, 256), 256, 0, st>>>(tets, ntet, keys.as<uint64_t>(), vals.as<int>(), nbr.as<int4>());
  size_t tmp_bytes = 0;
  BNX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, keys.as<uint64_t>(), keys2.as<uint64_t>(),
                                             vals.as<int>(), vals2.as<int>(), (int)nf, 0, 64, st));
  BNX_HIP(tmp.ensure(tmp_bytes));
  BNX_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.ptr, tmp_bytes, keys.as<uint64_t>(), keys2.as<uint64_t>(),
                                             vals.as<int>(), vals2.as<int>(), (int)nf, 0, 64, st));
  k_face_match<<<nblk((long)nf, 256), 256, 0, st>>>(tets, keys2.as<uint64_t>(), vals2.as<int>(), (long long)nf,
                                                   nbr.as<int4>());
  BNX_HIP(hipGetLastError());
  BNX_HIP(hipStreamSynchronize(st));
  return BNX_OK;
}

// ------------------------------------------------------------ fine grid
// The value ranges: every cell adds the range of its vertices' scalars to the
// grid cells that its box touches, grown by a twentieth of its extent and
// 1e-5 of its coordinates (a test accepts points outside the cell by far
// less, see k_cell_pack).  Values are means of the scalars with weights above
// -1e-3 (a Newton inversion's last step), so the ranges take in a thousandth
// of their width and 1e-5 of the scalars at either end.
//
// A tet adds less: only to the grid cells that reach past none of its planes
// by more than a hundredth of its size, and there only the values that its
// linear function takes between the cell's corners.  With its whole range in
// every grid cell of its box a mesh of few tets, whose boxes take in most of
// it, settled hardly a sample (jittered cubes of five tets, 1920x1080, 2 spp,
// isosurface and volume: 8^3 15.5 ms then, 11.4 now; 14^3 13.2 and 9.7; 40^3
// 12.5 and 10.0; 160^3 13.5 and 12.9).
//
// A cell with more than `most` grid cells in its box, and a tet too flat for
// its planes to bound where it is accepted, adds its whole range to the one
// that all grid cells share.  LANES threads work on a cell.
constexpr float FINE_SLACK = 1e-5f;
template <int LANES>
__global__ void k_fine_ranges(const int4 *tets, const int4 *ext, const uint8_t *types, const float4 *verts, int n,
                              VolumeDev d, long long most, int *lo, int *hi, int *all)
{
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int c = (int)(tid / LANES), sub = (int)(tid % LANES);
  if (c >= n) return;
  float4 l, h;
  cell_box(tets, ext, types, verts, c, l, h);
  const float size = fmx(fmx(h.x - l.x, h.y - l.y), h.z - l.z);
  const float far = fmx(fmx(fmx(fabsf(l.x), fabsf(h.x)), fmx(fabsf(l.y), fabsf(h.y))), fmx(fabsf(l.z), fabsf(h.z)));
  const float m = .05f * size + 1e-5f * far, slack = 2e-3f * (h.w - l.w) + FINE_SLACK * fmx(fabsf(l.w), fabsf(h.w));
  const int a = seed_cell(d, v3{l.x - m, l.y - m, l.z - m}), b = seed_cell(d, v3{h.x + m, h.y + m, h.z + m});
  const int nx = d.seed_dims[0], ny = d.seed_dims[1];
  const int ax = a % nx, ay = (a / nx) % ny, az = a / (nx * ny), bx = b % nx, by = (b / nx) % ny, bz = b / (nx * ny);
  const bool finite = slack < INFINITY;       // an infinite scalar: any value may come of it
  // A tet's planes, computed with an error e, accept the tet scaled by
  // (r + e) / r about its incentre, r the radius of its inscribed sphere: with
  // e below 1e-6 of the distance to it and r a thousandth of its size that is
  // well inside the margin.  A flatter one may accept any point of its leaf.
  const bool tet = !types || types[c] == CELL_TET;
  bool flat = false;
  v3 N[4], at[4], grad{0.f, 0.f, 0.f};
  float past[4], s[4], sum = 0.f;
  const float mid = .5f * l.w + .5f * h.w;
  if (tet) {
    float4 q[4];
    for (int k = 0; k < 4; k++) q[k] = cell_vertex(tets, ext, verts, c, k);
    // the planes of tet_planes: t[k] = dot(P - at[k], N[k])
    N[0] = cross(xyz(q[3]) - xyz(q[1]), xyz(q[2]) - xyz(q[1]));
    N[1] = cross(xyz(q[2]) - xyz(q[0]), xyz(q[3]) - xyz(q[0]));
    N[2] = cross(xyz(q[3]) - xyz(q[0]), xyz(q[1]) - xyz(q[0]));
    N[3] = cross(xyz(q[1]) - xyz(q[0]), xyz(q[2]) - xyz(q[0]));
    for (int k = 0; k < 4; k++) at[k] = xyz(q[k == 0 ? 1 : 0]);
    sum = dot(xyz(q[1]) - xyz(q[0]), N[1]);
    float area = 0.f;
    for (int k = 0; k < 4; k++) area += length(N[k]);
    flat = !(fabsf(sum) > 1e-3f * size * area);
    for (int k = 0; k < 4; k++) {
      s[k] = (q[k].w - mid) / sum;
      grad = grad + s[k] * N[k];
    }
  }
  const long long cells = (long long)(bx - ax + 1) * (by - ay + 1) * (bz - az + 1);
  if (!finite || flat || cells > most) {
    if (sub == 0) {
      atomicMin(all, f2o(finite ? l.w - slack : -INFINITY));
      atomicMax(all + 1, f2o(finite ? h.w + slack : INFINITY));
    }
    return;
  }
  // half the sides of a grid cell, with what the cell that a point is given
  // to may be off by
  const v3 side{1.f / d.seed_rcp[0], 1.f / d.seed_rcp[1], 1.f / d.seed_rcp[2]};
  const v3 half{.52f * side.x + 1e-5f * far, .52f * side.y + 1e-5f * far, .52f * side.z + 1e-5f * far};
  if (tet)
    for (int k = 0; k < 4; k++) past[k] = dot(vabs(N[k]), half) + 1e-2f * size * length(N[k]);
  // the linear function's rounding: each term's, however much they cancel
  float reach = dot(vabs(grad), half);
  if (tet)
    for (int k = 0; k < 4; k++) reach += 1e-6f * fabsf(s[k]) * dot(vabs(N[k]), half);
  const int wx = bx - ax + 1, wy = by - ay + 1;
  for (long long j = sub; j < cells; j += LANES) {
    const int x = ax + (int)(j % wx), y = ay + (int)((j / wx) % wy), z = az + (int)(j / ((long long)wx * wy));
    float vl = l.w, vh = h.w;
    if (tet) {
      const v3 C{d.seed_origin[0] + ((float)x + .5f) * side.x, d.seed_origin[1] + ((float)y + .5f) * side.y,
                 d.seed_origin[2] + ((float)z + .5f) * side.z};
      float f = mid, err = 0.f;
      bool out = false;
      for (int k = 0; k < 4; k++) {
        const float t = dot(C - at[k], N[k]);
        out |= t < -past[k];
        f += t * s[k];
        err += 1e-6f * fabsf(s[k]) * dot(vabs(C - at[k]), vabs(N[k]));
      }
      vl = fmx(vl, f - (reach + err));
      vh = fmn(vh, f + (reach + err));
      if (out || vl - slack > vh + slack) continue;
    }
    const int i = (z * ny + y) * nx + x;
    atomicMin(lo + i, f2o(vl - slack));
    atomicMax(hi + i, f2o(vh + slack));
  }
}

// per grid cell the tet (depth-first query) holding its centre, and its range
constexpr int SEED_TB = 256;
__global__ __launch_bounds__(SEED_TB) void k_fine_pack(VolumeDev d, int ncells, const int *lo, const int *hi,
                                                       const int *all, float4 *fine)
{
  __shared__ uint32_t ring[PQ_SHORT * SEED_TB];
  QueryCtx cx{ring + threadIdx.x, 0, 0};
  const int c = blockIdx.x * SEED_TB + threadIdx.x;
  if (c >= ncells) return;
  int seed = -1;
  if (d.field == FIELD_KIND_TETS) {
    const int nx = d.seed_dims[0], ny = d.seed_dims[1];
    const int ix = c % nx, iy = (c / nx) % ny, iz = c / (nx * ny);
    const v3 P = v3{d.seed_origin[0] + ((float)ix + .5f) / d.seed_rcp[0],
                    d.seed_origin[1] + ((float)iy + .5f) / d.seed_rcp[1],
                    d.seed_origin[2] + ((float)iz + .5f) / d.seed_rcp[2]};
    float f;
    seed = umesh_dfs<SEED_TB>(d, P, cx, f);
  }
  fine[c] = make_float4(__int_as_float(seed), o2f(min(lo[c], all[0])), o2f(max(hi[c], all[1])), 0.f);
}

// Fine grid over the bounds: of a mesh of tets about one cell per two tets, and
// no fewer than FINE_MC a side of a macrocell (a march's sub-steps are a tenth
// of one; 2: 14^3 10.2 ms and 40^3 11.7, 6: 10.7 and 9.6, in three times the
// memory), of another mesh eight per cell; at most 256 a side.  ext, types
// null: tets
constexpr int FINE_MC = 4;
int build_fine_grid(Volume *v, const int4 *tets, const int4 *ext, const uint8_t *types, const float4 *verts, int n)
{
  VolumeDev &d = v->dd;
  hipStream_t st = v->dev->stream;
  double size[3], vol = 1.0;
  bool flat = false;
  d.ufine = nullptr;
  for (int k = 0; k < 3; k++) {
    size[k] = (double)d.hi[k] - (double)d.lo[k];
    if (size[k] > 0.0) vol *= size[k];
    else flat = true;
  }
  if (flat) return BNX_OK;      // a flat mesh holds no cell with volume
  const double h = std::cbrt(vol / std::max(1.0, d.field == FIELD_KIND_TETS ? n / 2.0 : 8.0 * n));
  long long ncells = 1;
  for (int k = 0; k < 3; k++) {
    const double least = d.field == FIELD_KIND_TETS ? (double)FINE_MC * d.mc[k] : 1.0;
    d.seed_dims[k] = (int)std::min(256.0, std::max(least, std::ceil(size[k] / h)));
    d.seed_origin[k] = d.lo[k];
    d.seed_rcp[k] = (float)d.seed_dims[k] / (float)size[k];
    ncells *= d.seed_dims[k];
  }
  DevMem lo, hi;
  BNX_HIP(v->ufine.ensure(sizeof(float4) * (size_t)ncells));
  BNX_HIP(lo.ensure(sizeof(int) * (size_t)ncells));
  BNX_HIP(hi.ensure(sizeof(int) * (size_t)ncells));
  k_fill_ranges<<<nblk(ncells, 256), 256, 0, st>>>(lo.as<int>(), hi.as<int>(), (int)ncells);
  DevMem all;
  BNX_HIP(all.ensure(2 * sizeof(int)));
  k_fill_ranges<<<1, 64, 0, st>>>(all.as<int>(), all.as<int>() + 1, 1);
  // few cells meet many grid cells each: more of these, and more threads, for each
  const long long most = std::max(4096LL, (1LL << 26) / std::max(1, n));
  if (n < (1 << 18))
    k_fine_ranges<64><<<nblk(64L * n, 256), 256, 0, st>>>(tets, ext, types, verts, n, d, most, lo.as<int>(),
                                                          hi.as<int>(), all.as<int>());
  else
    k_fine_ranges<1><<<nblk(n, 256), 256, 0, st>>>(tets, ext, types, verts, n, d, most, lo.as<int>(), hi.as<int>(),
                                                   all.as<int>());
  k_fine_pack<<<nblk(ncells, SEED_TB), SEED_TB, 0, st>>>(d, (int)ncells, lo.as<int>(), hi.as<int>(), all.as<int>(),
                                                         v->ufine.as<float4>());
  BNX_HIP(hipGetLastError());
  BNX_HIP(hipStreamSynchronize(st));
  BNX_SET(d.ufine, v->ufine.ptr);
  return BNX_OK;
}

int volume_build_umesh(Volume *v, const int4 *tets4, const int4 *ext4, const uint8_t *types, int ntet,
                       const float4 *verts4, int nvert)
{
  Device *dev = v->dev;
  VolumeDev &d = v->dd;
  hipStream_t st = dev->stream;
  const bool mixed = types != nullptr;
  const BuildScope scope(dev->build);
  DevMem verts, tets, ext, typ, rlo, rhi;
  DevMem &lo = dev->build.box_lo, &hi = dev->build.box_hi;
  BNX_HIP(verts.ensure(sizeof(float4) * (size_t)nvert));
  BNX_HIP(hipMemcpyAsync(verts.ptr, verts4, sizeof(float4) * (size_t)nvert, hipMemcpyHostToDevice, st));
  BNX_HIP(tets.ensure(sizeof(int4) * (size_t)ntet));
  BNX_HIP(hipMemcpyAsync(tets.ptr, tets4, sizeof(int4) * (size_t)ntet, hipMemcpyHostToDevice, st));
  if (mixed) {
    BNX_HIP(ext.ensure(sizeof(int4) * (size_t)ntet));
    BNX_HIP(typ.ensure((size_t)ntet));
    BNX_HIP(hipMemcpyAsync(ext.ptr, ext4, sizeof(int4) * (size_t)ntet, hipMemcpyHostToDevice, st));
    BNX_HIP(hipMemcpyAsync(typ.ptr, types, (size_t)ntet, hipMemcpyHostToDevice, st));
  }
  const int4 *ext_d = mixed ? ext.as<int4>() : nullptr;
  const uint8_t *typ_d = mixed ? typ.as<uint8_t>() : nullptr;
  // element BVH over the cells' boxes; cells stored in its slot order
  BNX_HIP(lo.ensure(sizeof(float4) * (size_t)ntet));
  BNX_HIP(hi.ensure(sizeof(float4) * (size_t)ntet));
  k_cell_boxes<<<nblk(ntet, 256), 256, 0, st>>>(tets.as<int4>(), ext_d, typ_d, verts.as<float4>(), ntet,
                                                lo.as<float4>(), hi.as<float4>());
  BNX_HIP(hipGetLastError());
  int rc = build_bvh(dev, lo.as<float4>(), hi.as<float4>(), ntet, 4, v->ebvh);
  if (rc != BNX_OK) return rc;
  if (v->ebvh.max_depth + 1 > PQ_SHORT + PQ_DEEP) {
    set_error("bnx_volume_create_umesh: element BVH deeper than the point-query stack");
    return BNX_ERR_UNSUPPORTED;
  }
  BNX_SET(d.ebvh, v->ebvh.nodes.ptr);
  d.field = mixed ? FIELD_KIND_CELLS : FIELD_KIND_TETS;
  if (mixed) {
    // other cells than tets: point queries go depth first through the
    // element BVH (no tet walk)
    BNX_HIP(v->ucells.ensure(sizeof(float4) * 8 * (size_t)ntet));
    BNX_HIP(v->ucellbox.ensure(sizeof(float4) * 2 * (size_t)ntet));
    k_cell_pack<<<nblk(ntet, 256), 256, 0, st>>>(tets.as<int4>(), ext_d, typ_d, verts.as<float4>(),
                                                 v->ebvh.order.as<int>(), ntet, v->ucells.as<float4>(),
                                                 v->ucellbox.as<float4>());
    BNX_HIP(hipGetLastError());
    if ((rc = collapse_bvh4(dev, v->ebvh)) != BNX_OK) return rc;
    BNX_CHECK(v->ebvh.stack_need4 <= PQ_SHORT + PQ_DEEP4, BNX_ERR_UNSUPPORTED,
              "bnx_volume_create_umesh: element BVH deeper than the point-query stack");
    BNX_SET(d.ebvh4, v->ebvh.nodes4.ptr);
    BNX_SET(d.ucells, v->ucells.ptr);
    BNX_SET(d.ucellbox, v->ucellbox.ptr);
  } else {
    // the tet records: planes and face neighbours (for the walking point
    // query) in one 128-byte record per slot
    DevMem sorted, nbr;
    BNX_HIP(sorted.ensure(sizeof(int4) * (size_t)ntet));
    k_tet_sort<<<nblk(ntet, 256), 256, 0, st>>>(tets.as<int4>(), v->ebvh.order.as<int>(), ntet, sorted.as<int4>());
    BNX_HIP(hipGetLastError());
    if ((rc = build_tet_neighbors(dev, sorted.as<int4>(), ntet, nbr)) != BNX_OK) return rc;
    BNX_HIP(v->utetv.ensure(sizeof(float4) * TET_REC * (size_t)ntet));
    k_tet_pack<<<nblk(ntet, 256), 256, 0, st>>>(sorted.as<int4>(), verts.as<float4>(), nbr.as<int4>(), ntet,
                                                v3{d.lo[0], d.lo[1], d.lo[2]}, v3{d.hi[0], d.hi[1], d.hi[2]},
                                                v->utetv.as<float4>());
    BNX_HIP(hipGetLastError());
    BNX_SET(d.utetv, v->utetv.ptr);
    BNX_HIP(hipStreamSynchronize(st));
  }
  if ((rc = build_fine_grid(v, tets.as<int4>(), ext_d, typ_d, verts.as<float4>(), ntet)) != BNX_OK) return rc;
  // macrocell value ranges
  const int nmc = d.mc[0] * d.mc[1] * d.mc[2];
  BNX_HIP(rlo.ensure(sizeof(int) * (size_t)nmc));
  BNX_HIP(rhi.ensure(sizeof(int) * (size_t)nmc));
  BNX_HIP(v->ranges.ensure(sizeof(float2) * (size_t)nmc));
  BNX_HIP(v->majorants.ensure(sizeof(float) * (size_t)nmc));
  BNX_SET(d.ranges, v->ranges.ptr);
  BNX_SET(d.majorants, v->majorants.ptr);
  k_fill_ranges<<<nblk(nmc, 256), 256, 0, st>>>(rlo.as<int>(), rhi.as<int>(), nmc);
  k_umesh_raster<<<nblk(ntet, 128), 128, 0, st>>>(tets.as<int4>(), ext_d, typ_d, verts.as<float4>(), ntet, d,
                                                  rlo.as<int>(), rhi.as<int>());
  k_finish_ranges<<<nblk(nmc, 256), 256, 0, st>>>(rlo.as<int>(), rhi.as<int>(), nmc, v->ranges.as<float2>());
  k_majorants<<<nblk(nmc, 256), 256, 0, st>>>(d, v->ranges.as<float2>(), v->majorants.as<float>());
  BNX_HIP(hipStreamSynchronize(st));
  BNX_HIP(hipGetLastError());
  return BNX_OK;
}

int volume_rebuild_majorants(Volume *v)
{
  Device *dev = v->dev;
  const size_t nmc = (size_t)v->dd.mc[0] * v->dd.mc[1] * v->dd.mc[2];
  k_majorants<<<nblk((long)nmc, 256), 256, 0, dev->stream>>>(v->dd, v->ranges.as<float2>(),
                                                             v->majorants.as<float>());
  BNX_HIP(hipStreamSynchronize(dev->stream));
  BNX_HIP(hipGetLastError());
  return BNX_OK;
}

} // namespace bnx
