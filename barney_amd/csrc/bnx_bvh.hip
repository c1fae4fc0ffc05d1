// bnx_bvh.hip -- binned-SAH BVH builder on gfx950.
//
// Replaces cuBQL::gpuBuilder as called by rtcore/cuda/Group.cu:232,387,536
// (leaf <= 4 for triangles and user geometry, leaf == 1 for instances).
//
// Split rule (per task = node-to-be over a contiguous slot range):
//   16 bins per axis over the task's centroid bounds, bin index
//   (int)((c - lo) * (16 / extent)) clamped to 15; cost of plane j is
//   area(L_j)*|L_j| + area(R_j)*|R_j| with half-area surface measure; the
//   lowest cost wins (ties: lower axis, lower plane); stable partition.
//   Median split (first half in current order) when no axis has a valid
//   plane or depth >= 48.  Tasks of <= max_leaf prims become leaves.
//
// Structure:
//   phase A -- level-synchronous over the tasks with more than MID prims.
//     Slots are cut into windows of WIN <= MID, so at most two such tasks
//     meet a window (the one that holds its first slot and the one that
//     holds its last): every window reduces its bounds and its SAH bins in
//     registers and LDS and adds them to its tasks' totals with a few hundred
//     global atomics, and the stable partition needs two counts per window.
//     The boxes move with their slots, so every pass reads whole lines.
//   phase B -- one block per task of at most MID prims: boxes in LDS, one
//     wave per node, level by level down to the leaves.
// Min/max reductions and integer counts are exact, so the tree equals the
// CPU specification's tree node for node (numbering aside).
//
// What bounds it: phase B, by the latency of one wave's reductions per node
// (bounds, LDS bins, the sweep over 45 planes by 45 lanes); phase A moves
// about 200 bytes per slot and level.  Measured (MI355X): 33.5M triangles and
// 4M spheres in 68 ms, 1.05M triangles and 50k spheres in 3.9 ms.  Levels
// over all slots down to 32 prims, with bounds and bins gathered by atomics
// per prim and one thread per small task, took 720 and 39 ms: a wave's 64
// atomics on one address take 64 turns, and every level paid for all slots.
#include "bnx_internal.h"

#include <algorithm>
#include <chrono>
#include <cstring>

namespace bnx {
namespace {

constexpr int NB = 16;
constexpr int MAX_SAH_DEPTH = 48;
constexpr int BLOCK = 256;
// tasks of at most MID prims are built by one block: 24 bytes of box per
// prim in LDS, three blocks per CU
constexpr int MID = 1024;
constexpr int WIN = 1024;     // slots per window in phase A
static_assert(WIN <= MID, "a window must meet at most two tasks");

struct Task {
  int begin, end, depth, parent_side;   // parent_side = parent node * 2 + side, or -1
};
struct MidTask {
  int begin, end, depth, parent_side;
  int buf, pad0, pad1, pad2;            // which box buffer holds its slots
};
struct Split {
  int axis, bin, nl, begin;
  float lo, scale;
  int child[2];                         // the next level's task of each side, -1: not in phase A any more
};
// per task: box lo/hi and centroid lo/hi as ordered ints
struct TB {
  int v[12];
};
// per task: [axis][bin][count, lo xyz, hi xyz]
constexpr int BIN_INTS = 7;
constexpr int TASK_BIN_INTS = 3 * NB * BIN_INTS;
const int ORD_INF = 0x7f800000, ORD_NINF = (int)0x807fffff;   // f2o(+inf), f2o(-inf)
constexpr int STAT_NODE = 0, STAT_MID = 1, STAT_BIG = 2, STAT_DEPTH = 3;

__device__ __forceinline__ float cent(const float4 &lo, const float4 &hi, int a)
{
  float l = a == 0 ? lo.x : (a == 1 ? lo.y : lo.z);
  float h = a == 0 ? hi.x : (a == 1 ? hi.y : hi.z);
  return (l + h) * 0.5f;
}
__device__ __forceinline__ int bin_of(float c, float lo, float scale)
{
  int b = (int)((c - lo) * scale);
  return b > NB - 1 ? NB - 1 : b;
}
__device__ __forceinline__ float half_area(float lx, float ly, float lz, float hx, float hy, float hz)
{
  float dx = hx - lx, dy = hy - ly, dz = hz - lz;
  return (dx * dy + dy * dz) + dz * dx;
}

__device__ void write_child(Node *nodes, int parent_side, const float *box, int ref, int cnt)
{
  int node = parent_side >> 1, side = parent_side & 1;
  float *f = (float *)&nodes[node];
  for (int k = 0; k < 6; k++) f[side * 6 + k] = box[k];
  int *ip = (int *)&nodes[node];
  ip[12 + side] = ref;
  ip[14 + side] = cnt;
}

// ------------------------------------------------------- wave reductions
// Data-parallel moves inside a wave: shifts inside rows of 16 lanes, then
// the row totals passed on; lanes without a source take `id`.
template <int CTRL, int ROWS> __device__ __forceinline__ int dpp(int id, int x)
{
  return __builtin_amdgcn_update_dpp(id, x, CTRL, ROWS, 0xf, false);
}
constexpr int ROW_SHL = 0x100, ROW_SHR = 0x110, ROW_BCAST15 = 0x142, ROW_BCAST31 = 0x143;

template <typename Op> __device__ __forceinline__ int wave_reduce(int x, int id, Op op)
{
  x = op(x, dpp<ROW_SHR + 1, 0xf>(id, x));
  x = op(x, dpp<ROW_SHR + 2, 0xf>(id, x));
  x = op(x, dpp<ROW_SHR + 4, 0xf>(id, x));
  x = op(x, dpp<ROW_SHR + 8, 0xf>(id, x));
  x = op(x, dpp<ROW_BCAST15, 0xa>(id, x));
  x = op(x, dpp<ROW_BCAST31, 0xc>(id, x));
  return __builtin_amdgcn_readlane(x, 63);
}
__device__ __forceinline__ int wave_min(int x)
{
  return wave_reduce(x, 0x7fffffff, [](int a, int b) { return min(a, b); });
}
__device__ __forceinline__ int wave_max(int x)
{
  return wave_reduce(x, (int)0x80000000, [](int a, int b) { return max(a, b); });
}

// inclusive scans over the 16 lanes of a row, from its first lane (FWD) or
// from its last
template <bool FWD, typename Op> __device__ __forceinline__ int row_scan(int x, int id, Op op)
{
  constexpr int S = FWD ? ROW_SHR : ROW_SHL;
  x = op(x, dpp<S + 1, 0xf>(id, x));
  x = op(x, dpp<S + 2, 0xf>(id, x));
  x = op(x, dpp<S + 4, 0xf>(id, x));
  x = op(x, dpp<S + 8, 0xf>(id, x));
  return x;
}

// LDS written by this wave is read back by this wave: keep the order
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// The SAH sweep over a task's bins by one wave: lane axis * 16 + plane holds
// bin `plane` and gets the boxes and counts left and right of the plane from
// row scans.  Identical values to the CPU specification's sequential sweep
// (unions are exact); lowest cost, ties to the lower axis and plane.
struct Pick {
  int axis, bin, nl;
};
__device__ Pick wave_sah(const int *bins, const int *cb, bool sah)
{
  const int lane = lane_id();
  const int a = min(lane >> 4, 2), j = lane & 15;
  const int *q = bins + (a * NB + j) * BIN_INTS;
  int cnt = q[0], lo[3] = {q[1], q[2], q[3]}, hi[3] = {q[4], q[5], q[6]};
  const int clo = a == 0 ? cb[0] : (a == 1 ? cb[1] : cb[2]);
  const int chi = a == 0 ? cb[3] : (a == 1 ? cb[4] : cb[5]);
  const float ext = o2f(chi) - o2f(clo);
  auto mn = [](int x, int y) { return min(x, y); };
  auto mx = [](int x, int y) { return max(x, y); };
  auto ad = [](int x, int y) { return x + y; };
  float area[2];
  int num[2];
  for (int side = 0; side < 2; side++) {
    int l[3], h[3], c;
    for (int k = 0; k < 3; k++) {
      l[k] = side == 0 ? row_scan<true>(lo[k], ORD_INF, mn) : row_scan<false>(lo[k], ORD_INF, mn);
      h[k] = side == 0 ? row_scan<true>(hi[k], ORD_NINF, mx) : row_scan<false>(hi[k], ORD_NINF, mx);
    }
    c = side == 0 ? row_scan<true>(cnt, 0, ad) : row_scan<false>(cnt, 0, ad);
    if (side == 1) {
      // right of plane j: the bins from j + 1 on
      for (int k = 0; k < 3; k++) {
        l[k] = dpp<ROW_SHL + 1, 0xf>(ORD_INF, l[k]);
        h[k] = dpp<ROW_SHL + 1, 0xf>(ORD_NINF, h[k]);
      }
      c = dpp<ROW_SHL + 1, 0xf>(0, c);
    }
    num[side] = c;
    area[side] = half_area(o2f(l[0]), o2f(l[1]), o2f(l[2]), o2f(h[0]), o2f(h[1]), o2f(h[2]));
  }
  const bool ok = sah && lane < 48 && j < NB - 1 && ext >= 1e-30f && num[0] > 0 && num[1] > 0;
  float cost = area[0] * (float)num[0] + area[1] * (float)num[1];
  if (!ok || !(cost < INFINITY)) cost = INFINITY;
  const int key = f2o(cost);
  const int best = wave_min(key);
  Pick p{-1, -1, 0};
  if (best < ORD_INF) {
    const int w = __ffsll((unsigned long long)__ballot(key == best)) - 1;
    p.axis = w >> 4;
    p.bin = w & 15;
    p.nl = __builtin_amdgcn_readlane(num[0], w);
  }
  return p;
}

// one prim into a task's LDS bins; a wave whose lanes all meet one bin
// reduces first (a run of slots along a mesh row does, and 64 atomics on one
// address take 64 turns)
__device__ __forceinline__ void bin_add(int *bins, int a, int k, bool on, const int *lv, const int *hv)
{
  const uint64_t m = __ballot(on);
  if (m == 0) return;
  const int k0 = __builtin_amdgcn_readlane(k, __ffsll((unsigned long long)m) - 1);
  if (__popcll(m) > 8 && __ballot(on && k != k0) == 0) {
    int l[3], h[3];
    for (int q = 0; q < 3; q++) {
      l[q] = wave_min(on ? lv[q] : 0x7fffffff);
      h[q] = wave_max(on ? hv[q] : (int)0x80000000);
    }
    if (lane_id() == 0) {
      int *dst = bins + (a * NB + k0) * BIN_INTS;
      atomicAdd(&dst[0], __popcll(m));
      for (int q = 0; q < 3; q++) {
        atomicMin(&dst[1 + q], l[q]);
        atomicMax(&dst[4 + q], h[q]);
      }
    }
  } else if (on) {
    int *dst = bins + (a * NB + k) * BIN_INTS;
    atomicAdd(&dst[0], 1);
    for (int q = 0; q < 3; q++) {
      atomicMin(&dst[1 + q], lv[q]);
      atomicMax(&dst[4 + q], hv[q]);
    }
  }
}

__device__ __forceinline__ int bin_init(int i)
{
  const int w = i % BIN_INTS;
  return w == 0 ? 0 : (w < 4 ? ORD_INF : ORD_NINF);
}
__device__ __forceinline__ int tb_init(int i) { return (i % 6) < 3 ? ORD_INF : ORD_NINF; }

// ------------------------------------------------------------ phase A
// the root task; every slot belongs to it
__global__ void k_start(int n, int *slot_task, Task *tasks, int *task_node, TB *tb, int *bins, int *counters)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) slot_task[i] = 0;
  if (blockIdx.x == 0) {
    for (int k = threadIdx.x; k < TASK_BIN_INTS; k += blockDim.x) bins[k] = bin_init(k);
    if (threadIdx.x < 12) tb[0].v[threadIdx.x] = tb_init(threadIdx.x);
    if (threadIdx.x < 8) counters[threadIdx.x] = threadIdx.x == STAT_NODE ? 1 : 0;
    if (threadIdx.x == 0) {
      tasks[0] = Task{0, n, 0, -1};
      task_node[0] = 0;
    }
  }
}

// the (at most two) tasks of this block's window
__device__ __forceinline__ void window_tasks(int n, const int *slot_task, int &b, int &e, int *t)
{
  b = blockIdx.x * WIN;
  e = min(n, b + WIN);
  t[0] = slot_task[b];
  const int last = slot_task[e - 1];
  t[1] = last != t[0] ? last : -1;
}

__global__ __launch_bounds__(BLOCK) void k_bounds(int n, const int *slot_task, const float4 *lo, const float4 *hi,
                                                  TB *tb)
{
  __shared__ int s[2][12];
  int b, e, t[2];
  window_tasks(n, slot_task, b, e, t);
  if (t[0] < 0 && t[1] < 0) return;
  if (threadIdx.x < 24) s[threadIdx.x / 12][threadIdx.x % 12] = tb_init(threadIdx.x % 12);
  __syncthreads();
  for (int w = 0; w < 2; w++) {
    if (t[w] < 0) continue;
    int v[12];
    for (int k = 0; k < 12; k++) v[k] = tb_init(k);
    for (int i = b + threadIdx.x; i < e; i += BLOCK) {
      if (slot_task[i] != t[w]) continue;
      const float4 l = lo[i], h = hi[i];
      const float lv[3] = {l.x, l.y, l.z}, hv[3] = {h.x, h.y, h.z};
      for (int k = 0; k < 3; k++) {
        const int c = f2o((lv[k] + hv[k]) * 0.5f);
        v[k] = min(v[k], f2o(lv[k]));
        v[3 + k] = max(v[3 + k], f2o(hv[k]));
        v[6 + k] = min(v[6 + k], c);
        v[9 + k] = max(v[9 + k], c);
      }
    }
    for (int k = 0; k < 12; k++) v[k] = (k % 6) < 3 ? wave_min(v[k]) : wave_max(v[k]);
    if (lane_id() == 0)
      for (int k = 0; k < 12; k++) {
        if ((k % 6) < 3) atomicMin(&s[w][k], v[k]);
        else atomicMax(&s[w][k], v[k]);
      }
  }
  __syncthreads();
  if (threadIdx.x < 24) {
    const int w = threadIdx.x / 12, k = threadIdx.x % 12;
    if (t[w] >= 0) {
      if ((k % 6) < 3) atomicMin(&tb[t[w]].v[k], s[w][k]);
      else atomicMax(&tb[t[w]].v[k], s[w][k]);
    }
  }
}

__global__ __launch_bounds__(BLOCK) void k_bin(int n, const int *slot_task, const float4 *lo, const float4 *hi,
                                               const TB *tb, int *bins)
{
  __shared__ int s[2][TASK_BIN_INTS];
  int b, e, t[2];
  window_tasks(n, slot_task, b, e, t);
  if (t[0] < 0 && t[1] < 0) return;
  for (int i = threadIdx.x; i < 2 * TASK_BIN_INTS; i += BLOCK) s[i / TASK_BIN_INTS][i % TASK_BIN_INTS] = bin_init(i % TASK_BIN_INTS);
  __syncthreads();
  for (int w = 0; w < 2; w++) {
    if (t[w] < 0) continue;
    float clo[3], scale[3];
    for (int a = 0; a < 3; a++) {
      clo[a] = o2f(tb[t[w]].v[6 + a]);
      const float ext = o2f(tb[t[w]].v[9 + a]) - clo[a];
      scale[a] = (ext >= 1e-30f) ? (float)NB / ext : -1.f;
    }
    for (int base = b; base < e; base += BLOCK) {
      const int i = base + threadIdx.x;
      const bool on = i < e && slot_task[i] == t[w];
      float4 l = make_float4(0.f, 0.f, 0.f, 0.f), h = l;
      if (on) {
        l = lo[i];
        h = hi[i];
      }
      const int lv[3] = {f2o(l.x), f2o(l.y), f2o(l.z)}, hv[3] = {f2o(h.x), f2o(h.y), f2o(h.z)};
      for (int a = 0; a < 3; a++)
        if (scale[a] >= 0.f) bin_add(s[w], a, bin_of(cent(l, h, a), clo[a], scale[a]), on, lv, hv);
    }
  }
  __syncthreads();
  for (int w = 0; w < 2; w++) {
    if (t[w] < 0) continue;
    int *g = bins + (size_t)t[w] * TASK_BIN_INTS;
    for (int i = threadIdx.x; i < 3 * NB; i += BLOCK) {
      const int *q = s[w] + i * BIN_INTS;
      if (q[0] == 0) continue;
      atomicAdd(&g[i * BIN_INTS], q[0]);
      for (int k = 0; k < 3; k++) {
        atomicMin(&g[i * BIN_INTS + 1 + k], q[1 + k]);
        atomicMax(&g[i * BIN_INTS + 4 + k], q[4 + k]);
      }
    }
  }
}

// one wave per task: its own box into its parent, the plane, and the two
// children: the next level's tasks (bounds and bins reset here) or phase B's
__global__ __launch_bounds__(BLOCK) void k_split(int num_big, const Task *tasks, const int *task_node, const TB *tb,
                                                 const int *bins, Node *nodes, Split *split, Task *next,
                                                 int *next_node, TB *next_tb, int *next_bins, MidTask *mid,
                                                 int *counters, int next_buf)
{
  const int t = blockIdx.x * (BLOCK / 64) + (int)(threadIdx.x >> 6);
  if (t >= num_big) return;
  const int lane = lane_id();
  const Task tk = tasks[t];
  const int cnt = tk.end - tk.begin, node = task_node[t];
  const Pick p = wave_sah(bins + (size_t)t * TASK_BIN_INTS, tb[t].v + 6, tk.depth < MAX_SAH_DEPTH);
  const int nl = p.axis < 0 ? cnt / 2 : p.nl;
  Split sp{p.axis, p.bin, nl, tk.begin, 0.f, 0.f, {-1, -1}};
  if (p.axis >= 0) {
    sp.lo = o2f(tb[t].v[6 + p.axis]);
    sp.scale = (float)NB / (o2f(tb[t].v[9 + p.axis]) - sp.lo);
  }
  for (int side = 0; side < 2; side++) {
    const int b = side == 0 ? tk.begin : tk.begin + nl, e = side == 0 ? tk.begin + nl : tk.end;
    int c = -1;
    if (e - b > MID) {
      if (lane == 0) {
        c = atomicAdd(&counters[STAT_BIG], 1);
        next[c] = Task{b, e, tk.depth + 1, node * 2 + side};
        next_node[c] = atomicAdd(&counters[STAT_NODE], 1);
      }
      c = __builtin_amdgcn_readfirstlane(c);
      if (lane < 12) next_tb[c].v[lane] = tb_init(lane);
      for (int k = lane; k < TASK_BIN_INTS; k += 64) next_bins[(size_t)c * TASK_BIN_INTS + k] = bin_init(k);
    } else if (lane == 0) {
      mid[atomicAdd(&counters[STAT_MID], 1)] = MidTask{b, e, tk.depth + 1, node * 2 + side, next_buf, 0, 0, 0};
    }
    sp.child[side] = c;
  }
  if (lane == 0) {
    split[t] = sp;
    if (tk.parent_side >= 0) {
      float box[6];
      for (int k = 0; k < 6; k++) box[k] = o2f(tb[t].v[k]);
      write_child(nodes, tk.parent_side, box, node, 0);
    }
  }
}

__device__ __forceinline__ bool goes_left(const Split &sp, int i, const float4 &l, const float4 &h)
{
  if (sp.axis < 0) return i - sp.begin < sp.nl;
  return bin_of(cent(l, h, sp.axis), sp.lo, sp.scale) <= sp.bin;
}

// left slots of both tasks of every window
__global__ __launch_bounds__(BLOCK) void k_count(int n, const int *slot_task, const Split *split, const float4 *lo,
                                                 const float4 *hi, int *win)
{
  __shared__ int s[2];
  int b, e, t[2];
  window_tasks(n, slot_task, b, e, t);
  if (threadIdx.x < 2) s[threadIdx.x] = 0;
  __syncthreads();
  if (t[0] >= 0 || t[1] >= 0) {
    int c[2] = {0, 0};
    for (int i = b + threadIdx.x; i < e; i += BLOCK) {
      const int k = slot_task[i];
      if (k < 0) continue;
      const int f = goes_left(split[k], i, lo[i], hi[i]) ? 1 : 0;
      c[0] += k == t[0] ? f : 0;
      c[1] += k == t[0] ? 0 : f;
    }
    for (int w = 0; w < 2; w++)
      if (c[w]) atomicAdd(&s[w], c[w]);
  }
  __syncthreads();
  if (threadIdx.x < 2) win[2 * blockIdx.x + threadIdx.x] = s[threadIdx.x];
}

// exclusive prefix sums of the window counts, in slot order; one block
__global__ __launch_bounds__(1024) void k_scan_windows(int m, int *win)
{
  __shared__ int wsum[16];
  const int tid = (int)threadIdx.x, lane = tid & 63, w = tid >> 6;
  int carry = 0;
  for (int base = 0; base < m; base += 1024) {
    const int i = base + tid;
    const int v = i < m ? win[i] : 0;
    int x = v;
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int off = 0, tot = 0;
    for (int k = 0; k < 16; k++) {
      off += k < w ? wsum[k] : 0;
      tot += wsum[k];
    }
    __syncthreads();
    if (i < m) win[i] = carry + off + x - v;
    carry += tot;
  }
}

// stable partition: boxes and task of every slot to its place at the next
// level.  A task's slots before a window are the prefix sum there less the
// prefix sum where the task begins: the window's first entry when it begins
// with the window, else its second.
__global__ __launch_bounds__(BLOCK) void k_scatter(int n, const int *slot_task, const Split *split, const int *win,
                                                   const float4 *lo, const float4 *hi, float4 *lo_out, float4 *hi_out,
                                                   int *task_out)
{
  __shared__ int wl[BLOCK / 64][2];
  int b, e, t[2];
  window_tasks(n, slot_task, b, e, t);
  if (t[0] < 0 && t[1] < 0) {
    for (int i = b + threadIdx.x; i < e; i += BLOCK) task_out[i] = -1;
    return;
  }
  int run[2] = {0, 0};         // left slots of each task before this window's current row
  Split sp[2];
  for (int w = 0; w < 2; w++)
    if (t[w] >= 0) {
      sp[w] = split[t[w]];
      const int wb = sp[w].begin / WIN;
      run[w] = win[2 * blockIdx.x + w] - win[2 * wb + (sp[w].begin == wb * WIN ? 0 : 1)];
    }
  const int wave = threadIdx.x >> 6;
  for (int base = b; base < e; base += BLOCK) {
    const int i = base + threadIdx.x;
    const int k = i < e ? slot_task[i] : -1;
    const int w = k == t[0] ? 0 : 1;
    bool left = false;
    float4 l, h;
    if (k >= 0) {
      l = lo[i];
      h = hi[i];
      left = goes_left(sp[w], i, l, h);
    }
    const uint64_t m0 = __ballot(left && w == 0), m1 = __ballot(left && w == 1);
    if (lane_id() == 0) {
      wl[wave][0] = __popcll(m0);
      wl[wave][1] = __popcll(m1);
    }
    __syncthreads();
    int before[2] = {run[0], run[1]};
    for (int q = 0; q < BLOCK / 64; q++)
      for (int c = 0; c < 2; c++) {
        before[c] += q < wave ? wl[q][c] : 0;
        run[c] += wl[q][c];
      }
    __syncthreads();
    if (i < e && k < 0) task_out[i] = -1;
    if (k >= 0) {
      const int rank = before[w] + __popcll((w == 0 ? m0 : m1) & lanemask_lt());
      const int pos = left ? sp[w].begin + rank : sp[w].begin + sp[w].nl + ((i - sp[w].begin) - rank);
      lo_out[pos] = l;
      hi_out[pos] = h;
      task_out[pos] = sp[w].child[left ? 0 : 1];
    }
  }
}

// ------------------------------------------------------------ phase B
// One block builds the subtree of a task of at most MID prims: boxes in LDS
// (by local index), the slots' order as 16-bit local indices in two arrays
// used in turn, the level's nodes in a list.  Each wave takes nodes from the
// list: bounds, bins (its own 1.3 KB of LDS), sweep, stable partition by
// ballots; children of at most max_leaf prims become leaves at once.
__global__ __launch_bounds__(BLOCK) void k_mid(const MidTask *tasks, const float4 *lo0, const float4 *hi0,
                                               const float4 *lo1, const float4 *hi1, Node *nodes, int *order,
                                               int *counters, int max_leaf, TB *root_tb, int whole_n)
{
  __shared__ float bx[6][MID];
  __shared__ int prim[MID];
  __shared__ unsigned short perm[2][MID];
  __shared__ int2 list[2][MID / 2];          // begin | end << 16, parent_side
  __shared__ int num[2], base_node, deepest;
  __shared__ int wbins[BLOCK / 64][TASK_BIN_INTS];
  // whole_n >= 0: the whole build is this one task
  const MidTask mt = whole_n >= 0 ? MidTask{0, whole_n, 0, -1, 0, 0, 0, 0} : tasks[blockIdx.x];
  const int n = mt.end - mt.begin;
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  int *bins = wbins[wave];
  const float4 *lo = (mt.buf ? lo1 : lo0) + mt.begin, *hi = (mt.buf ? hi1 : hi0) + mt.begin;
  for (int i = threadIdx.x; i < n; i += BLOCK) {
    const float4 l = lo[i], h = hi[i];
    bx[0][i] = l.x; bx[1][i] = l.y; bx[2][i] = l.z;
    bx[3][i] = h.x; bx[4][i] = h.y; bx[5][i] = h.z;
    prim[i] = __float_as_int(l.w);
    perm[0][i] = (unsigned short)i;
  }
  if (threadIdx.x == 0) {
    list[0][0] = make_int2(n << 16, mt.parent_side);
    num[0] = 1;
    num[1] = 0;
    deepest = 0;
    if (whole_n >= 0) {
      for (int k = 0; k < 8; k++) counters[k] = k == STAT_NODE ? 1 : 0;
    }
  }
  __syncthreads();
  // box of local slots [b, e) of src, as ordered ints, in every lane
  auto bounds = [&](const unsigned short *src, int b, int e, int *v, bool centroids) {
    for (int k = 0; k < 12; k++) v[k] = tb_init(k);
    for (int i = b + lane; i < e; i += 64) {
      const int p = src[i];
      for (int k = 0; k < 3; k++) {
        const float l = bx[k][p], h = bx[3 + k][p];
        v[k] = min(v[k], f2o(l));
        v[3 + k] = max(v[3 + k], f2o(h));
        const int c = f2o((l + h) * 0.5f);
        v[6 + k] = min(v[6 + k], c);
        v[9 + k] = max(v[9 + k], c);
      }
    }
    for (int k = 0; k < (centroids ? 12 : 6); k++) v[k] = (k % 6) < 3 ? wave_min(v[k]) : wave_max(v[k]);
  };
  auto leaf = [&](const unsigned short *src, int b, int e, int parent_side) {
    int v[12];
    bounds(src, b, e, v, false);
    if (lane < e - b) order[mt.begin + b + lane] = prim[src[b + lane]];
    if (lane == 0) {
      float box[6];
      for (int k = 0; k < 6; k++) box[k] = o2f(v[k]);
      write_child(nodes, parent_side, box, mt.begin + b, e - b);
    }
  };
  if (whole_n >= 0 && wave == 0) {
    int v[12];
    bounds(perm[0], 0, n, v, true);
    if (lane < 12) {
      int x = v[0];
      for (int k = 1; k < 12; k++) x = lane == k ? v[k] : x;
      root_tb->v[lane] = x;
    }
  }
  if (n <= max_leaf) {
    if (wave == 0) {
      if (mt.parent_side >= 0) {
        leaf(perm[0], 0, n, mt.parent_side);
      } else {
        // the whole tree is one leaf (or empty): a root with one child
        const float empty[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (n > 0) leaf(perm[0], 0, n, 0);
        else if (lane == 0) write_child(nodes, 0, empty, 0, -1);
        if (lane == 0) write_child(nodes, 1, empty, 0, -1);
      }
      if (lane == 0) atomicMax(&counters[STAT_DEPTH], mt.parent_side >= 0 ? mt.depth : (n > 0 ? 1 : 0));
    }
    return;
  }
  // each level halves nothing in the worst case but always splits off at
  // least one prim per node, so at most n levels run
  int cur = 0;
  for (int level = 0; level < MID; level++) {
    const int nt = num[cur];
    if (nt == 0) break;
    const int depth = mt.depth + level;
    const unsigned short *src = perm[level & 1];
    unsigned short *dst = perm[(level & 1) ^ 1];
    if (threadIdx.x == 0)
      base_node = list[cur][0].y < 0 ? 0 : atomicAdd(&counters[STAT_NODE], nt);
    __syncthreads();
    for (int t = wave; t < nt; t += BLOCK / 64) {
      const int2 tk = list[cur][t];
      const int b = tk.x & 0xffff, e = tk.x >> 16, m = e - b, node = base_node + t;
      int v[12];
      bounds(src, b, e, v, true);
      if (lane == 0 && tk.y >= 0) {
        float box[6];
        for (int k = 0; k < 6; k++) box[k] = o2f(v[k]);
        write_child(nodes, tk.y, box, node, 0);
      }
      Pick p{-1, -1, 0};
      float clo[3], scale[3];
      if (depth < MAX_SAH_DEPTH) {
        for (int k = lane; k < TASK_BIN_INTS; k += 64) bins[k] = bin_init(k);
        wave_sync();
        for (int a = 0; a < 3; a++) {
          clo[a] = o2f(v[6 + a]);
          const float ext = o2f(v[9 + a]) - clo[a];
          scale[a] = (ext >= 1e-30f) ? (float)NB / ext : -1.f;
        }
        for (int i0 = b; i0 < e; i0 += 64) {
          const bool on = i0 + lane < e;
          const int q = on ? src[i0 + lane] : 0;
          float l[3], h[3];
          int lv[3], hv[3];
          for (int k = 0; k < 3; k++) {
            l[k] = bx[k][q];
            h[k] = bx[3 + k][q];
            lv[k] = f2o(l[k]);
            hv[k] = f2o(h[k]);
          }
          for (int a = 0; a < 3; a++)
            if (scale[a] >= 0.f) bin_add(bins, a, bin_of((l[a] + h[a]) * 0.5f, clo[a], scale[a]), on, lv, hv);
        }
        wave_sync();
        p = wave_sah(bins, v + 6, true);
      }
      const int nl = p.axis < 0 ? m / 2 : p.nl;
      int left = 0;
      for (int i0 = b; i0 < e; i0 += 64) {
        const int i = i0 + lane;
        const bool on = i < e;
        const int q = on ? src[i] : 0;
        bool f;
        if (p.axis < 0) {
          f = i - b < nl;
        } else {
          const float l = p.axis == 0 ? bx[0][q] : (p.axis == 1 ? bx[1][q] : bx[2][q]);
          const float h = p.axis == 0 ? bx[3][q] : (p.axis == 1 ? bx[4][q] : bx[5][q]);
          const float lo_a = p.axis == 0 ? clo[0] : (p.axis == 1 ? clo[1] : clo[2]);
          const float sc = p.axis == 0 ? scale[0] : (p.axis == 1 ? scale[1] : scale[2]);
          f = bin_of((l + h) * 0.5f, lo_a, sc) <= p.bin;
        }
        const uint64_t ml = __ballot(on && f);
        const int rank = left + __popcll(ml & lanemask_lt());
        if (on) dst[f ? b + rank : b + nl + (i - b - rank)] = (unsigned short)q;
        left += __popcll(ml);
      }
      wave_sync();
      for (int side = 0; side < 2; side++) {
        const int cb = side == 0 ? b : b + nl, ce = side == 0 ? b + nl : e;
        if (ce - cb <= max_leaf) {
          leaf(dst, cb, ce, node * 2 + side);
          if (lane == 0) atomicMax(&deepest, depth + 1);
        } else if (lane == 0) {
          list[cur ^ 1][atomicAdd(&num[cur ^ 1], 1)] = make_int2(cb | (ce << 16), node * 2 + side);
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) num[cur] = 0;
    cur ^= 1;
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMax(&counters[STAT_DEPTH], deepest);
}

inline int nblocks(long n, int bs) { return (int)((n + bs - 1) / bs); }

// ------------------------------------------------------- 4-wide collapse
// One thread per 4-wide node of the current level: start from the two
// children of its binary node, then repeatedly replace the inner child of
// largest half area by its two children, in place, until there are four
// children or only leaves.  The nodes of a level are numbered together after
// those of the levels above (cnt[level] counts them), and work[j] holds node
// j's binary node and need, the stack entries pushed on the way down to it;
// max_need collects the largest need at a leaf.  Every level is launched
// without a look at the one before: the host knows only that there are at
// most as many as the binary tree is deep.
constexpr int MAX_LEVELS = 128;
struct Cand {
  float lo[3], hi[3];
  int ref, cnt;
};

__device__ Cand cand_of(const Node &nd, int k)
{
  Cand c;
  if (k == 0) {
    c.lo[0] = nd.lo0x; c.lo[1] = nd.lo0y; c.lo[2] = nd.lo0z;
    c.hi[0] = nd.hi0x; c.hi[1] = nd.hi0y; c.hi[2] = nd.hi0z;
    c.ref = nd.ref0; c.cnt = nd.cnt0;
  } else {
    c.lo[0] = nd.lo1x; c.lo[1] = nd.lo1y; c.lo[2] = nd.lo1z;
    c.hi[0] = nd.hi1x; c.hi[1] = nd.hi1y; c.hi[2] = nd.hi1z;
    c.ref = nd.ref1; c.cnt = nd.cnt1;
  }
  return c;
}

__device__ float cand_area(const Cand &c)
{
  float dx = c.hi[0] - c.lo[0], dy = c.hi[1] - c.lo[1], dz = c.hi[2] - c.lo[2];
  return (dx * dy + dy * dz) + dz * dx;
}

__global__ __launch_bounds__(128) void k_collapse4(const Node *bin, int2 *work, int *cnt, int *max_need, int level,
                                                   Node4 *out, int cap4)
{
  int first = 0;
  for (int l = 0; l < level; l++) first += cnt[l];
  const int nwork = min(cnt[level], cap4 - first), next = first + cnt[level];
  int deepest = 0;
  for (int i0 = blockIdx.x * 128; i0 < nwork; i0 += gridDim.x * 128) {
    const int i = i0 + (int)threadIdx.x;
    const bool on = i < nwork;
    const int j = first + (on ? i : 0);
    const int b = work[j].x, need = work[j].y;
    Cand c[4];
    int m = 0;
    const Node root = bin[b];
    for (int k = 0; k < 2; k++) {
      Cand x = cand_of(root, k);
      if (x.cnt >= 0) c[m++] = x;
    }
    for (int round = 0; round < 3 && m < 4; round++) {
      int best = -1;
      float area = -1.f;
      for (int k = 0; k < m; k++)
        if (c[k].cnt == 0 && cand_area(c[k]) > area) {
          area = cand_area(c[k]);
          best = k;
        }
      if (best < 0) break;
      const Node nd = bin[c[best].ref];
      Cand a = cand_of(nd, 0), d = cand_of(nd, 1);
      if (a.cnt >= 0 && d.cnt >= 0) {
        // keep the binary tree's left-to-right order: a depth-first walk of
        // the 4-wide node in slot order meets the leaves in the same order
        for (int k = m; k > best + 1; k--) c[k] = c[k - 1];
        c[best] = a;
        c[best + 1] = d;
        m++;
      } else if (a.cnt >= 0 || d.cnt >= 0) {
        c[best] = a.cnt >= 0 ? a : d;
      } else {
        for (int k = best; k + 1 < m; k++) c[k] = c[k + 1];
        m--;
      }
    }
    // numbers for the inner children: one atomic per wave
    int inner = 0;
    for (int k = 0; k < m; k++) inner += on && c[k].cnt == 0 ? 1 : 0;
    int scan = inner;
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(scan, d, 64);
      if (lane_id() >= d) scan += y;
    }
    int idx = 0;
    if (lane_id() == 63 && scan > 0) idx = atomicAdd(cnt + level + 1, scan);
    idx = next + __builtin_amdgcn_readlane(idx, 63) + scan - inner;
    float lo[3][4], hi[3][4];
    uint32_t code[4];
    const int child_need = need + (m > 0 ? m - 1 : 0);
    for (int k = 0; k < 4; k++) {
      if (k < m) {
        for (int a = 0; a < 3; a++) {
          lo[a][k] = c[k].lo[a];
          hi[a][k] = c[k].hi[a];
        }
        if (c[k].cnt > 0) {
          code[k] = enc_child(c[k].ref, c[k].cnt);
          deepest = max(deepest, child_need);
        } else {
          if (on && idx < cap4) work[idx] = make_int2(c[k].ref, child_need);
          code[k] = (uint32_t)idx;
          idx++;
        }
      } else {
        for (int a = 0; a < 3; a++) {
          lo[a][k] = INFINITY;
          hi[a][k] = -INFINITY;
        }
        code[k] = EMPTY4;
      }
    }
    if (!on) continue;
    Node4 n4;
    n4.lox = make_float4(lo[0][0], lo[0][1], lo[0][2], lo[0][3]);
    n4.hix = make_float4(hi[0][0], hi[0][1], hi[0][2], hi[0][3]);
    n4.loy = make_float4(lo[1][0], lo[1][1], lo[1][2], lo[1][3]);
    n4.hiy = make_float4(hi[1][0], hi[1][1], hi[1][2], hi[1][3]);
    n4.loz = make_float4(lo[2][0], lo[2][1], lo[2][2], lo[2][3]);
    n4.hiz = make_float4(hi[2][0], hi[2][1], hi[2][2], hi[2][3]);
    n4.child = make_uint4(code[0], code[1], code[2], code[3]);
    n4.pad = make_uint4(0, 0, 0, 0);
    out[j] = n4;
  }
  deepest = wave_max(deepest);
  if (lane_id() == 0 && deepest > 0) atomicMax(max_need, deepest);
}

__global__ void k_collapse_start(int2 *work, int *cnt)
{
  for (int k = threadIdx.x; k < MAX_LEVELS + 2; k += blockDim.x) cnt[k] = k == 0 ? 1 : 0;
  if (threadIdx.x == 0) work[0] = make_int2(0, 0);
}

} // namespace

int collapse_bvh4(Device *dev, Bvh &bvh)
{
  hipStream_t st = dev->stream;
  BuildScratch &S = dev->build;
  // every 4-wide node but the root stands for a distinct inner binary node
  const int cap4 = bvh.num_nodes > 0 ? bvh.num_nodes : 1;
  const int levels = std::max(1, bvh.max_depth);
  BNX_CHECK(levels < MAX_LEVELS, BNX_ERR_STATE, "bvh collapse: too many levels");
  BNX_HIP(bvh.nodes4.ensure(sizeof(Node4) * (size_t)cap4));
  BNX_HIP(S.collapse.ensure(sizeof(int2) * (size_t)cap4));
  BNX_HIP(S.levels.ensure(sizeof(int) * (MAX_LEVELS + 2)));
  int *cnt = S.levels.as<int>(), *max_need = cnt + MAX_LEVELS + 1;
  k_collapse_start<<<1, 64, 0, st>>>(S.collapse.as<int2>(), cnt);
  for (int level = 0; level < levels; level++) {
    // a level holds at most four times the nodes of the one above
    const long long bound = level < 10 ? 1LL << (2 * level) : cap4;
    const int grid = nblocks((long)std::min<long long>(bound, cap4), 128);
    k_collapse4<<<std::min(grid, 8 * dev->num_cus), 128, 0, st>>>(bvh.nodes.as<Node>(), S.collapse.as<int2>(), cnt,
                                                                  max_need, level, bvh.nodes4.as<Node4>(), cap4);
  }
  int h[MAX_LEVELS + 2];
  BNX_HIP(hipMemcpyAsync(h, cnt, sizeof(h), hipMemcpyDeviceToHost, st));
  BNX_HIP(hipStreamSynchronize(st));
  BNX_HIP(hipGetLastError());
  long long total = 0;
  for (int l = 0; l <= MAX_LEVELS; l++) total += h[l];
  BNX_CHECK(total <= cap4 && h[levels] == 0, BNX_ERR_STATE, "bvh collapse: node overflow");
  bvh.num_nodes4 = (int)total;
  bvh.stack_need4 = h[MAX_LEVELS + 1];
  return BNX_OK;
}

int build_bvh(Device *dev, float4 *d_lo, float4 *d_hi, int n, int max_leaf, Bvh &out)
{
  auto t0 = std::chrono::steady_clock::now();
  hipStream_t st = dev->stream;
  BuildScratch &S = dev->build;
  const int ncap = n > 0 ? n : 1;
  BNX_HIP(out.nodes.ensure(sizeof(Node) * (size_t)ncap));
  BNX_HIP(out.order.ensure(sizeof(int) * (size_t)ncap));
  BNX_HIP(S.counters.ensure(sizeof(int) * 8 + sizeof(TB)));
  int *counters = S.counters.as<int>();
  TB *root_tb = (TB *)(counters + 8);
  Node *nodes = out.nodes.as<Node>();
  int *order = out.order.as<int>();
  struct {
    int ctr[8];
    TB tb;
  } host{};
  if (n <= MID) {
    k_mid<<<1, BLOCK, 0, st>>>(nullptr, d_lo, d_hi, d_lo, d_hi, nodes, order, counters, max_leaf, root_tb, n);
  } else {
    // at most n / MID tasks a level, each split into two; phase B gets one
    // task more than phase A has splits, over at most MAX_SAH_DEPTH levels of
    // SAH planes and then halves
    const int big = n / MID + 1;
    const long long mids = std::min<long long>(n, (MAX_SAH_DEPTH + 33LL) * big + 1);
    const int windows = nblocks(n, WIN);
    BNX_HIP(S.lo.ensure(sizeof(float4) * (size_t)n));
    BNX_HIP(S.hi.ensure(sizeof(float4) * (size_t)n));
    BNX_HIP(S.slot_task.ensure(2 * sizeof(int) * (size_t)n));
    BNX_HIP(S.windows.ensure(2 * sizeof(int) * (size_t)windows));
    BNX_HIP(S.tasks.ensure(2 * sizeof(Task) * (size_t)big));
    BNX_HIP(S.task_node.ensure(2 * sizeof(int) * (size_t)big));
    BNX_HIP(S.bounds.ensure(2 * sizeof(TB) * (size_t)big));
    BNX_HIP(S.bins.ensure(2 * sizeof(int) * TASK_BIN_INTS * (size_t)big));
    BNX_HIP(S.split.ensure(sizeof(Split) * (size_t)big));
    BNX_HIP(S.mid_tasks.ensure(sizeof(MidTask) * (size_t)mids));
    float4 *lo[2] = {d_lo, S.lo.as<float4>()}, *hi[2] = {d_hi, S.hi.as<float4>()};
    int *slot_task[2] = {S.slot_task.as<int>(), S.slot_task.as<int>() + n};
    Task *tasks[2] = {S.tasks.as<Task>(), S.tasks.as<Task>() + big};
    int *task_node[2] = {S.task_node.as<int>(), S.task_node.as<int>() + big};
    TB *tb[2] = {S.bounds.as<TB>(), S.bounds.as<TB>() + big};
    int *bins[2] = {S.bins.as<int>(), S.bins.as<int>() + (size_t)TASK_BIN_INTS * big};
    int *win = S.windows.as<int>();
    MidTask *mid = S.mid_tasks.as<MidTask>();
    k_start<<<nblocks(n, 256), 256, 0, st>>>(n, slot_task[0], tasks[0], task_node[0], tb[0], bins[0], counters);
    int num_big = 1, c = 0;
    for (int level = 0; num_big > 0; level++) {
      k_bounds<<<windows, BLOCK, 0, st>>>(n, slot_task[c], lo[c], hi[c], tb[c]);
      if (level == 0) BNX_HIP(hipMemcpyAsync(root_tb, tb[0], sizeof(TB), hipMemcpyDeviceToDevice, st));
      k_bin<<<windows, BLOCK, 0, st>>>(n, slot_task[c], lo[c], hi[c], tb[c], bins[c]);
      BNX_HIP(hipMemsetAsync(counters + STAT_BIG, 0, sizeof(int), st));
      k_split<<<nblocks(num_big, BLOCK / 64), BLOCK, 0, st>>>(num_big, tasks[c], task_node[c], tb[c], bins[c], nodes,
                                                             S.split.as<Split>(), tasks[c ^ 1], task_node[c ^ 1],
                                                             tb[c ^ 1], bins[c ^ 1], mid, counters, c ^ 1);
      k_count<<<windows, BLOCK, 0, st>>>(n, slot_task[c], S.split.as<Split>(), lo[c], hi[c], win);
      k_scan_windows<<<1, 1024, 0, st>>>(2 * windows, win);
      k_scatter<<<windows, BLOCK, 0, st>>>(n, slot_task[c], S.split.as<Split>(), win, lo[c], hi[c], lo[c ^ 1],
                                           hi[c ^ 1], slot_task[c ^ 1]);
      BNX_HIP(hipMemcpyAsync(host.ctr, counters, sizeof(host.ctr), hipMemcpyDeviceToHost, st));
      BNX_HIP(hipStreamSynchronize(st));
      num_big = host.ctr[STAT_BIG];
      if (num_big > big || host.ctr[STAT_MID] > mids) {
        set_error("bvh builder: task overflow");
        return BNX_ERR_STATE;
      }
      c ^= 1;
    }
    if (host.ctr[STAT_MID] > 0)
      k_mid<<<host.ctr[STAT_MID], BLOCK, 0, st>>>(mid, lo[0], hi[0], lo[1], hi[1], nodes, order, counters, max_leaf,
                                                  nullptr, -1);
  }
  BNX_HIP(hipMemcpyAsync(&host, counters, sizeof(host), hipMemcpyDeviceToHost, st));
  BNX_HIP(hipStreamSynchronize(st));
  BNX_HIP(hipGetLastError());
  auto back = [](int i) {
    i = i >= 0 ? i : (i ^ 0x7fffffff);
    float f;
    memcpy(&f, &i, 4);
    return f;
  };
  for (int k = 0; k < 3; k++) {
    out.root_lo[k] = back(host.tb.v[k]);
    out.root_hi[k] = back(host.tb.v[3 + k]);
  }
  out.num_nodes = host.ctr[STAT_NODE];
  out.num_prims = n;
  out.max_depth = host.ctr[STAT_DEPTH];
  out.build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return BNX_OK;
}

} // namespace bnx
