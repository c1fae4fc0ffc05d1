// bnx_claims.h -- how the waves of a persistent launch (march, trace) share
// a generation's rays, and scalar loads of wave-uniform records.
#pragma once
#include "bnx_device.h"
#include "bnx_render.h"

namespace bnx {
namespace {

// a record at a wave-uniform address that no running kernel writes: scalar
// loads, which the compiler may repeat where it is short of registers
#if defined(__HIP_DEVICE_COMPILE__)
#define BNX_CONST __attribute__((address_space(4)))
#else
#define BNX_CONST
#endif
template <typename T> BNX_D T uniform_load(const T BNX_G *p)
{
  static_assert(sizeof(T) % 4 == 0, "whole words");
  const uint32_t BNX_CONST *c = (const uint32_t BNX_CONST *)p;
  uint32_t w[sizeof(T) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); i++) w[i] = c[i];
  T r;
  __builtin_memcpy(&r, w, sizeof(T));
  return r;
}

// How the waves of a launch share its rays.  The generation's blocks of 256
// rays, each inside one segment, are cut into chunks: down to 64 rays until
// there are `balance` (a wave's first chunk is its own, and what no chunk is
// left for is time that waves with short rays wait for those with long ones),
// and down to 16 until there are `least` (so that a small generation still has
// some for every wave).  They are dealt to CLAIM_GROUPS
// groups of waves; a wave starts on a chunk of its own and then takes its
// group's next one from the group's counter, or another group's once its own
// is out.  One counter for all waves would be in the way: its atomics are
// served one after the other beyond the XCDs' caches (14 ns each, 3.4
// against 2.4 ms on the 256^3 volume).  Shares fixed beforehand would leave
// the waves with the long rays behind (isosurface of 20.5M tets: 19.6
// against 12.9 ms), and so do chunks as large as the waves are many: 82k
// triangles, 900x600, 2 spp, traces in 4219 chunks on 5120 waves, 1.92 ms a
// frame, and 1.57 in 16876; tets of 80^3 cubes, 1024x768, 2 spp, 5.77 and 3.99.
struct Claims {
  const Segment *segs;
  const int *blk;              // segment of each 256-ray block
  int *ctr;                    // this launch's counters, 0 when it begins
  int chunks, shift, per, waves;   // chunks of `per` = 256 >> shift rays
  int chunk, group, tries;     // the chunk in hand (-1: none left)
  int seg;                     // the segment being worked on
  int first, total;            // its first 256-ray block, its rays
  int base, next, stop;        // [next, stop) is in hand, segment-local, from queue index base
  bool dry;                    // none left in this segment

  BNX_D void begin(const SegView &sv, int nsegs, int program, int least, int balance)
  {
    segs = sv.segs;
    blk = sv.blk256;
    const Segment z = uniform_load((const Segment BNX_G *)(segs + nsegs - 1));
    deal(z.block256 + (z.count + 255) / 256, sv.claims + program * CLAIM_GROUPS * CLAIM_STRIDE, least, balance);
  }
  // n rays without segments
  BNX_D void begin(int n, int *counters, int least, int balance)
  {
    segs = nullptr;
    blk = nullptr;
    deal((n + 255) / 256, counters, least, balance);
    seg = first = base = 0;
    total = n;
    dry = chunk < 0;
    next = stop = 0;
    if (!dry) range();
    refill();
  }
  BNX_D void deal(int blocks, int *counters, int least, int balance)
  {
    ctr = counters;
    waves = (int)gridDim.x;
    shift = 0;
    while (shift < 2 && (blocks << shift) < balance) shift++;
    while (shift < 4 && (blocks << shift) < least) shift++;
    per = 256 >> shift;
    chunks = blocks << shift;
    chunk = (int)blockIdx.x < chunks ? (int)blockIdx.x : -1;
    group = (int)blockIdx.x % CLAIM_GROUPS;
    tries = chunks > waves ? 0 : CLAIM_GROUPS;   // every chunk is some wave's first
  }
  // the chunk after the one in hand
  BNX_D void advance()
  {
    chunk = -1;
    const int rounds = waves / CLAIM_GROUPS;   // the launch has whole rounds of waves
    while (chunk < 0 && tries < CLAIM_GROUPS) {
      int c = 0;
      if (lane_id() == 0) c = atomicAdd(ctr + group * CLAIM_STRIDE, 1);
      c = (rounds + __builtin_amdgcn_readfirstlane(c)) * CLAIM_GROUPS + group;
      if (c < chunks) {
        chunk = c;
      } else {
        group = (group + 1) % CLAIM_GROUPS;
        tries++;
      }
    }
  }
  // take up the segment of the chunk in hand
  BNX_D const Segment open()
  {
    seg = segment_of_chunk();
    const Segment sg = uniform_load((const Segment BNX_G *)(segs + seg));
    base = sg.begin;
    first = sg.block256;
    total = sg.count;
    dry = false;
    range();
    return sg;
  }
  BNX_D int segment_of_chunk() { return blk ? __builtin_amdgcn_readfirstlane(blk[chunk >> shift]) : 0; }
  BNX_D void range()
  {
    const int b = chunk >> shift;
    next = (b - first) * 256 + (chunk - (b << shift)) * per;
    stop = min(next + per, total);
  }
  // once the chunk in hand is taken: the next one, if it is of this segment
  BNX_D void refill()
  {
    while (next >= stop && !dry) {
      advance();
      if (chunk < 0 || segment_of_chunk() != seg) {
        dry = true;
      } else {
        range();
      }
    }
  }
  // the rays for the next `want` lanes in line: this lane's (place: its place
  // in the line), and whether there is one
  BNX_D int claim(int want, int place, bool &on)
  {
    on = next + place < stop;
    const int i = base + next + (on ? place : 0);
    next += want;
    refill();
    return i;
  }
};

} // namespace
} // namespace bnx
