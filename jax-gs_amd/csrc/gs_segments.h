// Segments of the tiles' lists: what the compositing forward leaves for its backward
// (gs_composite.hip) and where.
#pragma once

#include "gs_common.h"

namespace gs {

constexpr int kQuadTiles = 2048;  // images below are composited by composite_fwd_quad_kernel

// Segments of a tile's list.  The backward walks a tile's entries back to front, a serial
// chain like the forward's, and the longest tile's chain was most launches' time (2170 tiles
// of 274 entries on average: the one of 1046 took 283 us while the work of all would fill the
// GPU for 50).  The forward therefore cuts every list into segments, 1024/u of u entries, then
// 512/u of 2u and 512/u of 4u (4096 in all; log2 u = segment_shift), and leaves for each segment it
// completes, per pixel, the transmittance after it and the colour blended in it.  The backward
// then walks all segments at once: a segment starts from its own end's transmittance, and the
// colour behind it is the background's share plus the later segments' colours, summed from
// the back, so neither is recovered through the entries behind it.
// Backward, whole lists -> segments: 300k Gaussians at 979x546 283 -> 95 us, 200k at 504x378
// 217 -> 75, 50k at 640x479 170 -> 66, 2k at 96x64 90 -> 22, 2.1M at 1280x720 284 -> 197 (which
// zeroes 500 MB besides); the order of the items instead of the tiles' 4.8 -> 10 us, the slots
// add 5-8 us to the forward.
// Slot j of a tile (256 pixels, row by row): (T after segment j, colour r g b of segment j).  A
// tile's slots are those of its own entries where that is less than the most that a list can
// have (segment_slot).
// A pixel's slots are written for every segment it enters, except where its wave never leaves
// segment 0 (there the final T and the background say it all).
// The backward's work items are pieces: the segments of a coarser unit, the smallest of u, 2u,
// .. 512 at which the pieces of all tiles fit the launch's grid (segment_grid; every coarser
// unit's ends are ends of segments of u, and at 512 a tile has at most four).
struct Segments {
  int32_t* items;   // [0] = number of pieces, [1] = log2 of their unit + 256 packed, then tile * 32 + piece, longest first
  int32_t* met;     // per tile, the entries met by each of the forward's waves
  float4* slots;    // [segment_slots()][256]; NULL: the forward leaves none
  int lu;           // log2(u)
  bool packed;      // the forward's choice of slots (segments_packed); the backward reads items[1]
};
// From kFwdOneWaveTiles tiles on, one wave per tile fills the GPU several times over, and the
// slots' traffic and the pieces' set-up cost more than they balance (8160 tiles, the longest
// of 781 entries: backward 247 -> 255 us, its order 8 -> 13 us): no segments there.
constexpr int kFwdOneWaveTiles = 6 * 1024;
// Units: 64 entries where tiles are few (200k Gaussians, 504x378: 128 91 us, 64 75), 128 where
// they fill the GPU sooner and a piece's set-up has to be earned back (300k, 979x546: 64 99 us,
// 128 95, 256 121).
__host__ __device__ inline int segment_shift(int T) { return T < kQuadTiles ? 6 : 7; }  // log2(u)
__host__ __device__ inline int segment_count(int lu) { return 2048 >> lu; }
__host__ __device__ inline int segment_start(int j, int lu) {
  const int n0 = 1024 >> lu, n1 = n0 + (n0 >> 1);
  return j <= n0 ? j << lu : (j <= n1 ? 1024 + ((j - n0) << (lu + 1)) : 2048 + ((j - n1) << (lu + 2)));
}
// segments that hold the first k entries (k <= 4096)
__host__ __device__ inline int segments_within(int k, int lu) {
  const int n0 = 1024 >> lu, n1 = n0 + (n0 >> 1);
  const int up = (1 << lu) - 1, up1 = (2 << lu) - 1, up2 = (4 << lu) - 1;
  return k <= 1024 ? (k + up) >> lu : (k <= 2048 ? n0 + ((k - 1024 + up1) >> (lu + 1)) : n1 + ((k - 2048 + up2) >> (lu + 2)));
}
// Slots: 4 KB each, held from a render's forward to its backward.  A list of 4096 entries takes
// segment_count of them, so T tiles can take 128 KB (u = 64) or 64 KB (128) each, 101 MB at
// 504x378 and 236 MB at 1280x720.  A list of n entries takes at most n / u + 1, and tile t's entries
// start at ranges[t], so the slots of tile t from ranges[t] / u + t on are its own: T + capacity / u
// slots hold any set of lists of `capacity` entries.  The smaller of the two is taken (packed: the
// second): 2000 Gaussians (capacity 512,000) at 1440x1079 hold 41 MB instead of 401.
__host__ __device__ inline bool segments_packed(int T, int64_t capacity, int lu) {
  return T + (capacity >> lu) < (int64_t)T * segment_count(lu);
}
__host__ __device__ inline int64_t segment_slots(int T, int64_t capacity, int lu) {
  return segments_packed(T, capacity, lu) ? T + (capacity >> lu) : (int64_t)T * segment_count(lu);
}
// first slot of a tile whose entries start at `start`
__host__ __device__ inline int64_t segment_slot(bool packed, int tile, int start, int lu) {
  return packed ? (int64_t)(start >> lu) + tile : (int64_t)tile * segment_count(lu);
}
// Most pieces a launch takes.  Workgroups past the pieces' number exit at once, but each
// still costs its dispatch (3600 tiles with room for 16 pieces each, 57,600 workgroups of which
// 10,000 had work: 232 us against 203).
__host__ __device__ inline int segment_grid(int T) {
  const int all = T * segment_count(segment_shift(T)), some = 4 * T + 2048;
  return all < some ? all : some;
}

}  // namespace gs
