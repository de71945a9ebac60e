// Tile-window machinery shared by the FP64 and FP32 particle passes.
//
// One workgroup takes one sort tile (its particles are contiguous after the
// sort) or one chunk of the unsorted inflow tail.  It accumulates current
// and density in an LDS window around an anchor box: the tile's cells, or
// the bounding box of a few sampled particles of a tail chunk.  The window
// spans the anchor +- kMargin cells; a particle whose cell at the start of
// the step lies within the anchor +- (kMargin - 2) has all its gather and
// deposit nodes inside the window (it moves less than one cell per step and
// its stencils reach one node below and two above its cell).
#pragma once
#include <hip/hip_runtime.h>

#include "pic_internal.h"

namespace pic {

constexpr int kMargin = 3;
constexpr int kTailChunk = 2048;  // most slots per workgroup of the tail
constexpr int kStray = 8;

// Slots per workgroup of the unsorted tail of `tail` slots.  An inflow batch
// walks its two-layer slab in blocks of 4 x 4 x 2 cells (blocked) or along y
// in columns of 2 cells, ppc slots per cell; the window holds 3 blocks or 16
// columns (kStray cells to either side of the middle sample), so a chunk of
// more slots than that has no window and adds every contribution to the
// global planes.  A tail too short to give every place on the chip (3
// workgroups per CU) a chunk is cut finer: it runs last, so its longest chunk
// is what the launch waits for, and the overflow of the in-tile inflow, some
// hundred slots per slab tile in tile order, spans few tiles per chunk.  In
// chunks of 2048 that overflow cost 60 us of 330 us per launch at
// 64^3 x 32 ppc.
constexpr int kChipSlots = 768;

inline int tail_chunk(int ppc, bool blocked, int64_t tail) {
  const int64_t most = (int64_t)(blocked ? 64 : 32) * ppc;
  int c = kTailChunk;
  while (c > 256 && (c > most || tail < (int64_t)kChipSlots * c)) c >>= 1;
  return c;
}
// most workgroups that a store of cap slots can need for its tail
inline int64_t most_chunks(int ppc, int64_t cap) {
  const int64_t c = tail_chunk(ppc, false, cap);
  const int64_t few = (int64_t)kChipSlots * kTailChunk / 256;
  return ((cap + c - 1) / c > few ? (cap + c - 1) / c : few) + 1;
}

// Below this many workgroups of both species, their fused passes are one
// launch: the second species' workgroups take the places that the first one's
// last round leaves empty, and a launch's latency goes.  Above it the
// arguments' indirection by species costs more than that.  20 steps, one
// launch / two: FP32 31 x 27 x 45 x 8 ppc 1.62 / 1.82 ms, 64^3 x 32 ppc (4100
// workgroups) 14.1 / 14.6 ms, 128^3 x 64 ppc (33000) 154 / 149.5 ms; FP64
// 8 x 8 x 16 x 4 ppc 0.53 / 0.58 ms, 32^3 x 16 ppc (2000 to 4000) 4.66 /
// 4.80 ms, 128^3 x 64 ppc 332 / 294 ms (with a species per launch the force
// gathers its own E).
constexpr unsigned kBothBlocks = 8 * kChipSlots;

struct TileRun {
  const uint32_t *tile_start;  // ntiles + 1 entries (rows: one per cell, + 1)
  int ntiles;
  int64_t sorted_end;          // [0, sorted_end) is tile-sorted
  int64_t n;                   // stored slots
  int ntail;                   // tail chunks
  int chunk;                   // slots per tail chunk
  int split;                   // workgroups (parts) per tile
  __host__ __device__ inline int parts() const { return ntiles * split; }
};

// Workgroups per tile.  Where the tiles of a species are fewer than the
// places on the chip, a tile's particles go to several workgroups, each with
// a window of its own, as long as a part keeps 512 particles (down to 256 and
// up to 1024 the same within 3 %).  20 steps, whole tiles / parts:
// 128^2 x 64 ppc on 16^2 tiles FP32 6.35 / 2.68 ms and FP64 7.4 / 2.5 ms,
// 256^2 x 16 ppc 2.9 / 2.24 ms, 24 x 24 x 32 x 64 ppc on 4 x 4 x 8 tiles FP32
// 4.56 / 3.88 ms and FP64 6.1 / 4.6 ms.
inline int tile_split(int64_t ntiles, int64_t particles, int places) {
  int p = 1;
  while (p < 8 && ntiles * p < places && particles / (ntiles * 2 * p) >= 512) p *= 2;
  return p;
}

// part p of n of the slots [s, e): whole groups of four slots but for the ends
__device__ inline void part_range(int p, int n, int64_t &s, int64_t &e) {
  const int64_t b = s, len = e - s;
  if (p > 0) {
    const int64_t a = (b + len * p / n) & ~(int64_t)3;
    s = a > b ? a : b;
  }
  if (p + 1 < n) {
    const int64_t a = (b + len * (p + 1) / n) & ~(int64_t)3;
    e = a > b ? a : b;
  }
}

// A store sorted as one tile (the reference's order: cells along z, then y,
// then x) has no tile ranges of its own.  The pass takes it in boxes of
// TX x TY columns of TZ cells; a box's particles are TX * TY ranges of the
// store, found in the table of each cell's first slot that the sort leaves.
// Boxes may reach over the grid's upper faces (the sizes need not divide).
// 4 x 4 x 8 is the largest box whose window fits both forms; where that
// gives fewer than 300 boxes (both species' run together), 2 x 2 x 8.  20
// steps, small / large boxes: 336 large ones of 31 x 27 x 45 x 8 ppc FP32
// 3.25 / 2.28 ms, 500 of 40^3 x 4 ppc FP32 3.56 / 2.11 ms and FP64 3.3 /
// 2.54 ms; 256 of 32^3 x 16 ppc FP64 the same.
inline TileGeom row_geom(const TileGeom &one) {
  const auto up = [](int a, int b) { return (a + b - 1) / b; };
  TileGeom t = one;
  const int NX = one.TX, NY = one.TY, NZ = one.TZ;
  for (int w = 4; w >= 2; w -= 2) {
    t.TX = t.TY = w;
    t.TZ = 8;
    t.NTX = up(NX, w);
    t.NTY = up(NY, w);
    t.NTZ = up(NZ, 8);
    if (t.ntiles() >= 300) break;
  }
  t.LX = t.LY = t.LZ = -1;
  return t;
}

// Whether a store of n particles takes its boxes; else it goes in chunks, as
// an unsorted tail.  Every box pays for its window, so the store must hold 32
// particles per box: two steps, chunks / boxes, with 16 and with 32 per box:
// 128^3 FP64 1.85 / 1.88 and 2.73 / 1.93 ms, FP32 1.86 / 2.02 and 3.03 / 2.16
// ms; 32^3 FP64 0.127 / 0.129 and 0.162 / 0.128 ms; with 1 per box at 128^3
// 0.78 / 1.49 and 0.48 / 1.18 ms.  And one workgroup takes the fullest box
// (most particles): it must not hold more than 8 times a workgroup's share.
// 64^3, 500000 particles within a cube, chunks / boxes: 32^3 cells (3 times)
// FP64 0.58 / 0.45, FP32 0.46 / 0.36 ms; 16^3 cells (24 times) 0.40 / 1.11 and
// 0.35 / 0.76 ms; 4 x 4 x 8 cells 0.36 / 14 and 0.32 / 9.9 ms.
inline bool boxes_filled(int64_t n, int64_t boxes) { return n >= 32 * boxes; }
inline bool boxes_even(int64_t n, int64_t boxes, int64_t most) {
  return most * (boxes < kChipSlots ? boxes : kChipSlots) <= 8 * n;
}

// slot range of column r (< TX * TY) of box bid
__device__ inline void row_range(const TileRun &tr, const TileGeom &tg, int NX, int NY,
                                 int NZ, int bid, int r, int &s, int &e) {
  const int tz = bid % tg.NTZ, ty = (bid / tg.NTZ) % tg.NTY, tx = bid / (tg.NTZ * tg.NTY);
  const int k = tx * tg.TX + r / tg.TY, l = ty * tg.TY + r % tg.TY;
  s = e = 0;
  if (k >= NX || l >= NY) return;
  const int64_t c = ((int64_t)k * NY + l) * NZ;
  s = (int)tr.tile_start[c + tz * tg.TZ];
  e = (int)tr.tile_start[c + min((tz + 1) * tg.TZ, NZ)];
}

// LDS window: origin (cells) and extents (nodes), and the cell range whose
// stencils fit inside it
struct Win {
  int k0, l0, m0, WX, WY, WZ;
  int vk0, vk1, vl0, vl1, vm0, vm1;
  bool on;
};

// Between sorts the particles move with the bulk drift (vdrift) and leave
// their tile on its downstream side; those more than one cell out deposit
// through global atomics.  The tiles' windows follow the drift: after
// `halves` half-step drifts since the sort they are moved by the bulk
// displacement rounded to whole cells.
inline void add_drift_shift(TileGeom &t, const pic_config &c, int halves) {
  for (int a = 0; a < 3; ++a)
    t.shift[a] = (int)lround(c.vdrift[a] * 0.5 * c.dt * halves / c.dx);
}

__device__ inline int xcd_remap(int b, int nt, int nb) {
  // Workgroups are dealt round-robin over the 8 XCDs in launch order.  Each
  // XCD gets a contiguous range of the nt tiles (neighbouring tiles share its
  // L2) and then an equal share of the nb - nt tail chunks, so the light
  // chunk workgroups do not displace tiles onto the other XCDs.
  const int nc = nb - nt;
  const int qt = nt / 8, qc = nc / 8, q = qt + qc;
  if (b >= 8 * q) {  // remainders of both kinds, in order
    const int r = b - 8 * q, rt = nt - 8 * qt;
    return r < rt ? 8 * qt + r : nt + 8 * qc + (r - rt);
  }
  const int x = b % 8, s = b / 8;
  return s < qt ? x * qt + s : nt + x * qc + (s - qt);
}

// Range and window of workgroup bid.  cell_of(i, k, l, m) returns false for
// a dead slot.  Runs on one thread.  ROWS: the workgroups below ntiles are
// boxes of rows (row_geom), whose ranges row_range gives; s < e here.
template <bool ROWS, typename CellOf>
__device__ inline void tile_setup(int bid, const TileRun &tr, const TileGeom &tg,
                                  int win_max, CellOf cell_of, int64_t &s,
                                  int64_t &e, Win &w) {
  int ak0, ak1, al0, al1, am0, am1;  // anchor box (cells)
  if (bid < tr.parts()) {
    const int t = bid / tr.split;
    s = ROWS ? 0 : tr.tile_start[t];
    e = ROWS ? 1 : tr.tile_start[t + 1];
    if (!ROWS) part_range(bid % tr.split, tr.split, s, e);
    const int tz = t % tg.NTZ, ty = (t / tg.NTZ) % tg.NTY, tx = t / (tg.NTZ * tg.NTY);
    ak0 = 2 + tx * tg.TX + tg.shift[0];
    ak1 = ak0 + tg.TX - 1;
    al0 = 2 + ty * tg.TY + tg.shift[1];
    al1 = al0 + tg.TY - 1;
    am0 = 2 + tz * tg.TZ + tg.shift[2];
    am1 = am0 + tg.TZ - 1;
  } else {
    const int c = bid - tr.parts();
    s = tr.sorted_end + (int64_t)c * tr.chunk;
    e = s + tr.chunk < tr.n ? s + tr.chunk : tr.n;
    ak0 = al0 = am0 = 1 << 20;
    ak1 = al1 = am1 = -1;
    // 8 samples; those more than kStray cells from a middle sample on some
    // axis (a particle that wrapped across a periodic face, a straggler) are
    // left out of the box and deposit globally
    int ks[8], ls[8], ms[8];
    bool ok[8];
    for (int j = 0; j < 8; ++j) {
      const int64_t i = s + (e - s - 1) * j / 7;
      ok[j] = i >= s && i < e && cell_of(i, ks[j], ls[j], ms[j]);
    }
    int r = -1;
    for (int q = 0; q < 8 && r < 0; ++q) {
      const int j = (q & 1) ? 3 - (q >> 1) : 4 + (q >> 1);  // 4 3 5 2 6 1 7 0
      if (ok[j]) r = j;
    }
    for (int j = 0; j < 8 && r >= 0; ++j) {
      if (!ok[j] || abs(ks[j] - ks[r]) > kStray || abs(ls[j] - ls[r]) > kStray ||
          abs(ms[j] - ms[r]) > kStray)
        continue;
      ak0 = min(ak0, ks[j]); ak1 = max(ak1, ks[j]);
      al0 = min(al0, ls[j]); al1 = max(al1, ls[j]);
      am0 = min(am0, ms[j]); am1 = max(am1, ms[j]);
    }
  }
  w.on = ak1 >= ak0;
  if (w.on) {
    w.k0 = ak0 - kMargin;
    w.l0 = al0 - kMargin;
    w.m0 = am0 - kMargin;
    w.WX = ak1 - ak0 + 1 + 2 * kMargin;
    w.WY = al1 - al0 + 1 + 2 * kMargin;
    w.WZ = am1 - am0 + 1 + 2 * kMargin;
    w.vk0 = ak0 - (kMargin - 2);
    w.vk1 = ak1 + (kMargin - 2);
    w.vl0 = al0 - (kMargin - 2);
    w.vl1 = al1 + (kMargin - 2);
    w.vm0 = am0 - (kMargin - 2);
    w.vm1 = am1 + (kMargin - 2);
    if ((int64_t)w.WX * w.WY * w.WZ > win_max) w.on = false;
  }
}

}  // namespace pic
