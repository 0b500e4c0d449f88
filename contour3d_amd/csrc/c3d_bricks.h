// Index arithmetic of the bricks that a frame's tessellation walks, shared
// by the device kernels and a host-side brute-force check (compiled by hipcc
// for the device and by a plain C++ compiler for the CPU tests).
//
// A brick is a box of bw x bh x bz cells, one lane of a wave per cell column
// (bw * bh <= 64), compact so that its projection is: the order and the
// visibility of its triangles are decided brick by brick.  Bricks are taken
// in groups of 2^shift per axis, the unit in which a launch orders them by
// depth and shares them out over the XCDs.  The triangles of a frame carry
// their place in the drawing order in their ids, so bricks may run in any
// order.
#pragma once

#include <cstdint>

#include "c3d_tiles.h"

namespace c3d {

constexpr uint32_t kBrickColumns = 64;  // cell columns of a brick at most (a wave's lanes)
constexpr uint32_t kBrickSide = 8;      // cells per axis of a brick's plane, where the lattice has them
constexpr uint32_t kBrickPlanes = 8;    // planes of a brick at most

// The shapes a frame chooses from: columns per side of a brick, and planes.
struct BrickShape {
  uint32_t side, planes;
};
constexpr BrickShape kBrickShapes[] = {{8, 8}, {8, 4}, {8, 2}, {4, 4}, {4, 2}, {4, 1}, {2, 2}, {2, 1}};
constexpr uint32_t kNumBrickShapes = sizeof(kBrickShapes) / sizeof(kBrickShapes[0]);
constexpr uint32_t brick_volume(uint32_t s) { return kBrickShapes[s].side * kBrickShapes[s].side * kBrickShapes[s].planes; }

struct BrickGeo {
  uint32_t bw, bh, bz;     // cells per brick
  uint32_t nbx, nby, nbz;  // bricks per axis
  uint32_t nsx, nsy, nsz;  // groups per axis
  uint32_t shift;          // log2 of the bricks per axis of a group
  FastDiv div_bw, div_nsx, div_nsy;
};

// Bricks of an ncx x ncy x ncz cell lattice: balanced, at most side^2 columns,
// max_rows rows (0: as many as fit) and `planes` planes each.
inline BrickGeo make_brick_geo(uint32_t ncx, uint32_t ncy, uint32_t ncz, uint32_t max_rows, uint32_t planes,
                               uint32_t shift, uint32_t side = kBrickSide) {
  auto parts = [](uint32_t n, uint32_t of) { return (n + of - 1) / of; };
  BrickGeo g{};
  const uint32_t columns = side * side;
  uint32_t rows = ncy < side ? ncy : side;
  if (max_rows && rows > max_rows) rows = max_rows;
  g.nbx = parts(ncx, columns / rows);
  g.bw = parts(ncx, g.nbx);
  g.nbx = parts(ncx, g.bw);
  rows = columns / g.bw;
  if (max_rows && rows > max_rows) rows = max_rows;
  g.nby = parts(ncy, rows);
  g.bh = parts(ncy, g.nby);
  g.nby = parts(ncy, g.bh);
  if (planes < 1) planes = 1;
  if (planes > kBrickPlanes) planes = kBrickPlanes;
  g.nbz = parts(ncz, planes);
  g.bz = parts(ncz, g.nbz);
  g.nbz = parts(ncz, g.bz);
  g.shift = shift;
  g.nsx = (g.nbx + (1u << shift) - 1) >> shift;
  g.nsy = (g.nby + (1u << shift) - 1) >> shift;
  g.nsz = (g.nbz + (1u << shift) - 1) >> shift;
  g.div_bw = make_fastdiv(g.bw);
  g.div_nsx = make_fastdiv(g.nsx);
  g.div_nsy = make_fastdiv(g.nsy);
  return g;
}

C3D_TD uint32_t brick_groups(const BrickGeo& g) { return g.nsx * g.nsy * g.nsz; }

// a group's coordinates
C3D_TD void group_at(const BrickGeo& g, uint32_t s, uint32_t& x, uint32_t& y, uint32_t& z) {
  const uint32_t yz = fdiv(s, g.div_nsx);
  x = s - yz * g.nsx;
  z = fdiv(yz, g.div_nsy);
  y = yz - z * g.nsy;
}

// Cells [i0, i1) x [j0, j1) x [k0, k1) of brick b (0 .. 8^shift - 1) of group
// s, the group's bricks taken from their far end on the axes in `flip` (bits
// 0-2); false for a brick past the lattice.
struct BrickBox {
  uint32_t i0, i1, j0, j1, k0, k1;
};
C3D_TD bool brick_box(const BrickGeo& g, uint32_t ncx, uint32_t ncy, uint32_t ncz, uint32_t s, uint32_t b,
                      uint32_t flip, BrickBox& o) {
  uint32_t x, y, z;
  group_at(g, s, x, y, z);
  const uint32_t m = (1u << g.shift) - 1u;
  x = (x << g.shift) + ((b & m) ^ (flip & 1u ? m : 0u));
  y = (y << g.shift) + (((b >> g.shift) & m) ^ (flip & 2u ? m : 0u));
  z = (z << g.shift) + ((b >> (2u * g.shift)) ^ (flip & 4u ? m : 0u));
  if (x >= g.nbx || y >= g.nby || z >= g.nbz) return false;
  o.i0 = x * g.bw;
  o.j0 = y * g.bh;
  o.k0 = z * g.bz;
  o.i1 = o.i0 + g.bw < ncx ? o.i0 + g.bw : ncx;
  o.j1 = o.j0 + g.bh < ncy ? o.j0 + g.bh : ncy;
  o.k1 = o.k0 + g.bz < ncz ? o.k0 + g.bz : ncz;
  return true;
}

// The walk: XCD x takes groups x, x + 8, ... of the launch's ordered list,
// brick by brick; its positions are 0 .. brick_positions(...) - 1, position p
// being brick p mod 8^shift of its (p div 8^shift)-th group.
C3D_TD uint32_t brick_positions(uint32_t ngroups, uint32_t shift, uint32_t x) {
  return x < ngroups ? ((ngroups - x + 7u) >> 3) << (3u * shift) : 0u;
}

}  // namespace c3d
