// Brute-force check of the brick arithmetic of c3d_bricks.h (the header the
// device kernels use).  For each lattice given as "ncx ncy ncz max_rows
// planes shift" on the command line, and bricks of 8, 4 and 2 columns a
// side, walks every position of every XCD list and every lane of every brick
// as the kernel does, for all eight flips, and checks that every cell is
// visited exactly once, that a brick holds at most side^2 columns and
// kBrickPlanes planes inside the lattice, and that every position lies inside
// the ordered list.  Prints one line per lattice and side; exits 1 on the
// first failure.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "c3d_bricks.h"

using namespace c3d;

static int fail(const char* what, unsigned long long a, unsigned long long b) {
  std::printf("FAIL %s (%llu, %llu)\n", what, a, b);
  return 1;
}

static int check(uint32_t ncx, uint32_t ncy, uint32_t ncz, uint32_t rows, uint32_t planes, uint32_t shift,
                 uint32_t side) {
  const BrickGeo g = make_brick_geo(ncx, ncy, ncz, rows, planes, shift, side);
  const uint32_t ng = brick_groups(g), per = 1u << (3 * shift);
  if (g.bw * g.bh > side * side || g.bz > kBrickPlanes || !g.bw || !g.bh || !g.bz) return fail("size", g.bw, g.bh);
  if (rows && g.bh > rows) return fail("rows", g.bh, rows);
  for (uint32_t flip = 0; flip < 8; flip++) {
    std::vector<uint8_t> seen(uint64_t(ncx) * ncy * ncz, 0), taken(ng, 0);
    for (uint32_t x = 0; x < 8; x++) {
      const uint32_t n = brick_positions(ng, shift, x);
      for (uint32_t p = 0; p < n; p++) {
        const uint32_t s = x + 8u * (p >> (3u * shift));
        if (s >= ng) return fail("group", s, ng);
        if (p % per == 0 && taken[s]++) return fail("group twice", s, x);
        BrickBox b;
        if (!brick_box(g, ncx, ncy, ncz, s, p & (per - 1u), flip, b)) continue;
        if (b.i1 > ncx || b.j1 > ncy || b.k1 > ncz || b.k0 >= b.k1) return fail("box", s, p);
        for (uint32_t lane = 0; lane < 64; lane++) {
          const uint32_t row = fdiv(lane, g.div_bw), col = lane - row * g.bw;
          const uint32_t i = b.i0 + col, j = b.j0 + row;
          if (!(i < b.i1 && j < b.j1)) continue;
          for (uint32_t k = b.k0; k < b.k1; k++)
            if (seen[(uint64_t(k) * ncy + j) * ncx + i]++) return fail("cell twice", s, lane);
        }
      }
    }
    for (uint64_t c = 0; c < seen.size(); c++)
      if (!seen[c]) return fail("cell never visited", c, flip);
    for (uint32_t s = 0; s < ng; s++)
      if (!taken[s]) return fail("group never taken", s, ng);
  }
  std::printf("ok %u x %u x %u rows<=%u planes<=%u: bricks %u x %u x %u, groups %u\n", ncx, ncy, ncz, rows, planes, g.bw,
              g.bh, g.bz, ng);
  return 0;
}

int main(int argc, char** argv) {
  for (int a = 1; a + 5 < argc; a += 6) {
    uint32_t v[6];
    for (int q = 0; q < 6; q++) v[q] = uint32_t(std::atoi(argv[a + q]));
    for (uint32_t side = kBrickSide; side >= 2; side /= 2)
      if (check(v[0], v[1], v[2], v[3], v[4], v[5], side)) return 1;
  }
  return 0;
}
