// When a brick's triangles cannot reach the image: the arithmetic behind
// skipping them, shared by the device kernel and a host-side check (compiled
// by hipcc for the device and by a plain C++ compiler for the CPU tests).
//
// A triangle may be left out if every fragment it draws loses the z-test
// against what the z-buffer already holds (keys only grow).  Two things have
// to be known for that, both from the FP64 arithmetic as it is computed, not
// from exact geometry:
//   - which pixels its fragments fall on: those of the projection of its
//     brick's box, widened by three pixels (brick_limits);
//   - how near they can be: the harmonic depth of a fragment is the nearest
//     vertex's depth at most, up to a relative margin, provided that the
//     computed barycentric weights sum to one within kSlack (bound).
// The second is not true of every triangle.  One whose projection has next
// to no area (a sliver at a corner of its tetrahedron, a triangle seen edge
// on, vertices that fell together where a value equals the threshold) has
// weights of rounding noise, or exactly +-0, and then any depth up to
// +infinity, which the reference draws over everything.  So a cell is only
// skipped if it is regular (cell_regular): the doubled projected area of
// every triangle it can hold is at least `need`, chosen so that rounding
// moves the sum of the weights by at most kSlack.
//
// The area of a cell's triangles.  A triangle of a tetrahedron of volume
// H / 6 (H = hx hy hz) cuts three of its edges, and consecutive cut edges
// share a corner; with d = value - threshold at the corners, Delta the
// difference along a cut edge and F the tetrahedron's affine interpolant at
// the camera, minus the threshold, the triangle and the camera span
//   |det(r0, r1, r2)| = H |F| |d_a| |d_b| / (Delta0 Delta1 Delta2),
// a, b the shared corners (a = b when one corner is cut off).  With m the
// least |d| and M the range of the cell's eight values this is at least
// H |F| m^2 / M^3.  The projection q = (D / nr) ray . l / l.l (project.c)
// turns it into the doubled area
//   A = cv |det(r0, r1, r2)| / |nr0 nr1 nr2|,  cv = D^2 |lx x ly| / (lxx lyy),
// D the distance from the camera to the screen plane.
//
// What the area has to be.  Let u be the unit roundoff, g = 4.5 u, L a bound
// on the projected extent of the brick (x and y ranges added), p the larger
// and s the smaller pixel spacing and E a bound on the error of a projected
// vertex.  A candidate pixel lies within L + 6 p of every vertex, so each
// computed edge function is within g (L + 6 p) L of its exact value for the
// computed vertices, their sum is the exact area of the computed vertices, and
// that is within 6 E L of A.  Hence with
//   need = 2 (3 g (L + 6 p) L / kSlack + 6 E L),
// and at least 4e-16 (above the reference's clamp of the area at 1e-16),
// every A >= need gives weights whose sum is within kSlack of one, each within
// kSlack / 6 of its exact value.  Pixels farther than the widened box (the
// reference clamps boxes to the image) lie outside the triangle by more than
// s, where some exact weight is below -s / (3 L); with L < 10000 s that is
// beyond rounding.
// All of it needs vertices that are near where they should be: 24 E < L, so
// that L holds and the area's error is 6 E L at most, and E < s / 4, so that
// the widened box holds.  Where a lattice's spacing nears the last place of
// its coordinates neither is true, down to bricks whose corners all round
// onto one screen point (L = 0, with which any area would do).
#pragma once

#include "c3d_geom.h"

namespace c3d {

constexpr double kSlack = 1.0e-4;    // |sum of the computed weights - 1| of a regular cell's fragments
constexpr double kNearBy = 4.0e-4;   // relative margin of the depth bound, at least 3 kSlack

// projection of one corner of a brick's box: screen coordinates, depth, and
// the size of the coordinates that went into them; false when it is not
// safely between the camera and the screen's far side
struct CornerView {
  double x, y, nr;
  double size;  // |ray| (1-norm)
};

C3D_HD bool corner_view(const ViewDev<double>& v, double px, double py, double pz, CornerView& o) {
  const double rx = px - v.cam[0], ry = py - v.cam[1], rz = pz - v.cam[2];
  o.nr = v.nrm[0] * rx + v.nrm[1] * ry + v.nrm[2] * rz;
  const double t = (v.d - v.nc) / o.nr;
  const double dx = v.cam[0] + t * rx - v.ctr[0], dy = v.cam[1] + t * ry - v.ctr[1],
               dz = v.cam[2] + t * rz - v.ctr[2];
  o.x = (dx * v.lx[0] + dy * v.lx[1] + dz * v.lx[2]) / v.lxx;
  o.y = (dx * v.ly[0] + dy * v.ly[1] + dz * v.ly[2]) / v.lyy;
  o.size = fabs(rx) + fabs(ry) + fabs(rz);
  return fabs(o.nr) > 1.0e-6 && t > 1.0e-6 && t < 1.0 - 1.0e-6;
}

// ranges over the eight corners
struct BrickRange {
  double x0, x1, y0, y1, n0, n1, size;
};

struct BrickLimits {
  int32_t i0, i1, j0, j1;  // pixels its regular cells' fragments fall on (empty: i1 < i0 or j1 < j0)
  double bound;            // no fragment of a regular cell has a larger depth
  double scale;            // cell_volume's: cv / (need |nr|^3), per unit of cell volume
};

// false: nothing can be said of the brick
C3D_HD bool brick_limits(const ViewDev<double>& v, const BrickRange& r, BrickLimits& o) {
  const double u = 1.1102230246251565e-16, g = 4.5 * u;
  const double p = v.pitch;
  const double s = 1.0 / fmax(v.fw, v.fh);
  const double L = (r.x1 - r.x0) + (r.y1 - r.y0);
  if (!(L < fmin(2000.0 * p, 10000.0 * s))) return false;
  // one sign of depth, and not too wide a range of it
  if (!(r.n0 * r.n1 > 0.0)) return false;
  const double nmin = fmin(fabs(r.n0), fabs(r.n1)), nmax = fmax(fabs(r.n0), fabs(r.n1));
  if (!(nmax < 1000.0 * nmin)) return false;
  // error of a projected vertex: the rounding of the vertex, the ray, nr, t,
  // the screen offset and its products with lx and ly
  const double cam = fabs(v.cam[0]) + fabs(v.cam[1]) + fabs(v.cam[2]);
  const double S = 2.0 * cam + fabs(v.ctr[0]) + fabs(v.ctr[1]) + fabs(v.ctr[2]) + r.size;
  const double l = sqrt(fmin(v.lxx, v.lyy));
  const double q = fmax(fmax(fabs(r.x0), fabs(r.x1)), fmax(fabs(r.y0), fabs(r.y1)));
  const double E = 64.0 * u * (S * (1.0 + r.size / nmin) / l + 1.0 + q);
  // (false also where E is not a number)
  if (!(E < 0.25 * s && 24.0 * E < L)) return false;
  const double need = fmax(2.0 * (3.0 * g * (L + 6.0 * p) * L / kSlack + 6.0 * E * L), 4.0e-16);
  const double scale = v.cv / (need * nmax * nmax * nmax);
  if (!(scale > 0.0 && scale < 1.0e30)) return false;
  o.scale = scale;
  o.bound = r.n1 + kNearBy * fabs(r.n1);
  // boxes of pixel indices, widened by three; far off the image they are
  // clamped to a few pixels outside it
  const double fw = v.fw, fh = v.fh;
  const double a = fmin(fmax((r.x0 + 0.5) * fw - 3.5, -8.0), fw + 8.0), b = fmin(fmax((r.x1 + 0.5) * fw + 2.5, -8.0), fw + 8.0);
  const double c = fmin(fmax((r.y0 + 0.5) * fh - 3.5, -8.0), fh + 8.0), d = fmin(fmax((r.y1 + 0.5) * fh + 2.5, -8.0), fh + 8.0);
  o.i0 = int32_t(floor(a)) > 0 ? int32_t(floor(a)) : 0;
  o.i1 = int32_t(ceil(b)) < v.W - 1 ? int32_t(ceil(b)) : v.W - 1;
  o.j0 = int32_t(floor(c)) > 0 ? int32_t(floor(c)) : 0;
  o.j1 = int32_t(ceil(d)) < v.H - 1 ? int32_t(ceil(d)) : v.H - 1;
  return true;
}

// What the check needs of a cell besides a threshold: the affine
// interpolants of its six tetrahedra at the camera, and the range of its
// values, all relative to corner 0.
struct CellValues {
  float e[8];   // value - value of corner 0
  float at[6];  // the tetrahedra's interpolants at the camera
  float range;  // M
  float err;    // bound on the rounding of `at`, in units of the range
};

// v: corner values (corner i + 2j + 4k); (X, Y, Z): the camera in units of
// the cell, from corner 0
C3D_HD void cell_values(const double v[8], float X, float Y, float Z, CellValues& c) {
  float lo = 0.0f, hi = 0.0f, sum = 0.0f;
  c.e[0] = 0.0f;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
  for (int n = 1; n < 8; n++) {
    c.e[n] = float(v[n] - v[0]);
    lo = fminf(lo, c.e[n]);
    hi = fmaxf(hi, c.e[n]);
    sum += c.e[n];
  }
  // a value that is not a number (which min and max pass over) makes the range
  // one, too
  c.range = (hi - lo) * 1.000001f + 0.0f * sum;
  const float x1 = c.e[1] * X, y2 = c.e[2] * Y, z4 = c.e[4] * Z;
  c.at[0] = x1 + (c.e[3] - c.e[1]) * Y + (c.e[7] - c.e[3]) * Z;
  c.at[1] = x1 + (c.e[5] - c.e[1]) * Z + (c.e[7] - c.e[5]) * Y;
  c.at[2] = z4 + (c.e[5] - c.e[4]) * X + (c.e[7] - c.e[5]) * Y;
  c.at[3] = z4 + (c.e[6] - c.e[4]) * Y + (c.e[7] - c.e[6]) * X;
  c.at[4] = y2 + (c.e[6] - c.e[2]) * Z + (c.e[7] - c.e[6]) * X;
  c.at[5] = y2 + (c.e[3] - c.e[2]) * X + (c.e[7] - c.e[3]) * Z;
  // coordinates and differences are rounded once or twice each, products and
  // sums once: under 8 units of 2^-24 per term.  A camera so far off, in
  // cells, that a product could leave float's range (which a minimum passes
  // over once it is not a number) makes the bound one that nothing meets.
  const float far = fabsf(X) + fabsf(Y) + fabsf(Z);
  c.err = far < 1.0e15f ? 1.0e-6f * (far + 1.0f) : HUGE_VALF;
}

// scale * |hx hy hz| for cell_regular, from edges and a scale of any size: the
// product is formed in FP64 and cut off at 1e20 (a smaller volume makes fewer
// cells regular), and it is 0 where an edge, which the camera's place in cells
// is divided by in FP32, comes near the ends of that range.
C3D_HD float cell_volume(double hx, double hy, double hz, double scale) {
  const double x = fabs(hx), y = fabs(hy), z = fabs(hz), v = x * y * z * scale;
  if (!(fmin(fmin(x, y), z) > 1.0e-30 && fmax(fmax(x, y), z) < 1.0e30)) return 0.0f;
  return v < 1.0e20 ? float(v) * 0.999999f : 1.0e20f;
}

// Whether every triangle of the cell at a threshold is regular; d0: value of
// corner 0 minus the threshold; volume: cell_volume.  False for values that
// are not finite, and below 1e-8 (where the interpolation keeps a corner
// instead of a point between two).
C3D_HD bool cell_regular(const CellValues& c, float d0, float volume) {
  float m = fabsf(d0), f = fabsf(c.at[0] + d0);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
  for (int n = 1; n < 8; n++) m = fminf(m, fabsf(c.e[n] + d0));
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
  for (int n = 1; n < 6; n++) f = fminf(f, fabsf(c.at[n] + d0));
  m -= 1.0e-6f * c.range;
  f -= c.err * c.range;
  // the range also keeps the squares and quotients inside float's range
  if (!(c.range > 1.0e-12f && c.range < 1.0e12f && m > 1.0e-8f && f > 0.0f)) return false;
  const float a = m / c.range, b = f / c.range;
  return a * a * b * volume >= 1.00001f;
}

}  // namespace c3d
