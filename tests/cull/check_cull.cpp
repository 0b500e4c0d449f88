// Brute-force check of c3d_cull.h (the header the device kernel uses): for
// random bricks, values and cameras, every fragment of every triangle of a
// regular cell -- found by the reference's own box, coverage test and
// harmonic depth in FP64 (c3d_geom.h) -- must lie in the brick's pixel box
// and be no nearer than its bound.  The values include what breaks depths:
// corners equal to the threshold or within 10^-1 .. 10^-17 of it, exact
// planes seen edge on through pixel centres, steps below the 1e-8 rule,
// infinities and NaN; the cameras include axis-aligned ones on odd images,
// sheared screens and screens facing away.
// Usage: check_cull <seed> <bricks per kind>; prints one line per kind of
// values, exits 1 on a miss.
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>
#include <vector>

#include "c3d_cull.h"

using namespace c3d;

typedef V3<double> V;
static std::mt19937_64 rng;
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static int pick(int n) { return int(rng() % uint64_t(n)); }

static const int kTet[6][4] = {{0, 7, 3, 1}, {0, 7, 1, 5}, {0, 7, 5, 4}, {0, 7, 4, 6}, {0, 7, 6, 2}, {0, 7, 2, 3}};
static const int kNtri[8] = {0, 1, 1, 2, 1, 2, 2, 1};
static const int kPairs[8][2][3][2] = {
    {{{0, 0}, {0, 0}, {0, 0}}, {{0, 0}, {0, 0}, {0, 0}}}, {{{0, 1}, {0, 3}, {0, 2}}, {{0, 0}, {0, 0}, {0, 0}}},
    {{{1, 0}, {1, 2}, {1, 3}}, {{0, 0}, {0, 0}, {0, 0}}}, {{{0, 2}, {1, 3}, {0, 3}}, {{0, 2}, {1, 2}, {1, 3}}},
    {{{2, 0}, {2, 3}, {2, 1}}, {{0, 0}, {0, 0}, {0, 0}}}, {{{2, 1}, {0, 3}, {2, 3}}, {{2, 1}, {0, 1}, {0, 3}}},
    {{{0, 2}, {2, 3}, {1, 3}}, {{0, 2}, {1, 3}, {0, 1}}}, {{{3, 0}, {3, 2}, {3, 1}}, {{0, 0}, {0, 0}, {0, 0}}}};

static V interp(double thr, V p0, double v0, V p1, double v1) {
  if (fabs(v1 - v0) < 1.e-8) return p0;
  const double f = (thr - v0) / (v1 - v0);
  return vadd(p0, vscale(f, vsub(p1, p0)));
}

static ViewDev<double> camera(int kind) {
  ViewDev<double> v = {};
  V cam, ctr, lx, ly;
  const int W[] = {1, 7, 33, 64, 101, 640}, H[] = {1, 9, 31, 48, 75, 361};
  v.W = W[pick(6)];
  v.H = H[pick(6)];
  if (kind == 0) {  // straight at the origin along an axis
    const int a = pick(3);
    const double s = pick(2) ? 1 : -1, dist = 1.0 + pick(3);
    double c[3] = {0, 0, 0}, x[3] = {0, 0, 0}, y[3] = {0, 0, 0};
    c[a] = s * dist;
    x[(a + 1) % 3] = 1;
    y[(a + 2) % 3] = pick(2) ? 1 : -1;
    cam = {c[0], c[1], c[2]};
    ctr = vscale(0.5, cam);
    lx = {x[0], x[1], x[2]};
    ly = {y[0], y[1], y[2]};
  } else {
    cam = {uni(-2, 2), uni(-2, 2), uni(-2, 2)};
    const double r = sqrt(vdot(cam, cam));
    cam = vscale(uni(1.2, 3.0) / r, cam);
    ctr = vscale(uni(0.3, 0.9), cam);
    const V d = vunit(cam), up = {uni(-1, 1), uni(-1, 1), uni(-1, 1)};
    lx = vscale(uni(0.2, 2.0), vunit(vcross(up, d)));
    ly = vscale(uni(0.2, 2.0), vunit(vcross(d, lx)));
    if (kind == 2) ly = vadd(ly, vscale(uni(-0.8, 0.8), lx));
    if (pick(4) == 0) ly = vscale(-1.0, ly);
  }
  const V n = vunit(vcross(lx, ly));
  const double s[5][3] = {{cam.x, cam.y, cam.z}, {ctr.x, ctr.y, ctr.z}, {lx.x, lx.y, lx.z}, {ly.x, ly.y, ly.z},
                          {n.x, n.y, n.z}};
  double* t[5] = {v.cam, v.ctr, v.lx, v.ly, v.nrm};
  for (int q = 0; q < 5; q++)
    for (int d = 0; d < 3; d++) t[q][d] = s[q][d];
  v.nc = vdot(n, cam);
  v.d = vdot(n, ctr);
  v.lxx = vdot(lx, lx);
  v.lyy = vdot(ly, ly);
  v.fw = v.W;
  v.fh = v.H;
  set_pitch(v);
  set_cv(v);
  return v;
}

struct Stats {
  long bricks = 0, cut = 0, regular = 0, triangles = 0, fragments = 0, misses = 0;
};

static void one(int kind, Stats& st) {
  const int n[3] = {1 + pick(4), 1 + pick(4), 1 + pick(4)};
  const double h = std::pow(2.0, -1 - pick(9));
  std::vector<double> g[3];
  for (int d = 0; d < 3; d++) {
    double x = kind == 4 ? -h * 0.5 * n[d] : uni(-0.5, 0.5);
    for (int q = 0; q <= n[d]; q++) {
      g[d].push_back(x);
      x += kind == 4 ? h : h * uni(0.3, 1.7);
    }
    if (pick(5) == 0) g[d] = std::vector<double>(g[d].rbegin(), g[d].rend());
  }
  const double thr = kind == 4 ? 0.0 : uni(-0.3, 0.3);
  // values
  std::vector<double> f(size_t(n[0] + 1) * (n[1] + 1) * (n[2] + 1));
  const double a = uni(-1, 1), b = uni(-1, 1), c = uni(-1, 1), scale = std::pow(10.0, uni(-4, 4));
  const int axis = pick(3);
  auto at = [&](int i, int j, int k) -> double& { return f[(size_t(k) * (n[1] + 1) + j) * (n[0] + 1) + i]; };
  for (int k = 0; k <= n[2]; k++)
    for (int j = 0; j <= n[1]; j++)
      for (int i = 0; i <= n[0]; i++) {
        const int p[3] = {i, j, k};
        double x;
        switch (kind) {
          case 0: x = thr + scale * (a * (i - 0.5 * n[0]) + b * (j - 0.5 * n[1]) + c * (k - 0.5 * n[2]) + 0.3 * uni(-1, 1)); break;
          case 1: x = uni(-1, 1); break;
          case 2: x = pick(3) ? uni(-1, 1) : thr + (pick(4) ? uni(-1, 1) * std::pow(10.0, -pick(18)) : 0.0); break;
          case 3: x = thr + uni(-1, 1) * std::pow(10.0, -pick(18)); break;
          // exact planes through the origin, along an axis or a diagonal
          case 4: x = b > 0 ? g[axis][p[axis]] : g[axis][p[axis]] + (c > 0 ? g[(axis + 1) % 3][p[(axis + 1) % 3]] : -g[(axis + 1) % 3][p[(axis + 1) % 3]]); break;
          case 5: x = (i - 1) + (c > 0 ? j : 0); break;
          default:
            x = uni(-1, 1);
            if (pick(6) == 0) {
              const double bad[4] = {std::numeric_limits<double>::infinity(), -std::numeric_limits<double>::infinity(),
                                     std::numeric_limits<double>::quiet_NaN(), 1.0e300};
              x = bad[pick(4)];
            }
        }
        at(i, j, k) = x;
      }
  const ViewDev<double> v = camera(kind == 4 ? pick(2) : pick(3));
  BrickRange r = {};
  for (int q = 0; q < 8; q++) {
    CornerView o;
    if (!corner_view(v, g[0][q & 1 ? n[0] : 0], g[1][q & 2 ? n[1] : 0], g[2][q & 4 ? n[2] : 0], o)) return;
    if (!q) r = {o.x, o.x, o.y, o.y, o.nr, o.nr, o.size};
    r.x0 = fmin(r.x0, o.x);
    r.x1 = fmax(r.x1, o.x);
    r.y0 = fmin(r.y0, o.y);
    r.y1 = fmax(r.y1, o.y);
    r.n0 = fmin(r.n0, o.nr);
    r.n1 = fmax(r.n1, o.nr);
    r.size = fmax(r.size, o.size);
  }
  BrickLimits lim;
  if (!brick_limits(v, r, lim)) return;
  st.bricks++;
  for (int k = 0; k < n[2]; k++)
    for (int j = 0; j < n[1]; j++)
      for (int i = 0; i < n[0]; i++) {
        double w[8];
        V p[8];
        int code = 0;
        for (int q = 0; q < 8; q++) {
          const int x = i + (q & 1), y = j + ((q >> 1) & 1), z = k + (q >> 2);
          w[q] = at(x, y, z);
          p[q] = {g[0][x], g[1][y], g[2][z]};
          code |= (thr < w[q]) << q;
        }
        if (code == 0 || code == 255) continue;
        st.cut++;
        const double hx = g[0][i + 1] - g[0][i], hy = g[1][j + 1] - g[1][j], hz = g[2][k + 1] - g[2][k];
        const float fx = float(hx), fy = float(hy), fz = float(hz);
        CellValues cv;
        cell_values(w, float(v.cam[0] - g[0][i]) / fx, float(v.cam[1] - g[1][j]) / fy, float(v.cam[2] - g[2][k]) / fz,
                    cv);
        if (!cell_regular(cv, float(w[0] - thr), fabsf(fx * fy * fz) * 0.999999f * lim.scale)) continue;
        st.regular++;
        for (int t = 0; t < 6; t++) {
          int m = 0;
          for (int q = 0; q < 4; q++) m |= ((code >> kTet[t][q]) & 1) << q;
          const bool rev = m >= 8;
          if (rev) m = 15 - m;
          for (int s = 0; s < kNtri[m]; s++) {
            st.triangles++;
            Projected<double> P;
            bool ok = true;
            for (int q = 0; q < 3; q++) {
              const int* e = kPairs[m][s][rev ? 2 - q : q];
              ok = ok && project(v, interp(thr, p[kTet[t][e[0]]], w[kTet[t][e[0]]], p[kTet[t][e[1]]], w[kTet[t][e[1]]]),
                                 P.q[q]);
            }
            if (!ok) continue;
            raster_box(v, P);
            for (int32_t y = P.j0; y <= P.j1; y++)
              for (int32_t x = P.i0; x <= P.i1; x++) {
                double w0, w1, w2;
                if (!pixel_weights(P, pixel_centre<double>(x, v.fw), pixel_centre<double>(y, v.fh), w0, w1, w2))
                  continue;
                st.fragments++;
                const double dep = pixel_depth(P, w0, w1, w2);
                const bool in = x >= lim.i0 && x <= lim.i1 && y >= lim.j0 && y <= lim.j1;
                if (!in || !(dep <= lim.bound)) {
                  if (st.misses++ < 5)
                    std::printf("MISS kind %d pixel (%d, %d) box %d..%d %d..%d depth %.17g bound %.17g\n", kind, x, y,
                                lim.i0, lim.i1, lim.j0, lim.j1, dep, lim.bound);
                }
              }
          }
        }
      }
}

int main(int argc, char** argv) {
  rng.seed(argc > 1 ? uint64_t(std::atoll(argv[1])) : 1);
  const int per = argc > 2 ? std::atoi(argv[2]) : 2000;
  const char* name[] = {"smooth", "noise", "some near", "all near", "edge-on planes", "steps", "not finite"};
  long misses = 0;
  for (int kind = 0; kind < 7; kind++) {
    Stats st;
    for (int q = 0; q < per; q++) one(kind, st);
    std::printf("%s: %ld bricks, %ld cut cells, %ld regular, %ld triangles, %ld fragments, %ld misses\n", name[kind],
                st.bricks, st.cut, st.regular, st.triangles, st.fragments, st.misses);
    misses += st.misses;
  }
  return misses != 0;
}
