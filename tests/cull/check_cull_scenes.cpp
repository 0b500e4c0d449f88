// Brute-force check of c3d_cull.h, as check_cull.cpp's (whose cameras,
// tables and interpolation it uses), on whole scenes moved away from the
// origin, scaled and stretched: lattice spacings down to a few units in the
// last place of the coordinates, where a brick's corners may round onto one
// screen point; lengths and volumes near the ends of single precision; cells
// many times longer on one axis than on another.
// Usage: check_cull_scenes <seed> <bricks per scene and kind> <scene ...>
//   shift:<e>    10^e added to every coordinate
//   scale:<e>    every coordinate times 2^e
//   stretch:<e>  the lattice's x coordinates times 2^e about the camera's
//                axis, the camera and screen left as they are
// Prints one line per scene, exits 1 on a miss.
#include <cstring>

#define main check_cull_main
#include "check_cull.cpp"
#undef main

struct Scene {
  double shift = 0, scale = 1, stretch = 1;
  int wide = 0;
};

static V moved(const Scene& S, V p) {
  return {p.x * S.scale + S.shift, p.y * S.scale + S.shift, p.z * S.scale + S.shift};
}

static ViewDev<double> scene_camera(const Scene& S, int kind) {
  ViewDev<double> v = camera(kind);
  const V cam = moved(S, {v.cam[0], v.cam[1], v.cam[2]}), ctr = moved(S, {v.ctr[0], v.ctr[1], v.ctr[2]});
  const V lx = vscale(S.scale, V{v.lx[0], v.lx[1], v.lx[2]}), ly = vscale(S.scale, V{v.ly[0], v.ly[1], v.ly[2]});
  const V n = {v.nrm[0], v.nrm[1], v.nrm[2]};
  const double s[4][3] = {{cam.x, cam.y, cam.z}, {ctr.x, ctr.y, ctr.z}, {lx.x, lx.y, lx.z}, {ly.x, ly.y, ly.z}};
  double* t[4] = {v.cam, v.ctr, v.lx, v.ly};
  for (int q = 0; q < 4; q++)
    for (int d = 0; d < 3; d++) t[q][d] = s[q][d];
  v.nc = vdot(n, cam);
  v.d = vdot(n, ctr);
  v.lxx = vdot(lx, lx);
  v.lyy = vdot(ly, ly);
  if (S.wide) {
    v.W = S.wide;
    v.H = 1;
    if (pick(2)) std::swap(v.W, v.H);
    v.fw = v.W;
    v.fh = v.H;
  }
  set_pitch(v);
  set_cv(v);
  return v;
}

static void one_scene(const Scene& S, int kind, Stats& st) {
  // small cells of a uniform lattice that a camera along an axis sees edge on
  // through pixel centres, some values near the threshold
  const bool small = kind == 3;
  const int n[3] = {1 + pick(3), 1 + pick(3), 1 + pick(3)};
  const double h = std::pow(2.0, small ? -8 - pick(5) : -2 - pick(13));
  std::vector<double> g[3];
  for (int d = 0; d < 3; d++) {
    double x = small ? -h * 0.5 * n[d] : uni(-0.5, 0.5);
    for (int q = 0; q <= n[d]; q++) {
      g[d].push_back(x * S.scale * (d == 0 ? S.stretch : 1.0) + S.shift);
      x += small ? h : h * uni(0.3, 1.7);
    }
    if (pick(5) == 0) g[d] = std::vector<double>(g[d].rbegin(), g[d].rend());
  }
  const double thr = uni(-0.3, 0.3);
  std::vector<double> f(size_t(n[0] + 1) * (n[1] + 1) * (n[2] + 1));
  const double a = uni(-1, 1), b = uni(-1, 1), c = uni(-1, 1);
  auto at = [&](int i, int j, int k) -> double& { return f[(size_t(k) * (n[1] + 1) + j) * (n[0] + 1) + i]; };
  for (int k = 0; k <= n[2]; k++)
    for (int j = 0; j <= n[1]; j++)
      for (int i = 0; i <= n[0]; i++) {
        double x = thr + a * (i - 0.5 * n[0]) + b * (j - 0.5 * n[1]) + c * (k - 0.5 * n[2]) + 0.3 * uni(-1, 1);
        if (kind == 1) x = uni(-1, 1);
        if (kind == 2) x = pick(3) ? uni(-1, 1) : thr + uni(-1, 1) * std::pow(10.0, -pick(9));
        if (small) x = thr + (pick(2) ? 1 : -1) * (pick(3) ? uni(0.1, 1) : std::pow(10.0, -uni(4.5, 5.95)));
        at(i, j, k) = x;
      }
  const ViewDev<double> v = scene_camera(S, small ? 0 : pick(3));
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
        if (!cell_regular(cv, float(w[0] - thr), cell_volume(hx, hy, hz, lim.scale))) continue;
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
                  if (st.misses++ < 3)
                    std::printf("MISS kind %d pixel (%d, %d) box %d..%d %d..%d depth %.17g bound %.17g\n", kind, x, y,
                                lim.i0, lim.i1, lim.j0, lim.j1, dep, lim.bound);
                }
              }
          }
        }
      }
}

int main(int argc, char** argv) {
  const int per = argc > 2 ? std::atoi(argv[2]) : 2000;
  long misses = 0;
  for (int a = 3; a < argc; a++) {
    rng.seed(uint64_t(std::atoll(argv[1])));
    const char* colon = std::strchr(argv[a], ':');
    if (!colon) return 2;
    const double e = std::atof(colon + 1);
    Scene S;
    if (!std::strncmp(argv[a], "shift:", 6)) S.shift = std::pow(10.0, e);
    else if (!std::strncmp(argv[a], "scale:", 6)) S.scale = std::pow(2.0, e);
    else if (!std::strncmp(argv[a], "stretch:", 8)) S.stretch = std::pow(2.0, e);
    else if (!std::strncmp(argv[a], "wide:", 5)) S.wide = 1 << int(e);
    else return 2;
    Stats st;
    for (int kind = 0; kind < 4; kind++)
      for (int q = 0; q < per; q++) one_scene(S, kind, st);
    std::printf("%s: %ld bricks, %ld cut cells, %ld regular, %ld triangles, %ld fragments, %ld misses\n", argv[a],
                st.bricks, st.cut, st.regular, st.triangles, st.fragments, st.misses);
    misses += st.misses;
  }
  return misses != 0;
}
