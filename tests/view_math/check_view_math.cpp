// CPU check of the arithmetic by which a frame avoids divisions and boxes
// (c3d_geom.h, the header the device kernels use):
//   column_centre / row_centre  equal pixel_centre bit for bit
//   div_const (FP32)            equals the division bit for bit
//   pixel_box                   lies in the reference's box (raster_box) and
//                               holds every pixel that the coverage test accepts
// Usage: check_view_math <seed> <scale>; prints counts, exits 1 on a mismatch.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <random>

#include "c3d_geom.h"

using namespace c3d;

static std::mt19937_64 rng;
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static int32_t whole(double lo, double hi) { return int32_t(std::exp(uni(std::log(lo), std::log(hi)))); }

template <typename R>
static bool same(R a, R b) {
  return std::memcmp(&a, &b, sizeof(R)) == 0 || (a != a && b != b);
}

template <typename R>
static ViewDev<R> image(int32_t W, int32_t H) {
  ViewDev<R> v = {};
  v.W = W;
  v.H = H;
  v.fw = R(double(W));
  v.fh = R(double(H));
  v.lxx = v.lyy = R(1);
  set_pitch(v);
  set_recips(v);
  return v;
}

template <typename R>
static long centres(long n) {
  long bad = 0;
  // every column of small images, then random columns of all sizes
  for (int32_t W = 1; W <= 700; W++) {
    const ViewDev<R> v = image<R>(W, W);
    for (int32_t i = 0; i < W; i++) bad += !same(column_centre(v, i), pixel_centre<R>(i, v.fw)) + !same(row_centre(v, i), pixel_centre<R>(i, v.fh));
  }
  for (long q = 0; q < n; q++) {
    const ViewDev<R> v = image<R>(whole(1, 2147483000), whole(1, 70000));
    const int32_t i = int32_t(uni(0, 1) * v.W), j = int32_t(uni(0, 1) * v.H);
    bad += !same(column_centre(v, i), pixel_centre<R>(i, v.fw)) + !same(row_centre(v, j), pixel_centre<R>(j, v.fh));
  }
  return bad;
}

static float any_float() {
  const uint32_t u = uint32_t(rng());
  float x;
  std::memcpy(&x, &u, 4);
  return x;
}

static long quotients(long n) {
  const float inf = std::numeric_limits<float>::infinity();
  const float special[] = {0.0f, -0.0f, inf, -inf, std::numeric_limits<float>::quiet_NaN(), 1.4e-45f, 1.17549435e-38f, 3.4028235e38f};
  long bad = 0;
  for (long q = 0; q < n; q++) {
    const int kind = int(rng() % 5);
    float a = any_float(), b = any_float();
    if (kind == 1) a = float(uni(-4, 4)), b = float(uni(0.01, 4));
    if (kind == 2) b = float(std::exp(uni(-30, 30)));
    if (kind == 3) a = special[rng() % 8];
    if (kind == 4) b = float(std::exp(uni(-3, 3))), a = b * float(std::exp(uni(-88, -86)));  // near the subnormals
    bad += !same(div_const(a, b, 1.0 / double(b)), a / b);
  }
  return bad;
}

template <typename R>
static long boxes(long n, long& direct) {
  long bad = 0;
  for (long q = 0; q < n; q++) {
    const ViewDev<R> v = image<R>(whole(1, 4000), whole(1, 4000));
    Projected<R> P, T;
    const double cx = uni(-0.7, 0.7), cy = uni(-0.7, 0.7), s = std::pow(10.0, uni(-2, 1.2));
    for (int k = 0; k < 3; k++) {
      P.q[k].x = R(cx + s * uni(-1, 1) / v.W);
      P.q[k].y = R(cy + s * uni(-1, 1) / v.H);
      P.q[k].z = R(-1);
    }
    if (q % 7 == 0) P.q[2] = P.q[1];
    if (q % 7 == 1) {  // next to a line
      const double t = uni(0, 1), f = std::pow(10.0, -uni(0, 14));
      P.q[2].x += R((1 - f)) * (P.q[0].x + R(t) * (P.q[1].x - P.q[0].x) - P.q[2].x);
      P.q[2].y += R((1 - f)) * (P.q[0].y + R(t) * (P.q[1].y - P.q[0].y) - P.q[2].y);
    }
    if (q % 7 == 2)  // on pixel centres
      for (int k = 0; k < 3; k++) {
        P.q[k].x = pixel_centre<R>(int32_t((P.q[k].x + R(0.5)) * v.fw), v.fw);
        P.q[k].y = pixel_centre<R>(int32_t((P.q[k].y + R(0.5)) * v.fh), v.fh);
      }
    if (q % 7 == 3) P.q[0].x *= R(std::pow(10.0, uni(0, 30)));
    if (q % 97 == 0) P.q[q % 3].y = R(q % 2 ? std::numeric_limits<double>::infinity() : std::numeric_limits<double>::quiet_NaN());
    T = P;
    raster_box(v, P);
    pixel_box(v, T);
    if (!same(P.ainv, T.ainv)) bad++;
    const bool some = T.i1 >= T.i0 && T.j1 >= T.j0;
    if (some && (T.i0 < P.i0 || T.i1 > P.i1 || T.j0 < P.j0 || T.j1 > P.j1)) bad++;
    if (!some || T.i0 > P.i0 || T.i1 < P.i1 || T.j0 > P.j0 || T.j1 < P.j1) direct++;
    if (long(P.i1 - P.i0 + 1) * long(P.j1 - P.j0 + 1) > 4096) continue;
    for (int32_t j = P.j0; j <= P.j1; j++)
      for (int32_t i = P.i0; i <= P.i1; i++) {
        R w0, w1, w2;
        if (pixel_weights(P, pixel_centre<R>(i, v.fw), pixel_centre<R>(j, v.fh), w0, w1, w2) &&
            (i < T.i0 || i > T.i1 || j < T.j0 || j > T.j1))
          bad++;
      }
  }
  return bad;
}

int main(int argc, char** argv) {
  rng.seed(argc > 1 ? std::strtoull(argv[1], nullptr, 10) : 1);
  const long n = argc > 2 ? std::atol(argv[2]) : 300000;
  long narrow[2] = {0, 0};
  const long bad[5] = {centres<double>(n), centres<float>(n), quotients(20 * n), boxes<double>(n, narrow[0]),
                       boxes<float>(n, narrow[1])};
  std::printf("mismatches: centres %ld %ld, quotients %ld, boxes %ld %ld; narrowed %ld %ld of %ld\n", bad[0], bad[1],
              bad[2], bad[3], bad[4], narrow[0], narrow[1], n);
  return bad[0] || bad[1] || bad[2] || bad[3] || bad[4] ? 1 : 0;
}
