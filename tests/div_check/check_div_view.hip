// GPU check of the divisions by constants of a view (contour3d_amd/csrc/
// c3d_geom.h) as frames make them: set_recips rounds the reciprocals once on
// the host, and div_const and centre_quotient on the device must equal the
// compiler's divisions bit for bit, in FP64 and FP32.
//   div_const        2^23 numerators (any bit pattern; the projections' range;
//                    every exponent; zeros, subnormals, infinities, NaN) against
//                    divisors of a view's range, of every kind of significand
//                    (all ones, next to a power of two, random) and of extreme
//                    and subnormal size
//   centre_quotient  every half-integer numerator i + 1/2 below the extent, for
//                    image extents up to 2^20, and random i of extents up to 2^31
// Prints the counts; exit status 1 on any mismatch.  Built by
// __graft_entry__.build() next to this file.
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>
#include "c3d_geom.h"

template <typename R>
struct Divisor {
  R b;
  double rb;
};

__device__ bool differ(double p, double q) {
  return p != p ? q == q : __double_as_longlong(p) != __double_as_longlong(q);
}
__device__ bool differ(float p, float q) { return p != p ? q == q : __float_as_uint(p) != __float_as_uint(q); }

template <typename R>
__global__ void k_div(const R* a, uint32_t n, const Divisor<R>* d, int nd, unsigned long long* bad) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int k = 0; k < nd; k++) {
    const R b = d[k].b;
    if (differ(c3d::div_const(a[i], b, d[k].rb), a[i] / b)) atomicAdd(bad, 1ull);
  }
}

// numerators i + 1/2, i = first + t * step below the extent
template <typename R>
__global__ void k_centre(Divisor<R> d, uint32_t first, uint32_t step, uint32_t n, unsigned long long* bad) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const R a = R(int32_t(first + t * step)) + R(0.5);
  if (differ(c3d::centre_quotient(a, d.b, d.rb), a / d.b)) atomicAdd(bad, 1ull);
}

#define CHECK(x)            \
  do {                      \
    if (x) {                \
      printf("%s\n", #x);   \
      return 2;             \
    }                       \
  } while (0)

template <typename R>
static Divisor<R> divisor(R b) {
  c3d::ViewDev<R> v = {};
  v.lxx = b;
  v.lyy = v.fw = v.fh = R(1);
  c3d::set_recips(v);
  return {b, v.rlxx};
}

template <typename R>
static int check(const char* name) {
  constexpr int kBits = sizeof(R) == 8 ? 52 : 23, kMin = sizeof(R) == 8 ? -1074 : -149, kMax = sizeof(R) == 8 ? 1023 : 127;
  std::mt19937_64 g(11);
  const uint32_t n = 1u << 23;
  std::vector<R> a(n);
  const R sp[] = {R(0),  R(-0.0), R(1e-310), std::ldexp(R(-1), kMin), std::ldexp(R(1.5), kMax), -std::ldexp(R(1.25), kMax),
                  R(INFINITY), R(-INFINITY), R(NAN), R(1), R(3)};
  const auto significand = [&] { return R(1) + std::ldexp(R(g() >> (64 - kBits)), -kBits); };
  for (uint32_t i = 0; i < n; i++) {
    const uint64_t u = g();
    R x;
    switch (i % 4) {
      case 0: std::memcpy(&x, &u, sizeof(R)); break;
      case 1: x = std::ldexp(significand(), int(g() % 100) - 50); break;
      case 2: x = (u & 1 ? R(-1) : R(1)) * std::ldexp(significand(), int(g() % uint64_t(kMax - kMin + 1)) + kMin); break;
      default: x = sp[u % 11];
    }
    a[i] = x;
  }
  std::vector<R> bs = {R(1), R(3), R(0.7071067811865476), R(1.3333333333333333), R(1920), R(1080), R(2.5e-5), R(7.3e4),
                       std::ldexp(R(1), kMin), std::ldexp(R(3), kMin), std::ldexp(R(1), kMin + kBits), R(INFINITY),
                       std::ldexp(R(1.5), kMax), std::ldexp(R(1), kMax), std::ldexp(R(1.75), kMin / 2)};
  for (int e : {-40, -3, 0, 1, 17, 60}) {
    bs.push_back(std::ldexp(R(2) - std::ldexp(R(1), -kBits), e));  // all ones
    bs.push_back(std::ldexp(R(1) + std::ldexp(R(1), -kBits), e));  // next to a power of two
    bs.push_back(std::ldexp(R(2) - std::ldexp(R(1), 1 - kBits), e));
  }
  for (int k = 0; k < 31; k++) bs.push_back(std::ldexp(significand(), int(g() % 120) - 60));
  std::vector<Divisor<R>> d;
  for (R b : bs) d.push_back(divisor(b));
  R* da;
  Divisor<R>* dd;
  unsigned long long *dbad, bad = 0;
  CHECK(hipMalloc(&da, n * sizeof(R)));
  CHECK(hipMalloc(&dd, d.size() * sizeof(d[0])));
  CHECK(hipMalloc(&dbad, 8));
  CHECK(hipMemcpy(da, a.data(), n * sizeof(R), hipMemcpyHostToDevice));
  CHECK(hipMemcpy(dd, d.data(), d.size() * sizeof(d[0]), hipMemcpyHostToDevice));
  CHECK(hipMemcpy(dbad, &bad, 8, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_div<R>, dim3(n / 256), dim3(256), 0, 0, da, n, dd, int(d.size()), dbad);
  CHECK(hipGetLastError());
  unsigned long long count = (unsigned long long)n * d.size();
  for (int q = 0; q < 400; q++) {
    // extents of every size: all columns of an image, or 2^20 of them from a
    // random first one on
    const uint32_t top = q < 300 ? 1u << 20 : 0x7fffffffu;
    const uint32_t w = q < 40 ? q + 1u : uint32_t(1 + std::exp(std::log(double(top - 1)) * double(g() >> 11) * 0x1p-53));
    const uint32_t step = w >> 20 ? (w >> 20) + 1u : 1u, m = (w - 1u) / step;
    const uint32_t first = step > 1u ? uint32_t(g() % step) : 0u;
    // first + (m - 1) * step < w
    const uint32_t nt = step > 1u ? m : w;
    hipLaunchKernelGGL(k_centre<R>, dim3((nt + 255) / 256), dim3(256), 0, 0, divisor(R(double(w))), first, step, nt, dbad);
    CHECK(hipGetLastError());
    count += nt;
  }
  CHECK(hipDeviceSynchronize());
  CHECK(hipMemcpy(&bad, dbad, 8, hipMemcpyDeviceToHost));
  CHECK(hipFree(da));
  CHECK(hipFree(dd));
  CHECK(hipFree(dbad));
  printf("%s: divisions %llu mismatches %llu\n", name, count, bad);
  return bad != 0;
}

int main() {
  const int r = check<double>("fp64");
  return r ? r : check<float>("fp32");
}
