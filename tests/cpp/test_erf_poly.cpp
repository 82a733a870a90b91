// The GELU's erf polynomials (csrc/erf_poly.hpp) against the canonical Maclaurin series
// (in double, the divisions as products with double reciprocals): the same float for
// every 61st float of [0, 3) and every float within 4,096 of the interval bounds.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "../../moss-transcribe.cpp_amd/csrc/erf_poly.hpp"

template <int N>
static double poly(const double (&c)[N], double v) {
  double r = c[0];
  for (int i = 1; i < N; ++i) r = std::fma(r, v, c[i]);
  return r;
}
static double series(double a) {
  const int terms = a < 1.0 ? 28 : (a < 2.0 ? 44 : 60);
  const double a2 = a * a;
  double term = a, sum = 0.0;
  for (int n = 0; n < terms; ++n) {
    sum = sum + term * (1.0 / (double)(2 * n + 1));
    term = -((term * a2) * (1.0 / (double)(n + 1)));
  }
  return sum * 1.1283791670955126;
}
int main() {
  const uint32_t one = 0x3f800000u, two = 0x40000000u, three = 0x40400000u;
  long n = 0, bad = 0;
  auto check = [&](uint32_t b) {
    float z;
    std::memcpy(&z, &b, 4);
    const double a = z;
    const double p = a < 1.0 ? a * poly(mtg::kErfPoly0, a * a)
                     : a < 2.0 ? poly(mtg::kErfPoly1, a - 1.5) : poly(mtg::kErfPoly2, a - 2.5);
    ++n;
    bad += (float)p != (float)series(a);
  };
  for (uint32_t b = 0; b < three; b += 61) check(b);
  const uint32_t edges[] = {one, two, three};
  for (uint32_t e : edges)
    for (uint32_t b = e - 4096; b < e + 4096 && b < three; ++b) check(b);
  for (uint32_t b = 0; b < 4096; ++b) check(b);
  std::printf("{\"record\": \"erfPoly\", \"floats\": %ld, \"differ\": %ld}\n", n, bad);
  return bad ? 1 : 0;
}
