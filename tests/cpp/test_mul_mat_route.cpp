// Which kernels mtg_q8_mul_mat_dev launches, on the fake HIP runtime: the one-launch
// product where it may run, else the general path (conversion into a panel, then the
// product). k_mul_mat's workgroups read every row of x for themselves while others
// already store y, so operands that overlap belong on the general path, whose first
// launch has converted all of x before the second one writes y.
#include "fake_hip.hpp"

#include <cstdio>
#include <vector>

#include "mtg_verify.h"

static int failures = 0;
static void expect(bool ok, const char* what, long a = 0, long b = 0) {
  if (ok) return;
  std::fprintf(stderr, "%s (%ld, %ld)\n", what, a, b);
  ++failures;
}

struct Matrix {
  mtg_q8_packed* w = nullptr;
  Matrix(int k, int n) {
    std::vector<uint8_t> raw((size_t)n * (k / 32) * 34, 0);
    expect(mtg_q8_pack(raw.data(), k, n, &w) == MTG_OK, "pack", k, n);
  }
  ~Matrix() { mtg_q8_free(w); }
};
// 1: the one-launch kernel alone, 2: the general path alone
static int route(const Matrix& m, const float* x, int T, float* y) {
  fake::state().launches.clear();
  expect(mtg_q8_mul_mat_dev(m.w, x, T, y) == MTG_OK, "product", T);
  const int one = fake::count("k_mul_mat"), all = (int)fake::state().launches.size();
  return one == 1 && all == 1 ? 1 : one == 0 && all == 2 ? 2 : -1;
}

static void overlap() {
  const int k = 1024, n = 1024, other = 512;
  Matrix square(k, n), narrow(k, other);
  std::vector<float> buf(4 * 16 * 1024 + 4);
  float* at = (float*)(((uintptr_t)buf.data() + 15) & ~(uintptr_t)15);
  const int Ts[] = {1, 8, 9, 16};
  for (int T : Ts) {
    const int xs = T * k, ys = T * n, ns = T * other;
    expect(route(square, at, T, at + xs) == 1, "y behind x", T);
    expect(route(square, at + ys, T, at) == 1, "y ahead of x", T);
    expect(route(square, at, T, at) == 2, "y is x", T);
    expect(route(square, at, T, at + xs - 4) == 2, "y begins in x", T);
    expect(route(square, at + ys - 4, T, at) == 2, "y ends in x", T);
    expect(route(narrow, at, T, at + 4) == 2, "y inside x", T);
    expect(route(narrow, at + ns, T, at) == 1, "narrow y ahead of x", T);
    expect(route(narrow, at, T, at + xs) == 1, "narrow y behind x", T);
  }
}

// Panels of which a CU holds three, two or one: the one-launch kernel as long as all
// tiles' workgroups are on the chip at once, or for a few short rows.
static void large_panels() {
  const struct {
    int k, n, T, route;
  } cases[] = {{4160, 4096, 16, 1}, {4160, 4112, 16, 2}, {4096, 8192, 16, 1}, {5120, 4096, 9, 1},  {5120, 6144, 9, 2},
               {7168, 4096, 16, 1}, {7168, 8192, 16, 2}, {7168, 8192, 8, 1},  {8640, 8192, 7, 1},  {8704, 4096, 8, 1},
               {8704, 4112, 8, 2},  {9216, 8192, 8, 2},  {11264, 8192, 1, 1}, {12288, 8192, 1, 2}, {9216, 8192, 2, 1},
               {10240, 8192, 2, 2}, {14336, 4096, 8, 1}, {14336, 4112, 1, 2}, {4288, 8208, 1, 2}};
  for (const auto& c : cases) {
    Matrix m(c.k, c.n);
    std::vector<float> x((size_t)c.T * c.k + 4), y((size_t)c.T * c.n + 4);
    float* xa = (float*)(((uintptr_t)x.data() + 15) & ~(uintptr_t)15);
    float* ya = (float*)(((uintptr_t)y.data() + 15) & ~(uintptr_t)15);
    const int r = route(m, xa, c.T, ya);
    if (r != c.route) std::fprintf(stderr, "K %d N %d: ", c.k, c.n);
    expect(r == c.route, "route of T", c.T, r);
  }
}

// The LDS limit of the kernel is one value per process: another thread's call between
// this one's setting of it and its launch. A launch or an attribute that is refused
// sends the call to the general path and leaves no error behind.
static void limits() {
  const int n = 32, T = 16;
  Matrix large(7168, n), small(4160, n);
  std::vector<float> x(T * 7168 + 4), y(T * n + 4), y2(T * n + 4);
  auto at = [](std::vector<float>& v) { return (float*)(((uintptr_t)v.data() + 15) & ~(uintptr_t)15); };
  fake::State& f = fake::state();
  bool inside = false;
  int other = -1;
  f.attribute_set = [&] {
    if (inside) return;
    inside = true;
    other = mtg_q8_mul_mat_dev(small.w, at(x), T, at(y2));
  };
  f.launches.clear();
  expect(mtg_q8_mul_mat_dev(large.w, at(x), T, at(y)) == MTG_OK && other == MTG_OK, "two calls", other);
  f.attribute_set = nullptr;
  expect(inside && fake::count("k_mul_mat") == 2 && f.launches.size() == 2, "both launch", (long)f.launches.size());
  expect(f.last_error == 0, "an error left behind", f.last_error);

  f.launch_fails = [](const std::string& k) { return k.find("k_mul_mat") != std::string::npos; };
  expect(route(large, at(x), T, at(y)) == 2, "a refused launch");
  f.launch_fails = nullptr;
  expect(f.last_error == 0, "a refused launch leaves an error", f.last_error);
  f.attribute_fails = [](const std::string& k) { return k.find("k_mul_mat") != std::string::npos; };
  expect(route(large, at(x), T, at(y)) == 2, "a refused attribute");
  f.attribute_fails = nullptr;
  expect(f.last_error == 0, "a refused attribute leaves an error", f.last_error);
  f.last_error = 7;  // another call's, which this one does not report as its own
  expect(route(large, at(x), T, at(y)) == 1, "another call's error");
  f.last_error = 0;
}

int main() {
  limits();
  overlap();
  large_panels();
  std::printf("{\"record\": \"mulMatRoute\", \"failures\": %d}\n", failures);
  return failures ? 1 : 0;
}
