// Host checks of the fused kernels' arithmetic (exact.hpp), compiled with g++ by
// the CPU tests, under the address and undefined-behaviour sanitizers.
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <random>

#include "exact.hpp"
#include "params.hpp"

using namespace aoa;
typedef __int128 i128;

// The fail_in-th allocation of this thread from now on throws (0: none).
static thread_local int fail_in = 0;
void* operator new(size_t n) {
  if (fail_in && --fail_in == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static int failures = 0;
static void expect(bool ok, const char* what, const char* where = "") {
  if (ok) return;
  if (++failures <= 20) std::printf("FAIL %s %s\n", what, where);
}
static uint64_t residue(i128 v, uint64_t p) {
  const i128 r = v % (i128)p;
  return (uint64_t)(r < 0 ? r + p : r);
}
// 1/2 + 3 A p 2^-54, the bound of a product's remainder (times p)
static double M(double A, double p) { return 0.5 + 3 * A * std::ldexp(p, -54); }

// Products at the ends of their operands' ranges: exact, and within M.
static void products(const Fp64& f, uint64_t p, std::mt19937_64& rng) {
  for (int t = 0; t < 4000; ++t) {
    const double A = (const double[]){1, 2, 4, 8, 10, 13.4, 16, 17}[t % 8];
    const int64_t near = (int64_t)(rng() % 4096);
    const double a = (rng() & 1 ? 1 : -1) * (std::floor(A * f.p) - (double)near);
    const double w = (rng() & 1 ? 1 : -1) * (double)((int64_t)(p / 2) - (int64_t)(rng() % 4096));
    const double r = f.mul(a, w);
    expect(std::fabs(r) <= M(A, f.p) * f.p + 1, "product within its bound");
    expect(residue((i128)a * (i128)w - (i128)r, p) == 0, "product exact");
  }
}

// The last stage of the inverse columns: its operands are sums of two values of up
// to eight times what enters the columns (0.83 p), the first after before_last.
static void last_stage(const Fp64& f, uint64_t p, std::mt19937_64& rng) {
  const double top = std::floor(8 * 0.83 * f.p);
  double first = 0;
  for (int t = 0; t < 20000; ++t) {
    const double x = t < 64 ? top - (double)(rng() % (p / 2)) : std::floor((double)(rng() >> 11) * std::ldexp(1.0, -53) * top);
    first = std::max({first, std::fabs(f.before_last(x)), std::fabs(f.before_last(-x))});
  }
  expect(M((first + top) / f.p, f.p) < 1, "last stage's products below p");
  for (int t = 0; t < 4000; ++t) {
    const double sign = rng() & 1 ? 1 : -1;
    const int64_t x0 = (int64_t)(sign * (top - (double)(rng() % 65536))), x2 = (int64_t)(sign * (top - (double)(rng() % 65536)));
    const int64_t n0 = (int64_t)(p / 2) - (int64_t)(rng() % 65536), n1 = -(int64_t)(p / 2) + (int64_t)(rng() % 65536);
    double a = f.before_last((double)x0), b = (double)x2;
    f.inv_last(a, b, (double)n0, (double)n1);
    expect(f.out_last(a) == residue(((i128)x0 + x2) * n0, p) && f.out_last(b) == residue(((i128)x0 - x2) * n1, p),
           "last stage canonical");
  }
}

// The bounds that exact.hpp names, for the largest prime.
static void chains() {
  const double p = std::ldexp(1.0, 48);
  double x = 2, e = 2;
  for (int s = 0; s < 16; ++s) x += M(x, p);
  expect(x < 15.8, "forward stages");
  for (int r = 0; r < 4; ++r) e = std::max(0.51, M(8 * e, p));
  expect(e < 0.83, "inverse rows");
  const double s1 = 2 * e, s2 = 4 * e, s3 = std::max(8 * e, 2 * M(s2, p));
  expect(s3 < 6.7 && std::max({M(s1, p), M(s2, p), M(s3, p)}) < 0.83, "inverse columns");
  expect(M(2 * s3, p) > 1 && M(s3 + 0.51, p) < 0.85, "last stage");
}

static void fp64_forms() {
  std::mt19937_64 rng(1);
  for (int prec : {45, 48}) {
    HostParams H;
    if (!build_host_params(2048, prec == 45 ? 40 : 64, prec == 45 ? 40 : 2, prec, &H).empty()) {
      expect(false, "build_host_params");
      return;
    }
    for (const DevPrime& d : H.dprimes) {
      if (d.field != FIELD_FP64) continue;
      const Fp64 f(d.fp, d.fpinv);
      products(f, d.p, rng);
      last_stage(f, d.p, rng);
    }
  }
}

// parallel_for where the calling thread runs out of memory at its i-th allocation,
// the creation of threads among them: every call is made once, or the exception
// comes back; threads that were created are joined.
static void parallel_for_without_memory() {
  for (int i = 1; i <= 12; ++i) {
    std::atomic<int> calls{0};
    const std::function<void(int)> f = [&](int) { ++calls; };
    bool thrown = false;
    fail_in = i;
    try {
      parallel_for(64, 65536, f);
    } catch (const std::bad_alloc&) {
      thrown = true;
    }
    fail_in = 0;
    expect(thrown || calls == 64, "parallel_for without memory");
  }
}

int main() {
  chains();
  parallel_for_without_memory();
  fp64_forms();
  std::printf("fused host checks: %d failure(s)\n", failures);
  return failures ? 1 : 0;
}
