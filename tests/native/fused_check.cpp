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

struct Shape {
  int N, k, kl, prec;
};
static uint64_t mulm(uint64_t a, uint64_t b, uint64_t p) { return (uint64_t)((unsigned __int128)a * b % p); }

// The digit columns of output row m of block `blk` (T digits, kbs steps of 8
// inputs, of which kbn are used) for the input words in[], as the matrix
// instruction sums them.
static void columns(const uint8_t* blk, int T, int kbs, int kbn, int m, const uint64_t* in, int* S) {
  for (int t = 0; t < 8; ++t) S[t] = 0;
  for (int t = 0; t < T; ++t)
    for (int s = 0; s < 8 * kbn; ++s)
      for (int b = 0; b < 8; ++b) {
        const int lane = m + 16 * (s % 8 / 2), at = s % 2 * 8 + b;
        const int w = (int8_t)blk[(((size_t)t * kbs + s / 8) * 64 + lane) * 16 + at];
        S[t] += w * (int)(int8_t)(uint8_t)((in[s] >> (8 * b)) ^ 0x80);
        expect(S[t] > -(1 << 23) && S[t] < (1 << 23), "digit columns below 2^23");
      }
}
static uint64_t join(int T, const int* S, const ConvOut& o, uint64_t z) {
  auto c = [&](int t) { return S[t]; };
  return T == 6 ? conv_value<6>(c, o, z) : T == 7 ? conv_value<7>(c, o, z) : conv_value<8>(c, o, z);
}
static void conv_is(int T, const int* S, const ConvOut& o, uint64_t z, uint64_t want, const char* what) {
  const uint64_t v = join(T, S, o, z);
  expect(v % o.p == want % o.p, what, "congruent");
  expect((double)v < 1.3 * (double)o.p, what, "below 1.3 p");
  expect(join(8, S, o, z) == v, what, "in eight digits");
}
// Residues below p: random, at the ends, or of bytes at the ends.
static uint64_t sample(std::mt19937_64& rng, uint64_t p, int mode) {
  switch (mode) {
    case 0: return 0;
    case 1: return p - 1;
    case 2: return 0x8080808080808080ull % p;
    case 3: {
      uint64_t v = 0;
      for (int b = 0; b < 8; ++b) v |= (rng() & 1 ? 0xffull : 0) << (8 * b);
      return v % p;
    }
    default: return rng() % p;
  }
}

// ModUp's and ModDown's tables through conv_value against modular sums.
static void conversions(const Shape& sh, const HostParams& H, const FusedTables& F, std::mt19937_64& rng) {
  const int k = H.k, K = H.K;
  const uint64_t* q = H.primes.data();
  int S[8];
  std::vector<uint64_t> in(8 * (size_t)std::max(F.mu_kb, F.md_kb) + 8);
  auto garbage = [&] { for (uint64_t& x : in) x = rng(); };  // rows that no constant meets
  const int Tb = conv_digits((int)H.dprimes[k].nb);
  for (int l : {0, 1, 6, 7, 8, k / 2, k - 1}) {
    if (l >= k) continue;
    for (int mode = 0; mode < 6; ++mode) {
      garbage();
      for (int i = 0; i <= l; ++i) in[i] = sample(rng, q[i], mode);
      for (int j = 0; j < K; ++j) {
        uint64_t want = 0;
        for (int i = 0; i <= l; ++i)
          want = (want + mulm(in[i] % q[k + j], H.qhat_mod_b[((size_t)l * K + j) * k + i], q[k + j])) % q[k + j];
        columns(&F.mu_w[(size_t)l * F.mu_stride + (size_t)(j / 16) * Tb * F.mu_kb * 1024], Tb, F.mu_kb, (l + 8) / 8, j % 16,
                in.data(), S);
        conv_is(Tb, S, F.mu_out[(size_t)l * K + j], 0, want, "ModUp");
      }
    }
  }
  // set k: no rescale; set l: from level l, with the dropped limb as input K
  for (int set : {k, 1, 7, 16, k - 1}) {
    if (set < 1 || set > k) continue;
    for (int mode = 0; mode < 6; ++mode) {
      garbage();
      for (int j = 0; j < K; ++j) in[j] = sample(rng, q[k + j], mode);
      if (set < k) in[K] = sample(rng, q[set], mode);
      for (int i = 0; i < (set < k ? set : k); ++i) {
        const uint64_t p = q[i], f = set < k ? H.md_fin[((size_t)set * k + i) * 2] : H.inv_b_mod_q[2 * i];
        const uint64_t z = sample(rng, p, (mode + i) % 6);
        uint64_t take = set < k ? mulm(in[K] % p, H.inv_ql_mod_qi[((size_t)set * k + i) * 2], p) : 0;
        for (int j = 0; j < K; ++j)
          take = (take + mulm(in[j] % p, mulm(H.bhat_mod_q[((size_t)i * K + j) * 2], f, p), p)) % p;
        columns(&F.md_w[(size_t)set * F.md_stride + (size_t)(i / 16) * 8 * F.md_kb * 1024],
                conv_digits((int)H.dprimes[i / 16 * 16].nb), F.md_kb, F.md_kb, i % 16, in.data(), S);
        conv_is(conv_digits((int)H.dprimes[i / 16 * 16].nb), S, F.md_out[(size_t)set * k + i], z, (z + (p - take)) % p,
                "ModDown");
      }
    }
  }
  // twiddles and the last stage's constants, as the prime's form reads them
  for (int r = 0; r < k + K; ++r) {
    const DevPrime& d = H.dprimes[r];
    for (int dir = 0; dir < 2; ++dir)
      for (int n = 0; n < 50; ++n) {
        const size_t e = (size_t)r * sh.N + rng() % sh.N;
        const uint64_t want = (dir ? H.tw_inv : H.tw_fwd)[2 * e];
        const uint64_t* t = &F.tw[dir][(size_t)r * sh.N * 2];
        if (d.field == FIELD_FP64) {
          const double w = bits_to_double(t[e - (size_t)r * sh.N]);
          expect(std::fabs(w) <= d.fp / 2 && residue((i128)w, d.p) == want, "balanced twiddle");
        } else {
          expect(t[2 * (e - (size_t)r * sh.N)] == want, "twiddle");
        }
      }
  }
}

// Every product whose reduction deviates passes the screen, at the window's edges
// and inside it; products built as in chk_moddown_terms.
static void screen(const HostParams& H, const FusedTables& F, std::mt19937_64& rng) {
  const int k = H.k, K = H.K;
  int deviating = 0;
  for (int i = 0; i < k; ++i) {
    const DevPrime& d = H.dprimes[i];
    const uint64_t thr = d.quirk_thr < d.p ? d.quirk_thr : d.p;
    for (int t = 0; t < 3000; ++t) {
      const int j = (int)(rng() % K);
      const uint64_t b = H.primes[k + j], c = H.bhat_mod_q[((size_t)i * K + j) * 2];
      uint64_t a = rng() % b;
      if (t % 4 && c) {
        const uint64_t edge[4] = {0, d.quirk_lo + rng() % 3 - 1, thr + rng() % 3 - 1,
                                  d.quirk_lo + rng() % (thr > d.quirk_lo ? thr - d.quirk_lo : 1)};
        const uint64_t base = mulm(edge[t % 4] % d.p, inv_mod(c, d.p), d.p);
        const uint64_t most = base < b ? (b - 1 - base) / d.p : 0;
        a = base < b ? base + (t & 8 ? most : most ? rng() % (most + 1) : 0) * d.p : base % b;
      }
      const double al = (double)(a & ((1u << 28) - 1)), ah = (double)(a >> 28);
      const double* e = &F.scr[((size_t)j * 64 + i) * 2];
      const double fine = screen_fine(al, ah, e[0], e[1]);
      const bool half = screen_half(al, ah, e[0], e[1]) <= screen_bound(F.scr_thr[i]);
      const bool in = half && fine - std::floor(fine) < F.scr_thr[i];
      const uint64_t exact = mulm(a, c, d.p);
      const bool dev = ref_barrett(mulhi64(a, c), a * c, d.p, d.mu, (int)d.nb) != exact;
      deviating += dev;
      expect(in || !dev, "deviating product passes the screen");
      expect(in || exact >= thr, "remainder below the threshold passes the screen");
    }
  }
  if (H.prec == 48 || H.prec == 52) expect(deviating > 0, "products that deviate");
}

static void tables() {
  std::mt19937_64 rng(2);
  for (const Shape& s : {Shape{2048, 2, 1, 55}, Shape{2048, 4, 5, 48}, Shape{4096, 9, 7, 52}, Shape{2048, 18, 16, 48},
                         Shape{2048, 30, 31, 48}, Shape{2048, 48, 52, 45}, Shape{2048, 64, 64, 55}, Shape{16384, 10, 15, 45}}) {
    HostParams H;
    FusedTables F;
    if (!build_host_params(s.N, s.k, s.kl, s.prec, &H).empty()) {
      expect(false, "build_host_params");
      continue;
    }
    build_fused_tables(H, &F);
    conversions(s, H, F, rng);
    screen(H, F, rng);
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
  tables();
  std::printf("fused host checks: %d failure(s)\n", failures);
  return failures ? 1 : 0;
}
