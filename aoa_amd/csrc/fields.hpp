// Residue arithmetic of the 16 x M transforms and the key products
// (fused_rows.hip, fused_cols.hip, fused_ntt.hip): one form per size of prime,
// behind one interface.
//
//  FieldLazy    p < 2^56: 64-bit residues left below 2^8 p.  A Shoup product
//               takes any 64-bit value and drops the lowest of the quotient's
//               four partial products (result below 4p), so a butterfly needs no
//               conditional correction: 15 vector instructions (compiled alone).
//  FieldFp64    p <= 2^48: signed FP64 integers (exact.hpp).  A butterfly is eight
//               FP64 instructions and its twiddle one double.
//  FieldStrict  wider primes (the 63-bit q0, p = 2^63 - c): 64-bit values, with
//               2^63 = c and a carry out of 64 bits = 2c; below 2p in the inverse.
//
// Bounds (FP64: exact.hpp).  Forward: every stage adds at most 4p, 16 stages stay
// below 72 p.  Inverse: a stage doubles the sums; after each register round
// inv_reduce brings the grown values back below 8p, so that the next four stages
// stay below 128 p.
#pragma once
#include "device_common.hpp"
#include "exact.hpp"

namespace aoa {

// Entry at byte `o` of a wave-uniform base: a 32-bit offset from a scalar
// pointer, which keeps 64-bit addresses out of the vector registers.
template <class T>
__device__ __forceinline__ T at_byte(const void* base, uint32_t o) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o);
}
// The same for a wave-uniform offset, as a scalar load.
template <class T>
__device__ __forceinline__ T at_byte_u(const void* base, uint32_t o) {
  constexpr int W = (int)(sizeof(T) / 8);
  const cptr<uint64_t> w = as_const(reinterpret_cast<const uint64_t*>(reinterpret_cast<const char*>(base) + o));
  uint64_t t[W];
#pragma unroll
  for (int i = 0; i < W; ++i) t[i] = w[i];
  T v;
  __builtin_memcpy(&v, t, sizeof(T));
  return v;
}
__device__ __forceinline__ void put_byte(void* base, uint32_t o, uint64_t v) {
  *reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(base) + o) = v;
}

__device__ __forceinline__ uint32_t mulhi32(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }

// x w mod p in [0, 4p), any x; wq = floor(w 2^64 / p), np = -p mod 2^64.  The
// quotient leaves out the low partial product and the two middle ones' low
// words, so it is at most 3 below floor(x w / p).
__device__ __forceinline__ uint64_t shoup4(uint64_t x, uint64_t w, uint64_t wq, uint64_t np) {
  const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32), g0 = (uint32_t)wq, g1 = (uint32_t)(wq >> 32);
  const uint64_t q = (uint64_t)x1 * g1 + ((uint64_t)mulhi32(x0, g1) + mulhi32(x1, g0));
  const uint32_t q0 = (uint32_t)q, q1 = (uint32_t)(q >> 32);
  const uint32_t w0 = (uint32_t)w, w1 = (uint32_t)(w >> 32), n0 = (uint32_t)np, n1 = (uint32_t)(np >> 32);
  uint64_t acc = (uint64_t)x0 * w0;
  acc = (uint64_t)q0 * n0 + acc;
  // the high words' sum stays in 32 bits (left to itself the compiler widens
  // it into a 64-bit add of a register pair with a zero)
  uint32_t hi;
  asm("v_add3_u32 %0, %1, %2, %3"
      : "=v"(hi)
      : "v"((uint32_t)(acc >> 32)), "v"(x0 * w1 + x1 * w0), "v"(q0 * n1 + q1 * n0));
  return ((uint64_t)hi << 32) | (uint32_t)acc;
}

// u - v + off, off1 = off + 1: without a borrow chain, whose carry would have
// to wait two instructions.
__device__ __forceinline__ uint64_t diff(uint64_t u, uint64_t v, uint64_t off1) { return u + off1 + ~v; }

// x - p where that is not negative, else x: the borrow is the condition.
__device__ __forceinline__ uint64_t csub(uint64_t x, uint64_t p) {
  unsigned b0, b1;
  const uint32_t l = __builtin_subc((uint32_t)x, (uint32_t)p, 0u, &b0);
  const uint32_t h = __builtin_subc((uint32_t)(x >> 32), (uint32_t)(p >> 32), b0, &b1);
  return b1 ? x : ((uint64_t)h << 32) | l;
}

// Words of caller data.  The forms below take values of up to the prime's nb
// bits; aoa_eltwise_scalar leaves wider ones, since it uses its scalar as given.
struct Words {
  uint32_t hi = 0;
  __device__ __forceinline__ uint64_t operator()(uint64_t x) {
    hi |= (uint32_t)(x >> 32);
    return x;
  }
};
// form(w, k, set) for each of a thread's V values, which reads caller data of
// prime pr through w and keeps what it makes of it by set(array, value): with
// Words and, where one of the wave was too wide, again with Residues.  That rare
// loop stays rolled and its results are selected into place: unrolled, its
// registers cost the key products of 928 limbs of 48 bits at N = 2^16 754 us
// instead of 682.  then() follows either way, the first time before the test, so
// that what it loads is requested with the words.  U: pr is the same for the whole
// wave.
template <int V, bool U = true, class F, class Form, class Then>
__device__ __forceinline__ void with_caller_words(const F& f, const DevPrime* primes, int pr, Form&& form, Then&& then) {
  Words w;
#pragma unroll
  for (int k = 0; k < V; ++k) form(w, k, [&](auto& x, auto v) { x[k] = v; });
  then();
  if constexpr (!F::kAnyWord) {
    if (__builtin_amdgcn_ballot_w64(w.hi >> (f.bits() - 32) != 0)) {
      const Residues r(U ? ld_prime(primes, pr) : primes[pr]);
#pragma unroll 1
      for (int k = 0; k < V; ++k) {
        form(r, k, [&](auto& x, auto v) {
#pragma unroll
          for (int c = 0; c < V; ++c) x[c] = c == k ? v : x[c];
        });
      }
      then();
    }
  }
}
template <int V, bool U = true, class F, class Form>
__device__ __forceinline__ void with_caller_words(const F& f, const DevPrime* primes, int pr, Form&& form) {
  with_caller_words<V, U>(f, primes, pr, form, [] {});
}

struct FieldLazy {
  static constexpr bool kAnyWord = false;
  using V = uint64_t;
  struct W {
    uint64_t w, q;
  };
  uint64_t p, np, mu2;
  uint32_t mu32;  // floor(2^64 / p), p > 2^44
  int nb;
  __device__ __forceinline__ explicit FieldLazy(const DevPrime& d)
      : p(d.p), np(0 - d.p), mu2(d.mu2), mu32((uint32_t)(d.mu >> (2 * (int)d.nb - 64))), nb((int)d.nb) {}
  __device__ __forceinline__ int bits() const { return nb; }
  // canonical residue in; raw / raw_in: the 64-bit pattern between two kernels of one path
  __device__ __forceinline__ V in(uint64_t x) const { return x; }
  __device__ __forceinline__ V raw_in(uint64_t x) const { return x; }
  __device__ __forceinline__ uint64_t raw(V x) const { return x; }
  __device__ __forceinline__ W tw(const uint64_t* T, uint32_t i) const {
    const tw2 t = at_byte<tw2>(T, i * 16);
    return W{t.w, t.q};
  }
  __device__ __forceinline__ W tw_u(const uint64_t* T, uint32_t i) const { return at_byte_u<W>(T, i * 16); }
  // entries i .. i + C - 1
  template <int C>
  __device__ __forceinline__ void tws(W (&t)[C], const uint64_t* T, uint32_t i) const {
#pragma unroll
    for (int c = 0; c < C; ++c) t[c] = tw(T, i + c);
  }
  __device__ __forceinline__ V mul(V x, W w) const { return shoup4(x, w.w, w.q, np); }
  __device__ __forceinline__ void fwd(V& a, V& b, W w) const {
    const V v = mul(b, w), u = a;
    a = u + v;
    b = diff(u, v, 4 * p + 1);
  }
  // stage S of an inverse round, values below (8 << S) p
  template <int S>
  __device__ __forceinline__ void inv(V& a, V& b, W w) const {
    const V u = a, v = b;
    a = u + v;
    b = mul(diff(u, v, ((8 * p) << S) + 1), w);
  }
  __device__ __forceinline__ V before_last(V x) const { return x; }
  // the last stage, values below 64p: canonical
  __device__ __forceinline__ void inv_last(V& a, V& b, W w0, W w1) const {
    const V u = a, v = b;
    a = fix4(shoup4(u + v, w0.w, w0.q, np));
    b = fix4(shoup4(diff(u, v, 64 * p + 1), w1.w, w1.q, np));
  }
  __device__ __forceinline__ uint64_t fix4(uint64_t x) const {
    return csub(csub(x, 2 * p), p);
  }
  // any value -> [0, 3p): the quotient from the high word
  __device__ __forceinline__ V red(V x) const {
    const uint32_t q = mulhi32((uint32_t)(x >> 32), mu32);
    return x + (uint64_t)q * np;
  }
  static constexpr int kGrow = 2;  // doublings a value may keep after a round
  __device__ __forceinline__ uint64_t out(V x) const { return fix4(red(x)); }
  __device__ __forceinline__ uint64_t out_last(V x) const { return x; }  // after inv_last
  // factor of two products: canonical
  __device__ __forceinline__ V factor(V x) const { return out(x); }
  __device__ __forceinline__ V add(V a, V b) const { return a + b; }  // up to 2^8 p
  __device__ __forceinline__ V key(V x, uint64_t k) const { return mul_barrett62_lazy(x, k, p, mu2, nb); }
  // HomMul's products d2 = a1 b1, d0 = a0 b0, d1 = a0 b1 + a1 b0 and their
  // relinearisation d2 key + (B mod q) d
  __device__ __forceinline__ V d2(uint64_t a1, uint64_t b1) const { return mul_barrett62(a1, b1, p, mu2, nb); }
  __device__ __forceinline__ V d0(uint64_t a0, uint64_t b0) const { return key(a0, b0); }
  __device__ __forceinline__ V d1(uint64_t a0, uint64_t a1, uint64_t b0, uint64_t b1) const {
    return key(a0, b1) + key(a1, b0);
  }
  __device__ __forceinline__ V relin(V d2, uint64_t k, V d, W bq) const { return key(d2, k) + mul(d, bq); }
};

struct FieldFp64 : Fp64 {
  static constexpr bool kAnyWord = false;
  using V = double;
  using W = double;
  __device__ __forceinline__ explicit FieldFp64(const DevPrime& d) : Fp64(d.fp, d.fpinv) {}
  __device__ __forceinline__ int bits() const { return __builtin_amdgcn_frexp_exp(p); }
  __device__ __forceinline__ V raw_in(uint64_t x) const { return __longlong_as_double((long long)x); }
  __device__ __forceinline__ uint64_t raw(V x) const { return (uint64_t)__double_as_longlong(x); }
  __device__ __forceinline__ W tw(const uint64_t* T, uint32_t i) const { return at_byte<double>(T, i * 8); }
  __device__ __forceinline__ W tw_u(const uint64_t* T, uint32_t i) const { return at_byte_u<double>(T, i * 8); }
  struct alignas(16) Two {
    double a, b;
  };
  template <int C>
  __device__ __forceinline__ void tws(W (&t)[C], const uint64_t* T, uint32_t i) const {  // i a multiple of C
    if constexpr (C == 1) {
      t[0] = tw(T, i);
    } else {
#pragma unroll
      for (int c = 0; c < C; c += 2) {
        const Two v = at_byte<Two>(T, (i + c) * 8);
        t[c] = v.a;
        t[c + 1] = v.b;
      }
    }
  }
  static constexpr int kGrow = 1;
  __device__ __forceinline__ V factor(V x) const { return red(x); }
  __device__ __forceinline__ V add(V a, V b) const { return a + b; }  // up to 17 p
  __device__ __forceinline__ V key(V x, uint64_t k) const { return mul(x, in(k)); }
  __device__ __forceinline__ V d2(uint64_t a1, uint64_t b1) const { return mul(in(a1), in(b1)); }
  __device__ __forceinline__ V d0(uint64_t a0, uint64_t b0) const { return mul(in(a0), in(b0)); }
  __device__ __forceinline__ V d1(uint64_t a0, uint64_t a1, uint64_t b0, uint64_t b1) const {
    return mul(in(a0), in(b1)) + mul(in(a1), in(b0));
  }
  __device__ __forceinline__ V relin(V d2, uint64_t k, V d, W bq) const { return mul(d2, in(k)) + mul(d, bq); }
};

// Of a small call's limbs this one ends last: a butterfly is 32 vector
// instructions compiled alone (a Shoup product and canonical sums: about 45).
struct FieldStrict {
  static constexpr bool kAnyWord = true;
  using V = uint64_t;
  using W = uint64_t;
  uint64_t p;
  uint32_t c, c2;  // p = 2^63 - c, c < 2^26 (build_host_params checks it); 2c
  __device__ __forceinline__ explicit FieldStrict(const DevPrime& d) : p(d.p), c((uint32_t)d.eps), c2(2 * (uint32_t)d.eps) {}
  __device__ __forceinline__ V in(uint64_t x) const { return x; }
  __device__ __forceinline__ V raw_in(uint64_t x) const { return x; }
  __device__ __forceinline__ uint64_t raw(V x) const { return x; }
  __device__ __forceinline__ W tw(const uint64_t* T, uint32_t i) const { return at_byte<uint64_t>(T, i * 16); }
  __device__ __forceinline__ W tw_u(const uint64_t* T, uint32_t i) const { return at_byte_u<uint64_t>(T, i * 16); }
  template <int C>
  __device__ __forceinline__ void tws(W (&t)[C], const uint64_t* T, uint32_t i) const {
#pragma unroll
    for (int k = 0; k < C; ++k) t[k] = tw(T, i + k);
  }
  // x w mod p, any x, w < p: below 2^63 + 2^54, by folding at bit 63 (2^63 = c).
  // x w = z 2^63 + lo with z c = t 2^63 + m (t < 2^27 + 1), s = lo + m < 2^64.
  __device__ __forceinline__ V mul(V x, W w) const {
    constexpr uint64_t M63 = ~0ull >> 1;
    uint64_t hi, lo;
    mul128(x, w, &hi, &lo);
    const uint64_t z = (hi << 1) | (lo >> 63);
    const uint64_t u = (uint64_t)(uint32_t)z * c, v = (z >> 32) * c + (u >> 32);  // z c = v 2^32 + low word of u
    const uint64_t s = (lo & M63) + (((v << 32) & M63) | (uint32_t)u);
    return (uint64_t)((uint32_t)(v >> 31) + (uint32_t)(s >> 63)) * c + (s & M63);
  }
  // u + v and u - v as 64-bit values, v < 2p: a carry is 2^64 = 2c mod p.  No
  // second one: u + v - 2^64 < 2p and u - v + 2^64 > 2c.
  __device__ __forceinline__ V plus(V u, V v) const {
    unsigned b0, b1;
    const uint32_t l = __builtin_addc((uint32_t)u, (uint32_t)v, 0u, &b0);
    const uint32_t h = __builtin_addc((uint32_t)(u >> 32), (uint32_t)(v >> 32), b0, &b1);
    return (((uint64_t)h << 32) | l) + (b1 ? c2 : 0u);
  }
  __device__ __forceinline__ V minus(V u, V v) const {
    unsigned b0, b1;
    const uint32_t l = __builtin_subc((uint32_t)u, (uint32_t)v, 0u, &b0);
    const uint32_t h = __builtin_subc((uint32_t)(u >> 32), (uint32_t)(v >> 32), b0, &b1);
    return (((uint64_t)h << 32) | l) - (b1 ? c2 : 0u);
  }
  // u + v below 2p for u, v < 2p
  __device__ __forceinline__ V add(V u, V v) const {
    unsigned b0, b1, b2, b3;
    const uint32_t l = __builtin_addc((uint32_t)u, (uint32_t)v, 0u, &b0);
    const uint32_t h = __builtin_addc((uint32_t)(u >> 32), (uint32_t)(v >> 32), b0, &b1);
    const uint32_t tl = __builtin_addc(l, c2, 0u, &b2), th = __builtin_addc(h, 0u, b2, &b3);
    return b1 | b3 ? ((uint64_t)th << 32) | tl : ((uint64_t)h << 32) | l;
  }
  __device__ __forceinline__ void fwd(V& a, V& b, W w) const {
    const V v = mul(b, w), u = a;
    a = plus(u, v);
    b = minus(u, v);
  }
  template <int S>
  __device__ __forceinline__ void inv(V& a, V& b, W w) const {
    const V u = a, v = b;
    a = add(u, v);
    b = mul(minus(u, v), w);
  }
  __device__ __forceinline__ V before_last(V x) const { return x; }
  __device__ __forceinline__ void inv_last(V& a, V& b, W w0, W w1) const {
    const V u = a, v = b;
    a = csub(mul(add(u, v), w0), p);
    b = csub(mul(minus(u, v), w1), p);
  }
  __device__ __forceinline__ V red(V x) const { return x; }
  static constexpr int kGrow = 64;
  __device__ __forceinline__ uint64_t out(V x) const {
    return csub((x & (~0ull >> 1)) + (x >> 63 ? c : 0u), p);
  }
  __device__ __forceinline__ uint64_t out_last(V x) const { return x; }  // after inv_last
  __device__ __forceinline__ V factor(V x) const { return x; }
  __device__ __forceinline__ V key(V x, uint64_t k) const { return mul(x, k); }
  __device__ __forceinline__ V d2(uint64_t a1, uint64_t b1) const { return mul(a1, b1); }
  __device__ __forceinline__ V d0(uint64_t a0, uint64_t b0) const { return mul(a0, b0); }
  __device__ __forceinline__ V d1(uint64_t a0, uint64_t a1, uint64_t b0, uint64_t b1) const {
    return add(mul(a0, b1), mul(a1, b0));
  }
  __device__ __forceinline__ V relin(V d2, uint64_t k, V d, W bq) const { return add(mul(d2, k), mul(d, bq)); }
};

// Brings the values that an inverse round of NB stages has doubled more than
// kGrow times back into a butterfly's range.  Value j (its NB active bits)
// left a product at the stage of its highest set bit and was doubled by the
// stages after it; j = 0 was doubled by all.
template <int NB, int V, class F>
__device__ __forceinline__ void inv_reduce(const F& f, typename F::V (&x)[V]) {
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int j = k & ((1 << NB) - 1);
    const int hb = j ? 31 - __builtin_clz(j) : -1;
    if ((j == 0 ? 64 : NB - 1 - hb) >= F::kGrow && F::kGrow < 64) x[k] = f.red(x[k]);
  }
}

// ----------------------------------------------------------------- columns --
// The 16 rows of a column over four threads q = 0..3 of four values: rows q +
// 4k for the first two stages, rows 4q + k for the last two.  T: the prime's
// FusedDev::tw block.  U: T and q are the same for a whole wave.
template <bool U, class F>
__device__ __forceinline__ typename F::W col_tw(const F& f, const uint64_t* T, int i) {
  if constexpr (U) return f.tw_u(T, i);
  return f.tw(T, i);
}
template <bool U, class F>
__device__ __forceinline__ void col_tw2(const F& f, typename F::W (&w)[2], const uint64_t* T, int i) {
  if constexpr (U) {
    w[0] = f.tw_u(T, i);
    w[1] = f.tw_u(T, i + 1);
  } else {
    f.tws(w, T, i);
  }
}
template <bool U = false, class F>
__device__ __forceinline__ void col_fwd_a(const F& f, typename F::V (&x)[4], const uint64_t* T) {
  const typename F::W w1 = col_tw<U>(f, T, 1), w2 = col_tw<U>(f, T, 2), w3 = col_tw<U>(f, T, 3);
  f.fwd(x[0], x[2], w1);
  f.fwd(x[1], x[3], w1);
  f.fwd(x[0], x[1], w2);
  f.fwd(x[2], x[3], w3);
}
template <bool U = false, class F>
__device__ __forceinline__ void col_fwd_b(const F& f, typename F::V (&x)[4], const uint64_t* T, int q) {
  typename F::W w[2];
  const typename F::W w4 = col_tw<U>(f, T, 4 + q);
  col_tw2<U>(f, w, T, 8 + 2 * q);
  f.fwd(x[0], x[2], w4);
  f.fwd(x[1], x[3], w4);
  f.fwd(x[0], x[1], w[0]);
  f.fwd(x[2], x[3], w[1]);
}
template <bool U = false, class F>
__device__ __forceinline__ void col_inv_b(const F& f, typename F::V (&x)[4], const uint64_t* T, int q) {
  typename F::W w[2];
  const typename F::W w4 = col_tw<U>(f, T, 4 + q);
  col_tw2<U>(f, w, T, 8 + 2 * q);
  f.template inv<0>(x[0], x[1], w[0]);
  f.template inv<0>(x[2], x[3], w[1]);
  f.template inv<1>(x[0], x[2], w4);
  f.template inv<1>(x[1], x[3], w4);
}
// Outputs through F::out_last; lc: the last stage's constants.
template <bool U = false, class F>
__device__ __forceinline__ void col_inv_a(const F& f, typename F::V (&x)[4], const uint64_t* T, const uint64_t* lc) {
  const typename F::W w2 = col_tw<U>(f, T, 2), w3 = col_tw<U>(f, T, 3), n0 = col_tw<U>(f, lc, 0), n1 = col_tw<U>(f, lc, 1);
  f.template inv<2>(x[0], x[1], w2);
  f.template inv<2>(x[2], x[3], w3);
  x[0] = f.before_last(x[0]);
  f.inv_last(x[0], x[2], n0, n1);
  f.inv_last(x[1], x[3], n0, n1);
}

// -------------------------------------------------------------------- rows --
// A row of M = 2^LOGM elements on M / V threads of V = 2^LOGV values, in
// register rounds of LOGV stages (the last one what is left) with an exchange
// through LDS between them.  Round I's value j of thread s is the element
// whose bits from LO up are j's, the others s's: strided s + TS j in the first
// round, packed V s + j in the last.
template <int LOGM, int LOGV>
struct Row {
  static constexpr int M = 1 << LOGM, V = 1 << LOGV, TS = M / V;
  static constexpr int ROUNDS = (LOGM + LOGV - 1) / LOGV;
  static constexpr int THREADS = TS < 64 ? 64 : TS, ROWS = THREADS / TS;
  static constexpr int PITCH = M + M / V, LDS = ROWS * PITCH;
  template <int I>
  struct Round {
    static constexpr int D = I * LOGV, R = LOGM - D < LOGV ? LOGM - D : LOGV, LO = LOGM - D - R;
    // a row's twiddles of this round are the same for a whole wave
    static constexpr bool UNIFORM = ROWS == 1 && LO >= 6;
    // LDS word (one word of padding per V): a part of the thread and a constant of j
    static __device__ __forceinline__ int at(int s, int j) {
      if constexpr (LO == 0) return (V + 1) * s + j;
      const int b = ((s >> LO) << (LO + LOGV)) + (s & ((1 << LO) - 1));
      return b + (b >> LOGV) + (j << LO) + (LO >= LOGV ? j << (LO >= LOGV ? LO - LOGV : 0) : j >> (LO >= LOGV ? 0 : LOGV - LO));
    }
  };
};

// The round's twiddles, stage by stage: entry ((16 + row) << (D + r)) + (high << r) + n,
// n < 2^r, for each of the V >> R groups of values.
template <int LOGM, int LOGV, int I, class F>
struct RoundTw {
  using G = Row<LOGM, LOGV>;
  using Q = typename G::template Round<I>;
  static constexpr int GROUPS = G::V >> Q::R, PER = (1 << Q::R) - 1;
  typename F::W w[GROUPS * PER];
  template <int R>
  __device__ __forceinline__ void stage(const F& f, const uint64_t* T, int row, int s) {
    if constexpr (R < Q::R) {
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        const int high = Q::LO == 0 ? s * GROUPS + g : s >> Q::LO;
        uint32_t i = ((16u + row) << (Q::D + R)) + ((uint32_t)high << R);
        typename F::W t[1 << R];
        if constexpr (Q::UNIFORM) {
          i = __builtin_amdgcn_readfirstlane(i);
#pragma unroll
          for (int n = 0; n < (1 << R); ++n) t[n] = f.tw_u(T, i + n);
        } else {
          f.tws(t, T, i);
        }
#pragma unroll
        for (int n = 0; n < (1 << R); ++n) w[g * PER + (1 << R) - 1 + n] = t[n];
      }
      stage<R + 1>(f, T, row, s);
    }
  }
  __device__ __forceinline__ RoundTw(const F& f, const uint64_t* T, int row, int s) { stage<0>(f, T, row, s); }
};

template <int LOGM, int LOGV, int I, class F>
__device__ __forceinline__ void round_fwd(const F& f, typename F::V (&x)[1 << LOGV], const RoundTw<LOGM, LOGV, I, F>& t) {
  using Q = typename Row<LOGM, LOGV>::template Round<I>;
#pragma unroll
  for (int r = 0; r < Q::R; ++r) {
    const int half = 1 << (Q::R - 1 - r);
#pragma unroll
    for (int k = 0; k < (1 << LOGV); ++k)
      if (!(k & half))
        f.fwd(x[k], x[k + half], t.w[(k >> Q::R) * t.PER + (1 << r) - 1 + ((k & ((1 << Q::R) - 1)) >> (Q::R - r))]);
  }
}

template <int LOGM, int LOGV, int I, int S, class F>
__device__ __forceinline__ void round_inv(const F& f, typename F::V (&x)[1 << LOGV], const RoundTw<LOGM, LOGV, I, F>& t) {
  using Q = typename Row<LOGM, LOGV>::template Round<I>;
  if constexpr (S < Q::R) {
    constexpr int r = Q::R - 1 - S, half = 1 << S;
#pragma unroll
    for (int k = 0; k < (1 << LOGV); ++k)
      if (!(k & half))
        f.template inv<S>(x[k], x[k + half],
                          t.w[(k >> Q::R) * t.PER + (1 << r) - 1 + ((k & ((1 << Q::R) - 1)) >> (Q::R - r))]);
    round_inv<LOGM, LOGV, I, S + 1>(f, x, t);
  } else {
    inv_reduce<Q::R>(f, x);
  }
}

// From round A's layout to round B's: out, and in after a barrier.
template <int LOGM, int LOGV, int A, class F>
__device__ __forceinline__ void row_put(const F& f, const typename F::V (&x)[1 << LOGV], int s, uint64_t* L) {
  using G = Row<LOGM, LOGV>;
#pragma unroll
  for (int k = 0; k < G::V; ++k) L[G::template Round<A>::at(s, k)] = f.raw(x[k]);
}
template <int LOGM, int LOGV, int B, class F>
__device__ __forceinline__ void row_get(const F& f, typename F::V (&x)[1 << LOGV], int s, const uint64_t* L) {
  using G = Row<LOGM, LOGV>;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < G::V; ++k) x[k] = f.raw_in(L[G::template Round<B>::at(s, k)]);
}
template <int LOGM, int LOGV, int A, int B, class F>
__device__ __forceinline__ void row_turn(const F& f, typename F::V (&x)[1 << LOGV], int s, uint64_t* L) {
  row_put<LOGM, LOGV, A>(f, x, s, L);
  row_get<LOGM, LOGV, B>(f, x, s, L);
}

// Strided in, packed out.  A thread writes to LDS only where it read last, so
// one barrier per exchange is enough.  Each round's twiddles are requested
// before the round that precedes it.
template <int LOGM, int LOGV, int I, class F>
__device__ __forceinline__ void row_fwd_from(const F& f, typename F::V (&x)[1 << LOGV], const RoundTw<LOGM, LOGV, I, F>& t,
                                             const uint64_t* T, int row, int s, uint64_t* L) {
  if constexpr (I + 1 >= Row<LOGM, LOGV>::ROUNDS) {
    round_fwd<LOGM, LOGV, I>(f, x, t);
  } else {
    const RoundTw<LOGM, LOGV, I + 1, F> n(f, T, row, s);
    round_fwd<LOGM, LOGV, I>(f, x, t);
    row_turn<LOGM, LOGV, I, I + 1>(f, x, s, L);
    row_fwd_from<LOGM, LOGV, I + 1>(f, x, n, T, row, s, L);
  }
}
template <int LOGM, int LOGV, class F>
__device__ __forceinline__ void row_fwd(const F& f, typename F::V (&x)[1 << LOGV], const uint64_t* T, int row, int s,
                                        uint64_t* L) {
  const RoundTw<LOGM, LOGV, 0, F> t(f, T, row, s);
  row_fwd_from<LOGM, LOGV, 0>(f, x, t, T, row, s, L);
}

// Packed in (with the last round's twiddles), strided out.
template <int LOGM, int LOGV, int I, class F>
__device__ __forceinline__ void row_inv_from(const F& f, typename F::V (&x)[1 << LOGV], const RoundTw<LOGM, LOGV, I, F>& t,
                                             const uint64_t* T, int row, int s, uint64_t* L) {
  if constexpr (I == 0) {
    round_inv<LOGM, LOGV, I, 0>(f, x, t);
  } else {
    const RoundTw<LOGM, LOGV, I - 1, F> n(f, T, row, s);
    round_inv<LOGM, LOGV, I, 0>(f, x, t);
    row_turn<LOGM, LOGV, I, I - 1>(f, x, s, L);
    row_inv_from<LOGM, LOGV, I - 1>(f, x, n, T, row, s, L);
  }
}

}  // namespace aoa
