// Arithmetic of the fused kernels whose exactness rests on bounds, in a form that
// the host checks compile too: the FP64 residues of the transforms and key
// products (FieldFp64), the join of a basis conversion's digit columns and the
// screen of ModDown's products.
//
// FP64.  A residue modulo p <= 2^48 is a signed integer in a double.  a w mod p =
// fma(-q, p, h) + l with h = a w rounded, l = a w - h exact, q = rint(h / p).  For
// |a| <= A p and |w| <= p / 2 the quotient is off by at most A p 2^-53 (1/p and
// the product, rounded) and l is at most A p^2 2^-54, so that the result stays within
//     M(A) = 1/2 + 3 A p 2^-54 <= 0.5 + 0.047 A   (times p),
// all integers below 2^53 = 32 p.  A caller's word is below 2^nb < 2 p.
//
// Forward: a stage takes x to x + M(x): 16 of them from 2 stay below 15.8.
// Inverse rows, from 2: a round of R <= 3 stages from E multiplies up to 2^R E <=
// 16, after which inv_reduce brings what was doubled below 0.51; the others left a
// product, M(2^R E): 1.26, 0.98, 0.87 and 0.83 after four rounds of three, less
// after rounds of two.  Inverse columns, from 0.83: the sums reach 3.4 and 6.7, the
// products stay below M(6.7) = 0.82.  The last stage would take 2 x 6.7, and
// M(13.4) is above 1: out_last needs |x| < p.  before_last brings the first of its
// operands below 0.51, and M(7.2) = 0.84.
#pragma once
#include "params.hpp"

#if defined(__HIPCC__)
#define AOA_HDM __host__ __device__ __forceinline__
#else
#define AOA_HDM inline
#endif

namespace aoa {

AOA_HD double bits_to_double(uint64_t x) {
  double d;
  __builtin_memcpy(&d, &x, 8);
  return d;
}
AOA_HD uint64_t double_to_bits(double d) {
  uint64_t x;
  __builtin_memcpy(&x, &d, 8);
  return x;
}

struct Fp64 {
  double p, pinv;
  AOA_HDM Fp64(double p_, double pinv_) : p(p_), pinv(pinv_) {}
  AOA_HDM double in(uint64_t x) const {  // x < 2^52
    return bits_to_double(x | 0x4330000000000000ull) - 4503599627370496.0;
  }
  AOA_HDM double mul(double x, double w) const {
    const double h = x * w, q = __builtin_rint(h * pinv);
    const double l = __builtin_fma(x, w, -h);
    return __builtin_fma(-q, p, h) + l;
  }
  AOA_HDM void fwd(double& a, double& b, double w) const {
    const double v = mul(b, w), u = a;
    a = u + v;
    b = u - v;
  }
  template <int S>
  AOA_HDM void inv(double& a, double& b, double w) const {
    const double u = a, v = b;
    a = u + v;
    b = mul(u - v, w);
  }
  AOA_HDM double before_last(double x) const { return red(x); }
  AOA_HDM void inv_last(double& a, double& b, double w0, double w1) const {
    const double u = a, v = b;
    a = mul(u + v, w0);
    b = mul(u - v, w1);
  }
  AOA_HDM double red(double x) const { return __builtin_fma(-__builtin_rint(x * pinv), p, x); }
  AOA_HDM uint64_t out(double x) const { return out_last(red(x)); }
  // |x| < p -> canonical
  AOA_HDM uint64_t out_last(double x) const {
    x = x < 0 ? x + p : x;
    return double_to_bits(x + 4503599627370496.0) & 0x000fffffffffffffull;
  }
};

// A basis conversion's sum plus z < p modulo p = o.p, in [0, 1.3 p), from its T
// digit columns S(t).  The columns stay below 2^23 (at most 65 x 7 bytes, or 63 x
// 7 + 8, of products of two signed bytes), pairs of them fit 32 bits; z's high word
// is below 2^31.
template <int T, class Columns>
AOA_HD uint64_t conv_value(const Columns& column, const ConvOut& o, uint64_t z) {
  auto S = [&](int t) -> int { return t < T ? column(t < T ? t : 0) : 0; };
  const int A01 = S(0) + S(1) * 256, A23 = S(2) + S(3) * 256, A45 = S(4) + S(5) * 256, A67 = S(6) + S(7) * 256;
  float f = __builtin_fmaf((float)A45 + (float)(int)(z >> 32), o.c_32, __builtin_fmaf((float)A23, o.c_16, o.c_b));
  uint64_t v = o.off + z + (uint64_t)((int64_t)A01 + (int64_t)A23 * 65536);
  uint32_t hi = (uint32_t)A45;
  if (T > 6) {
    f = __builtin_fmaf((float)A67, o.c_48, f);
    hi += (uint32_t)A67 << 16;
  }
  v += (uint64_t)hi << 32;
  return v - (uint64_t)(uint32_t)f * o.p;
}

// The screen of ModDown's products a c mod q, a = al + ah 2^28 < 2^56, for
// remainders below thr q: frac(a c / q) = frac(al c/q + ah frac(2^28 c/q)), e0 and
// e1 the two constants (FusedDev::scr).  Onto 1.5 2^36 + 2^-16 the sum's first 16
// bits (one unit off at most, one unit added) end up in the low half word, which
// is at most screen_bound where the remainder is below thr q.
AOA_HD uint16_t screen_half(double al, double ah, double e0, double e1) {
  return (uint16_t)(uint32_t)double_to_bits(
      __builtin_fma(ah, e1, __builtin_fma(al, e0, 103079215104.0000152587890625)));
}
AOA_HD uint32_t screen_bound(double thr) {
  const uint32_t b = (uint32_t)(thr * 65536.0 + 2.1);
  return b < 65535u ? b : 65535u;
}
// The same to 2^-22 (bias 2^-21; FusedDev::scr_thr holds thr + 2^-20): its fraction
// is below scr_thr there.
AOA_HD double screen_fine(double al, double ah, double e0, double e1) {
  return __builtin_fma(ah, e1, __builtin_fma(al, e0, 4.76837158203125e-07));
}

}  // namespace aoa
