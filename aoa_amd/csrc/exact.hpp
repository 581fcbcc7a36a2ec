// FP64 residue arithmetic of the transforms and key products (FieldFp64), in a
// form that the host checks compile too: its exactness rests on bounds.
//
// A residue modulo p <= 2^48 is a signed integer in a double.  a w mod p =
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
#include "modarith.hpp"

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

}  // namespace aoa
