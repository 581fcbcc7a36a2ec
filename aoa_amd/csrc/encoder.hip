// CKKS encoder on the GPU (FP64): the canonical-embedding FFT and the
// conversions between slot values and residues (aoa-ntt/src/ckks/encoder.cu:33-298).
//
// The FFT follows the reference's loop structure (HEAAN's fftSpecial /
// fftSpecialInv): a bit reversal and log2(n) radix-2 stages whose twiddle
// for butterfly j of a block of length len is exp(+-2 pi i (5^j mod 4 len) /
// (4 len)).  Entry len/2 + j of a direction's table holds it (DevParams::enc_t),
// so a stage's twiddles are consecutive.  The arithmetic is written operation
// by operation with contraction off, so each value is rounded exactly as the
// host loops round it.
#include "device_common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace aoa {

struct cplx {
  double re, im;
};

__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
  const double re = a.re * b.re - a.im * b.im;
  const double im = a.re * b.im + a.im * b.re;
  return cplx{re, im};
}

// In-place bit reversal: the thread of the smaller index of each pair swaps
// it (arrayBitReverse, encoder.cu:11-23); with inv_n != 0 every value is
// also divided by n, the last step of fftSpecialInv (encoder.cu:117-124).
__global__ __launch_bounds__(256) void k_enc_bitrev(cplx* v, int n, int logn, int div) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int j = logn ? (int)(__brev((unsigned)i) >> (32 - logn)) : 0;
  if (i > j) return;
  cplx a = v[i], b = v[j];
  if (div) {
    const double dn = (double)n;
    a = cplx{a.re / dn, a.im / dn};
    b = cplx{b.re / dn, b.im / dn};
  }
  v[i] = b;
  if (i != j) v[j] = a;
}

// fftSpecial's butterfly (encoder.cu:56-70): u = v[a], t = v[b] * ksi; v[a] = u + t, v[b] = u - t.
__device__ __forceinline__ void bfly_fwd(cplx& a, cplx& b, cplx w) {
  const cplx u = a, t = cmul(b, w);
  a = cplx{u.re + t.re, u.im + t.im};
  b = cplx{u.re - t.re, u.im - t.im};
}
// fftSpecialInv's (encoder.cu:96-110): u = v[a] + v[b], t = (v[a] - v[b]) * ksi^-1.
__device__ __forceinline__ void bfly_inv(cplx& a, cplx& b, cplx w) {
  const cplx x = a, y = b;
  a = cplx{x.re + y.re, x.im + y.im};
  b = cmul(cplx{x.re - y.re, x.im - y.im}, w);
}

// Residues of the encoded plaintext on limbs 0..k-1 (encoder.cu:166-221):
// value s (already divided by n) times the scale, truncated to int64, at
// coefficient s*gap (real part) and N/2 + s*gap (imaginary part), zero
// elsewhere; negative values map to p - (|v| mod p).
__global__ __launch_bounds__(256) void k_enc_pack(DevParams P, uint64_t* out, const cplx* u, int slots,
                                                  double scale, int k) {
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (size_t)k * P.N) return;
  const int l = (int)(e >> P.logN);
  const int pos = (int)(e & (size_t)(P.N - 1));
  const int half = P.N / 2, gap = half / slots;
  uint64_t r = 0;
  const int off = pos < half ? pos : pos - half;
  if (off % gap == 0) {
    const int s = off / gap;
    const double x = pos < half ? u[s].re : u[s].im;
    const int64_t v = (int64_t)(x * scale);
    const uint64_t p = P.primes[l].p;
    r = v >= 0 ? (uint64_t)v % p : (p - ((uint64_t)(-v) % p)) % p;
  }
  out[e] = r;
}

// Slot values from limb 0 in the coefficient domain (encoder.cu:223-257):
// the residue x <= p/2 gives x / scale, a larger one (x - p) / scale, both
// converted to double before the subtraction as the reference does.
struct DecodeIn {
  const uint64_t* in;  // limb 0, or null: the values are in memory
  int slots;
  double scale;
};
__device__ __forceinline__ cplx dec_value(const DevParams& P, const DecodeIn& d, int s) {
  const int half = P.N / 2, gap = half / d.slots;
  const uint64_t p = ld_prime_p(P.primes, 0);
  const uint64_t a = d.in[(size_t)s * gap], b = d.in[(size_t)s * gap + half];
  return cplx{a <= (p >> 1) ? (double)a / d.scale : ((double)a - (double)p) / d.scale,
              b <= (p >> 1) ? (double)b / d.scale : ((double)b - (double)p) / d.scale};
}

static int ilog2(int n) {
  int g = 0;
  while ((1 << g) < n) ++g;
  return g;
}

static unsigned blocks(size_t n) { return (unsigned)((n + 255) / 256); }

// The stages of length <= B inside aligned blocks of B <= 4096 values, one
// workgroup of B / 4 threads per block: four values a thread and two stages a
// round (after a first, or before a last, round of one stage if log2 B is odd),
// with one exchange through LDS between rounds, where a thread writes only what
// it read last; each round's twiddles are requested a round earlier.  Latency
// bound: the chain of rounds sets the time (2048 values: 12.0 us with a stage a
// barrier and the twiddles looked up through 5^j, 5.9 now).
// rev: the bit reversal over n values, on the way in (forward) or out
// (inverse, with the division by n: a product with 1/n, exact).
constexpr int kFftBlock = 4096;
__device__ __forceinline__ int fft_pad(int i) { return i + (i >> 2); }
__device__ __forceinline__ int fft_at(int lo, int t, int k) {
  return ((t >> lo) << (lo + 2)) + (t & ((1 << lo) - 1)) + (k << lo);
}
__device__ __forceinline__ int brev(int i, int logn) { return logn ? (int)(__brev((unsigned)i) >> (32 - logn)) : 0; }

template <bool INV>
__global__ __launch_bounds__(kFftBlock / 4) void k_enc_fft(DevParams P, const cplx* src, cplx* dst, int logB, int logn, int rev,
                                                           DecodeIn d) {
  extern __shared__ double fft_lds[];
  const int B = 1 << logB, t = threadIdx.x, base = blockIdx.x << logB;
  double *re = fft_lds, *im = fft_lds + B + (B >> 2);
  const cplx* T = reinterpret_cast<const cplx*>(P.enc_t[INV]);
  const bool on = 4 * t < B;
  cplx x[4], w[3];
  // entry of a round's first stage, then the two of its second (double rounds)
  auto twiddles = [&](int lo, int low) {
    w[0] = T[(1 << lo) + low];
    w[1] = T[(2 << lo) + low];
    w[2] = T[(3 << lo) + low];
  };
  auto exchange = [&](int from, int to) {
    if (on) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = fft_pad(fft_at(from, t, k));
        re[i] = x[k].re;
        im[i] = x[k].im;
      }
    }
    __syncthreads();
    if (on) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = fft_pad(fft_at(to, t, k));
        x[k] = cplx{re[i], im[i]};
      }
    }
  };
  const bool odd = logB & 1;
  if (!INV) {
    if (on) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = 4 * t + k;
        if (i < B) {
          const int s = rev ? brev(base + i, logn) : base + i;
          x[k] = d.in ? dec_value(P, d, s) : src[s];
        }
      }
    }
    int lo = 0;
    if (odd) {
      const cplx w1 = T[1];
      if (on && logB > 1) twiddles(1, t & 1);
      bfly_fwd(x[0], x[1], w1);
      if (logB > 1) {
        bfly_fwd(x[2], x[3], w1);
        exchange(0, 1);
        lo = 1;
      }
    } else if (on && logB > 0) {
      twiddles(0, 0);
    }
    while (logB > 1) {
      const cplx w0 = w[0], w1 = w[1], w2 = w[2];
      const bool last = lo + 2 >= logB;
      if (on && !last) twiddles(lo + 2, t & ((4 << lo) - 1));
      bfly_fwd(x[0], x[1], w0);
      bfly_fwd(x[2], x[3], w0);
      bfly_fwd(x[0], x[2], w1);
      bfly_fwd(x[1], x[3], w2);
      if (last) break;
      exchange(lo, lo + 2);
      lo += 2;
    }
    if (on) {
      if (logB < 2) lo = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = fft_at(lo, t, k);
        if (i < B) dst[base + i] = x[k];
      }
    }
  } else {
    int lo = logB > 2 ? logB - 2 : 0;
    if (on) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = fft_at(lo, t, k);
        if (i < B) x[k] = src[base + i];
      }
      if (logB > 1) twiddles(lo, t & ((1 << lo) - 1));
    }
    while (logB > 1) {
      const cplx w0 = w[0], w1 = w[1], w2 = w[2];
      if (on && lo >= 2) twiddles(lo - 2, t & ((1 << (lo - 2)) - 1));
      bfly_inv(x[0], x[2], w1);
      bfly_inv(x[1], x[3], w2);
      bfly_inv(x[0], x[1], w0);
      bfly_inv(x[2], x[3], w0);
      if (lo < 2) break;
      exchange(lo, lo - 2);
      lo -= 2;
    }
    if (odd) {
      const cplx w1 = T[1];
      if (logB > 1) {
        exchange(1, 0);
        bfly_inv(x[2], x[3], w1);
      }
      bfly_inv(x[0], x[1], w1);
    }
    if (on) {
      const double f = rev ? 1.0 / (double)(1 << logn) : 1.0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = 4 * t + k;
        if (i < B) {
          if (rev)
            dst[brev(base + i, logn)] = cplx{x[k].re * f, x[k].im * f};
          else
            dst[base + i] = x[k];
        }
      }
    }
  }
}

// The last (forward) or first (inverse) three stages of n = 8 B values, eight
// values a thread in registers: a launch for three.  Encoding 2^14 values (with
// the residues): 15 us in three launches, 38 us in five before; decoding them 14
// for 40.
template <bool INV>
__global__ __launch_bounds__(64) void k_enc_outer(DevParams P, const cplx* src, cplx* dst, int B) {
  const int j = blockIdx.x * 64 + threadIdx.x;
  const cplx* T = reinterpret_cast<const cplx*>(P.enc_t[INV]) + j;
  cplx x[8], w[7];
#pragma unroll
  for (int m = 0; m < 8; ++m) x[m] = src[j + (size_t)m * B];
#pragma unroll
  for (int m = 0; m < 7; ++m) w[m] = T[(size_t)(m + 1) * B];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const int h = INV ? 4 >> s : 1 << s;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      if (m & h) continue;
      const cplx tw = w[h - 1 + (m & (h - 1))];
      if (INV)
        bfly_inv(x[m], x[m + h], tw);
      else
        bfly_fwd(x[m], x[m + h], tw);
    }
  }
#pragma unroll
  for (int m = 0; m < 8; ++m) dst[j + (size_t)m * B] = x[m];
}

template <bool INV>
static void fft_blocks(const DevParams& P, const cplx* src, cplx* dst, int n, int rev, const DecodeIn& d, hipStream_t st) {
  const int B = n <= kFftBlock ? n : n / 8;
  const int threads = B / 4 < 64 ? 64 : B / 4;
  k_enc_fft<INV><<<(unsigned)(n / B), threads, (size_t)(B + B / 4) * 16, st>>>(P, src, dst, ilog2(B), ilog2(n), rev, d);
}
template <bool INV>
static void fft_outer(const DevParams& P, const cplx* src, cplx* dst, int n, hipStream_t st) {
  k_enc_outer<INV><<<(unsigned)(n / 8 / 64), 64, 0, st>>>(P, src, dst, n / 8);
}

// A vector of at most 4096 values takes one launch; a longer one the blocks,
// the outer stages and, in place, a bit reversal.
void launch_special_fft(const DevParams& P, double* vals, int n, int inverse, hipStream_t st) {
  cplx* v = reinterpret_cast<cplx*>(vals);
  const DecodeIn none{nullptr, 1, 1.0};
  const bool whole = n <= kFftBlock;
  if (!inverse) {
    if (!whole) k_enc_bitrev<<<blocks(n), 256, 0, st>>>(v, n, ilog2(n), 0);
    fft_blocks<false>(P, v, v, n, whole, none, st);
    if (!whole) fft_outer<false>(P, v, v, n, st);
  } else {
    if (!whole) fft_outer<true>(P, v, v, n, st);
    fft_blocks<true>(P, v, v, n, whole, none, st);
    if (!whole) k_enc_bitrev<<<blocks(n), 256, 0, st>>>(v, n, ilog2(n), 1);
  }
}

// The inverse FFT in place and the residues of its values.  A long vector goes
// through the first limb of the output (at most N/2 values: N words) between
// its two launches, so that the second one's bit reversal meets no other block.
void launch_encode(const DevParams& P, uint64_t* out, double* vals, int slots, double scale, int k, hipStream_t st) {
  cplx* v = reinterpret_cast<cplx*>(vals);
  cplx* src = v;
  if (slots > kFftBlock) {
    src = reinterpret_cast<cplx*>(out);
    fft_outer<true>(P, v, src, slots, st);
  }
  fft_blocks<true>(P, src, v, slots, 1, DecodeIn{nullptr, 1, 1.0}, st);
  k_enc_pack<<<blocks((size_t)k * P.N), 256, 0, st>>>(P, out, v, slots, scale, k);
}

// The blocks read their values from limb 0 in bit-reversed order.
void launch_decode(const DevParams& P, double* vals, const uint64_t* in, int slots, double scale, hipStream_t st) {
  cplx* v = reinterpret_cast<cplx*>(vals);
  fft_blocks<false>(P, nullptr, v, slots, 1, DecodeIn{in, slots, scale}, st);
  if (slots > kFftBlock) fft_outer<false>(P, v, v, slots, st);
}

}  // namespace aoa
