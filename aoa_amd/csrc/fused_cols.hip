// Column kernels of the fused key switching (fused.hpp): the column stages of
// both transforms with the basis conversion between or after them.
#include "fused.hpp"

namespace aoa {

// A tile is eight columns (64-byte segments of a row) of all limbs: LDS for 62
// limbs of 128 coefficients, two workgroups a CU.  Wider tiles leave one; 16 limbs
// at a time and three a CU read the constants twice and chain seven barriers:
// ModDown of 64 polynomials at N = 2^16 2.75 ms against 1.75.

// Sums of basis conversions run as products of signed bytes on the matrix
// cores: input byte s of residue i against the digits of 256^s c_ij mod q_j
// (FusedDev::mu_w, md_w).
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int FZ_COLS = 8;               // columns of a tile: 64-byte row segments
constexpr int FZ_TILE = 16 * FZ_COLS;    // coefficients of a tile
constexpr int FZ_PITCH = FZ_TILE + 8;    // LDS words between limbs (limbs of a wave on different banks)
constexpr int FZ_THREADS = 512;

__device__ __forceinline__ int up8(int x) { return (x + 7) & ~7; }

// Orders a wave's LDS accesses: the four threads of a column are lanes of one
// wave, whose LDS instructions run in order, so an exchange between them needs
// no barrier.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A column's values between its two pairs of stages, through its place in LDS:
// from rows 4q + k to q + 4k, or back.
template <bool TO_A, class F>
__device__ __forceinline__ void col_turn(const F& f, typename F::V (&x)[4], uint64_t* t, int q) {
#pragma unroll
  for (int k = 0; k < 4; ++k) t[(TO_A ? 4 * q + k : q + 4 * k) * FZ_COLS] = f.raw(x[k]);
  wave_order();
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = f.raw_in(t[(TO_A ? q + 4 * k : 4 * q + k) * FZ_COLS]);
}

// ------------------------------------------------- conversions by matrix --
// One step of 8 inputs per instruction: lane (n, g) holds the bytes of inputs
// 8 kb + 2 g and + 1 of coefficient n, and of the same inputs' constants for
// output row n; byte - 128 as the signed digit (ConvOut::off makes up for it).
template <int T, int NB>
__device__ __forceinline__ void conv_acc(v4i (&acc)[T][NB], const uint8_t* W, int kbs, int kbn, const uint64_t* tl, int nb0,
                                         int lane) {
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[t][b] = v4i{0, 0, 0, 0};
  const v4i* w = reinterpret_cast<const v4i*>(W) + lane;
  const int n = lane & 15, g = lane >> 4;
#pragma unroll 2
  for (int kb = 0; kb < kbn; ++kb) {
    v4i in[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint64_t* q = tl + (8 * kb + 2 * g) * FZ_PITCH + (nb0 + b) * 16 + n;
      const uint64_t v0 = q[0] ^ 0x8080808080808080ull, v1 = q[FZ_PITCH] ^ 0x8080808080808080ull;
      in[b] = v4i{(int)(uint32_t)v0, (int)(v0 >> 32), (int)(uint32_t)v1, (int)(v1 >> 32)};
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const v4i a = w[(size_t)(t * kbs + kb) * 64];
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[t][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, in[b], acc[t][b], 0, 0, 0);
    }
  }
}

// conv_value of component r.
template <int T, int NB>
__device__ __forceinline__ uint64_t conv_join(const v4i (&acc)[T][NB], int b, int r, const ConvOut& o, uint64_t z) {
  return conv_value<T>([&](int t) { return acc[t][b][r]; }, o, z);
}

__device__ __forceinline__ ConvOut ld_conv(const ConvOut* t) {
  ConvOut o;
  const uint4* s = reinterpret_cast<const uint4*>(t);
  uint4 v[2] = {s[0], s[1]};
  __builtin_memcpy(&o, v, sizeof(o));
  return o;
}

// ------------------------------------------------------------------ ModUp --
// MUL: the item's D (inverse rows of d2) is brought to coefficients; otherwise
// the item's d holds coefficients, whose Q limbs also start their forward NTT
// here.  v_i = x_i (Q_l/q_i)^-1 into LDS, the conversion, the forward columns
// of the special limbs.  32 items at N = 2^16: 540 us (ModUp alone 430 before, the
// inverse and forward column passes 240 and 260); the chain of a workgroup's
// phases bounds it, 0.47 vector instructions a busy CU and cycle.
template <class F, bool MUL>
__device__ __forceinline__ void up_in(const DevParams& P, const FzItem& it, int i, int M, int col, int q, int c,
                                      uint64_t* tl) {
  const DevPrime dp = P.primes[i];
  const F f(dp);
  const uint64_t* src = glob(MUL ? it.D : it.d) + (size_t)i * P.N + col;
  uint64_t* t = tl + i * FZ_PITCH + c;
  typename F::V x[4];
  if constexpr (MUL) {
    const uint64_t* T = P.fz.tw[1] + (size_t)i * P.N * 2;
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = f.raw_in(src[(size_t)(4 * q + k) * M]);
    col_inv_b(f, x, T, q);
    col_turn<true>(f, x, t, q);
    col_inv_a(f, x, T, P.fz.lc_up + 4 * ((size_t)it.level * P.k + i));
#pragma unroll
    for (int k = 0; k < 4; ++k) t[(q + 4 * k) * FZ_COLS] = f.out_last(x[k]);
  } else {
    const uint64_t* T = P.fz.tw[0] + (size_t)i * P.N * 2;
    const tw2 w = reinterpret_cast<const tw2*>(P.inv_qhat)[(size_t)it.level * P.k + i];
    uint64_t v[4];
    with_caller_words<4, false>(f, P.primes, i, [&](auto& words, int k, auto set) {
      const uint64_t u = words(src[(size_t)(q + 4 * k) * M]);
      set(v, mul_shoup(u, w.w, w.q, dp.p));
      set(x, f.in(u));
    }, [&] { col_fwd_a(f, x, T); });
    col_turn<false>(f, x, t, q);
    wave_order();
#pragma unroll
    for (int k = 0; k < 4; ++k) t[(q + 4 * k) * FZ_COLS] = v[k];
    col_fwd_b(f, x, T, q);
    uint64_t* dst = glob(it.XQ) + (size_t)i * P.N + col;
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[(size_t)(4 * q + k) * M] = f.raw(x[k]);
  }
}

template <class F>
__device__ __forceinline__ void up_out(const DevParams& P, const FzItem& it, int j, int M, int col, int q, int c,
                                       uint64_t* tl) {
  const F f(P.primes[P.k + j]);
  const uint64_t* T = P.fz.tw[0] + (size_t)(P.k + j) * P.N * 2;
  typename F::V x[4];
  uint64_t* t = tl + j * FZ_PITCH + c;
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = f.in(t[(q + 4 * k) * FZ_COLS]);
  col_fwd_a(f, x, T);
  col_turn<false>(f, x, t, q);
  col_fwd_b(f, x, T, q);
  uint64_t* dst = glob(it.X) + (size_t)j * P.N + col;
#pragma unroll
  for (int k = 0; k < 4; ++k) dst[(size_t)(4 * q + k) * M] = f.raw(x[k]);
}

// Special limbs 16 jb.. of coefficients 16 nb0..: the conversion into LDS.
template <int T, int NB>
__device__ __forceinline__ void up_conv(const DevParams& P, const FzItem& it, int jb, int nb0, const uint64_t* tl,
                                        uint64_t* to, int lane) {
  const FusedDev& Z = P.fz;
  v4i acc[T][NB];
  const uint8_t* W = Z.mu_w + (size_t)it.level * Z.mu_stride + (size_t)jb * T * Z.mu_kb * 1024;
  conv_acc<T, NB>(acc, W, Z.mu_kb, (it.level + 8) / 8, tl, nb0, lane);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = jb * 16 + 4 * (lane >> 4) + r;
    if (j < P.K) {
      const ConvOut o = ld_conv(Z.mu_out + (size_t)it.level * P.K + j);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        to[j * FZ_PITCH + (nb0 + b) * 16 + (lane & 15)] = conv_join<T, NB>(acc, b, r, o, 0);
    }
  }
}

template <bool MUL, bool ARG>
__global__ __launch_bounds__(FZ_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void k_fz_up(DevParams P, FzItem arg,
                                                                                                  const FzItem* items) {
  extern __shared__ uint64_t fz_lds[];
  const int M = P.N / 16, per = M / FZ_COLS;
  const int w = xcd_chunk_id(blockIdx.x, gridDim.x);
  const FzItem it = fz_item<ARG>(arg, items, w / per);
  const int col0 = (w % per) * FZ_COLS, L = it.level + 1;
  uint64_t* to = fz_lds + up8(L) * FZ_PITCH;
  for (int t = threadIdx.x; t < L * 32; t += FZ_THREADS) {
    const int i = t / 32, q = t / FZ_COLS % 4, c = t % FZ_COLS;
#define CALL(F) up_in<F, MUL>(P, it, i, M, col0 + c, q, c, fz_lds)
    switch (P.primes[i].field) {
      case FIELD_FP64: CALL(FieldFp64); break;
      case FIELD_LAZY: CALL(FieldLazy); break;
      default: CALL(FieldStrict); break;
    }
#undef CALL
  }
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int units = ((P.K + 15) / 16) * 4;
  const bool fp = ld_prime_field(P.primes, P.k) == FIELD_FP64;
  for (int u = wave; u < units; u += FZ_THREADS / 64) {
    if (fp)
      up_conv<6, 2>(P, it, u / 4, (u % 4) * 2, fz_lds, to, lane);
    else
      up_conv<7, 2>(P, it, u / 4, (u % 4) * 2, fz_lds, to, lane);
  }
  __syncthreads();
  for (int t = threadIdx.x; t < P.K * 32; t += FZ_THREADS) {
    const int j = t / 32, q = t / FZ_COLS % 4, c = t % FZ_COLS;
    if (fp)
      up_out<FieldFp64>(P, it, j, M, col0 + c, q, c, to);
    else
      up_out<FieldLazy>(P, it, j, M, col0 + c, q, c, to);
  }
}

// ---------------------------------------------------------------- ModDown --
// Inverse columns of every limb into LDS, the screen, the dropped limb, the
// conversion.  64 polynomials at N = 2^16, L = 30, K = 31: 1.711 ms, 7.0e8 vector
// instructions, 0.72 a busy CU and cycle: issue bound (integer sums before: 1.75 ms
// for ModDown and 1.0 for the column pass).  Of a workgroup's cycles about a third
// each are the columns, the screen and the conversion.
template <class F>
__device__ __forceinline__ void down_in(const DevParams& P, const uint64_t (&u)[4], int pr, const uint64_t* lc, int q,
                                        uint64_t* t) {
  const F f(P.primes[pr]);
  const uint64_t* T = P.fz.tw[1] + (size_t)pr * P.N * 2;
  typename F::V x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = f.raw_in(u[k]);
  col_inv_b(f, x, T, q);
  col_turn<true>(f, x, t, q);
  col_inv_a(f, x, T, lc);
#pragma unroll
  for (int k = 0; k < 4; ++k) t[(q + 4 * k) * FZ_COLS] = f.out_last(x[k]);
}

// f_i (ref(a c) - (a c mod q)) mod q of one product, c = (B/b_j) mod q_i: what
// the reference's reduction of it takes off the result, f_i as in lc_down.
__device__ __forceinline__ uint64_t down_deviation(const DevParams& P, uint64_t a, int i, int j, int set) {
  const DevPrime dq = ld_prime(P.primes, i);
  const tw2 w = ld_tw2(reinterpret_cast<const tw2*>(P.bhat_mod_q) + (size_t)i * P.K, j);
  const tw2 f = i < set && set < P.k ? ld_tw2(reinterpret_cast<const tw2*>(P.md_fin) + (size_t)set * P.k, i)
                                     : ld_tw2(reinterpret_cast<const tw2*>(P.inv_b_mod_q), i);
  const uint64_t x = mul_shoup(a, w.w, w.q, dq.p);
  const uint64_t r = ref_barrett(mulhi64(a, w.w), a * w.w, dq.p, dq.mu, (int)dq.nb);
  return mul_shoup(sub_mod(r, x, dq.p), f.w, f.q, dq.p);
}

// Looks for the products a_j c_ij of the limbs i0 <= i < i0 + NL whose
// remainder may lie in the reference's deviation window and takes what they
// deviate by off the results.  Each product takes two FP64 multiply-adds
// (screen_half); the least of a term's NL halves is compared with the widest
// window.  About one wave in twenty looks closer: at each limb's half word, then
// to 2^-22 (screen_fine), then with the exact formulas.
template <int NL>
__device__ __forceinline__ void down_screen(const DevParams& P, const uint64_t* aux, uint64_t* xq, int i0, int c, int set) {
  const cptr<double> tab = as_const(P.fz.scr) + i0 * 2;
  const cptr<double> thr = as_const(P.fz.scr_thr) + i0;
  double widest = thr[0];
#pragma unroll
  for (int n = 1; n < NL; ++n) widest = __builtin_fmax(widest, thr[n]);
  const uint32_t bound = __builtin_amdgcn_readfirstlane(screen_bound(widest));
  for (int j = 0; j < P.K; ++j) {
    const uint64_t a = aux[j * FZ_PITCH + c];
    const double al = (double)((uint32_t)a & ((1u << 28) - 1)), ah = (double)(uint32_t)(a >> 28);
    const cptr<double> e = tab + (size_t)j * 128;
    uint16_t h[NL], least = 65535;
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      h[n] = screen_half(al, ah, e[2 * n], e[2 * n + 1]);
      least = __builtin_elementwise_min(least, h[n]);
    }
    if (__builtin_amdgcn_ballot_w64(least <= bound)) {
      // opaque, so that this branch's addresses are not carried around the loop
      int jo = j;
      asm volatile("" : "+s"(jo));
#pragma unroll
      for (int n = 0; n < NL; ++n) {
        if (__builtin_amdgcn_ballot_w64(h[n] <= bound)) {
          if (__builtin_amdgcn_fract(screen_fine(al, ah, e[2 * n], e[2 * n + 1])) < thr[n]) {
            const int i = i0 + n;
            uint64_t* x = xq + i * FZ_PITCH + c;
            *x = sub_mod(*x, down_deviation(P, a, i, jo, set), ld_prime_p(P.primes, i));
          }
        }
      }
    }
  }
}

// Limbs 16 ib.. of coefficients 16 nb0..: the conversion and the result
// f_i x_i - sum (xq holds f_i x_i; with a rescale the dropped limb is input K of
// the sum), canonical, + add_i
// (caller data, canonical or not).
template <int T, int NB>
__device__ __forceinline__ void down_out(const DevParams& P, int set, const uint64_t* add, uint64_t* out, int ib, int nb0,
                                         int lout, const uint64_t* aux, const uint64_t* xq, int M, int col0, int lane) {
  const FusedDev& Z = P.fz;
  v4i acc[T][NB];
  conv_acc<T, NB>(acc, Z.md_w + (size_t)set * Z.md_stride + (size_t)ib * 8 * Z.md_kb * 1024, Z.md_kb, Z.md_kb, aux, nb0,
                  lane);
  // addends requested together (none with a rescale)
  uint64_t w[4][NB];
  if (add) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = min(ib * 16 + 4 * (lane >> 4) + r, lout - 1);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int n = (nb0 + b) * 16 + (lane & 15);
        w[r][b] = add[(size_t)i * P.N + (size_t)(n / FZ_COLS) * M + col0 + n % FZ_COLS];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = ib * 16 + 4 * (lane >> 4) + r;
    if (i < lout) {
      const ConvOut o = ld_conv(Z.md_out + (size_t)set * P.k + i);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int n = (nb0 + b) * 16 + (lane & 15);
        uint64_t v = conv_join<T, NB>(acc, b, r, o, xq[i * FZ_PITCH + n]);
        v = csub(v, o.p);
        const size_t at = (size_t)i * P.N + (size_t)(n / FZ_COLS) * M + col0 + n % FZ_COLS;
        if (add) {
          uint64_t a = w[r][b];
          if (__builtin_amdgcn_ballot_w64(a >= o.p)) a = Residues(P.primes[i])(a);
          v = add_mod(v, a, o.p);
        }
        out[at] = v;
      }
    }
  }
}

// The dropped limb's sum for coefficients 16 nb..: one output, so the rows of a
// product are its digits (row n: digit n & 7, by the same constants).  Digits 0..3
// stay in the first 16 lanes, digits 4..7 in the next.
__device__ __forceinline__ v4i down_top_sum(const DevParams& P, int level, const uint64_t* aux, int nb, int lane) {
  const FusedDev& Z = P.fz;
  const int n = lane & 15, g = lane >> 4;
  const uint8_t* W = Z.md_w + (size_t)P.k * Z.md_stride + ((size_t)(level / 16) * 8 + (n & 7)) * Z.md_kb * 1024;
  const v4i* w = reinterpret_cast<const v4i*>(W) + (level & 15) + 16 * g;
  const uint64_t* q = aux + 2 * g * FZ_PITCH + nb * 16 + n;
  v4i acc{0, 0, 0, 0};
#pragma unroll 4
  for (int kb = 0; kb < Z.md_kb; ++kb, q += 8 * FZ_PITCH) {
    const uint64_t v0 = q[0] ^ 0x8080808080808080ull, v1 = q[FZ_PITCH] ^ 0x8080808080808080ull;
    const v4i in{(int)(uint32_t)v0, (int)(v0 >> 32), (int)(uint32_t)v1, (int)(v1 >> 32)};
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[(size_t)kb * 64], in, acc, 0, 0, 0);
  }
  return acc;
}
// ... and the limb itself into input K of the other limbs' sums.
__device__ __forceinline__ void down_top(const DevParams& P, int level, v4i sum, const uint64_t* xq, uint64_t* aux, int nb,
                                         int lane) {
  v4i acc[8][1];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    acc[r][0][0] = sum[r];
    acc[r + 4][0][0] = __shfl(sum[r], (lane & 15) + 16);
  }
  if (lane < 16) {
    const ConvOut o = ld_conv(P.fz.md_out + (size_t)P.k * P.k + level);
    const int n = nb * 16 + lane;
    const uint64_t z = xq[level * FZ_PITCH + n];
    const uint64_t v = conv_join<8, 1>(acc, 0, 0, o, z);  // unused digits are 0
    aux[P.K * FZ_PITCH + n] = csub(v, o.p);
  }
}

__host__ __device__ inline int down_aux_rows(int K) { return (K + 8) & ~7; }

template <bool ARG>
__global__ __launch_bounds__(FZ_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void k_fz_down(DevParams P, FzItem arg,
                                                                                                const FzItem* items) {
  extern __shared__ uint64_t fz_lds[];  // special limbs (and the dropped limb), Q limbs
  const int M = P.N / 16, per = M / FZ_COLS, K = P.K;
  const int w = xcd_chunk_id(blockIdx.x, gridDim.x);
  const FzItem it = fz_item<ARG>(arg, items, w / (2 * per));
  const int y = (w / per) & 1, col0 = (w % per) * FZ_COLS, L = it.level + 1;
  const int rescale = it.rescale, lout = rescale ? it.level : L, set = rescale ? it.level : P.k;
  const uint64_t* p = glob(y ? it.P1 : it.P0) + col0;
  uint64_t* aux = fz_lds;
  uint64_t* xq = aux + down_aux_rows(K) * FZ_PITCH;
  // inverse columns: Q limbs, then from a wave boundary the special limbs
  const int L2 = (L + 1) & ~1, tasks = (L2 + K) * 32;
  const int q = threadIdx.x / FZ_COLS % 4, cc = threadIdx.x % FZ_COLS;
  // the next round's values are requested before this round's are used
  auto load = [&](int t, uint64_t (&u)[4]) {
    const int m = t / 32, row = m < L2 ? min(m, L - 1) : m - L2 + L;
    const uint64_t* s = p + (size_t)row * P.N + cc;
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = s[(size_t)(4 * q + k) * M];
  };
  uint64_t u[4];
  if ((int)threadIdx.x < tasks) load(threadIdx.x, u);
  for (int t = threadIdx.x; t < tasks; t += FZ_THREADS) {
    uint64_t un[4] = {0, 0, 0, 0};
    if (t + FZ_THREADS < tasks) load(t + FZ_THREADS, un);
    const int m = t / 32;
    if (m < L2) {
      if (m < L) {
#define CALL(F) down_in<F>(P, u, m, P.fz.lc_down + 4 * ((size_t)set * P.k + m), q, xq + m * FZ_PITCH + cc)
        switch (P.primes[m].field) {
          case FIELD_FP64: CALL(FieldFp64); break;
          case FIELD_LAZY: CALL(FieldLazy); break;
          default: CALL(FieldStrict); break;
        }
#undef CALL
      }
    } else {
      const int j = m - L2;
      if (ld_prime_field(P.primes, P.k) == FIELD_FP64)
        down_in<FieldFp64>(P, u, P.k + j, P.fz.lc_b + 4 * j, q, aux + j * FZ_PITCH + cc);
      else
        down_in<FieldLazy>(P, u, P.k + j, P.fz.lc_b + 4 * j, q, aux + j * FZ_PITCH + cc);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = un[k];
  }
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  v4i top{0, 0, 0, 0};
  if (rescale) top = down_top_sum(P, it.level, aux, wave, lane);
  if (!P.moddown_exact) {
    // two waves of 64 coefficients for each quarter of the limbs
    const int g = wave >> 1, c = (wave & 1) * 64 + lane, per_g = (L + 3) / 4;
    const int end = min(L, (g + 1) * per_g);
    for (int i = g * per_g; i < end;) {
      const int left = end - i;
      if (left >= 8) {
        down_screen<8>(P, aux, xq, i, c, set);
        i += 8;
        continue;
      }
      switch (left) {
        case 7: down_screen<7>(P, aux, xq, i, c, set); break;
        case 6: down_screen<6>(P, aux, xq, i, c, set); break;
        case 5: down_screen<5>(P, aux, xq, i, c, set); break;
        case 4: down_screen<4>(P, aux, xq, i, c, set); break;
        case 3: down_screen<3>(P, aux, xq, i, c, set); break;
        case 2: down_screen<2>(P, aux, xq, i, c, set); break;
        default: down_screen<1>(P, aux, xq, i, c, set); break;
      }
      break;
    }
    __syncthreads();
  }
  const uint64_t* add = glob(y ? it.add1 : it.add0);
  uint64_t* out = glob(y ? it.out1 : it.out0);
  if (rescale) {
    down_top(P, it.level, top, xq, aux, wave, lane);
    __syncthreads();
  }
  const int units = ((lout + 15) / 16) * 4;
  for (int u = wave; u < units; u += FZ_THREADS / 64) {
    const int ib = u / 4, nb0 = (u % 4) * 2, nb = ld_prime_nb(P.primes, ib * 16);
    if (nb > 56)
      down_out<8, 2>(P, set, add, out, ib, nb0, lout, aux, xq, M, col0, lane);
    else if (nb > 48)
      down_out<7, 2>(P, set, add, out, ib, nb0, lout, aux, xq, M, col0, lane);
    else
      down_out<6, 2>(P, set, add, out, ib, nb0, lout, aux, xq, M, col0, lane);
  }
}

// ---------------------------------------------------------------- launch ---

template <bool ARG>
static void fz_up(const DevParams& P, const FzItem& arg, const FzItem* items, int n, int max_level, bool mul,
                  hipStream_t st) {
  const size_t lds = (size_t)(((max_level + 8) & ~7) + P.K) * FZ_PITCH * 8;
  const dim3 grid((unsigned)(n * (P.N / FZ_TILE)));
  if (mul)
    k_fz_up<true, ARG><<<grid, FZ_THREADS, lds, st>>>(P, arg, items);
  else
    k_fz_up<false, ARG><<<grid, FZ_THREADS, lds, st>>>(P, arg, items);
}

template <bool ARG>
static void fz_down(const DevParams& P, const FzItem& arg, const FzItem* items, int n, int max_level, hipStream_t st) {
  const size_t lds = ((size_t)(down_aux_rows(P.K) + ((max_level + 8) & ~7)) * FZ_PITCH) * 8;
  k_fz_down<ARG><<<dim3((unsigned)(2 * n * (P.N / FZ_TILE))), FZ_THREADS, lds, st>>>(P, arg, items);
}

void fz_up_item(const DevParams& P, const FzItem& it, bool mul, hipStream_t st) {
  fz_up<true>(P, it, nullptr, 1, it.level, mul, st);
}
void fz_down_item(const DevParams& P, const FzItem& it, hipStream_t st) { fz_down<true>(P, it, nullptr, 1, it.level, st); }
void fz_up_desc(const DevParams& P, const FzItem* items, int n, int max_level, bool mul, hipStream_t st) {
  fz_up<false>(P, FzItem{}, items, n, max_level, mul, st);
}
void fz_down_desc(const DevParams& P, const FzItem* items, int n, int max_level, hipStream_t st) {
  fz_down<false>(P, FzItem{}, items, n, max_level, st);
}

int fz_mul(const DevParams& P, const FzItem& it, hipStream_t st) {
  if (fz_rows_item(P, it, st)) return -1;
  fz_up_item(P, it, true, st);
  if (fz_key_item(P, it, st)) return -1;
  fz_down_item(P, it, st);
  return 0;
}

int fz_switch(const DevParams& P, const FzItem& it, hipStream_t st) {
  fz_up_item(P, it, false, st);
  if (fz_key_item(P, it, st)) return -1;
  fz_down_item(P, it, st);
  return 0;
}

}  // namespace aoa
