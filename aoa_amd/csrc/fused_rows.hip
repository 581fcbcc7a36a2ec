// Row kernels of the fused key switching (fused.hpp): the forward and inverse
// row stages with the products between them.
#include <type_traits>

#include "fused.hpp"

namespace aoa {

// ------------------------------------------------------ d2 = a b, its rows --
// Memory bound: two operands in, one out.  960 limbs at N = 2^16: 321 us, 4.8
// TB/s of counter traffic (a tensor pass and the inverse pass of d2 before: 370
// and more traffic).
template <class F, int LOGM>
__device__ __forceinline__ void rows_body(const DevParams& P, const uint64_t* a, const uint64_t* b, uint64_t* dst, int pr,
                                          int tile, uint64_t* lds) {
  using G = RowOf<LOGM>;
  constexpr int LV = kLogV<LOGM>;
  const F f(ld_prime(P.primes, pr));
  const uint64_t* T = P.fz.tw[1] + (size_t)pr * P.N * 2;
  const RowId<LOGM> id(tile, lds);
  typename F::V x[G::V];
  with_caller_words<G::V>(f, P.primes, pr, [&](auto& w, int k, auto set) {
    const uint32_t o = id.off + G::TS * 8 * k;
    set(x, f.key(f.in(w(at_byte<uint64_t>(a, o))), w(at_byte<uint64_t>(b, o))));
  });
  row_turn<LOGM, LV, 0, G::ROUNDS - 1>(f, x, id.s, id.L);
  rows_out<F, LOGM>(f, x, T, dst, id);
}

template <int LOGM, bool ARG, int FIELD>
__global__ __launch_bounds__(RowOf<LOGM>::THREADS) void k_fz_rows(DevParams P, FzItem arg, const FzItem* items,
                                                                  const uint32_t* list) {
  __shared__ uint64_t lds[RowOf<LOGM>::LDS];
  constexpr int per = 16 / RowOf<LOGM>::ROWS;
  const int w = fz_work(P, blockIdx.x, gridDim.x);
  const uint32_t e = fz_entry<ARG>(list, w / per);
  const FzItem it = fz_item<ARG>(arg, items, e >> 8);
  const int i = (int)(e & 255), tile = w % per;
  const size_t o = (size_t)i * P.N;
  const uint64_t *a = glob(it.a1) + o, *b = glob(it.b1) + o;
  uint64_t* d = glob(it.D) + o;
#define CALL(F) rows_body<F, LOGM>(P, a, b, d, i, tile, lds)
  FZ_FIELD(i, CALL)
#undef CALL
}

// ---------------------------------------------------------- key products --
// Limb m of an item: Q limbs 0..level, then the special limbs.  HomMul's Q
// limbs take their NTT-domain input d2 and addends d0, d1 from the operands;
// other limbs come as forward columns and take the forward rows here, once for
// both key halves.  BOTH: this
// workgroup forms both key halves, otherwise half y0; a kernel each, since with
// the choice at run time the halves' code and registers added up (hommul at
// N = 2^16, k = 30: 199 us, now 190).

template <class F, int LOGM, bool BOTH>
__device__ __forceinline__ void key_body_tensor(const DevParams& P, const FzItem& it, int m, int tile, int y0,
                                                uint64_t* lds) {
  using G = RowOf<LOGM>;
  constexpr int LV = kLogV<LOGM>;
  const F f(ld_prime(P.primes, m));
  const uint64_t* T = P.fz.tw[1] + (size_t)m * P.N * 2;
  const RowId<LOGM> id(tile, lds);
  const size_t o = (size_t)m * P.N;
  const uint64_t *a0 = glob(it.a0) + o, *a1 = glob(it.a1) + o, *b0 = glob(it.b0) + o, *b1 = glob(it.b1) + o;
  const uint64_t *kb = glob(it.kb) + o, *ka = glob(it.ka) + o;
  const typename F::W bq = f.tw_u(P.fz.bq + 2 * m, 0);
  // both halves' products from one reading of the operands; the second waits
  // in registers while the first is transformed
  typename F::V x[G::V], x1[G::V];
  auto form = [&](auto first, auto second) {
    with_caller_words<G::V>(f, P.primes, m, [&](auto& w, int k, auto set) {
      const uint32_t i = id.off + G::TS * 8 * k;
      const uint64_t va0 = w(at_byte<uint64_t>(a0, i)), va1 = w(at_byte<uint64_t>(a1, i));
      const uint64_t vb0 = w(at_byte<uint64_t>(b0, i)), vb1 = w(at_byte<uint64_t>(b1, i));
      const auto d2 = f.d2(va1, vb1);
      if (first) set(x, f.relin(d2, at_byte<uint64_t>(kb, i), f.d0(va0, vb0), bq));
      if (second) set(x1, f.relin(d2, at_byte<uint64_t>(ka, i), f.d1(va0, va1, vb0, vb1), bq));
    });
  };
  // Which halves, decided once: with a branch per value the loads went out a
  // value at a time (928 limbs of 48 bits at N = 2^16 796 us against 682).
  if constexpr (BOTH)
    form(std::true_type(), std::true_type());
  else if (y0 == 0)
    form(std::true_type(), std::false_type());
  else
    form(std::false_type(), std::true_type());
#pragma unroll 1
  for (int y = BOTH ? 0 : y0; y < (BOTH ? 2 : y0 + 1); ++y) {
    if (y) {
#pragma unroll
      for (int k = 0; k < G::V; ++k) x[k] = x1[k];
    }
    row_turn<LOGM, LV, 0, G::ROUNDS - 1>(f, x, id.s, id.L);
    rows_out<F, LOGM>(f, x, T + opaque_zero(), glob(y ? it.P1 : it.P0) + o, id);
  }
}

// Two words of a key, which need no more than a word's alignment.
struct KeyPair {
  uint64_t a, b;
};

template <class F, int LOGM, bool BOTH>
__device__ __forceinline__ void key_body(const DevParams& P, const FzItem& it, int m, int pr, int tile, int y0,
                                         uint64_t* lds) {
  using G = RowOf<LOGM>;
  constexpr int LV = kLogV<LOGM>;
  const F f(ld_prime(P.primes, pr));
  const int N = P.N, L = it.level + 1;
  const uint64_t* T = P.fz.tw[1] + (size_t)pr * N * 2;
  const RowId<LOGM> id(tile, lds);
  typename F::V x0[G::V];
  const uint64_t* src = m < L ? glob(it.XQ) + (size_t)m * N : glob(it.X) + (size_t)(m - L) * N;
#pragma unroll
  for (int k = 0; k < G::V; ++k) x0[k] = f.raw_in(at_byte<uint64_t>(src, id.off + G::TS * 8 * k));
  row_fwd<LOGM, LV>(f, x0, P.fz.tw[0] + (size_t)pr * N * 2, id.row, id.s, id.L);
#pragma unroll
  for (int k = 0; k < G::V; ++k) x0[k] = f.factor(x0[k]);
#pragma unroll 1
  for (int y = BOTH ? 0 : y0; y < (BOTH ? 2 : y0 + 1); ++y) {
    const uint32_t z = opaque_zero();
    // packed, as the inverse rows begin: a thread's values are 16-byte loads
    const uint64_t* kp = glob(y ? it.ka : it.kb) + (size_t)pr * N;
    typename F::V x[G::V];
#pragma unroll
    for (int k = 0; k < G::V; k += 2) {
      const KeyPair v = at_byte<KeyPair>(kp, id.poff + 8 * k);
      x[k] = f.key(x0[k], v.a);
      x[k + 1] = f.key(x0[k + 1], v.b);
    }
    if (BOTH && y) __syncthreads();  // the first half's last exchange has been read
    rows_out<F, LOGM>(f, x, T + z, glob(y ? it.P1 : it.P0) + (size_t)m * N, id);
  }
}

// Special limbs at N = 2^16 (992 of 55 bits): 826 us, 0.90 vector instructions a
// busy CU and cycle: issue bound.  Q limbs (928 of 48 bits): 667 us, 4.8 TB/s, 47
// for the 32 of q0.  (The split form's row pass took 1.6 ms for all of them and its
// columns 1.0, now in k_fz_down.)
//
// !BOTH: one workgroup per key half (the two halves of a tile `n` blocks apart).
// SPECIAL: every limb is a special one.
template <int LOGM, bool ARG, int FIELD, bool SPECIAL, bool BOTH>
__global__ __launch_bounds__(RowOf<LOGM>::THREADS) __attribute__((amdgpu_waves_per_eu(4))) void k_fz_key(
    DevParams P, FzItem arg, const FzItem* items, const uint32_t* list, int n) {
  __shared__ uint64_t lds[RowOf<LOGM>::LDS];
  constexpr int per = 16 / RowOf<LOGM>::ROWS;
  const int y = BOTH ? 0 : (int)blockIdx.x / n;
  const int w = fz_work(P, BOTH ? (int)blockIdx.x : (int)blockIdx.x % n, n);
  const uint32_t e = fz_entry<ARG>(list, w / per);
  const FzItem it = fz_item<ARG>(arg, items, e >> 8);
  const int m = (int)(e & 255), L = it.level + 1, pr = m < L ? m : P.k + m - L;
  if (!SPECIAL && it.a0 && m < L) {
#define CALL(F) key_body_tensor<F, LOGM, BOTH>(P, it, m, w % per, y, lds)
    FZ_FIELD(pr, CALL)
#undef CALL
  } else {
#define CALL(F) key_body<F, LOGM, BOTH>(P, it, m, pr, w % per, y, lds)
    FZ_FIELD(pr, CALL)
#undef CALL
  }
}

// ---------------------------------------------------------------- launch ---

template <bool ARG, int FIELD>
static int fz_rows(const DevParams& P, const FzItem& arg, const FzItem* items, const uint32_t* list, int n, hipStream_t st) {
  if (n <= 0) return 0;
#define CALL(LM) k_fz_rows<LM, ARG, FIELD><<<dim3(n * 16 / RowOf<LM>::ROWS), RowOf<LM>::THREADS, 0, st>>>(P, arg, items, list)
  FZ_DISPATCH_M(CALL)
#undef CALL
  return 0;
}

// One workgroup per key half while both halves together leave the chip
// partly idle: the forward rows are then done twice, on idle units.  With and
// without: 7.3 and 10.3 us (N = 2^13, 288 waves), 10.2 and 12.7 (N = 2^14, 1088),
// 24.6 and 21.2 (N = 2^15, 3584), 90 and 74 (N = 2^16, 7808).
template <bool ARG, int FIELD, bool SPECIAL>
static int fz_key(const DevParams& P, const FzItem& arg, const FzItem* items, const uint32_t* list, int n, hipStream_t st) {
  if (n <= 0) return 0;
#define CALL(LM)                                                                                                       \
  {                                                                                                                    \
    const int blocks = n * 16 / RowOf<LM>::ROWS;                                                                       \
    if (blocks * (RowOf<LM>::THREADS / 64) <= 2048)                                                                    \
      k_fz_key<LM, ARG, FIELD, SPECIAL, false>                                                                         \
          <<<dim3(2 * blocks), RowOf<LM>::THREADS, 0, st>>>(P, arg, items, list, blocks);                              \
    else                                                                                                               \
      k_fz_key<LM, ARG, FIELD, SPECIAL, true>                                                                          \
          <<<dim3(blocks), RowOf<LM>::THREADS, 0, st>>>(P, arg, items, list, blocks);                                  \
  }
  FZ_DISPATCH_M(CALL)
#undef CALL
  return 0;
}

int fz_rows_item(const DevParams& P, const FzItem& it, hipStream_t st) {
  return fz_rows<true, FZ_ANY>(P, it, nullptr, nullptr, it.level + 1, st);
}
int fz_key_item(const DevParams& P, const FzItem& it, hipStream_t st) {
  return fz_key<true, FZ_ANY, false>(P, it, nullptr, nullptr, it.level + 1 + P.K, st);
}
int fz_rows_desc(const DevParams& P, const FzItem* items, const uint32_t* list, int n, int nstrict, int field,
                 hipStream_t st) {
  const FzItem z{};
  if (nstrict < 0) return fz_rows<false, FZ_ANY>(P, z, items, list, n, st);
  if (fz_rows<false, FIELD_STRICT>(P, z, items, list, nstrict, st)) return -1;
  if (field == FIELD_FP64) return fz_rows<false, FIELD_FP64>(P, z, items, list + nstrict, n - nstrict, st);
  return fz_rows<false, FIELD_LAZY>(P, z, items, list + nstrict, n - nstrict, st);
}
int fz_key_desc(const DevParams& P, const FzItem* items, const uint32_t* list, int n, int nstrict, int field,
                hipStream_t st) {
  const FzItem z{};
  if (nstrict < 0) return fz_key<false, FZ_ANY, false>(P, z, items, list, n, st);
  if (fz_key<false, FIELD_STRICT, false>(P, z, items, list, nstrict, st)) return -1;
  if (field == FIELD_FP64) return fz_key<false, FIELD_FP64, false>(P, z, items, list + nstrict, n - nstrict, st);
  return fz_key<false, FIELD_LAZY, false>(P, z, items, list + nstrict, n - nstrict, st);
}
int fz_key_special_desc(const DevParams& P, const FzItem* items, const uint32_t* list, int n, int field, hipStream_t st) {
  const FzItem z{};
  if (field == FIELD_FP64) return fz_key<false, FIELD_FP64, true>(P, z, items, list, n, st);
  return fz_key<false, FIELD_LAZY, true>(P, z, items, list, n, st);
}

}  // namespace aoa
