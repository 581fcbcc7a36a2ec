// Fused key switching on N = 16 x M: HomMul and rotations in three or four
// launches, and the plain transforms on the same split.
//
// A polynomial limb is 16 rows of M = N/16 contiguous elements.  Its forward
// NTT is four stages down the columns (16 values of one thread's registers)
// and log2 M stages along each row (LDS); the inverse runs them backwards.
// Both basis conversions work on one coefficient of every limb, and so do the
// column stages, so the columns are done where the conversions are:
//
//   k_fz_rows  d2 = a1 b1, inverse row stages
//   k_fz_up    inverse columns of d2, ModUp, forward columns of the special limbs
//   k_fz_key   forward rows, both key products, inverse rows
//   k_fz_down  inverse columns of the key products, ModDown, rescale
//
// Output values are those of the reference's sequence
// (aoa-ntt/src/ckks/ckks.cpp:273-358, :982-1009): every step is exact, and the
// ModDown products that the reference's Barrett reduction gets wrong
// (aoa-ntt/src/cuda/manager.cu:331-334) are found and corrected one by one.
#pragma once
#include "fields.hpp"
#include "kernels.hpp"

namespace aoa {

// ------------------------------------------------------------ work lookup --
// ARG: one item given by value, the launch's limbs in order; otherwise entry
// w / per of `list`: item << 8 | limb.
template <bool ARG>
__device__ __forceinline__ FzItem fz_item(const FzItem& arg, const FzItem* items, uint32_t i) {
  if constexpr (ARG) return arg;
  constexpr int W = (int)(sizeof(FzItem) / 8);
  const cptr<uint64_t> w = as_const(reinterpret_cast<const uint64_t*>(items + i));
  uint64_t t[W];
#pragma unroll
  for (int x = 0; x < W; ++x) t[x] = w[x];
  FzItem it;
  __builtin_memcpy(&it, t, sizeof(it));
  return it;
}
template <bool ARG>
__device__ __forceinline__ uint32_t fz_entry(const uint32_t* list, uint32_t i) {
  if constexpr (ARG) return i;
  return as_const(list)[i];
}

// ------------------------------------------------------------------- rows --
// FIELD: the form of every limb of the launch, or FZ_ANY, which looks it up;
// a kernel of one form holds fewer registers.
constexpr int FZ_ANY = -1;
#define FZ_FIELD(pr_, CALL)                                                            \
  switch (FIELD == FZ_ANY ? (int)ld_prime_field(P.primes, pr_) : FIELD) {              \
    case FIELD_FP64: if constexpr (FIELD == FZ_ANY || FIELD == FIELD_FP64) CALL(FieldFp64); break;      \
    case FIELD_LAZY: if constexpr (FIELD == FZ_ANY || FIELD == FIELD_LAZY) CALL(FieldLazy); break;      \
    default: if constexpr (FIELD == FZ_ANY || FIELD == FIELD_STRICT) CALL(FieldStrict); break;          \
  }

// Work item of a workgroup: its index, or with P.xcd_chunks the XCD chunk map.
__device__ __forceinline__ int fz_work(const DevParams& P, int w, int n) { return P.xcd_chunks ? xcd_chunk_id(w, n) : w; }

// Values per thread: four (two stages a round) up to rows of 2048, so that a
// small call's few rows spread over many waves; eight above.  Rows of 2048: the
// product of 11 limbs at N = 2^15 58.4 us with four against 63.1 with eight, a
// batch of 96 the same.  Rows of 4096: a batch of 32 products 4.66 ms with four
// (workgroups of 1024 threads) against 4.16 with eight.
template <int LOGM>
constexpr int kLogV = LOGM <= 11 ? 2 : 3;
template <int LOGM>
using RowOf = Row<LOGM, kLogV<LOGM>>;

template <int LOGM>
struct RowId {
  using G = RowOf<LOGM>;
  int s, row;
  uint32_t off;   // byte offset of the thread's first strided element in its limb
  uint32_t poff;  // of its first packed one
  uint64_t* L;
  __device__ __forceinline__ RowId(int tile, uint64_t* lds) {
    const int rl = G::ROWS == 1 ? 0 : threadIdx.x / G::TS;
    s = G::ROWS == 1 ? threadIdx.x : threadIdx.x % G::TS;
    row = tile * G::ROWS + rl;
    off = (row * G::M + s) * 8;
    poff = (row * G::M + s * G::V) * 8;
    L = lds + rl * G::PITCH;
  }
};

// A zero that the compiler does not see through: what depends on it is formed
// again where it is used instead of staying in registers from one use to the next.
__device__ __forceinline__ uint32_t opaque_zero() {
  uint32_t z = 0;
  asm volatile("" : "+s"(z));
  return z;
}

// The forward rows of x: u, canonical, strided.
template <class F, int LOGM>
__device__ __forceinline__ void rows_fwd_all(const F& f, typename F::V (&x)[RowOf<LOGM>::V],
                                             uint64_t (&u)[RowOf<LOGM>::V], const uint64_t* T, const RowId<LOGM>& id) {
  using G = RowOf<LOGM>;
  row_fwd<LOGM, kLogV<LOGM>>(f, x, T, id.row, id.s, id.L);
#pragma unroll
  for (int k = 0; k < G::V; ++k) id.L[G::template Round<G::ROUNDS - 1>::at(id.s, k)] = f.out(x[k]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < G::V; ++k) u[k] = id.L[G::template Round<0>::at(id.s, k)];
}

// The inverse rows of x (packed) and the store.
template <class F, int LOGM>
__device__ __forceinline__ void rows_out(const F& f, typename F::V (&x)[RowOf<LOGM>::V], const uint64_t* T, uint64_t* dst,
                                         const RowId<LOGM>& id) {
  using G = RowOf<LOGM>;
  constexpr int LV = kLogV<LOGM>;
  const RoundTw<LOGM, LV, G::ROUNDS - 1, F> t(f, T, id.row, id.s);
  row_inv_from<LOGM, LV, G::ROUNDS - 1>(f, x, t, T, id.row, id.s, id.L);
#pragma unroll
  for (int k = 0; k < G::V; ++k) put_byte(dst, id.off + G::TS * 8 * k, f.raw(x[k]));
}

inline int log2_of(int n) {
  int g = 0;
  while ((1 << g) < n) ++g;
  return g;
}

#define FZ_DISPATCH_M(CALL)          \
  switch (log2_of(P.N) - 4) {        \
    case 7: CALL(7); break;          \
    case 8: CALL(8); break;          \
    case 9: CALL(9); break;          \
    case 10: CALL(10); break;        \
    case 11: CALL(11); break;        \
    case 12: CALL(12); break;        \
    default: return -1;              \
  }

}  // namespace aoa
