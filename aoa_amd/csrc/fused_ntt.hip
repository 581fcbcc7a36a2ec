// Plain transforms on N = 16 x M (fused.hpp): a column and a row launch, and
// encryption's and decryption's row stages with their products.
#include "fused.hpp"

namespace aoa {

// Limb l of polynomial blockIdx.y of a launch, or entry l of a table.  FIRST: of
// a transform's first launch; the second one is in place.
struct NtLimb {
  const uint64_t* src;
  uint64_t* dst;
  int pr;
};
template <bool FIRST>
__device__ __forceinline__ NtLimb nt_table(const NttDesc* d, int l) {
  const cptr<uint64_t> w = as_const(reinterpret_cast<const uint64_t*>(d + l));
  return NtLimb{glob((const uint64_t*)w[FIRST ? 0 : 1]), glob((uint64_t*)w[1]), (int)(uint32_t)w[2]};
}
#define NT_LIMB(FIRST, l_)                                                                                  \
  ARG ? NtLimb{(FIRST ? m.src[blockIdx.y] : m.base[blockIdx.y]) + (size_t)(l_) * P.N,                       \
               m.base[blockIdx.y] + (size_t)(l_) * P.N, limb_prime(m, P.k, l_)}                             \
      : nt_table<FIRST>(d, l_)

// ----------------------------------------------------------------- columns --
// Memory bound: 64 columns on 256 threads, where a wave holds one quarter of
// the rows of all of them, so its loads are whole 512-byte row segments and its
// twiddles scalar; the quarters change hands in LDS.  61 limbs at N = 2^16: 13.3
// us, the time of a copy (the split by 256: 22.1 forward, 24.2 inverse).
constexpr int NT_COLS = 64;

template <class F, bool INV>
__device__ __forceinline__ void nt_cols(const DevParams& P, const uint64_t* src, uint64_t* dst, int pr, int q, int c,
                                        uint64_t* lds) {
  const int M = P.N / 16;
  const F f(ld_prime(P.primes, pr));
  const uint64_t* T = P.fz.tw[INV ? 1 : 0] + (size_t)pr * P.N * 2;
  uint64_t* t = lds + c;
  typename F::V x[4];
  if constexpr (INV) {
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = f.raw_in(src[(size_t)(4 * q + k) * M]);
    col_inv_b<true>(f, x, T, q);
  } else {
    with_caller_words<4>(
        f, P.primes, pr, [&](auto& w, int k, auto set) { set(x, f.in(w(src[(size_t)(q + 4 * k) * M]))); },
        [&] { col_fwd_a<true>(f, x, T); });
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) t[(INV ? 4 * q + k : q + 4 * k) * NT_COLS] = f.raw(x[k]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = f.raw_in(t[(INV ? q + 4 * k : 4 * q + k) * NT_COLS]);
  if constexpr (INV) {
    col_inv_a<true>(f, x, T, P.fz.lc + 4 * pr);
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[(size_t)(q + 4 * k) * M] = f.out_last(x[k]);
  } else {
    col_fwd_b<true>(f, x, T, q);
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[(size_t)(4 * q + k) * M] = f.raw(x[k]);
  }
}

template <bool INV, bool ARG>
__global__ __launch_bounds__(256) void k_nt_cols(DevParams P, LimbMap m, const NttDesc* d) {
  constexpr int FIELD = FZ_ANY;
  __shared__ uint64_t lds[16 * NT_COLS];
  const int per = P.logN - 10, li = blockIdx.x >> per;  // log2 of a limb's N / 16 / NT_COLS tiles
  const NtLimb l = NT_LIMB(!INV, li);
  const int q = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), c = threadIdx.x & 63;
  const int col = (blockIdx.x & ((1 << per) - 1)) * NT_COLS + c;
#define CALL(F) nt_cols<F, INV>(P, l.src + col, l.dst + col, l.pr, q, c, lds)
  FZ_FIELD(l.pr, CALL)
#undef CALL
}

// -------------------------------------------------------------------- rows --
// Rows as in the key products' kernel, here between two passes over memory;
// vector work and twiddle latency bound.  61 limbs at N = 2^16: 21.6 us forward
// and 23.1 inverse (25.1 and 28.6 for rows of 256).
template <class F, int LOGM, bool INV>
__device__ __forceinline__ void nt_rows(const DevParams& P, const uint64_t* src, uint64_t* dst, int pr, int tile,
                                        uint64_t* lds) {
  using G = RowOf<LOGM>;
  constexpr int LV = kLogV<LOGM>;
  const RowId<LOGM> id(tile, lds);
  const F f(ld_prime(P.primes, pr));
  const uint64_t* T = P.fz.tw[INV ? 1 : 0] + (size_t)pr * P.N * 2;
  typename F::V x[G::V];
  if constexpr (INV) {
    with_caller_words<G::V>(
        f, P.primes, pr,
        [&](auto& w, int k, auto set) { set(x, f.in(w(at_byte<uint64_t>(src, id.off + G::TS * 8 * k)))); },
        [&] { row_put<LOGM, LV, 0>(f, x, id.s, id.L); });
    row_get<LOGM, LV, G::ROUNDS - 1>(f, x, id.s, id.L);
    rows_out<F, LOGM>(f, x, T, dst, id);
  } else {
    uint64_t u[G::V];
#pragma unroll
    for (int k = 0; k < G::V; ++k) x[k] = f.raw_in(at_byte<uint64_t>(src, id.off + G::TS * 8 * k));
    rows_fwd_all<F, LOGM>(f, x, u, T, id);
#pragma unroll
    for (int k = 0; k < G::V; ++k) put_byte(dst, id.off + G::TS * 8 * k, u[k]);
  }
}

template <int LOGM, bool INV, bool ARG>
__global__ __launch_bounds__(RowOf<LOGM>::THREADS) void k_nt_rows(DevParams P, LimbMap m, const NttDesc* d) {
  constexpr int FIELD = FZ_ANY;
  __shared__ uint64_t lds[RowOf<LOGM>::LDS];
  constexpr int per = 16 / RowOf<LOGM>::ROWS;
  const int li = blockIdx.x / per;
  const NtLimb l = NT_LIMB(INV, li);
#define CALL(F) nt_rows<F, LOGM, INV>(P, l.src, l.dst, l.pr, blockIdx.x % per, lds)
  FZ_FIELD(l.pr, CALL)
#undef CALL
}

// Decryption's rows: both components' forward rows (stored, as the transforms
// leave them), c0 + c1 s and its inverse rows.  A chain of three row transforms
// in one launch: 16.4 us at N = 2^15, 12 limbs, for the 31 of two launches of
// rows and the product between them.
template <class F, int LOGM>
__device__ __forceinline__ void nt_decrypt(const DevParams& P, uint64_t* c0, uint64_t* c1, const uint64_t* s, uint64_t* out,
                                           int pr, int tile, uint64_t* lds) {
  using G = RowOf<LOGM>;
  constexpr int LV = kLogV<LOGM>;
  const RowId<LOGM> id(tile, lds);
  const F f(ld_prime(P.primes, pr));
  const uint64_t* T = P.fz.tw[0] + (size_t)pr * P.N * 2;
  typename F::V x[G::V], z[G::V];
  uint64_t u[G::V];
#pragma unroll
  for (int k = 0; k < G::V; ++k) {
    z[k] = f.raw_in(at_byte<uint64_t>(c1, id.off + G::TS * 8 * k));
    x[k] = f.raw_in(at_byte<uint64_t>(c0, id.off + G::TS * 8 * k));
  }
  rows_fwd_all<F, LOGM>(f, z, u, T, id);
#pragma unroll
  for (int k = 0; k < G::V; ++k) put_byte(c1, id.off + G::TS * 8 * k, u[k]);
  uint64_t v[G::V];
  with_caller_words<G::V>(f, P.primes, pr, [&](auto& w, int k, auto set) {
    set(v, w(at_byte<uint64_t>(s, id.off + G::TS * 8 * k)));
  });
#pragma unroll
  for (int k = 0; k < G::V; ++k) z[k] = f.key(f.in(u[k]), v[k]);
  rows_fwd_all<F, LOGM>(f, x, u, T + opaque_zero(), id);
#pragma unroll
  for (int k = 0; k < G::V; ++k) {
    put_byte(c0, id.off + G::TS * 8 * k, u[k]);
    x[k] = f.add(f.in(u[k]), z[k]);
  }
  row_turn<LOGM, LV, 0, G::ROUNDS - 1>(f, x, id.s, id.L);
  rows_out<F, LOGM>(f, x, P.fz.tw[1] + (size_t)pr * P.N * 2, out, id);
}

template <int LOGM>
__global__ __launch_bounds__(RowOf<LOGM>::THREADS) void k_nt_decrypt(DevParams P, uint64_t* c0, uint64_t* c1,
                                                                     const uint64_t* s, uint64_t* out) {
  constexpr int FIELD = FZ_ANY;
  __shared__ uint64_t lds[RowOf<LOGM>::LDS];
  constexpr int per = 16 / RowOf<LOGM>::ROWS;
  const int i = blockIdx.x / per;
  const size_t o = (size_t)i * P.N;
#define CALL(F) nt_decrypt<F, LOGM>(P, c0 + o, c1 + o, s + o, out + o, i, blockIdx.x % per, lds)
  FZ_FIELD(i, CALL)
#undef CALL
}

// Encryption's rows, from forward columns: c0 = pk_b u + e0 (e0 with m added),
// c1 = pk_a u + e1 and m in place, a workgroup each: the rows of u twice, on
// idle units, for two transforms in a chain instead of four.
template <class F, int LOGM>
__device__ __forceinline__ void nt_encrypt(const DevParams& P, const NtEncrypt& a, int y, int i, int tile, uint64_t* lds) {
  using G = RowOf<LOGM>;
  const RowId<LOGM> id(tile, lds);
  const size_t o = (size_t)i * P.N;
  const F f(ld_prime(P.primes, i));
  const uint64_t* T = P.fz.tw[0] + (size_t)i * P.N * 2;
  typename F::V x[G::V], z[G::V];
  uint64_t u[G::V];
  const uint64_t* e = (y == 0 ? a.e0 : y == 1 ? a.e1 : a.m) + o;
#pragma unroll
  for (int k = 0; k < G::V; ++k) x[k] = f.raw_in(at_byte<uint64_t>(e, id.off + G::TS * 8 * k));
  if (y < 2) {
#pragma unroll
    for (int k = 0; k < G::V; ++k) z[k] = f.raw_in(at_byte<uint64_t>(a.u + o, id.off + G::TS * 8 * k));
    rows_fwd_all<F, LOGM>(f, z, u, T, id);
    const uint64_t* pk = (y == 0 ? a.pkb : a.pka) + o;
    uint64_t v[G::V];
    with_caller_words<G::V>(f, P.primes, i, [&](auto& w, int k, auto set) {
      set(v, w(at_byte<uint64_t>(pk, id.off + G::TS * 8 * k)));
    });
#pragma unroll
    for (int k = 0; k < G::V; ++k) z[k] = f.key(f.in(u[k]), v[k]);
  }
  rows_fwd_all<F, LOGM>(f, x, u, T + opaque_zero(), id);
  uint64_t* out = (y == 0 ? a.c0 : y == 1 ? a.c1 : a.m) + o;
#pragma unroll
  for (int k = 0; k < G::V; ++k)
    put_byte(out, id.off + G::TS * 8 * k, y < 2 ? f.out(f.add(f.in(u[k]), z[k])) : u[k]);
}

template <int LOGM>
__global__ __launch_bounds__(RowOf<LOGM>::THREADS) void k_nt_encrypt(DevParams P, NtEncrypt a) {
  constexpr int FIELD = FZ_ANY;
  __shared__ uint64_t lds[RowOf<LOGM>::LDS];
  constexpr int per = 16 / RowOf<LOGM>::ROWS;
  const int i = blockIdx.x / per;
#define CALL(F) nt_encrypt<F, LOGM>(P, a, blockIdx.y, i, blockIdx.x % per, lds)
  FZ_FIELD(i, CALL)
#undef CALL
}

// ------------------------------------------------------------------ launch --
template <bool INV, bool ARG>
static void nt_run_cols(const DevParams& P, const LimbMap& m, const NttDesc* d, int n, hipStream_t st) {
  k_nt_cols<INV, ARG><<<dim3((unsigned)(n * (P.N / 16 / NT_COLS)), ARG ? m.npolys : 1), 256, 0, st>>>(P, m, d);
}
template <bool INV, bool ARG>
static int nt_run(const DevParams& P, const LimbMap& m, const NttDesc* d, int n, hipStream_t st) {
  if (n <= 0) return -1;
  if (!INV) nt_run_cols<INV, ARG>(P, m, d, n, st);
#define CALL(LM)                                                                                                    \
  k_nt_rows<LM, INV, ARG>                                                                                           \
      <<<dim3(n * 16 / RowOf<LM>::ROWS, ARG ? m.npolys : 1), RowOf<LM>::THREADS, 0, st>>>(P, m, d)
  FZ_DISPATCH_M(CALL)
#undef CALL
  if (INV) nt_run_cols<INV, ARG>(P, m, d, n, st);
  return 0;
}

bool nt_default(const DevParams& P) { return !P.ntt_n1 && P.N >= 2048 && P.N <= 65536; }

int nt_forward(const DevParams& P, const LimbMap& m, hipStream_t st) {
  return nt_run<false, true>(P, m, nullptr, m.nlimbs, st);
}
int nt_inverse(const DevParams& P, const LimbMap& m, hipStream_t st) {
  return nt_run<true, true>(P, m, nullptr, m.nlimbs, st);
}
int nt_forward_desc(const DevParams& P, const NttDesc* d, int n, hipStream_t st) {
  return nt_run<false, false>(P, LimbMap{}, d, n, st);
}
int nt_inverse_desc(const DevParams& P, const NttDesc* d, int n, hipStream_t st) {
  return nt_run<true, false>(P, LimbMap{}, d, n, st);
}

void nt_forward_cols(const DevParams& P, const LimbMap& m, hipStream_t st) {
  nt_run_cols<false, true>(P, m, nullptr, m.nlimbs, st);
}
int nt_encrypt_rows(const DevParams& P, const NtEncrypt& a, int nlimbs, hipStream_t st) {
#define CALL(LM) k_nt_encrypt<LM><<<dim3(nlimbs * 16 / RowOf<LM>::ROWS, 3), RowOf<LM>::THREADS, 0, st>>>(P, a)
  FZ_DISPATCH_M(CALL)
#undef CALL
  return 0;
}

int nt_decrypt(const DevParams& P, uint64_t* m, uint64_t* c0, uint64_t* c1, const uint64_t* s, int nlimbs, hipStream_t st) {
  LimbMap c{};
  c.src[0] = c.base[0] = c0;
  c.src[1] = c.base[1] = c1;
  c.nlimbs = c.qlimbs = nlimbs;
  c.npolys = 2;
  nt_run_cols<false, true>(P, c, nullptr, nlimbs, st);
#define CALL(LM) k_nt_decrypt<LM><<<dim3(nlimbs * 16 / RowOf<LM>::ROWS), RowOf<LM>::THREADS, 0, st>>>(P, c0, c1, s, m)
  FZ_DISPATCH_M(CALL)
#undef CALL
  c.base[0] = m;
  c.npolys = 1;
  nt_run_cols<true, true>(P, c, nullptr, nlimbs, st);
  return 0;
}

}  // namespace aoa
