// Shared device-side definitions for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "modarith.hpp"
#include "params.hpp"

namespace aoa {

struct alignas(16) tw2 {
  uint64_t w, q;  // constant and its Shoup quotient
};

// Read-only tables seen through the constant address space: loads at a
// wave-uniform index become scalar loads, which the compiler cannot prove
// safe through a generic pointer once the kernel also stores to memory.
// The tables are written only by aoa_params_create, before any kernel runs.
template <class T>
using cptr = const T __attribute__((address_space(4)))*;
template <class T>
__device__ __forceinline__ cptr<T> as_const(const T* p) {
  return (cptr<T>)p;
}

// A pointer read from a descriptor in memory, marked as pointing to global
// memory.  The compiler otherwise treats it as generic and accesses it with
// flat instructions, which count against the LDS / scalar-load counter as
// well, so that every wait for an LDS exchange or a scalar load also waits
// for them, and take 64-bit addresses in vector registers.  The cast is
// undone at once; the compiler carries the address space to every use.
template <class T>
__device__ __forceinline__ T* glob(T* p) {
  return (T*)(T __attribute__((address_space(1)))*)(uintptr_t)p;
}

// Entry i of a read-only table of tw2 / DevPrime through the constant
// address space (word by word: structs cannot be copied out of it).
__device__ __forceinline__ tw2 ld_tw2(const tw2* base, size_t i) {
  const cptr<uint64_t> w = as_const(reinterpret_cast<const uint64_t*>(base + i));
  return tw2{w[0], w[1]};
}
__device__ __forceinline__ uint64_t ld_u64(const uint64_t* base, size_t i) { return as_const(base)[i]; }
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup w runs on
// XCD w % 8).  This map deals the n work items out in 8 contiguous chunks,
// one per XCD (the first n % 8 chunks one item longer): XCD x receives
// exactly the ids w < n with w % 8 == x, as many as its chunk holds, so the
// map is a bijection of [0, n).
__device__ __forceinline__ int xcd_chunk_id(unsigned w, unsigned n) {
  const unsigned q = n >> 3, r = n & 7, x = w & 7;
  return (int)(x * q + (x < r ? x : r) + (w >> 3));
}

// One field of a DevPrime at a wave-uniform index, as a scalar load.
__device__ __forceinline__ uint64_t ld_prime_p(const DevPrime* base, int i) { return as_const(&base[i].p)[0]; }
__device__ __forceinline__ int ld_prime_nb(const DevPrime* base, int i) { return (int)as_const(&base[i].nb)[0]; }
__device__ __forceinline__ uint32_t ld_prime_field(const DevPrime* base, int i) { return as_const(&base[i].field)[0]; }
__device__ __forceinline__ DevPrime ld_prime(const DevPrime* base, int i) {
  constexpr int W = (int)(sizeof(DevPrime) / 8);
  const cptr<uint64_t> w = as_const(reinterpret_cast<const uint64_t*>(base + i));
  uint64_t t[W];
#pragma unroll
  for (int x = 0; x < W; ++x) t[x] = w[x];
  DevPrime d;
  __builtin_memcpy(&d, t, sizeof(d));
  return d;
}

// Canonical residues of any words, one from 2^63 up read as that minus 2^64: what
// aoa_eltwise_scalar leaves of a residue smaller than a constant above the prime.
struct Residues {
  uint64_t p, wq;  // floor(2^64 / p)
  __device__ __forceinline__ explicit Residues(const DevPrime& d) : p(d.p), wq(d.mu >> (2 * (int)d.nb - 64)) {}
  __device__ __forceinline__ uint64_t operator()(uint64_t x) const {
    const bool neg = x >> 63;
    const uint64_t r = mul_shoup(neg ? 0 - x : x, 1, wq, p);
    return neg ? neg_mod(r, p) : r;
  }
};

// Where the limbs of one launch live.  Limb li of poly y is at
// base[y] + li * N and uses prime index prime_of(li): the first `qlimbs`
// limbs are Q limbs prime0, prime0+1, ..., the rest are special limbs
// k, k+1, ...
struct LimbMap {
  uint64_t* base[4];
  const uint64_t* src[4];  // optional separate input (out-of-place first pass), else == base
  int nlimbs;
  int qlimbs;
  int npolys;
  int prime0;  // prime index of limb 0 when it is a Q limb
};

__device__ __forceinline__ int limb_prime(const LimbMap& m, int k, int li) {
  return li < m.qlimbs ? m.prime0 + li : k + (li - m.qlimbs);
}

// Descriptor tables of the batched (stage-fused) launches: one entry per
// limb.
struct NttDesc {
  const uint64_t* src;  // first-pass input limb (== dst for in place)
  uint64_t* dst;        // output limb
  int prime;
  int pad;
};

struct AutoDesc {
  const uint64_t* in;      // limb of the input (coefficient domain)
  uint64_t* out;           // limb of the output
  const uint64_t* addsrc;  // optional limb added to sigma(in)
  uint64_t ginv;           // inverse Galois element mod 2N
  int prime;
  int pad;
};

// One HomMul (a0 set) or key switching of the fused kernels (fused.hpp).
// Limb-major buffers, stride N; P0 and P1 hold level + 1 + K limbs.
struct FzItem {
  const uint64_t *a0, *a1, *b0, *b1;  // HomMul's operands (NTT domain)
  const uint64_t* d;                  // key switching's input (coefficient domain)
  const uint64_t *kb, *ka;            // switching key, limb of prime r at + r N
  uint64_t* D;                        // HomMul: d2 after the inverse rows (level + 1 limbs)
  uint64_t* XQ;                       // key switching: the input's forward columns (level + 1 limbs)
  uint64_t* X;                        // the special limbs' forward columns (K limbs)
  uint64_t *P0, *P1;                  // key products after the inverse rows
  const uint64_t *add0, *add1;        // added to the result (coefficient domain), or null
  uint64_t *out0, *out1;
  int level;
  int rescale;
};

__device__ __forceinline__ tw2 load_tw(const uint64_t* table, size_t idx) {
  return reinterpret_cast<const tw2*>(table)[idx];
}

}  // namespace aoa
