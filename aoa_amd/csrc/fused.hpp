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

}  // namespace aoa
