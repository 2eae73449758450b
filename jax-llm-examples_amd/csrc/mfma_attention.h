// What the attention kernels on the matrix cores share: operand types, sums over a column's lanes, where a page
// tile's pieces lie in shared memory.
#pragma once
#include "common.h"

namespace jle {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;  // (register arrays of HIP's uint4 may end up in scratch)

constexpr float kLog2e = 1.4426950408889634f;

// Maximum / sum over the four lanes that hold one column (equal lane % 16), in all of them.  The two swaps
// exchange the halves of the wavefront and neighbouring rows of 16 lanes: no trip through shared memory.
__device__ __forceinline__ float column_max(float v) {
  uint32_t u = __float_as_uint(v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  u = __float_as_uint(v);
  r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float column_sum(float v) {
  uint32_t u = __float_as_uint(v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  u = __float_as_uint(v);
  r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// where piece p of key row r of a page tile lies: p ^ key_swizzle(r); the eight rows that eight neighbouring lanes read
// (r % 4, r / 8 varying) then differ in the low three bits
__device__ __forceinline__ int key_swizzle(int r) { return (r & 3) | ((r >> 3) << 2) | (((r >> 2) & 1) << 3); }

}  // namespace jle
