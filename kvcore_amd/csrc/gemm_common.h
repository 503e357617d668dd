// Operand vectors of the bfloat16 matrix instructions and guarded stores of four results,
// shared by the weight-streaming products.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_utils.h"

namespace kvc {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Sixteen bytes; ONCE: of a matrix that the whole launch reads once.  Such loads are marked as streaming ones: 512 MB in
// runs of 64 KB a wave are read at 6.6 TB/s with the mark and at 6.25 without (the caches need not make room for
// them, and keep the rows).  Steps with them in the products of few and of some dozen rows, in the experts' tiles and on
// keys and values of single tokens: 8B shape, 8 tokens 3,478 -> 3,271 us, 64 tokens 5,005 -> 4,835, 1B, one token 901 ->
// 856.  A model's size does not matter much: matrices of up to 256 MB in all, which the memory-side cache holds, read one after
// the other by nothing but these products take 1.04 to 1.2 times as long with the mark (2048 x 2048 in 128 MB, one row 4.05 -> 4.48 us),
// but whole decode steps of six models with 60 to 200 MB 0.95 to 1.01 up to 16 tokens and 0.97 to 1.04 at 32 and 64.
// Where several blocks share a matrix through the L2, or a load takes
// part of a line whose rest comes with another, the mark costs more than it brings.
template <bool ONCE>
__device__ __forceinline__ bf16x8_t read8(const void* p) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  const u32x4_t* from = static_cast<const u32x4_t*>(p);
  return __builtin_bit_cast(bf16x8_t, ONCE ? __builtin_nontemporal_load(from) : *from);
}

__device__ __forceinline__ bf16x8_t zero8() {
  bf16x8_t z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = static_cast<__bf16>(0.f);
  return z;
}

// four results to a place that is aligned for all of them
__device__ __forceinline__ void store4_whole(float* p, f32x4_t v) { *reinterpret_cast<f32x4_t*>(p) = v; }
// (the conversion in hardware rounds to nearest, ties to even, and keeps NaN, as f32_to_bf16_bits does)
__device__ __forceinline__ void store4_whole(bf16_t* p, f32x4_t v) {
  typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
  *reinterpret_cast<bf16x4_t*>(p) = __builtin_convertvector(v, bf16x4_t);
}

template <typename OutT>
__device__ __forceinline__ void store4(OutT* p, f32x4_t v, int n_left);
template <>
__device__ __forceinline__ void store4<float>(float* p, f32x4_t v, int n_left) {
  if (n_left >= 4 && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    store4_whole(p, v);
  } else {
    for (int i = 0; i < 4 && i < n_left; ++i) p[i] = v[i];
  }
}
template <>
__device__ __forceinline__ void store4<bf16_t>(bf16_t* p, f32x4_t v, int n_left) {
  if (n_left >= 4 && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
    store4_whole(p, v);
  } else {
    for (int i = 0; i < 4 && i < n_left; ++i) p[i].bits = f32_to_bf16_bits(v[i]);
  }
}

}  // namespace kvc
