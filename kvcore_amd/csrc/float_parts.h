// Float32 operands of the bfloat16 matrix instructions: each value the sum of three bfloat16 parts, and six of the nine products
// of parts, for kernels whose sums must not be less precise than on the float32 matrix instructions.  (Splitting a number
// into parts of a shorter format goes back to Dekker 1971; with bfloat16 parts: Henry, Tang and Heinecke 2019.)
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gemm_common.h"

namespace kvc {

// Eight float32 values times 2^16 as sums of three bfloat16 values, rounded to nearest one after the other: 24 significand bits
// in three times eight, and the least bit of float32, 2^-149, comes to the least of bfloat16, 2^-133, so nothing is left over
// of any value below 2^111.  (Without the factor values below 2^-110 lost bits, which a large value on the other side
// showed: 1e-38 x 1e36 was off by 3e-3.  The factor costs 122 rows of 16384 x 2048 67 -> 70 us; with v_dot2c_f32_bf16, which takes
// out a part and subtracts it in one instruction and gives the same bits, they took 74.)  Sums of products are to be
// multiplied by kPartsUnscale; what goes beyond float32 on the way, operands from 2^111 or sums from 2^96 on, comes out as no
// finite number and is to be summed again without parts.
constexpr float kPartsScale = 0x1p16f, kPartsUnscale = 0x1p-32f;
struct split_t {
  bf16x8_t part[3];
};
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ split_t split8(const f32x4_t* v) {
  u32x4_t out[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // two values at a time: one conversion makes both halves of a register
    f32x2_t x = {v[i >> 1][2 * (i & 1)] * kPartsScale, v[i >> 1][2 * (i & 1) + 1] * kPartsScale};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t bits = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2_t));
      out[p][i] = bits;
      if (p < 2) {
        x[0] -= __uint_as_float(bits << 16);
        x[1] -= __uint_as_float(bits & 0xffff0000u);
      }
    }
  }
  split_t s;
#pragma unroll
  for (int p = 0; p < 3; ++p) s.part[p] = __builtin_bit_cast(bf16x8_t, out[p]);
  return s;
}

// Which parts the six products take, the smallest first.  A second part is at most 2^-8 of the value and a third one 2^-17, so the
// three products left out are at most 2^-24 of the product, half a unit in its last place (both operands 0x1.00ff8p+0 come
// to that; operands at random to 2^-27.5 in the root mean square).
constexpr int kOrder[6][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}, {0, 0}};

// What is summed again without parts is summed by a whole wave, every lane of which takes these calls with the same
// arguments: a lane its values 64 apart, the lanes' sums in one fixed order.  (A lane that walks along a row alone waits for
// each of its values: with one NaN in a row 122 rows of 2048 x 8192 took 4.5 ms, not 40 us, and a step of 2 x 61 tokens of
// which one holds a NaN 210 ms, not 3; so 46 us and 4.8 ms.)
__device__ __forceinline__ bool wave_holds_nan(const float* __restrict__ a, int K) {
  bool holds = false;
#pragma unroll 8
  for (int k = threadIdx.x & 63; k < K; k += 64) holds |= a[k] != a[k];
  return __ballot(holds) != 0;
}
// S products of the row a with rows of their own
template <int S>
__device__ __forceinline__ void wave_products(float (&sum)[S], const float* __restrict__ a, const float* const (&w)[S], int K) {
#pragma unroll
  for (int i = 0; i < S; ++i) sum[i] = 0.f;
#pragma unroll 4
  for (int k = threadIdx.x & 63; k < K; k += 64) {
    const float x = a[k];
#pragma unroll
    for (int i = 0; i < S; ++i) sum[i] = fmaf(x, w[i][k], sum[i]);
  }
#pragma unroll
  for (int i = 0; i < S; ++i) sum[i] = wave_sum(sum[i]);
}

}  // namespace kvc
