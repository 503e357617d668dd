// C[M, N] = A[M, K] * W[N, K]^T (+ bias) in true float32: float32 products, float32 sums (the matrix
// instructions whose operands are float32), no mode of reduced precision.
//
// Every element of C is made in one way, whatever M, its tile or its row's place in the batch: K is cut into
// chunks of 32; wave w of a block's eight adds up the chunks w, w + 8, ... in order (a chunk is eight
// 16 x 16 x 4 instructions, of which number j takes the values k + j, k + 8 + j, k + 16 + j, k + 24 + j); the
// eight sums are added in wave order, then the bias.  So the tile may follow the sizes of a call and the bits
// do not.
//
// A block takes NT x MT tiles of 16 columns x 16 rows of C and all its waves take all of them, each its part
// of K: the operands go from memory to registers (a lane 32 contiguous bytes, the four lanes of a row 128), a
// fetched weight meets 16 MT rows and a fetched row 16 NT columns.  Bound by the float32 matrix rate
// (157 TFLOP/s) from some 30 rows on and by reading W below that.  Against a tile of 64 x 64 through LDS whose
// threads multiplied and added: 122 rows of 16384 x 2048 262 -> 118 us (70 TFLOP/s), of 2048 x 8192 875 -> 62;
// 2,048 rows of 16384 x 2048 3.64 -> 1.68 ms (82 TFLOP/s); one row of 16384 x 2048 196 -> 33 us (4.0 TB/s).  It was
// the faster only for hundreds of rows whose K is short and no multiple of 8 (300 rows of 8192 x 100 17 and 23 us).

#include <hip/hip_runtime.h>

#include "device_utils.h"
#include "gemm_common.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

constexpr int kWaves = 8;
constexpr int kChunk = 32;

// Eight values of a row from k on, loaded in pieces of PIECE (8: two of four): K a multiple of PIECE and the rows
// aligned to it (16 bytes at most), so a piece is in or out as a whole; `whole` (the same for the wave): the chunk
// lies inside K.
template <int PIECE>
__device__ __forceinline__ void load8(f32x4_t* v, const float* row, int k, int K, bool whole) {
  if constexpr (PIECE == 8) {
    const float* p = row + (k < K ? k : 0);
    v[0] = *reinterpret_cast<const f32x4_t*>(p);
    v[1] = *reinterpret_cast<const f32x4_t*>(p + 4);
    if (!whole && k >= K) v[0] = v[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  } else if constexpr (PIECE == 2) {  // for many tiles: with a piece a value 300 rows of 8192 x 100 take 27.5 us, 22.7 so
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float2 x = *reinterpret_cast<const float2*>(row + (k + i < K ? k + i : 0));
      v[i >> 2][i & 3] = whole || k + i < K ? x.x : 0.f;
      v[i >> 2][(i & 3) + 1] = whole || k + i < K ? x.y : 0.f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i >> 2][i & 3] = k + i < K ? row[k + i] : 0.f;
  }
}

template <int NT, int MT, int AHEAD, int PIECE>
__global__ __launch_bounds__(kWaves * 64) void gemm_f32_kernel(float* __restrict__ C, const float* __restrict__ A,
                                                               const float* __restrict__ W,
                                                               const float* __restrict__ bias, int M, int N, int K,
                                                               int64_t lda, int64_t ldc) {
  __shared__ f32x4_t part[kWaves][MT][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
  // columns and rows beyond the matrix read its last ones and are not stored
  const float* wp[NT];
  const float* ap[MT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wp[n] = W + static_cast<int64_t>(n0 + 16 * n + li < N ? n0 + 16 * n + li : N - 1) * K;
#pragma unroll
  for (int m = 0; m < MT; ++m) ap[m] = A + static_cast<int64_t>(m0 + 16 * m + li < M ? m0 + 16 * m + li : M - 1) * lda;
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int chunks = (K + kChunk - 1) / kChunk;
  f32x4_t wv[AHEAD][NT][2], av[AHEAD][MT][2];
  // no branch around the loads: a chunk that is not there is one that reads zeros
  auto fetch = [&](int slot, int c) {
    const int k = c * kChunk + 8 * lk;
    const bool whole = (c + 1) * kChunk <= K;
#pragma unroll
    for (int n = 0; n < NT; ++n) load8<PIECE>(wv[slot][n], wp[n], k, K, whole);
#pragma unroll
    for (int m = 0; m < MT; ++m) load8<PIECE>(av[slot][m], ap[m], k, K, whole);
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) fetch(s, wave + kWaves * s);
  for (int c = wave; c < chunks; c += kWaves * AHEAD) {  // scalar
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      f32x4_t w[NT][2], a[MT][2];
#pragma unroll
      for (int n = 0; n < NT; ++n) w[n][0] = wv[s][n][0], w[n][1] = wv[s][n][1];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m][0] = av[s][m][0], a[m][1] = av[s][m][1];
      fetch(s, c + kWaves * (s + AHEAD));
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[n][j >> 2][j & 3], a[m][j >> 2][j & 3], acc[n][m], 0, 0, 0);
    }
  }
  // the waves' sums, 16 columns at a time: lane holds row li, columns 4 lk .. of its tiles
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    if (n > 0) __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m) part[wave][m][lane] = acc[n][m];
    __syncthreads();
    for (int idx = threadIdx.x; idx < MT * 64; idx += kWaves * 64) {
      const int m = idx >> 6, l = idx & 63;
      f32x4_t v = part[0][m][l];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) v += part[w][m][l];
      const int row = m0 + 16 * m + (l & 15), col = n0 + 16 * n + 4 * (l >> 4);
      if (row >= M || col >= N) continue;
      if (bias != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += bias[col + i < N ? col + i : N - 1];
      }
      store4<float>(C + static_cast<int64_t>(row) * ldc + col, v, N - col);
    }
  }
}

// The same for K of at most eight chunks, of which every wave above would have one: a wave takes all of them of NT x MT
// tiles of its own, each summed up from zero and added in order, so the bits are the same and nothing is left to meet
// in LDS.  The four waves of a block lie side by side along the columns.  Bound by storing C (at K of 32) and by the
// matrix rate (at 256).
template <int NT, int MT, int PIECE>
__global__ __launch_bounds__(256) void gemm_f32_short_kernel(float* __restrict__ C, const float* __restrict__ A,
                                                             const float* __restrict__ W, const float* __restrict__ bias,
                                                             int M, int N, int K, int64_t lda, int64_t ldc) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int n0 = (blockIdx.x * 4 + wave) * 16 * NT, m0 = blockIdx.y * 16 * MT;
  if (n0 >= N) return;  // scalar
  // columns and rows beyond the matrix read its last ones and are not stored
  const float* wp[NT];
  const float* ap[MT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wp[n] = W + static_cast<int64_t>(n0 + 16 * n + li < N ? n0 + 16 * n + li : N - 1) * K;
#pragma unroll
  for (int m = 0; m < MT; ++m) ap[m] = A + static_cast<int64_t>(m0 + 16 * m + li < M ? m0 + 16 * m + li : M - 1) * lda;
  f32x4_t sum[NT][MT], wv[NT][2], av[MT][2];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) sum[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int c) {  // a chunk that is not there is one that reads zeros
    const int k = c * kChunk + 8 * lk;
    const bool whole = (c + 1) * kChunk <= K;
#pragma unroll
    for (int n = 0; n < NT; ++n) load8<PIECE>(wv[n], wp[n], k, K, whole);
#pragma unroll
    for (int m = 0; m < MT; ++m) load8<PIECE>(av[m], ap[m], k, K, whole);
  };
  fetch(0);
  for (int c = 0; c * kChunk < K; ++c) {  // scalar
    f32x4_t w[NT][2], a[MT][2], acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n][0] = wv[n][0], w[n][1] = wv[n][1];
#pragma unroll
    for (int m = 0; m < MT; ++m) a[m][0] = av[m][0], a[m][1] = av[m][1];
    fetch(c + 1);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[n][j >> 2][j & 3], a[m][j >> 2][j & 3], acc[n][m], 0, 0, 0);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) sum[n][m] += acc[n][m];
  }
  // lane holds row li, columns 4 lk .. of its tiles
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m0 + 16 * m + li;
    if (row >= M) continue;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int col = n0 + 16 * n + 4 * lk;
      if (col >= N) continue;
      f32x4_t v = sum[n][m];
      if (bias != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += bias[col + i < N ? col + i : N - 1];
      }
      store4<float>(C + static_cast<int64_t>(row) * ldc + col, v, N - col);
    }
  }
}

}  // namespace

extern "C" int kvc_gemm_f32(float* C, const float* A, const float* W, const float* bias, int M,
                            int N, int K, int64_t lda, int64_t ldc, kvc_stream stream) {
  if (M < 0 || N <= 0 || K <= 0 || lda < K || ldc < N) return kvc_fail("kvc_gemm_f32: bad sizes");
  if (M == 0) return 0;
  const int64_t units = kvc_device_compute_units();
  const uintptr_t ends = reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W);
  const int piece = K % 8 == 0 && lda % 4 == 0 && (ends & 15) == 0 ? 8 : K % 2 == 0 && lda % 2 == 0 && (ends & 7) == 0 ? 2 : 1;
#define KVC_F32_LAUNCH(KERNEL, THREADS)                                                                        \
  hipLaunchKernelGGL(KERNEL, grid, dim3(THREADS), 0, reinterpret_cast<hipStream_t>(stream), C, A, W, bias, M, N, K, lda, ldc)
  // Which of the two: 16 x 16 tiles of C a unit from which a wave with all of K pays.  Eight waves / one, us: 122 rows
  // of 8192 x 32 8.5 / 6.0, 2,048 rows 84 / 29; 122 rows of 2048 x 96 5.0 / 5.8, 1,000 rows 14.6 / 12.4; 122 rows of
  // 8192 x 256 13.4 / 15.0, 300 rows 33.3 / 27.1.  (Rows that load in smaller pieces: 300 rows of 2048 x 70 11.9 / 11.3.)
  const int chunks = (K + kChunk - 1) / kChunk;
  const int64_t tiles = static_cast<int64_t>((N + 15) / 16) * ((M + 15) / 16);
  const int from = chunks > 6 || (piece != 8 && chunks > 1) ? 24 : chunks > 2 ? 5 : chunks > 1 ? 3 : 0;
  if (chunks <= kWaves && tiles >= from * units) {
    // 64 rows a wave where the operands' way to it counts and two blocks a unit are left: 4,096 rows of 8192 x 100 209 ->
    // 157 us, of 8192 x 256 196 -> 189; of 8192 x 32, bound by C, 46 -> 55
    int mt = M <= 16 ? 1 : 2, nt = 4;
    if (chunks > 2 && static_cast<int64_t>((N + 255) / 256) * ((M + 63) / 64) >= 2 * units) mt = 4;
    auto short_blocks = [&]() { return static_cast<int64_t>((N + 64 * nt - 1) / (64 * nt)) * ((M + 16 * mt - 1) / (16 * mt)); };
    while (nt > 1 && short_blocks() < 2 * units) nt /= 2;
    const dim3 grid((N + 64 * nt - 1) / (64 * nt), (M + 16 * mt - 1) / (16 * mt));
    if (grid.y > 65535) return kvc_fail("kvc_gemm_f32: M too large for one launch");
#define KVC_F32(NT, MT)                                                                     \
  do {                                                                                      \
    if (piece == 8) KVC_F32_LAUNCH((gemm_f32_short_kernel<NT, MT, 8>), 256);                \
    else if (piece == 2) KVC_F32_LAUNCH((gemm_f32_short_kernel<NT, MT, 2>), 256);           \
    else KVC_F32_LAUNCH((gemm_f32_short_kernel<NT, MT, 1>), 256);                           \
  } while (0)
    if (mt == 1) {
      if (nt == 4) KVC_F32(4, 1);
      else if (nt == 2) KVC_F32(2, 1);
      else KVC_F32(1, 1);
    } else if (mt == 2) {
      if (nt == 4) KVC_F32(4, 2);
      else if (nt == 2) KVC_F32(2, 2);
      else KVC_F32(1, 2);
    } else {
      KVC_F32(4, 4);  // blocks enough
    }
#undef KVC_F32
    return kvc_check_launch("kvc_gemm_f32");
  }
  // tiles of 64 x 64 where they give every compute unit a block, narrower ones otherwise (122 rows of 2048 x 2048
  // are 64 blocks of 64 x 64 and 256 of 32 x 32); rows in sixteens up to the batch's size
  int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if (mt == 4 && M < 256 && (M + 63) / 64 * 64 >= M + 32) mt = 2;  // the last 64 rows would be half empty
  int nt = 4;
  auto blocks = [&]() { return static_cast<int64_t>((N + 16 * nt - 1) / (16 * nt)) * ((M + 16 * mt - 1) / (16 * mt)); };
  while (blocks() < units && (nt > 1 || mt > 2)) {
    if (nt >= mt && nt > 1) nt /= 2;
    else if (mt > 2) mt /= 2;
    else nt /= 2;
  }
  const dim3 grid((N + 16 * nt - 1) / (16 * nt), (M + 16 * mt - 1) / (16 * mt));
  if (grid.y > 65535) return kvc_fail("kvc_gemm_f32: M too large for one launch");
#define KVC_F32(NT, MT, AHEAD)                                                                      \
  do {                                                                                              \
    if (piece == 8) KVC_F32_LAUNCH((gemm_f32_kernel<NT, MT, AHEAD, 8>), kWaves * 64);               \
    else KVC_F32_LAUNCH((gemm_f32_kernel<NT, MT, 1, 1>), kWaves * 64);                              \
  } while (0)
  if (mt == 4) {  // from (2, 4) the loop above goes on to (2, 2)
    if (nt == 4) KVC_F32(4, 4, 1);
    else KVC_F32(2, 4, 1);
  } else if (mt == 2) {
    if (nt == 4) KVC_F32(4, 2, 1);
    else if (nt == 2) KVC_F32(2, 2, 2);
    else KVC_F32(1, 2, 2);
  } else {
    if (nt == 4) KVC_F32(4, 1, 2);
    else if (nt == 2) KVC_F32(2, 1, 2);
    else KVC_F32(1, 1, 4);
  }
#undef KVC_F32
#undef KVC_F32_LAUNCH
  return kvc_check_launch("kvc_gemm_f32");
}
