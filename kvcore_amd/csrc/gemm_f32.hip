// C[M, N] = A[M, K] * W[N, K]^T (+ bias) in float32, its products on the bfloat16 matrix instructions: an operand is
// the sum of three bfloat16 values, and the six largest products of parts are added up in float32 (float_parts.h).  That
// is no mode of reduced precision: over 1 to 2,048 rows and K of 64 to 8,192 the error against 64 bits is 0.43 to 0.89 of
// what the float32 matrix instructions leave (122 rows of 16384 x 2048: 2.4e-7 and 2.9e-7 of the result, of 2048 x 8192
// 5.1e-7 and 5.7e-7), and a chunk of 32 values takes 96 cycles of a matrix core, not 256.
//
// Every element of C is made in one way, whatever M, its tile or its row's place in the batch: K is cut into
// chunks of 32; eight chains take the chunks w, w + 8, ... in order (a chunk is six 16 x 16 x 32 instructions); the
// eight sums are added in order, then the bias.  So the tile may follow the sizes of a call and the bits do not.
//
// Few rows: a block takes NT x MT tiles of 16 columns x 16 rows of C and all its waves take all of them, each a chain
// of K: the operands go from memory to registers (the four lanes of a row read 64 contiguous bytes at a time).  Bound by
// reading W (one row of 16384 x 2048 31 us, 4.4 TB/s).  More than 32 rows: these, or gemm_f32_shared_kernel (shared_shape).

#include <hip/hip_runtime.h>

#include "device_utils.h"
#include "float_parts.h"
#include "gemm_common.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

constexpr int kWaves = 8;
constexpr int kChunk = 32;

// Read by lanes whose values lie beyond K: an address, so that no select stands between a load and its use (one that
// does makes the compiler wait for every load in flight).
__device__ f32x4_t kNothing[2];

// A lane's eight values of a chunk, four from k = 4 lk on and four from k + 16 on, so that the four lanes of a row read
// 64 contiguous bytes at a time; loaded in pieces of PIECE (8: two of four): K a multiple of PIECE and the rows aligned to
// it (16 bytes at most), so a piece is in or out as a whole; `whole` (the same for the wave): the chunk lies inside K.
template <int PIECE>
__device__ __forceinline__ void load8(f32x4_t* v, const float* row, int k, int K, bool whole) {
  if constexpr (PIECE == 8) {
    v[0] = *(k < K ? reinterpret_cast<const f32x4_t*>(row + k) : kNothing);
    v[1] = *(k + 16 < K ? reinterpret_cast<const f32x4_t*>(row + k + 16) : kNothing);
  } else if constexpr (PIECE == 2) {  // for many tiles: with a piece a value 300 rows of 8192 x 100 take 27.5 us, 22.7 so
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const int at = k + i + (i < 4 ? 0 : 12);
      const float2 x = *reinterpret_cast<const float2*>(row + (at < K ? at : 0));
      v[i >> 2][i & 3] = whole || at < K ? x.x : 0.f;
      v[i >> 2][(i & 3) + 1] = whole || at < K ? x.y : 0.f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = k + i + (i < 4 ? 0 : 12);
      v[i >> 2][i & 3] = at < K ? row[at] : 0.f;
    }
  }
}

// acc += the sums over a chunk of w x a, the smallest of the six products first.
template <int NT, int MT>
__device__ __forceinline__ void multiply(f32x4_t (&acc)[NT][MT], const split_t* w, const split_t* a) {
#pragma unroll
  for (int p = 0; p < 6; ++p)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[n].part[kOrder[p][0]], a[m].part[kOrder[p][1]], acc[n][m], 0, 0, 0);
}

// Four sums of parts' products that lie side by side in C, as they leave; every lane of a wave comes here, `live` or not.  A value
// beyond what the parts hold, an infinity or a NaN among the operands leaves a sum that is not finite: such an element is
// summed again by the wave, or, where its row holds a NaN (which is looked up once a row), is one.
__device__ __forceinline__ void leave(bool live, f32x4_t v, float* __restrict__ C, const float* __restrict__ A,
                                      const float* __restrict__ W, const float* __restrict__ bias, int row, int col, int N,
                                      int K, int64_t lda, int64_t ldc) {
  v *= kPartsUnscale;
  // 0 x each: a NaN unless all are finite
  const float none = fmaf(v[0], 0.f, fmaf(v[1], 0.f, fmaf(v[2], 0.f, v[3] * 0.f)));
  uint64_t todo = __ballot(live && none != none);
  while (todo != 0) {  // scalar, as all that decides here
    const int r = __builtin_amdgcn_readlane(row, __builtin_ctzll(todo));
    const float* a = A + static_cast<int64_t>(r) * lda;
    const bool nan = wave_holds_nan(a, K);
    uint64_t same = __ballot(row == r) & todo;
    todo &= ~same;
    for (; same != 0; same &= same - 1) {
      const int lane = __builtin_ctzll(same), c = __builtin_amdgcn_readlane(col, lane);
      float sum[4] = {NAN, NAN, NAN, NAN};
      if (!nan) {
        const float* w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = W + static_cast<int64_t>(c + i < N ? c + i : N - 1) * K;
        wave_products<4>(sum, a, w, K);
      }
      if ((threadIdx.x & 63) == lane) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fabsf(v[i]) < INFINITY ? v[i] : sum[i];
      }
    }
  }
  if (!live) return;
  if (bias != nullptr) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += bias[col + i < N ? col + i : N - 1];
  }
  store4<float>(C + static_cast<int64_t>(row) * ldc + col, v, N - col);
}

// ONCE: K is at most kWaves * AHEAD chunks, so all of it is on its way from the start and nothing is asked for behind it (one row
// of 4096 x 512 5.7 us with four chunks ahead and loads of nothing behind the two that there are, 4.5 so)
template <int NT, int MT, int AHEAD, int PIECE, bool ONCE>
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
  auto fetch = [&](int slot, int c) {  // a chunk that is not there is one that reads zeros
    const int k = c * kChunk + 4 * lk;
    const bool whole = (c + 1) * kChunk <= K;
#pragma unroll
    for (int n = 0; n < NT; ++n) load8<PIECE>(wv[slot][n], wp[n], k, K, whole);
#pragma unroll
    for (int m = 0; m < MT; ++m) load8<PIECE>(av[slot][m], ap[m], k, K, whole);
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) {
    fetch(s, wave + kWaves * s);
    __builtin_amdgcn_sched_barrier(0);  // in the order of their use, which the waits count on
  }
  for (int c = wave; c < chunks; c += kWaves * AHEAD) {  // scalar; no branch inside, which would drain the loads
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      split_t w[NT], a[MT];
#pragma unroll
      for (int n = 0; n < NT; ++n) w[n] = split8(wv[s][n]);
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = split8(av[s][m]);
      // the loads leave after the registers that they fill have been read (or they would fill others and be copied,
      // which waits for them) and before the products
      __builtin_amdgcn_sched_barrier(0);
      if (!ONCE) fetch(s, c + kWaves * (s + AHEAD));
      __builtin_amdgcn_sched_barrier(0);
      multiply<NT, MT>(acc, w, a);
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
      leave(row < M && col < N, v, C, A, W, bias, row, col, N, K, lda, ldc);
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
    const int k = c * kChunk + 4 * lk;
    const bool whole = (c + 1) * kChunk <= K;
#pragma unroll
    for (int n = 0; n < NT; ++n) load8<PIECE>(wv[n], wp[n], k, K, whole);
#pragma unroll
    for (int m = 0; m < MT; ++m) load8<PIECE>(av[m], ap[m], k, K, whole);
  };
  fetch(0);
  for (int c = 0; c * kChunk < K; ++c) {  // scalar
    split_t w[NT], a[MT];
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n] = split8(wv[n]);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      a[m] = split8(av[m]);
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch(c + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    multiply<NT, MT>(acc, w, a);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) sum[n][m] += acc[n][m];
  }
  // lane holds row li, columns 4 lk .. of its tiles
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m0 + 16 * m + li;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int col = n0 + 16 * n + 4 * lk;
      leave(row < M && col < N, sum[n][m], C, A, W, bias, row, col, N, K, lda, ldc);
    }
  }
}

// The same for more rows than a wave's registers take at a time: the waves of a block take 16 NT columns each of 16 MT
// rows, whose chunk along K goes through LDS, split by the threads that fetch it and laid out as the matrix
// instructions want it (a wave's load is one contiguous kilobyte); a wave splits the weights of its own columns in
// registers.  The eight chains of K are walked one after the other, each from zero, and added in order, or (where C
// has too few tiles for the chip) dealt out to gridDim.z blocks, which leave every chain's sums in `parts`
// [chain][M][round4(N)] for gemm_f32_parts_kernel.  The bits are those of the kernels above.
//
// Bound by the matrix and the vector instructions of a wave together (a step of 4 x 2 tiles is 48 matrix instructions of
// 16 cycles beside the split of 24 values a lane, 6.5 instructions each; with every operand hot in the cache the kernel is
// 5 to 10% faster, no more).  With the float32 matrix instructions on operands straight from the cache and now: 122 rows of
// 16384 x 2048 115 and 70 us (117 TFLOP/s), of 2048 x 8192 62 and 40, of 3072 x 2048 35 and 25, of 2048 x 2048 18.9 and 17.9;
// 1,000 rows of 2048 x 2048 110 and 69, 2,048 rows of 16384 x 2048 1,668 and 834 (165 TFLOP/s).  Tiles of 128 rows and one
// column block a wave read LDS twice as often: 74, 38, 24, 18, 68 and 860 us before an operand's factor (float_parts.h), where
// these took 64, 39, 24, 17, 58 and 824.
// HALVES 2: a block of eight waves whose halves walk every other chain each, with LDS of their own for the rows; the second
// half's sums go to the first by LDS after each chain and are added in the same order.  Where the launch gives a unit one
// block of four waves, a SIMD has a single one, whose splits, reads of LDS and products wait for one another (122 rows of 16384 x
// 2048: 57 of 60 us remain without five of the six products); with two they overlap: 69 -> 60 us.  Where a unit has two
// blocks of four waves anyway, those do it better (700 rows 306 and 317 us).
template <int MT, int NT, bool LEAVE, int HALVES>
__global__ __launch_bounds__(256 * HALVES, 2) void gemm_f32_shared_kernel(
    float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
    float* __restrict__ parts, int M, int N, int K, int64_t lda, int64_t ldc) {
  constexpr int UN = MT / 4;  // pieces of 16 rows that a wave brings
  __shared__ u32x4_t all_rows_s[HALVES][2][MT][3][64];
  __shared__ f32x4_t meet_s[HALVES == 2 ? 4 * NT * MT : 1][64];
  static_assert(HALVES == 1 || !LEAVE, "chains that stay in memory need not meet");
  const int of_block = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wave = of_block & 3, second = HALVES == 2 ? of_block >> 2 : 0;
  u32x4_t(&rows_s)[2][MT][3][64] = all_rows_s[second];
  const int li = lane & 15, lk = lane >> 4;
  const int n0 = (blockIdx.x * 4 + wave) * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const int chunks = K / kChunk;  // a multiple of 16: both halves of a block make the same steps
  const int per = kWaves / gridDim.z;
  const int first = blockIdx.z * per + second, last = blockIdx.z * per + per;  // this half's chains, HALVES apart
  // columns and rows beyond the matrix read its last ones and are not stored
  const float* wp[NT];
  const float* ap[UN];
#pragma unroll
  for (int n = 0; n < NT; ++n)
    wp[n] = W + static_cast<int64_t>(n0 + 16 * n + li < N ? n0 + 16 * n + li : N - 1) * K + 4 * lk;
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    const int row = m0 + 16 * (wave + 4 * u) + li;
    ap[u] = A + static_cast<int64_t>(row < M ? row : M - 1) * lda + 4 * lk;
  }
  f32x4_t wv[2][NT][2], av[2][UN][2];
  split_t ws[2][NT];
  auto fetch = [&](int slot, int c) {
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) av[slot][u][i] = *reinterpret_cast<const f32x4_t*>(ap[u] + c * kChunk + 16 * i);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 2; ++i) wv[slot][n][i] = *reinterpret_cast<const f32x4_t*>(wp[n] + c * kChunk + 16 * i);
  };
  auto stash = [&](int slot) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const split_t s = split8(av[slot][u]);
#pragma unroll
      for (int p = 0; p < 3; ++p) rows_s[slot][wave + 4 * u][p][lane] = __builtin_bit_cast(u32x4_t, s.part[p]);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) ws[slot][n] = split8(wv[slot][n]);
  };
  // the chunk after c: the next of its chain, or the first of the next chain, or (at the end) any
  auto after = [&](int c) {
    const int next = (c & (kWaves - 1)) + HALVES;
    return c + kWaves < chunks ? c + kWaves : next < last ? next : first;
  };
  f32x4_t acc[NT][MT], sum[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = sum[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int ahead = first;  // the chunk to be fetched next
  fetch(0, ahead);
  __builtin_amdgcn_sched_barrier(0);  // in the order of their use, which the waits count on
  ahead = after(ahead);
  fetch(1, ahead);
  __builtin_amdgcn_sched_barrier(0);
  stash(0);
  ahead = after(ahead);
  __builtin_amdgcn_sched_barrier(0);
  fetch(0, ahead);
  for (int chain = first; chain < last; chain += HALVES) {
    for (int c = chain; c < chunks; c += 2 * kWaves) {  // scalar; no branch inside, which would drain the loads
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        __syncthreads();  // this chunk's rows are in LDS buffer s, the other buffer has been read by all
        split_t a[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
          for (int p = 0; p < 3; ++p) a[m].part[p] = __builtin_bit_cast(bf16x8_t, rows_s[s][m][p][lane]);
        }
#pragma unroll
        for (int g = 0; g < MT / 2; ++g)
#pragma unroll
          for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
              for (int i = 0; i < 2; ++i)
                acc[n][2 * g + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws[s][n].part[kOrder[p][0]], a[2 * g + i].part[kOrder[p][1]],
                                                                            acc[n][2 * g + i], 0, 0, 0);
        stash(s ^ 1);
        ahead = after(ahead);
        // after the registers that they fill have been read, or they would fill others and be copied, which waits for them
        __builtin_amdgcn_sched_barrier(0);
        fetch(s ^ 1, ahead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if constexpr (LEAVE) {
          const int row = m0 + 16 * m + li, col = n0 + 16 * n + 4 * lk, wide = (N + 3) & ~3;
          if (row < M && col < N)
            *reinterpret_cast<f32x4_t*>(parts + (static_cast<int64_t>(chain) * M + row) * wide + col) = acc[n][m];
        } else if (second) {
          meet_s[(wave * NT + n) * MT + m][lane] = acc[n][m];
        } else {
          sum[n][m] = chain == first ? acc[n][m] : sum[n][m] + acc[n][m];
        }
        acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    if constexpr (HALVES == 2) {
      __syncthreads();
      if (!second) {  // read before this half comes to the next chain's first barrier, and so before it is written again
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) sum[n][m] += meet_s[(wave * NT + n) * MT + m][lane];
      }
    }
  }
  if (LEAVE || second) return;
  // lane holds row li, columns 4 lk .. of its tiles
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m0 + 16 * m + li;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int col = n0 + 16 * n + 4 * lk;
      leave(row < M && col < N, sum[n][m], C, A, W, bias, row, col, N, K, lda, ldc);
    }
  }
}

// Adds up what the blocks above left: a thread four columns.
__global__ __launch_bounds__(256) void gemm_f32_parts_kernel(float* __restrict__ C, const float* __restrict__ A,
                                                             const float* __restrict__ W, const float* __restrict__ bias,
                                                             const float* __restrict__ parts, int chains, int M, int N, int K,
                                                             int64_t lda, int64_t ldc) {
  const int quads = (N + 3) >> 2;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const bool live = idx < static_cast<int64_t>(M) * quads;
  const int row = static_cast<int>(idx / quads), col = 4 * static_cast<int>(idx - static_cast<int64_t>(row) * quads);
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(parts) + (live ? idx : 0);
  const int64_t step = static_cast<int64_t>(M) * quads;
  f32x4_t v[kWaves];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) v[w] = p[(w < chains ? w : 0) * step];
#pragma unroll
  for (int w = 1; w < kWaves; ++w)
    if (w < chains) v[0] += v[w];  // scalar
  leave(live, v[0], C, A, W, bias, row, col, N, K, lda, ldc);
}

// Tiles of 16 columns and 16 rows a block of gemm_f32_kernel: 64 x 64 where they give every compute unit a block, narrower ones
// otherwise (122 rows of 2048 x 2048 are 64 blocks of 64 x 64 and 256 of 32 x 32); rows in sixteens up to the batch's size.
struct FewShape {
  int nt, mt;
  int64_t blocks;
};
FewShape few_shape(int M, int N) {
  const int64_t units = kvc_device_compute_units();
  int nt = 4, mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if (mt == 4 && M < 256 && (M + 63) / 64 * 64 >= M + 32) mt = 2;  // the last 64 rows would be half empty
  auto blocks = [&]() { return (static_cast<int64_t>(N) + 16 * nt - 1) / (16 * nt) * ((M + 16 * mt - 1) / (16 * mt)); };
  while (blocks() < units && (nt > 1 || mt > 2)) {  // from (2, 4) on to (2, 2)
    if (nt >= mt && nt > 1) nt /= 2;
    else if (mt > 2) mt /= 2;
    else nt /= 2;
  }
  return {nt, mt, blocks()};
}

// How the sizes of a call are dealt out to the kernel with rows in LDS: column blocks of 16 a wave, chains to how many
// blocks; nt 0: not at all.  By an estimate in us of each way, fitted to 155 sizes (33 to 1,500 rows, N of 256 to 16,384, K of
// 512 to 8,192; weights that no cache holds) within some 6%: a round of blocks on the units has a start and its share of K, and chains left
// in memory cost another kernel and their bytes.  gemm_f32_kernel / here, 64 columns, chains in one block / 128 columns in one /
// the better of those dealt out, in us:
//   64 rows of 2048 x 512     6.1 / 13.1 / 21.1 /  9.6      122 of 2048 x 2048    18.6 / 37 / 62 / 18.5
//   64 rows of 8192 x 512    10.4 / 13.6 / 21.2 / 18.5      64 of 16384 x 2048    42 / 47 / 69 / 52
//   256 of 2048 x 1024       15.8 / 22.1 / 36.0 / 22.1      128 of 3072 x 8192    93 / 133 / 223 / 58
//   400 of 2048 x 1024       28.6 / 22.4 / 36.7 / 30.1      400 of 3072 x 4096   124 / 119 / 121 / 93
//   100 of 16384 x 512       26.2 / 21.2 / 23.8 / 41.4      200 of 8192 x 8192   347 / 261 / 257 / 229
// Chains are dealt out up to the workspace that 64 x 128 of C a unit need.
constexpr int kSharedRows = 4;  // row blocks of 16 a block
struct SharedShape {
  int nt, groups, halves;
};
SharedShape shared_shape(int M, int N, int K) {
  if (M <= 32 || K % (2 * kWaves * kChunk)) return {0, 0, 1};
  const int64_t units = kvc_device_compute_units();
  auto rounds = [&](int64_t blocks) { return static_cast<double>((blocks + units - 1) / units); };
  const FewShape few = few_shape(M, N);
  const int live = few.mt < (M + 15) / 16 ? few.mt : (M + 15) / 16;  // row blocks that are not copies of the last
  double least = 2.7 + rounds(few.blocks) * (0.3 * few.nt * few.mt + 0.45 * (K / (kWaves * kChunk)) * (few.nt + live));
  SharedShape best{0, 0, 1};
  for (int nt = 1; nt <= 2; ++nt) {
    const int64_t blocks = (static_cast<int64_t>(N) + 64 * nt - 1) / (64 * nt) * ((M + 63) / 64);
    for (int groups = 1; groups <= kWaves; groups *= 2) {
      if (groups > 1 && static_cast<int64_t>(M) * N > units * 64 * 128) break;
      const double r = rounds(blocks * groups);
      double us = 5.3 + 0.8 * r + K / kChunk / groups * (nt == 1 ? 0.49 + 0.45 * (r - 1) : 0.89 + 0.735 * (r - 1));
      if (groups > 1) us += 1.1 + 12e-6 * M * N;
      if (us < least) least = us, best = {nt, groups, 1};
      if (groups == 1 && nt == 2 && r == 1) {
        us = 7.4 + K / kChunk * 0.79;
        if (us < least) least = us, best = {nt, groups, 2};
      }
    }
  }
  return best;
}

}  // namespace

extern "C" int64_t kvc_gemm_f32_parts_floats(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || shared_shape(M, N, K).groups < 2) return 0;
  return static_cast<int64_t>(kWaves) * M * ((static_cast<int64_t>(N) + 3) & ~3);
}

extern "C" int kvc_gemm_f32(float* C, const float* A, const float* W, const float* bias, int M,
                            int N, int K, int64_t lda, int64_t ldc, float* parts, int64_t parts_floats, kvc_stream stream) {
  if (M < 0 || N <= 0 || K <= 0 || lda < K || ldc < N) return kvc_fail("kvc_gemm_f32: bad sizes");
  if (parts_floats < kvc_gemm_f32_parts_floats(M, N, K) || (reinterpret_cast<uintptr_t>(parts) & 15) != 0)
    return kvc_fail("kvc_gemm_f32: the workspace is too small or not 16-byte aligned");
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
    // 64 rows a wave where the operands' way to it counts and two blocks a unit are left: 4,096 rows of 8192 x 256 185 ->
    // 172 us (in smaller pieces, of 8192 x 100, 146 -> 167)
    int mt = M <= 16 ? 1 : 2, nt = 4;
    if (piece == 8 && chunks > 2 && static_cast<int64_t>((N + 255) / 256) * ((M + 63) / 64) >= 2 * units) mt = 4;
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
      KVC_F32_LAUNCH((gemm_f32_short_kernel<4, 4, 8>), 256);  // blocks enough
    }
#undef KVC_F32
    return kvc_check_launch("kvc_gemm_f32");
  }
  const SharedShape shape = piece == 8 ? shared_shape(M, N, K) : SharedShape{0, 0, 1};
  if (shape.nt) {
    const int cols = 64 * shape.nt, rows = 16 * kSharedRows;
    const dim3 grid((N + cols - 1) / cols, (M + rows - 1) / rows, shape.groups);
    if (grid.y > 65535) return kvc_fail("kvc_gemm_f32: M too large for one launch");
    const bool left = shape.groups > 1;
#define KVC_F32_SHARED(NT, LEAVE, HALVES)                                                                                   \
  hipLaunchKernelGGL((gemm_f32_shared_kernel<kSharedRows, NT, LEAVE, HALVES>), grid, dim3(256 * HALVES), 0,                 \
                     reinterpret_cast<hipStream_t>(stream), C, A, W, bias, parts, M, N, K, lda, ldc)
    if (left && shape.nt == 2) KVC_F32_SHARED(2, true, 1);
    else if (left) KVC_F32_SHARED(1, true, 1);
    else if (shape.nt == 2 && shape.halves == 2) KVC_F32_SHARED(2, false, 2);
    else if (shape.nt == 2) KVC_F32_SHARED(2, false, 1);
    else KVC_F32_SHARED(1, false, 1);
#undef KVC_F32_SHARED
    if (left) {
      const int64_t quads = static_cast<int64_t>(M) * ((N + 3) / 4);
      hipLaunchKernelGGL(gemm_f32_parts_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0,
                         reinterpret_cast<hipStream_t>(stream), C, A, W, bias, parts, chunks < kWaves ? chunks : kWaves, M, N,
                         K, lda, ldc);
    }
    return kvc_check_launch("kvc_gemm_f32");
  }
  const FewShape few = few_shape(M, N);
  const int nt = few.nt, mt = few.mt;
  const dim3 grid((N + 16 * nt - 1) / (16 * nt), (M + 16 * mt - 1) / (16 * mt));
  if (grid.y > 65535) return kvc_fail("kvc_gemm_f32: M too large for one launch");
#define KVC_F32(NT, MT, AHEAD)                                                                                        \
  do {                                                                                                                \
    if (piece != 8) KVC_F32_LAUNCH((gemm_f32_kernel<NT, MT, 1, 1, false>), kWaves * 64);                              \
    else if (chunks <= kWaves * AHEAD) KVC_F32_LAUNCH((gemm_f32_kernel<NT, MT, AHEAD, 8, true>), kWaves * 64);        \
    else KVC_F32_LAUNCH((gemm_f32_kernel<NT, MT, AHEAD, 8, false>), kWaves * 64);                                     \
  } while (0)
  if (mt == 4) {
    if (nt == 4) KVC_F32(4, 4, 1);
    else KVC_F32(2, 4, 1);
  } else if (mt == 2) {
    if (nt == 4) KVC_F32(4, 2, 1);
    else if (nt == 2) KVC_F32(2, 2, 2);
    else KVC_F32(1, 2, 2);
  } else {
    if (nt == 4) KVC_F32(4, 1, 2);
    else if (nt == 2) KVC_F32(2, 1, 2);
    else if (chunks <= 2 * kWaves) KVC_F32(1, 1, 2);
    else KVC_F32(1, 1, 4);
  }
#undef KVC_F32
#undef KVC_F32_LAUNCH
  return kvc_check_launch("kvc_gemm_f32");
}
