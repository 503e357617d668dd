// Matrix states whose decay changes from token to token, over portions of prompts: chunks of 64 tokens side by
// side instead of token by token.
//
//   kScalar  S <- g_t S + b_t k_t v_t^T         (g_t and b_t a number a head; a column of ones beside v if wanted)
//   kSpace   the same with g_t = exp(-exp(A_log) dt), b_t = dt = softplus(dt_raw + dt_bias), k = B, q = C, v = x,
//            and D x added to the result (the state-space recurrence; its state lies row by row)
//   o_t = S^T (q_scale q_t), read after the token's write.  For the tokens i of a chunk, S the state before it:
//
//   o_i = (g_0 .. g_i) S^T q_i + sum_{j <= i} (g_(j+1) .. g_i) b_j (k_j . q_i) v_j
//   S_after = (g_0 .. g_(n-1)) S + sum_j (g_(j+1) .. g_(n-1)) b_j k_j v_j^T
//
// Three kernels, as for a fixed decay (chunked_state.hip): every chunk's own sum into a workspace, with the
// chunk's whole decay; a walk over a request's chunks, which leaves the state before each of them in the
// workspace and the last one in the request's slot; every chunk's results.  Products are float32 matrix
// instructions with float32 operands, and every decay between two tokens is a product of the factors between
// them (inside a run of 16 tokens one by one, across runs by the runs' own products), never a quotient and never
// an exponential of a sum, so no decay is too fast for a chunk and a factor of zero is one.  Inside a chunk the products
// are made in 64 bits and rounded once, and no sum has more than eight terms in a row (a matrix instruction's four
// count as one): in 32 bits the decays left 4e-7 of error where the scan has 2e-7, and with the runs' products in 32
// bits and sums in one chain the results of 64 heads of 128 x 64 had 1.1 to 1.3 times the scan's error (256 tokens 0.90e-7
// and 0.69e-7; now 0.69e-7; matrix memories of 64 x 129 1.77e-7 and 1.74e-7; now 1.20e-7).  The walk from chunk to
// chunk rounds to 32 bits, once a chunk where the scan does once a token.  Chunks are counted from a request's first
// token in the step.
//
// The scan walks 2,048 tokens one after the other, some 180 ns each, on as many blocks as there are heads times
// tiles of values; here a chunk of a head is a block.  2,048 tokens of one request: 16 heads of 64 x 129 405 -> 59 us
// (sums 16, walk 9, results 33), 64 heads of 128 x 64 in 8 groups 376 -> 133 us (sums 49, walk 24, scores 7, results
// 53; the states' way to and from the workspace is 67 MB four times).  Loading the state before the chunk ahead of
// the chunk's own keys cost more waves than it hid (results 105 -> 122 us); scores once for the heads that share
// them brought 105 -> 56; two running sums for the state's part of the results, as the chunks' sums have them, instead
// of sums of eight terms took registers that cost waves (16 heads of 64 x 129 58.6 -> 70.1 us).

#include <hip/hip_runtime.h>

#include "device_utils.h"
#include "gemm_common.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

#define S(stream) reinterpret_cast<hipStream_t>(stream)

constexpr int kChunk = 64;
constexpr int kRun = 16;        // tokens whose decays are multiplied one by one
constexpr int kRuns = kChunk / kRun;
constexpr int kPad = 4;         // floats between rows in LDS
constexpr int kMostKeys = 128;  // rows of a state
constexpr int kScalar = 1, kSpace = 2, kChannel = 3;

__device__ __forceinline__ float softplus_of(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

struct GatedArgs {
  float* out;         // [T, nh * dv]
  const float* q;     // rows of nqk heads of d
  int64_t q_stride;
  const float* k;
  int64_t k_stride;
  const float* v;     // rows of nh heads of dv - ones values
  int64_t v_stride;
  const float* keep;  // kScalar: g [T, nh]; kChannel: [T, nh * d]
  int64_t keep_stride;
  const float* take;  // kScalar: b [T, nh], none: ones
  int64_t take_stride;
  const void* dt;     // kSpace: [T, nh] float32 or bfloat16
  int64_t dt_stride;
  int dt_bf16;
  const float* dt_bias;
  const float* a_log;
  const float* skip;
  float* work;        // [chunks][nh][dpad / 4][dv][4], then the chunks' whole decays [chunks][nh]
  float* decays;      // kChannel: [chunks][nh][dpad]
  float* scores;      // [chunks][nqk][64 queries][64 keys]: k . q of the heads that share both (else unused)
  float* state;       // [slots][nh][dpad / 4][dv][4]; kSpace: [slots][nh][d][dv]
  const int32_t* positions;
  const int32_t* token_req;
  const int32_t* q_start;
  const int32_t* slots;
  int R, nh, nqk, d, dv, dpad, ones;
  int from;           // requests of fewer tokens are left out
  float q_scale;
};

// Which request and which of its chunks the block `index` works on: first token and token count (0: none).
// Every lane looks at a request.
struct ChunkPlace {
  int t0, n;
};
__device__ __forceinline__ ChunkPlace find_chunk(const GatedArgs& a, int index) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int base = 0; base < a.R; base += kWave) {
    const int r = base + lane;
    const int b = r < a.R ? a.q_start[r] : 0, e = r < a.R ? a.q_start[r + 1] : 0;
    const int mine = e - b >= a.from ? (e - b + kChunk - 1) / kChunk : 0;
    int upto = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int other = __shfl_up(upto, o, kWave);
      if (lane >= o) upto += other;
    }
    const uint64_t has = __ballot(index < upto);
    if (has) {
      const int who = __ffsll(static_cast<unsigned long long>(has)) - 1;
      const int t0 = __builtin_amdgcn_readlane(b + (index - (upto - mine)) * kChunk, who);
      const int end = __builtin_amdgcn_readlane(e, who);
      return {t0, end - t0 < kChunk ? end - t0 : kChunk};
    }
    index -= __builtin_amdgcn_readlane(upto, kWave - 1);
  }
  return {0, 0};
}

// g and b of token i (threads 0 to 63) of the chunk; tokens that are not there neither decay nor write
template <int GATES>
__device__ __forceinline__ void gates_of(const GatedArgs& a, const ChunkPlace& at, int h, int i, float& g, float& b) {
  g = 1.f;
  b = 0.f;
  if (i >= at.n) return;
  const int64_t t = at.t0 + i;
  if constexpr (GATES == kSpace) {
    const int64_t idx = t * a.dt_stride + h;
    const float raw = a.dt_bf16 ? to_float(static_cast<const bf16_t*>(a.dt)[idx]) : static_cast<const float*>(a.dt)[idx];
    b = softplus_of(raw + a.dt_bias[h]);
    g = expf(-expf(a.a_log[h]) * b);
  } else {
    g = a.keep[t * a.keep_stride + h];
    b = a.take != nullptr ? a.take[t * a.take_stride + h] : 1.f;
  }
}

// Rows of the chunk's tokens (in sixteens), `size` columns of a head, into LDS rows of PADDED + kPad floats, zeros
// where there is no token or no column; with `one` >= 0 that column is a one for every token that is there.  In two
// halves, so that a thread's loads are all on their way before the first of them is waited for.
template <int VEC, int PADDED>
struct Staged {
  static constexpr int kGroups = PADDED / 4, kEach = (kChunk * kGroups + 255) / 256;
  f32x4_t x[kEach];
  __device__ __forceinline__ void fetch(const float* src, int64_t stride, const ChunkPlace& at, int size) {
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int idx = threadIdx.x + 256 * j, i = idx / kGroups, c = 4 * (idx - i * kGroups);
      x[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (i < at.n) {
        const float* p = src + (at.t0 + i) * stride + c;
        if (VEC) {
          if (c < size) x[j] = *reinterpret_cast<const f32x4_t*>(p);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < size) x[j][e] = p[e];
        }
      }
    }
  }
  // returns whether a value that is not finite went by
  __device__ __forceinline__ bool stash(float* dst, const ChunkPlace& at, int one) const {
    const int rows = (at.n + 15) & ~15;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int idx = threadIdx.x + 256 * j, i = idx / kGroups, c = 4 * (idx - i * kGroups);
      if (i >= rows) continue;
      f32x4_t v = x[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bad |= !(fabsf(v[e]) < INFINITY);
        if (c + e == one && i < at.n) v[e] = 1.f;
      }
      *reinterpret_cast<f32x4_t*>(dst + i * (PADDED + kPad) + c) = v;
    }
    return bad;
  }
};

// Sixteen terms of a product's sums, four of each lane's, in two sums of eight (all of a result's terms in a row would
// round too often).
template <typename TA, typename TB>
__device__ __forceinline__ f32x4_t sixteen_terms(const TA& x, const TB& y) {
  f32x4_t t[2] = {};
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], t[i & 1], 0, 0, 0);
  return t[0] + t[1];
}

// ---- every chunk's own sum.  Wave w takes the key channels 16 (w + 4 m) .., all of the block's columns.
template <int GATES, int NM, int NC, int VEC>
__global__ __launch_bounds__(256) void gated_sums_kernel(const GatedArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int kCols = 16 * NC, kVRow = kCols + kPad;
  const ChunkPlace at = find_chunk(a, blockIdx.x);
  if (at.n == 0 || a.token_req[at.t0] < 0) return;  // nothing here, or padding: the same for the whole block
  const int h = blockIdx.y, c0 = blockIdx.z * kCols;
  const int hk = h / (a.nh / a.nqk);
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int kKeys = 64 * NM, krow = kKeys + kPad;
  const int dvin = a.dv - a.ones;
  const int cols = dvin - c0 < kCols ? dvin - c0 : kCols;
  Staged<VEC, kKeys> keys;
  Staged<VEC, kCols> values;
  keys.fetch(a.k + static_cast<int64_t>(hk) * a.d, a.k_stride, at, a.d);
  values.fetch(a.v + static_cast<int64_t>(h) * dvin + c0, a.v_stride, at, cols);
  float* k_s = lds;                  // [64][krow]
  float* v_s = k_s + kChunk * krow;  // [64][kVRow]
  float* pw = v_s + kChunk * kVRow;  // [64] weight of token j
  if (tid < kChunk) {  // the first wave: the product of the factors behind each token
    float g, b;
    gates_of<GATES>(a, at, h, tid, g, b);
    double p = g;  // of this token's factor and those behind it
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const double other = __shfl_down(p, o, kWave);
      if (tid + o < kWave) p *= other;
    }
    const double behind = __shfl_down(p, 1, kWave);
    pw[tid] = static_cast<float>(tid < kWave - 1 ? behind : 1.0) * b;
    if (tid == 0 && blockIdx.z == 0) a.decays[static_cast<int64_t>(blockIdx.x) * a.nh + h] = static_cast<float>(p);
  }
  keys.stash(k_s, at, -1);
  values.stash(v_s, at, a.ones ? dvin - c0 : -1);
  __syncthreads();
  f32x4_t acc[NM][NC][2] = {};  // two sums, so that none has all of the terms in a row
  const int steps = (at.n + 15) / 16;
  for (int s = 0; s < steps; ++s) {
    float ka[NM][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = 16 * s + 4 * lk + i;
      const float w = pw[j];
#pragma unroll
      for (int m = 0; m < NM; ++m) ka[m][i] = k_s[j * krow + 16 * (wave + 4 * m) + li] * w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float vb[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) vb[c] = v_s[(16 * s + 4 * lk + i) * kVRow + 16 * c + li];
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          acc[m][c][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[m][i], vb[c], acc[m][c][i & 1], 0, 0, 0);
    }
  }
  // lane holds column li and key channels 4 lk .. of its tiles: four rows of one column, one 16-byte store
  float* dst = a.work + (static_cast<int64_t>(blockIdx.x) * a.nh + h) * a.dpad * a.dv;
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const int n = 16 * (wave + 4 * m) + 4 * lk;
    if (n >= a.dpad) continue;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int col = c0 + 16 * c + li;
      if (col < a.dv) *reinterpret_cast<f32x4_t*>(dst + (static_cast<int64_t>(n >> 2) * a.dv + col) * 4) = acc[m][c][0] + acc[m][c][1];
    }
  }
}

// ---- the walk over a request's chunks: a thread four rows of one column
template <int GATES>
__global__ __launch_bounds__(256) void gated_walk_kernel(const GatedArgs a) {
  const int r = blockIdx.x, h = blockIdx.y;
  const int b = a.q_start[r], e = a.q_start[r + 1];
  if (e <= b || e - b < a.from || a.token_req[b] < 0) return;
  // the request's first chunk in the workspace: the wave's lanes count the requests before it
  int first = 0;
  for (int p = threadIdx.x & (kWave - 1); p < r; p += kWave) {
    const int n = a.q_start[p + 1] - a.q_start[p];
    first += n >= a.from ? (n + kChunk - 1) / kChunk : 0;
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) first += __shfl_xor(first, o, kWave);
  const int fours = a.dpad / 4 * a.dv;
  const int idx = blockIdx.z * blockDim.x + threadIdx.x;
  if (idx >= fours) return;
  const int chunks = (e - b + kChunk - 1) / kChunk;
  const int n = idx / a.dv * 4, col = idx - idx / a.dv * a.dv;
  const int64_t head = static_cast<int64_t>(a.slots[r]) * a.nh + h;
  float* st = a.state + (GATES == kSpace ? head * a.d * a.dv + static_cast<int64_t>(n) * a.dv + col
                                         : head * a.dpad * a.dv + static_cast<int64_t>(idx) * 4);
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  if (a.positions[b] != 0) {  // the same for the whole block
    if (GATES == kSpace) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < a.d) s[i] = st[static_cast<int64_t>(i) * a.dv];
    } else {
      s = *reinterpret_cast<const f32x4_t*>(st);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i >= a.d) s[i] = 0.f;  // rows that pad the state are never written by anyone else
    }
  }
  const int64_t step = static_cast<int64_t>(a.nh) * a.dpad * a.dv;
  float* w = a.work + (static_cast<int64_t>(first) * a.nh + h) * a.dpad * a.dv + static_cast<int64_t>(idx) * 4;
  constexpr bool kFours = GATES == kChannel;  // a factor for each of the four rows
  const float* whole = kFours ? a.decays + (static_cast<int64_t>(first) * a.nh + h) * a.dpad + n
                              : a.decays + static_cast<int64_t>(first) * a.nh + h;
  constexpr int kAhead = 8;
  for (int c0 = 0; c0 < chunks; c0 += kAhead) {
    f32x4_t own[kAhead], g[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = c0 + i < chunks ? c0 + i : chunks - 1;
      own[i] = *reinterpret_cast<const f32x4_t*>(w + c * step);
      if (kFours) {
        g[i] = *reinterpret_cast<const f32x4_t*>(whole + static_cast<int64_t>(c) * a.nh * a.dpad);
      } else {
        const float one = whole[static_cast<int64_t>(c) * a.nh];
        g[i] = f32x4_t{one, one, one, one};
      }
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = c0 + i;
      if (c < chunks) {
        *reinterpret_cast<f32x4_t*>(w + c * step) = s;
        s = s * g[i] + own[i];
      }
    }
  }
  if (GATES == kSpace) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < a.d) st[static_cast<int64_t>(i) * a.dv] = s[i];
  } else {
    *reinterpret_cast<f32x4_t*>(st) = s;
  }
}

// A query's values in registers: NS runs of sixteen channels, of which a lane holds four (zeros for a query that is
// not there).
template <int NS, int VEC>
__device__ __forceinline__ void fetch_query(f32x4_t* qv, const GatedArgs& a, const ChunkPlace& at, int hk, int query, int lk) {
  const bool live = query < at.n;
  const float* p = a.q + (at.t0 + (live ? query : 0)) * a.q_stride + static_cast<int64_t>(hk) * a.d + 4 * lk;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    qv[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int n = 16 * s + 4 * lk;
    if (VEC) {
      if (n < a.d) qv[s] = *reinterpret_cast<const f32x4_t*>(p + 16 * s);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < a.d) qv[s][e] = p[16 * s + e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) qv[s][e] = live ? qv[s][e] * a.q_scale : 0.f;
  }
}
// k . q of sixteen keys (k_s: the first one's row) and the wave's sixteen queries; eight running sums: an instruction
// does not wait for the one before it, and no sum is long.  Lane holds query li, keys 4 lk + i.
template <int NS>
__device__ __forceinline__ f32x4_t score_tile(const float* k_s, const f32x4_t* qv, int d, int li, int lk) {
  constexpr int krow = 16 * NS + kPad;
  f32x4_t sum[4][2] = {};
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (16 * s < d) {  // scalar
      const f32x4_t kv = *reinterpret_cast<const f32x4_t*>(k_s + li * krow + 16 * s + 4 * lk);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sum[s & 3][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i], qv[s][i], sum[s & 3][i & 1], 0, 0, 0);
    }
  }
  return ((sum[0][0] + sum[0][1]) + (sum[1][0] + sum[1][1])) + ((sum[2][0] + sum[2][1]) + (sum[3][0] + sum[3][1]));
}

// ---- the scores of a chunk for heads that share queries and keys, once for all of them
template <int NS, int VEC>
__global__ __launch_bounds__(256) void gated_scores_kernel(const GatedArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const ChunkPlace at = find_chunk(a, blockIdx.x);
  if (at.n == 0 || a.token_req[at.t0] < 0) return;
  const int hk = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int krow = 16 * NS + kPad;
  f32x4_t qv[NS];
  fetch_query<NS, VEC>(qv, a, at, hk, 16 * wave + li, lk);
  {
    Staged<VEC, 16 * NS> keys;
    keys.fetch(a.k + static_cast<int64_t>(hk) * a.d, a.k_stride, at, a.d);
    keys.stash(lds, at, -1);
  }
  __syncthreads();
  if (16 * wave >= at.n) return;  // scalar
  float* dst = a.scores + ((static_cast<int64_t>(blockIdx.x) * a.nqk + hk) * kChunk + 16 * wave + li) * kChunk + 4 * lk;
  for (int kt = 0; kt <= wave; ++kt)  // scalar
    *reinterpret_cast<f32x4_t*>(dst + 16 * kt) = score_tile<NS>(lds + 16 * kt * krow, qv, a.d, li, lk);
}

// For token `tid` of a chunk: the factors between it and each later token of its run (`inside`, a row a later token),
// those from the run's start on (`from_start`) and those behind it (`to_end`).
__device__ __forceinline__ void run_products(const float* g_s, float* inside, double* from_start, double* to_end, int tid) {
  const int run = tid / kRun * kRun, j = tid - run;
  const double first = g_s[run];
  double p = 1.0;
#pragma unroll
  for (int i = 0; i < kRun; ++i) {
    if (i > j) p *= static_cast<double>(g_s[run + i]);
    inside[(run + i) * (kRun + 1) + j] = i >= j ? static_cast<float>(p) : 0.f;
    if (j == 0) from_start[run + i] = first * p;
  }
  to_end[tid] = p;
}

// ---- every chunk's results.  Wave w takes the queries 16 w .. 16 w + 15 (an operand's columns).  SHARED: the
// scores are there already.
template <int GATES, int NS, int NC, int VEC, int SHARED>
__global__ __launch_bounds__(256) void gated_results_kernel(const GatedArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int kCols = 16 * NC, kVRow = kCols + kPad;
  const ChunkPlace at = find_chunk(a, blockIdx.x);
  if (at.n == 0) return;
  const int h = blockIdx.y, c0 = blockIdx.z * kCols;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int out_cols = a.dv - c0 < kCols ? a.dv - c0 : kCols;
  const int width = a.nh * a.dv;
  if (a.token_req[at.t0] < 0) {  // padding rows: zeros
    for (int idx = tid; idx < at.n * out_cols; idx += blockDim.x) {
      const int i = idx / out_cols, c = idx - i * out_cols;
      a.out[static_cast<int64_t>(at.t0 + i) * width + h * a.dv + c0 + c] = 0.f;
    }
    return;
  }
  const int hk = h / (a.nh / a.nqk);
  constexpr int krow = 16 * NS + kPad;
  float* v_s = lds;                      // [64][kVRow]
  float* g_s = v_s + kChunk * kVRow;     // [64] factors
  float* b_s = g_s + kChunk;             // [64] what a token writes with
  double* from_start = reinterpret_cast<double*>(b_s + kChunk);  // [64] factors from the run's start to the token
  double* to_end = from_start + kChunk;  // [64] factors behind the token to the run's end
  float* inside = reinterpret_cast<float*>(to_end + kChunk);  // [64][17] factors between a token and each one before it in its run
  float* k_s = inside + kChunk * (kRun + 1);  // [64][krow], not with SHARED
  const int query = 16 * wave + li;
  const bool live = query < at.n;
  f32x4_t qv[NS];
  fetch_query<NS, VEC>(qv, a, at, hk, query, lk);
  const int dvin = a.dv - a.ones;
  const int cols = dvin - c0 < kCols ? dvin - c0 : kCols;
  bool bad;
  {
    Staged<VEC, SHARED ? 4 : 16 * NS> keys;
    Staged<VEC, kCols> values;
    if (!SHARED) keys.fetch(a.k + static_cast<int64_t>(hk) * a.d, a.k_stride, at, a.d);
    values.fetch(a.v + static_cast<int64_t>(h) * dvin + c0, a.v_stride, at, cols);
    if (tid < kChunk) gates_of<GATES>(a, at, h, tid, g_s[tid], b_s[tid]);
    if (!SHARED) keys.stash(k_s, at, -1);
    bad = values.stash(v_s, at, a.ones ? dvin - c0 : -1);
  }
  bad = __syncthreads_or(bad);  // the same for the whole block
  if (tid < kChunk) run_products(g_s, inside, from_start, to_end, tid);
  __syncthreads();
  if (16 * wave >= at.n) return;  // scalar; no barrier follows

  // the state before the chunk: S^T q
  const float* st = a.work + (static_cast<int64_t>(blockIdx.x) * a.nh + h) * a.dpad * a.dv;
  f32x4_t far[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) far[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (16 * s < a.d) {  // scalar
      const int n = 16 * s + 4 * lk;
      const int row = n < a.dpad ? n >> 2 : 0;  // rows beyond read the first: their q is zero
      f32x4_t sv[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int col = c0 + 16 * c + li;
        sv[c] = *reinterpret_cast<const f32x4_t*>(st + (static_cast<int64_t>(row) * a.dv + (col < a.dv ? col : c0)) * 4);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) far[c] += sixteen_terms(sv[c], qv[s]);
    }
  }
  // the chunk's own keys up to the query, run by run, the query's own run first
  f32x4_t own[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) own[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const float* shared = a.scores + ((static_cast<int64_t>(blockIdx.x) * a.nqk + hk) * kChunk + query) * kChunk + 4 * lk;
  double reach = from_start[query];  // factors from the start of the run after kt to the query
  for (int kt = wave; kt >= 0; --kt) {  // scalar
    // lane holds query li, keys 4 lk + i of the run: the operand order of the next product
    f32x4_t score = SHARED ? *reinterpret_cast<const f32x4_t*>(shared + 16 * kt)
                           : score_tile<NS>(k_s + 16 * kt * krow, qv, a.d, li, lk);
    const f32x4_t b = *reinterpret_cast<const f32x4_t*>(b_s + 16 * kt + 4 * lk);
    if (kt == wave) {  // scalar
#pragma unroll
      for (int i = 0; i < 4; ++i)
        score[i] = 4 * lk + i <= li ? score[i] * inside[query * (kRun + 1) + 4 * lk + i] * b[i] : 0.f;
      if (bad) {
        // a value that is not finite: a later key's zero times it would reach this query, so key by key
        for (int j = 0; j < kRun; ++j) {
          const float mine = __shfl(j & 2 ? (j & 1 ? score[3] : score[2]) : (j & 1 ? score[1] : score[0]), 16 * (j >> 2) + li, kWave);
          if (j <= li)
#pragma unroll
            for (int c = 0; c < NC; ++c) own[c] += mine * *reinterpret_cast<const f32x4_t*>(v_s + (16 * kt + j) * kVRow + 16 * c + 4 * lk);
        }
        continue;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) score[i] *= static_cast<float>(reach * to_end[16 * kt + 4 * lk + i]) * b[i];
      reach *= from_start[16 * kt + kRun - 1];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float vb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) vb[i] = v_s[(16 * kt + 4 * lk + i) * kVRow + 16 * c + li];
      own[c] += sixteen_terms(vb, score);
    }
  }
  if (!live) return;
  float* o = a.out + static_cast<int64_t>(at.t0 + query) * width + static_cast<int64_t>(h) * a.dv + c0;
  const bool vec_out = (a.dv & 3) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
  const float skip = GATES == kSpace ? a.skip[h] : 0.f, all = static_cast<float>(reach);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    f32x4_t y = far[c] * all + own[c];
    const int col = 16 * c + 4 * lk;
    if (GATES == kSpace) y += skip * *reinterpret_cast<const f32x4_t*>(v_s + query * kVRow + col);
    if (vec_out) {
      if (col < out_cols) *reinterpret_cast<f32x4_t*>(o + col) = y;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < out_cols) o[col + e] = y[e];
    }
  }
}

// ================================================= a factor per key channel: S <- diag(a_t) S + k_t v_t^T
// The same three kernels.  A wave takes a run of 16 tokens into registers as an operand lies (lane: token li, channels
// 16 s + 4 lk + e), so that products of factors along the run are scans over the 16 lanes of a row.  Scores of a run
// with an earlier one: (q . factors from the run's start) (k . factors to its run's end) with the whole runs between
// multiplied into the query on the way; inside a run, pair by pair on the vector unit, the key's row multiplied by one
// more factor for each later query.  Products of factors and the pairs' sums are made in 64 bits and rounded once, and
// no product's sum has more than eight terms in a row: in 32 bits and in long sums the results' error was 1.7 times the
// scan's, so they are the same (0.95e-7 and 0.94e-7 at 683 tokens of 64 x 128 with factors sigmoid(z)^(1/8)).
//
// 16 heads of 64 x 128, three requests of 683 tokens: 152 -> 82 us (sums 22, walk 9, results 50), 2,048 tokens of one
// 357 -> 68, 512 tokens 88 -> 39; bound by what a block does one after the other (a single chunk's results take 20 us,
// half of it the pairs) on two blocks a compute unit.

template <int NS, int VEC>
__device__ __forceinline__ void fetch_lane(f32x4_t* x, const float* row, bool live, int lk, int size, float none) {
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    x[s] = f32x4_t{none, none, none, none};
    const int n = 16 * s + 4 * lk;
    if (!live) continue;
    if (VEC) {
      if (n < size) x[s] = *reinterpret_cast<const f32x4_t*>(row + n);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < size) x[s][e] = row[n + e];
    }
  }
}
// a value from another lane of the row of 16, one where there is none
template <int CTRL>
__device__ __forceinline__ double row_or_one(double v) {
  const int64_t bits = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(bits), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0x3ff00000, static_cast<int>(bits >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(static_cast<int64_t>(hi) << 32 | static_cast<uint32_t>(lo));
}
__device__ __forceinline__ double product_up_to(double v) {  // of this lane's value and those before it in its row
  v *= row_or_one<0x111>(v);  // row_shr 1, 2, 4, 8
  v *= row_or_one<0x112>(v);
  v *= row_or_one<0x114>(v);
  v *= row_or_one<0x118>(v);
  return v;
}
__device__ __forceinline__ double product_behind(double v) {  // of the values behind this lane's in its row
  v = row_or_one<0x101>(v);  // row_shl 1, then 1, 2, 4, 8
  v *= row_or_one<0x101>(v);
  v *= row_or_one<0x102>(v);
  v *= row_or_one<0x104>(v);
  v *= row_or_one<0x108>(v);
  return v;
}

template <int NS, int NC, int VEC>
__global__ __launch_bounds__(256) void channel_sums_kernel(const GatedArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int kCols = 16 * NC, kVRow = kCols + kPad, kKeys = 16 * NS, krow = kKeys + kPad, NM = NS / 4;
  const ChunkPlace at = find_chunk(a, blockIdx.x);
  if (at.n == 0 || a.token_req[at.t0] < 0) return;
  const int h = blockIdx.y, c0 = blockIdx.z * kCols, hk = h / (a.nh / a.nqk);
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cols = a.dv - c0 < kCols ? a.dv - c0 : kCols;
  float* k_s = lds;                      // [64][krow], times the factors behind each token in the chunk
  float* v_s = k_s + kChunk * krow;      // [64][kVRow]
  double* whole = reinterpret_cast<double*>(v_s + kChunk * kVRow);  // [4][kKeys] a run's factors
  {
    const bool live = 16 * wave + li < at.n;
    const int64_t t = at.t0 + (live ? 16 * wave + li : 0);
    f32x4_t kv[NS], av[NS];
    fetch_lane<NS, VEC>(kv, a.k + t * a.k_stride + static_cast<int64_t>(hk) * a.d, live, lk, a.d, 0.f);
    fetch_lane<NS, VEC>(av, a.keep + t * a.keep_stride + static_cast<int64_t>(h) * a.d, live, lk, a.d, 1.f);
    Staged<VEC, kCols> values;
    values.fetch(a.v + static_cast<int64_t>(h) * a.dv + c0, a.v_stride, at, cols);
    double behind[NS][4];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        behind[s][e] = product_behind(av[s][e]);
        if (li == 0) whole[wave * kKeys + 16 * s + 4 * lk + e] = av[s][e] * behind[s][e];
      }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        for (int r = wave + 1; r < kRuns; ++r) behind[s][e] *= whole[r * kKeys + 16 * s + 4 * lk + e];  // scalar
        kv[s][e] = static_cast<float>(kv[s][e] * behind[s][e]);
      }
      *reinterpret_cast<f32x4_t*>(k_s + (16 * wave + li) * krow + 16 * s + 4 * lk) = kv[s];
    }
    values.stash(v_s, at, -1);
  }
  __syncthreads();
  f32x4_t acc[NM][NC];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[m][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; 16 * s < at.n; ++s) {  // scalar
    float ka[4][NM];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int m = 0; m < NM; ++m) ka[i][m] = k_s[(16 * s + 4 * lk + i) * krow + 16 * (wave + 4 * m) + li];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float vb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) vb[i] = v_s[(16 * s + 4 * lk + i) * kVRow + 16 * c + li];
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const float mine[4] = {ka[0][m], ka[1][m], ka[2][m], ka[3][m]};
        acc[m][c] += sixteen_terms(mine, vb);
      }
    }
  }
  const int64_t place = static_cast<int64_t>(blockIdx.x) * a.nh + h;
  float* dst = a.work + place * a.dpad * a.dv;
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const int tile = 16 * (wave + 4 * m);
    if (blockIdx.z == 0 && lk == 0 && tile + li < a.dpad) {
      const double* w = whole + tile + li;
      a.decays[place * a.dpad + tile + li] = static_cast<float>(w[0] * w[kKeys] * (w[2 * kKeys] * w[3 * kKeys]));
    }
    if (tile + 4 * lk >= a.dpad) continue;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int col = c0 + 16 * c + li;
      if (col < a.dv) *reinterpret_cast<f32x4_t*>(dst + (static_cast<int64_t>((tile >> 2) + lk) * a.dv + col) * 4) = acc[m][c];
    }
  }
}

// The pairs of a run whose query lies BY tokens behind the key, key li in lane li, over 64 channels: its row p takes that
// query's factors, and its products with the query are added up, in 64 bits.  (Lanes whose query would lie outside the
// run end up with zeros.)
template <int BY>
__device__ __forceinline__ void pair_step(float* sums, double (&p)[4][4], const f32x4_t* av, const f32x4_t* qv) {
  if constexpr (BY < kRun) {
    double sum[2] = {0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float query = qv[s][e];
        if constexpr (BY > 0) {  // row_shl: from the lane BY further on
          p[s][e] *= __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(av[s][e]), 0x100 + BY, 0xF, 0xF, true));
          query = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(query), 0x100 + BY, 0xF, 0xF, true));
        }
        sum[e & 1] = fma(p[s][e], static_cast<double>(query), sum[e & 1]);
      }
    float v = static_cast<float>(sum[0] + sum[1]);
    v += __shfl_xor(v, 16, kWave);
    v += __shfl_xor(v, 32, kWave);
    sums[BY] += v;
    pair_step<BY + 1>(sums, p, av, qv);
  }
}

template <int NS, int NC, int VEC>
__global__ __launch_bounds__(256) void channel_results_kernel(const GatedArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int kCols = 16 * NC, kVRow = kCols + kPad, kKeys = 16 * NS, krow = kKeys + kPad, kPairRow = kRun + 4;
  const ChunkPlace at = find_chunk(a, blockIdx.x);
  if (at.n == 0) return;
  const int h = blockIdx.y, c0 = blockIdx.z * kCols, hk = h / (a.nh / a.nqk);
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cols = a.dv - c0 < kCols ? a.dv - c0 : kCols;
  const int width = a.nh * a.dv;
  if (a.token_req[at.t0] < 0) {  // padding rows: zeros
    for (int idx = tid; idx < at.n * cols; idx += blockDim.x) {
      const int i = idx / cols, c = idx - i * cols;
      a.out[static_cast<int64_t>(at.t0 + i) * width + h * a.dv + c0 + c] = 0.f;
    }
    return;
  }
  float* k_s = lds;                        // [64][krow], times the factors behind each token in its run
  float* v_s = k_s + kChunk * krow;        // [64][kVRow]
  double* whole = reinterpret_cast<double*>(v_s + kChunk * kVRow);  // [4][kKeys] a run's factors
  float* pairs = reinterpret_cast<float*>(whole + 4 * kKeys);  // [64][kPairRow] scores of a query with its run's keys
  const int query = 16 * wave + li;
  const bool live = query < at.n;
  f32x4_t qv[NS];
  double far_q[NS][4];  // the query times the factors from the run at hand to it
  bool bad;
  {
    const int64_t t = at.t0 + (live ? query : 0);
    f32x4_t kv[NS], av[NS];
    fetch_lane<NS, VEC>(qv, a.q + t * a.q_stride + static_cast<int64_t>(hk) * a.d, live, lk, a.d, 0.f);
    fetch_lane<NS, VEC>(kv, a.k + t * a.k_stride + static_cast<int64_t>(hk) * a.d, live, lk, a.d, 0.f);
    fetch_lane<NS, VEC>(av, a.keep + t * a.keep_stride + static_cast<int64_t>(h) * a.d, live, lk, a.d, 1.f);
    Staged<VEC, kCols> values;
    values.fetch(a.v + static_cast<int64_t>(h) * a.dv + c0, a.v_stride, at, cols);
#pragma unroll
    for (int s = 0; s < NS; ++s) qv[s] = qv[s] * a.q_scale;
    float sums[kRun] = {};
#pragma unroll
    for (int half = 0; half < NS / 4; ++half) {
      double p[4][4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[s][e] = kv[4 * half + s][e];
      pair_step<0>(sums, p, av + 4 * half, qv + 4 * half);
    }
    // lane: key li of every query; of four neighbouring distances it stores number lk, and that distance's zeros for
    // the queries before the key
#pragma unroll
    for (int i = 0; i < kRun; i += 4) {
      const float mine = lk & 2 ? (lk & 1 ? sums[i + 3] : sums[i + 2]) : (lk & 1 ? sums[i + 1] : sums[i]);
      const int by = i + lk;
      if (li + by < kRun) pairs[(query + by) * kPairRow + li] = mine;
      if (by > 0 && li - by >= 0) pairs[(query - by) * kPairRow + li] = 0.f;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double upto = product_up_to(av[s][e]);
        far_q[s][e] = qv[s][e] * upto;
        if (li == kRun - 1) whole[wave * kKeys + 16 * s + 4 * lk + e] = upto;
        kv[s][e] = static_cast<float>(kv[s][e] * product_behind(av[s][e]));
        qv[s][e] = static_cast<float>(far_q[s][e]);
      }
      *reinterpret_cast<f32x4_t*>(k_s + query * krow + 16 * s + 4 * lk) = kv[s];
    }
    bad = values.stash(v_s, at, -1);
  }
  bad = __syncthreads_or(bad);  // the same for the whole block
  if (16 * wave >= at.n) return;  // scalar; no barrier follows
  f32x4_t own[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) own[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int kt = wave; kt >= 0; --kt) {  // scalar
    // lane holds query li, keys 4 lk + i of the run: the operand order of the next product
    f32x4_t score;
    if (kt == wave) {  // scalar
      score = *reinterpret_cast<const f32x4_t*>(pairs + query * kPairRow + 4 * lk);
      if (bad) {  // key by key: see gated_results_kernel
        for (int j = 0; j < kRun; ++j) {
          const float mine = pairs[query * kPairRow + j];
          if (j <= li)
#pragma unroll
            for (int c = 0; c < NC; ++c) own[c] += mine * *reinterpret_cast<const f32x4_t*>(v_s + (16 * kt + j) * kVRow + 16 * c + 4 * lk);
        }
        continue;
      }
    } else {
      score = score_tile<NS>(k_s + 16 * kt * krow, qv, a.d, li, lk);
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          far_q[s][e] *= whole[kt * kKeys + 16 * s + 4 * lk + e];
          qv[s][e] = static_cast<float>(far_q[s][e]);
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float vb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) vb[i] = v_s[(16 * kt + 4 * lk + i) * kVRow + 16 * c + li];
      own[c] += sixteen_terms(vb, score);
    }
  }
  // the state before the chunk; the queries carry every factor since by now
  const float* st = a.work + (static_cast<int64_t>(blockIdx.x) * a.nh + h) * a.dpad * a.dv;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (16 * s < a.d) {  // scalar
      const int n = 16 * s + 4 * lk;
      const int row = n < a.dpad ? n >> 2 : 0;  // rows beyond read the first: their q is zero
      f32x4_t sv[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int col = c0 + 16 * c + li;
        sv[c] = *reinterpret_cast<const f32x4_t*>(st + (static_cast<int64_t>(row) * a.dv + (col < a.dv ? col : c0)) * 4);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) own[c] += sixteen_terms(sv[c], qv[s]);
    }
  }
  if (!live) return;
  float* o = a.out + static_cast<int64_t>(at.t0 + query) * width + static_cast<int64_t>(h) * a.dv + c0;
  const bool vec_out = (a.dv & 3) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int col = 16 * c + 4 * lk;
    if (vec_out) {
      if (col < cols) *reinterpret_cast<f32x4_t*>(o + col) = own[c];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < cols) o[col + e] = own[c][e];
    }
  }
}

size_t gated_lds(int keys, int nc) {
  return sizeof(float) * (kChunk * (keys + kPad) + kChunk * (16 * nc + kPad) + 6 * kChunk + kChunk * (kRun + 1));
}

template <typename K>
int launch(K kernel, const GatedArgs& a, const dim3& grid, size_t lds, hipStream_t stream) {
  if (lds > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
    return kvc_fail("gated chunks: the kernel's LDS size was refused");
  hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, a);
  return 0;
}

template <int GATES, int NS, int NC, int VEC>
int run_results(const GatedArgs& a, const dim3& grid, hipStream_t stream) {
  if (a.nqk == a.nh) return launch(gated_results_kernel<GATES, NS, NC, VEC, 0>, a, grid, gated_lds(16 * NS, NC), stream);
  const size_t lds = sizeof(float) * kChunk * (16 * NS + kPad);
  const int code = launch(gated_scores_kernel<NS, VEC>, a, dim3(grid.x, a.nqk), lds, stream);
  return code ? code : launch(gated_results_kernel<GATES, NS, NC, VEC, 1>, a, grid, gated_lds(-kPad, NC), stream);
}

template <int GATES, int NC, int VEC>
int run_chunks(const GatedArgs& a, int chunks, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(chunks), a.nh, (a.dv + 16 * NC - 1) / (16 * NC));
  int code = 0;
  if (a.d <= 64) code = launch(gated_sums_kernel<GATES, 1, NC, VEC>, a, grid, gated_lds(64, NC), stream);
  else code = launch(gated_sums_kernel<GATES, 2, NC, VEC>, a, grid, gated_lds(128, NC), stream);
  if (code) return code;
  const int fours = a.dpad / 4 * a.dv;
  hipLaunchKernelGGL(gated_walk_kernel<GATES>, dim3(a.R, a.nh, (fours + 255) / 256), dim3(256), 0, stream, a);
  if (a.d <= 32) return run_results<GATES, 2, NC, VEC>(a, grid, stream);
  if (a.d <= 64) return run_results<GATES, 4, NC, VEC>(a, grid, stream);
  return run_results<GATES, 8, NC, VEC>(a, grid, stream);
}

template <int NS, int NC, int VEC>
int run_channel(const GatedArgs& a, int chunks, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(chunks), a.nh, (a.dv + 16 * NC - 1) / (16 * NC));
  const size_t lds = sizeof(float) * (kChunk * (16 * NS + kPad) + kChunk * (16 * NC + kPad) + 2 * 4 * 16 * NS);
  int code = launch(channel_sums_kernel<NS, NC, VEC>, a, grid, lds, stream);
  if (code) return code;
  const int fours = a.dpad / 4 * a.dv;
  hipLaunchKernelGGL(gated_walk_kernel<kChannel>, dim3(a.R, a.nh, (fours + 255) / 256), dim3(256), 0, stream, a);
  return launch(channel_results_kernel<NS, NC, VEC>, a, grid, lds + sizeof(float) * kChunk * (kRun + 4), stream);
}

int64_t channel_floats(int nh, int d, int dv) { return nh * (static_cast<int64_t>((d + 3) & ~3) * (dv + 1)); }

int64_t chunk_floats(int nh, int nqk, int d, int dv) {
  const int64_t all = nh * (static_cast<int64_t>((d + 3) & ~3) * dv + 1) + (nqk < nh ? static_cast<int64_t>(nqk) * kChunk * kChunk : 0);
  return (all + 3) & ~3;
}

// Tiles of 64 columns, or of 144 where they hold all of a head's columns in one: scores and staging are then paid
// for once.
template <int GATES>
int run(const GatedArgs& a, int64_t work_floats, int chunks, const char* who, hipStream_t stream) {
  if (a.work == nullptr || work_floats < chunks * chunk_floats(a.nh, a.nqk, a.d, a.dv))
    return kvc_fail("gated chunks: the workspace is too small");
  if (((reinterpret_cast<uintptr_t>(a.state) | reinterpret_cast<uintptr_t>(a.work)) & 15) != 0)
    return kvc_fail("gated chunks: state and workspace must be 16-byte aligned");
  GatedArgs b = a;
  b.scores = a.work + static_cast<int64_t>(chunks) * a.nh * a.dpad * a.dv;  // a multiple of four floats
  b.decays = b.scores + (a.nqk < a.nh ? static_cast<int64_t>(chunks) * a.nqk * kChunk * kChunk : 0);
  const bool vec = a.d % 4 == 0 && (a.dv - a.ones) % 4 == 0 && a.q_stride % 4 == 0 && a.k_stride % 4 == 0 &&
                   a.v_stride % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) | reinterpret_cast<uintptr_t>(a.v)) & 15) == 0;
  int code;
  if (a.dv > 64 && a.dv <= 144 && a.d <= 64)
    code = vec ? run_chunks<GATES, 9, 1>(b, chunks, stream) : run_chunks<GATES, 9, 0>(b, chunks, stream);
  else
    code = vec ? run_chunks<GATES, 4, 1>(b, chunks, stream) : run_chunks<GATES, 4, 0>(b, chunks, stream);
  return code ? code : kvc_check_launch(who);
}

}  // namespace

extern "C" int kvc_gated_chunk_tokens(void) { return kChunk; }
extern "C" int64_t kvc_gated_chunk_floats(int nh, int nqk, int d, int dv) { return chunk_floats(nh, nqk, d, dv); }

extern "C" int kvc_scalar_gate_chunks(float* out, const float* q, int64_t q_stride, const float* k, int64_t k_stride,
                                      const float* v, int64_t v_stride, const float* keep, int64_t keep_stride,
                                      const float* take, int64_t take_stride, float* state, float* work,
                                      int64_t work_floats, const int32_t* positions, const int32_t* token_req,
                                      const int32_t* q_start, const int32_t* slots, int chunks, int from, int R, int nh,
                                      int nqk, int d, int dv, float q_scale, int ones_column, kvc_stream stream) {
  if (chunks < 0 || R < 0 || nh <= 0 || nqk <= 0 || nh % nqk || d <= 0 || dv <= 0 || nh > 65535 || (ones_column && dv < 2))
    return kvc_fail("kvc_scalar_gate_chunks: bad sizes");
  if (d > kMostKeys) return kvc_fail("kvc_scalar_gate_chunks: at most 128 key channels a head");
  const int ones = ones_column ? 1 : 0;
  if (q_stride < static_cast<int64_t>(nqk) * d || k_stride < static_cast<int64_t>(nqk) * d ||
      v_stride < static_cast<int64_t>(nh) * (dv - ones) || keep_stride < nh || take_stride < nh)
    return kvc_fail("kvc_scalar_gate_chunks: rows too short for the heads");
  if (chunks == 0 || R == 0) return 0;
  GatedArgs a{};
  a.out = out; a.q = q; a.q_stride = q_stride; a.k = k; a.k_stride = k_stride; a.v = v; a.v_stride = v_stride;
  a.keep = keep; a.keep_stride = keep_stride; a.take = take; a.take_stride = take_stride;
  a.work = work; a.state = state;
  a.positions = positions; a.token_req = token_req; a.q_start = q_start; a.slots = slots;
  a.from = from; a.R = R; a.nh = nh; a.nqk = nqk; a.d = d; a.dv = dv; a.dpad = (d + 3) & ~3; a.ones = ones; a.q_scale = q_scale;
  return run<kScalar>(a, work_floats, chunks, "kvc_scalar_gate_chunks", S(stream));
}

extern "C" int64_t kvc_channel_chunk_floats(int nh, int d, int dv) { return channel_floats(nh, d, dv); }

extern "C" int kvc_channel_gate_chunks(float* out, const float* q, int64_t q_stride, const float* k, int64_t k_stride,
                                       const float* v, int64_t v_stride, const float* decay, int64_t decay_stride,
                                       float* state, float* work, int64_t work_floats, const int32_t* positions,
                                       const int32_t* token_req, const int32_t* q_start, const int32_t* slots, int chunks,
                                       int from, int R, int nh, int nqk, int d, int dv, float q_scale, kvc_stream stream) {
  if (chunks < 0 || R < 0 || nh <= 0 || nqk <= 0 || nh % nqk || d <= 0 || dv <= 0 || nh > 65535)
    return kvc_fail("kvc_channel_gate_chunks: bad sizes");
  if (d > kMostKeys) return kvc_fail("kvc_channel_gate_chunks: at most 128 key channels a head");
  if (q_stride < static_cast<int64_t>(nqk) * d || k_stride < static_cast<int64_t>(nqk) * d ||
      v_stride < static_cast<int64_t>(nh) * dv || decay_stride < static_cast<int64_t>(nh) * d)
    return kvc_fail("kvc_channel_gate_chunks: rows too short for the heads");
  if (chunks == 0 || R == 0) return 0;
  if (work == nullptr || work_floats < chunks * channel_floats(nh, d, dv))
    return kvc_fail("gated chunks: the workspace is too small");
  if (((reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(work)) & 15) != 0)
    return kvc_fail("gated chunks: state and workspace must be 16-byte aligned");
  GatedArgs a{};
  a.out = out; a.q = q; a.q_stride = q_stride; a.k = k; a.k_stride = k_stride; a.v = v; a.v_stride = v_stride;
  a.keep = decay; a.keep_stride = decay_stride; a.work = work; a.state = state;
  a.positions = positions; a.token_req = token_req; a.q_start = q_start; a.slots = slots;
  a.from = from; a.R = R; a.nh = nh; a.nqk = nqk; a.d = d; a.dv = dv; a.dpad = (d + 3) & ~3; a.q_scale = q_scale;
  a.decays = work + static_cast<int64_t>(chunks) * nh * a.dpad * dv;
  const bool vec = d % 4 == 0 && dv % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 &&
                   decay_stride % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                     reinterpret_cast<uintptr_t>(decay)) & 15) == 0;
  // all of a head's columns in one tile where it holds them: the pairs inside a run are then paid for once
  int code;
  if (d <= 64) {
    if (dv <= 64) code = vec ? run_channel<4, 4, 1>(a, chunks, S(stream)) : run_channel<4, 4, 0>(a, chunks, S(stream));
    else code = vec ? run_channel<4, 8, 1>(a, chunks, S(stream)) : run_channel<4, 8, 0>(a, chunks, S(stream));
  } else {
    code = vec ? run_channel<8, 8, 1>(a, chunks, S(stream)) : run_channel<8, 8, 0>(a, chunks, S(stream));
  }
  return code ? code : kvc_check_launch("kvc_channel_gate_chunks");
}

extern "C" int kvc_ssm_chunks(float* y, const float* xbc, int64_t xbc_stride, const void* dt_raw, int64_t dt_stride,
                              int dt_dtype, const float* dt_bias, const float* a_log, const float* d_skip, float* state,
                              float* work, int64_t work_floats, const int32_t* positions, const int32_t* token_req,
                              const int32_t* q_start, const int32_t* slots, int chunks, int from, int R, int nh, int P, int N,
                              int G, kvc_stream stream) {
  if (chunks < 0 || R < 0 || nh <= 0 || P <= 0 || N <= 0 || G <= 0 || nh % G || nh > 65535)
    return kvc_fail("kvc_ssm_chunks: bad sizes");
  if (N > kMostKeys) return kvc_fail("kvc_ssm_chunks: a state of more than 128 rows a head");
  if (dt_dtype != 0 && dt_dtype != 1) return kvc_fail("kvc_ssm_chunks: unknown dtype code");
  if (xbc_stride < static_cast<int64_t>(nh) * P + 2 * static_cast<int64_t>(G) * N || dt_stride < nh)
    return kvc_fail("kvc_ssm_chunks: rows too short");
  if (chunks == 0 || R == 0) return 0;
  GatedArgs a{};
  const int64_t inner = static_cast<int64_t>(nh) * P;
  a.out = y; a.v = xbc; a.k = xbc + inner; a.q = xbc + inner + static_cast<int64_t>(G) * N;
  a.q_stride = a.k_stride = a.v_stride = xbc_stride;
  a.dt = dt_raw; a.dt_stride = dt_stride; a.dt_bf16 = dt_dtype; a.dt_bias = dt_bias; a.a_log = a_log; a.skip = d_skip;
  a.work = work; a.state = state;
  a.positions = positions; a.token_req = token_req; a.q_start = q_start; a.slots = slots;
  a.from = from; a.R = R; a.nh = nh; a.nqk = G; a.d = N; a.dv = P; a.dpad = (N + 3) & ~3; a.ones = 0; a.q_scale = 1.f;
  return run<kSpace>(a, work_floats, chunks, "kvc_ssm_chunks", S(stream));
}
