// Routed experts: the router's choice, the arrangement of (token, choice) pairs by expert, the
// experts' two products over their own rows, and the weighted sum.
//
// Everything is decided on the device and every grid is sized by bounds known on the host (pairs =
// tokens x choices, tiles <= pairs / 16 + experts), so a step neither waits for the routing nor
// changes its launches with it: a captured step replays for any routing.
//
//   kvc_moe_route    scores = softmax(logits), sigmoid(logits) or the logits themselves in float32 (an
//                    optional bias per expert joins the logits); the choice is made on the scores plus
//                    an optional correction per expert: the `keep` groups that are worth most (a
//                    group's best choice score, or the sum of its best two); the `top` best experts of
//                    those groups (the lower index on a tie); weights = the chosen experts' plain
//                    scores / (their sum + 1e-20) * weight_scale, or (renormalize 0) the scores as they
//                    are * weight_scale, or, where the scores are the logits, the softmax over the chosen
//                    logits * weight_scale.  A wave a token.
//   kvc_moe_router   the router's product (float32 sums in one fixed order over rows of either dtype)
//                    and the choice in one kernel; a further row of the router's matrix may give one
//                    number a token, a sigmoid gate for an expert that every token runs.
//   kvc_moe_router_spread  the same and kvc_moe_align in kernels that spread the product over the chip.
//   kvc_moe_align    pairs sorted by expert: sorted[i] = pair index (token * top + choice), and a
//                    list of tiles of up to 16 (or 64, or 128) sorted rows that belong to one expert each.
//   kvc_moe_gemm     for every tile, rows x that expert's matrix.  Gated: gate and up rows of the
//                    expert side by side in one pass, and the activation
//                    min(g, limit) * sigmoid(alpha * g) * (clamp(u, -limit, limit) + up_shift) on the way
//                    out (an infinite limit, alpha 1 and up_shift 0: silu(g) * u).  Not gated: the rows as
//                    they are, or their square of relu.  row_scale: a number a pair that multiplies the
//                    pair's input (the sums, before any activation).
//                    bfloat16 operands go through the matrix cores (16 x 16 x 32, the expert's rows as
//                    the A operand, the tokens as B) with float32 sums; float32 operands, and rows
//                    that 16-byte loads do not divide, are summed in float32 in index order.  A row's sums do
//                    not depend on its place in a tile or on the rows beside it.  In bfloat16 their order is that of
//                    the kernel which the step's size chose (four shares of K added up, or one chain that starts at
//                    a place its expert and columns decide); in float32 it is the same in every step.
//   kvc_moe_combine  out[t] = sum_c weight[t, c] * y[t * top + c] (without weights: the plain sum) (+ up to two more row sets, the second
//                    times a number a token where one is given), float32, in the order of the
//                    choices; or added into out (the residual stream).
//   kvc_moe_combine_norm  the same added into the residual stream, and the RMS norm of its new rows

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "device_utils.h"
#include "gemm_common.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

#define S(stream) reinterpret_cast<hipStream_t>(stream)

constexpr int kTileRows = 16;
constexpr int kMidTileRows = 64;
constexpr int kBigTileRows = 128;
constexpr int kWideTileRows = 384;

bool known_tile_rows(int rows) {
  return rows == kTileRows || rows == kMidTileRows || rows == kBigTileRows || rows == kWideTileRows;
}

// What happens to the sums of an ungated product on their way out (the codes of kvc_activation; -1: nothing).
__device__ __forceinline__ float plain_act(float v, int act) {
  if (act == 0) {
    v = fmaxf(v, 0.f);
    return v * v;
  }
  return v;
}

// the lane that holds the largest value (the lowest index among equals) tells everyone
__device__ __forceinline__ void wave_argmax(float& val, int& idx) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(val, o, kWave);
    const int oi = __shfl_xor(idx, o, kWave);
    if (ov > val || (ov == val && oi < idx)) {
      val = ov;
      idx = oi;
    }
  }
}

// How a token's experts are chosen from its logits (+ bias[e], which may be null).  score_fn 0: softmax
// over the experts, 1: a sigmoid of each logit, 2: the logit itself.  The choice is made on score +
// correction[e] (correction may be null) and may so be negative; the weights are the plain scores of
// the chosen, over their sum (+ 1e-20) where `renormalize` is set, or (2) the softmax over the chosen
// logits, times weight_scale.
// With keep < groups only the experts of the best `keep` of `groups` equal
// groups of neighbours may be chosen; a group is worth the sum of its `group_best` (1 or 2) largest
// choice scores.  The lower index wins a tie.
struct RouteRule {
  int top, groups, keep, score_fn, group_best, renormalize;
  const float* bias;
  const float* correction;
  float weight_scale;
};

// The expert that every token runs, multiplied in the routed experts' launches: its tiles name kSharedExpert, its pair of
// token t is first_pair + t, and its matrix (of their sizes and their order of storage) lies at w.
constexpr int kSharedExpert = -1;
struct SharedExpert {
  const void* w;
  int first_pair;
  float limit;
};

// One token's choice by one wave: z [E] logits (global or LDS), sc [E], pk [E] and gs [groups] LDS
// scratch (sc may be z itself).
__device__ __forceinline__ void route_one(int32_t* __restrict__ choice, float* __restrict__ weight, const float* z,
                                          float* sc, float* pk, float* gs, int lane, int E, const RouteRule& rule) {
  const int top = rule.top, groups = rule.groups, keep = rule.keep;
  auto logit = [&](int e) -> float { return rule.bias != nullptr ? z[e] + rule.bias[e] : z[e]; };
  if (rule.score_fn == 0) {
    float mx = -INFINITY;
    for (int e = lane; e < E; e += kWave) mx = fmaxf(mx, logit(e));
    mx = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < E; e += kWave) {
      const float p = expf(logit(e) - mx);
      sc[e] = p;
      sum += p;
    }
    sum = wave_sum(sum);
    const float inv = 1.f / sum;
    for (int e = lane; e < E; e += kWave) sc[e] *= inv;
  } else if (rule.score_fn == 1) {
    for (int e = lane; e < E; e += kWave) sc[e] = 1.f / (1.f + expf(-logit(e)));
  } else {
    for (int e = lane; e < E; e += kWave) sc[e] = logit(e);
  }
  for (int e = lane; e < E; e += kWave) pk[e] = sc[e] + (rule.correction != nullptr ? rule.correction[e] : 0.f);
  __builtin_amdgcn_wave_barrier();
  const int per = E / groups;
  if (keep < groups) {
    for (int g = lane; g < groups; g += kWave) {
      float best = -INFINITY, second = -INFINITY;
      for (int i = 0; i < per; ++i) {
        const float s = pk[g * per + i];
        if (s > best) {
          second = best;
          best = s;
        } else if (s > second) {
          second = s;
        }
      }
      gs[g] = (rule.group_best >= 2 && per >= 2) ? best + second : best;
    }
    __builtin_amdgcn_wave_barrier();
    // the best `keep` groups are marked with +inf; the others' experts are taken out
    for (int r = 0; r < keep; ++r) {
      float val = -INFINITY;
      int idx = 0x7fffffff;
      for (int g = lane; g < groups; g += kWave) {
        const float s = gs[g];
        if (s != INFINITY && (s > val || (s == val && g < idx))) {
          val = s;
          idx = g;
        }
      }
      wave_argmax(val, idx);
      if (lane == 0 && idx < groups) gs[idx] = INFINITY;
      __builtin_amdgcn_wave_barrier();
    }
    for (int e = lane; e < E; e += kWave)
      if (gs[e / per] != INFINITY) pk[e] = -INFINITY;  // choice scores may be negative: minus infinity, not zero
    __builtin_amdgcn_wave_barrier();
  }
  float total = 0.f;
  float mine = 0.f;  // lane c keeps the c-th choice's score
  int mine_idx = 0;
  bool mine_ok = false;
  for (int c = 0; c < top; ++c) {
    float val = -INFINITY;
    int idx = 0x7fffffff;
    for (int e = lane; e < E; e += kWave) {
      const float s = pk[e];
      if (s > val || (s == val && e < idx)) {
        val = s;
        idx = e;
      }
    }
    wave_argmax(val, idx);
    if (idx >= E) idx = 0;
    // fewer allowed experts than choices: a weight of zero
    const float plain = (val == -INFINITY) ? 0.f : sc[idx];
    total += plain;
    if (lane == c) {
      mine = plain;
      mine_idx = idx;
      mine_ok = val != -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) pk[idx] = -INFINITY;
    __builtin_amdgcn_wave_barrier();
  }
  float norm = rule.renormalize ? rule.weight_scale / (total + 1e-20f) : rule.weight_scale;
  if (rule.score_fn == 2) {  // the softmax over the chosen logits alone
    const float mx = wave_max(mine_ok ? mine : -INFINITY);
    mine = mine_ok ? expf(mine - mx) : 0.f;
    norm = rule.weight_scale / wave_sum(mine);
  }
  if (lane < top) {
    choice[lane] = mine_idx;
    weight[lane] = mine * norm;
  }
}

// The same choice for at most 64 experts, one a lane (`z`: the lane's logit, lanes beyond E anything): an expert's
// place among the choices is the number of experts that come before it, counted against each in turn, so no
// wave-wide maximum has to be found choice by choice.
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ void route_lanes(int32_t* choice, float* weight, float z, int lane, int E, const RouteRule& rule) {
  const int top = rule.top, groups = rule.groups, keep = rule.keep;
  const bool live = lane < E;
  const int le = live ? lane : 0;
  if (rule.bias != nullptr) z += rule.bias[le];
  float sc = 0.f;
  if (rule.score_fn == 0) {
    const float mx = wave_max(live ? z : -INFINITY);
    const float p = live ? expf(z - mx) : 0.f;
    sc = p * (1.f / wave_sum(p));
  } else if (rule.score_fn == 1) {
    sc = 1.f / (1.f + expf(-z));
  } else {
    sc = z;
  }
  float pk = live ? sc + (rule.correction != nullptr ? rule.correction[le] : 0.f) : -INFINITY;
  if (keep < groups) {  // the same for the whole grid
    const int per = E / groups;
    const int base = lane < groups ? lane * per : 0;
    float best = -INFINITY, second = -INFINITY;  // lane g: of group g
    for (int i = 0; i < per; ++i) {
      const float s = __shfl(pk, base + i, kWave);
      if (s > best) {
        second = best;
        best = s;
      } else if (s > second) {
        second = s;
      }
    }
    const float worth = (rule.group_best >= 2 && per >= 2) ? best + second : best;
    int before = 0;
    for (int g = 0; g < groups; ++g) {
      const float s = lane_value(worth, g);
      before += s != INFINITY && (s > worth || (s == worth && g < lane));
    }
    const int kept = lane < groups && (worth == INFINITY || (worth == worth && before < keep));
    if (!__shfl(kept, le / per, kWave)) pk = -INFINITY;  // choice scores may be negative: minus infinity, not zero
  }
  int before = 0;
#pragma unroll 8
  for (int e = 0; e < E; ++e) {
    const float s = lane_value(pk, e);
    before += s > pk || (s == pk && e < lane);
  }
  const bool allowed = live && pk > -INFINITY;  // not for a score that is no number
  const int count = __popcll(__ballot(allowed));
  const uint64_t numbers = __ballot(live && pk == pk);
  const int spare = numbers ? __ffsll(static_cast<unsigned long long>(numbers)) - 1 : 0;
  float total = 0.f, mine = 0.f;  // lane c keeps the c-th choice's score
  int mine_idx = 0;
  bool mine_ok = false;
  for (int c = 0; c < top; ++c) {  // scalar
    // fewer allowed experts than choices: a weight of zero
    const bool ok = c < count;
    const uint64_t who = __ballot(allowed && before == c);
    const int idx = ok && who ? __ffsll(static_cast<unsigned long long>(who)) - 1 : spare;
    const float plain = ok ? lane_value(sc, idx) : 0.f;
    total += plain;
    if (lane == c) {
      mine = plain;
      mine_idx = idx;
      mine_ok = ok;
    }
  }
  float norm = rule.renormalize ? rule.weight_scale / (total + 1e-20f) : rule.weight_scale;
  if (rule.score_fn == 2) {  // the softmax over the chosen logits alone
    const float mx = wave_max(mine_ok ? mine : -INFINITY);
    mine = mine_ok ? expf(mine - mx) : 0.f;
    norm = rule.weight_scale / wave_sum(mine);
  }
  if (lane < top) {
    choice[lane] = mine_idx;
    weight[lane] = mine * norm;
  }
}

__global__ __launch_bounds__(256) void moe_route_kernel(int32_t* __restrict__ choice, float* __restrict__ weight,
                                                        const float* __restrict__ logits, int T, int E,
                                                        RouteRule rule) {
  extern __shared__ float lds[];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  float* sc = lds + wave * (2 * E + rule.groups);  // scores, choice scores, then the groups' worth
  const int t = blockIdx.x * 4 + wave;
  if (t >= T) return;  // the whole wave
  int32_t* ct = choice + static_cast<int64_t>(t) * rule.top;
  float* wt = weight + static_cast<int64_t>(t) * rule.top;
  const float* zt = logits + static_cast<int64_t>(t) * E;
  if (E <= kWave) route_lanes(ct, wt, zt[lane < E ? lane : 0], lane, E, rule);  // the same for the whole grid
  else route_one(ct, wt, zt, sc, sc + E, sc + 2 * E, lane, E, rule);
}

// The router whole: logits = x W^T with float32 products and sums (x of either dtype, its values as
// they are) on the matrix cores, then the choice as in moe_route_kernel.  A block of sixteen waves takes
// 16 tokens (the B operand's columns) and up to kRouterRows experts at a time (two A tiles of 16).  The
// waves share K: wave w takes the pieces of 32 values w, w + 16, ..., of which lane (expert or token li,
// lk) holds the values from 8 lk on (both operands are dealt the same way, so the eight 16 x 16 x 4
// products of a piece sum over all of it).  The waves' partial sums are added in wave order through LDS:
// one fixed order, whatever the batch.  Every wave then chooses for one token.  With `gate` the matrix
// has a row behind the experts', whose product's sigmoid goes to gate[t]; the lanes multiply that one
// themselves.
constexpr int kRouterWaves = 16;
constexpr int kRouterTokens = 16;
constexpr int kRouterRows = 32;
constexpr int kRouterPad = kRouterTokens + 1;

// Eight values of a row from k on.  VEC: rows of a multiple of 8 values, 16-byte aligned, so a piece is in
// or out as a whole; a piece that is out reads the row's last one (no branch around a load) and the
// caller drops it.  Otherwise element by element, zeros beyond H.
template <int VEC, typename T>
__device__ __forceinline__ void router_load(const T* row, int k, int H, float* v) {
  if constexpr (VEC) {
    const T* p = row + (k < H ? k : H - 8);
    if constexpr (sizeof(T) == 2) {
      const uint4 a = *reinterpret_cast<const uint4*>(p);
      const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
      }
    } else {
      const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
      v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (k + i < H) ? to_float(row[k + i]) : 0.f;
  }
}

template <typename T, int VEC>
__global__ __launch_bounds__(kRouterWaves * 64) void moe_router_kernel(
    int32_t* __restrict__ choice, float* __restrict__ weight, const T* __restrict__ x, int64_t x_stride,
    const float* __restrict__ wr, float* __restrict__ gate, int T_, int H, int E, RouteRule rule) {
  constexpr int NT = kRouterRows / 16;
  extern __shared__ float lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int li = lane & 15, lk = lane >> 4;
  float* part = lds;                                         // [waves][kRouterRows][kRouterPad]
  float* part_g = lds + kRouterWaves * kRouterRows * kRouterPad;  // [waves][kRouterTokens]
  float* z = part_g + kRouterWaves * kRouterTokens;          // [kRouterTokens][2 E + groups]
  const int zrow = 2 * E + rule.groups;
  const int t0 = blockIdx.x * kRouterTokens;
  const T* xr = x + static_cast<int64_t>(t0 + li < T_ ? t0 + li : T_ - 1) * x_stride;  // rows beyond are dropped
  float acc_g = 0.f;
  for (int e0 = 0; e0 < E; e0 += kRouterRows) {
    const int ne = (E - e0 < kRouterRows) ? E - e0 : kRouterRows;
    const bool with_gate = gate != nullptr && e0 == 0;
    const float* wp[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wp[n] = wr + static_cast<int64_t>(e0 + (16 * n + li < ne ? 16 * n + li : 0)) * H;
    const float* wg = wr + static_cast<int64_t>(with_gate ? E : e0) * H;
    f32x4_t acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float xn[8], wn[NT][8], gn[8];
    auto fetch = [&](int k) {
      router_load<VEC>(xr, k + 8 * lk, H, xn);
#pragma unroll
      for (int n = 0; n < NT; ++n) router_load<VEC>(wp[n], k + 8 * lk, H, wn[n]);
      router_load<VEC>(wg, k + 8 * lk, H, gn);
    };
    int k = 32 * wave;
    if (k < H) fetch(k);
    for (; k < H; k += 32 * kRouterWaves) {  // the same for the whole wave
      float xc[8], wc[NT][8];
      const bool in = !VEC || k + 8 * lk < H;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        xc[i] = in ? xn[i] : 0.f;
#pragma unroll
        for (int n = 0; n < NT; ++n) wc[n][i] = wn[n][i];
        if (with_gate) acc_g = fmaf(xc[i], gn[i], acc_g);
      }
      if (k + 32 * kRouterWaves < H) fetch(k + 32 * kRouterWaves);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[n][i], xc[i], acc[n], 0, 0, 0);
    }
    if (e0 > 0) __syncthreads();  // the partial sums of the experts before have been added up
    // lane holds token li, experts 16 n + 4 lk + i
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[(wave * kRouterRows + 16 * n + 4 * lk + i) * kRouterPad + li] = acc[n][i];
    if (with_gate) {
      acc_g += __shfl_xor(acc_g, 16, kWave);
      acc_g += __shfl_xor(acc_g, 32, kWave);
      if (lk == 0) part_g[wave * kRouterTokens + li] = acc_g;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < ne * kRouterTokens; idx += kRouterWaves * kWave) {
      const int e = idx / kRouterTokens, j = idx - e * kRouterTokens;
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kRouterWaves; ++w) sum += part[(w * kRouterRows + e) * kRouterPad + j];
      z[j * zrow + e0 + e] = sum;
    }
  }
  __syncthreads();
  const int t = t0 + wave;
  if (t >= T_) return;  // the whole wave
  if (gate != nullptr && lane == 0) {
    float sum = 0.f;
    for (int w = 0; w < kRouterWaves; ++w) sum += part_g[w * kRouterTokens + wave];
    gate[t] = 1.f / (1.f + expf(-sum));
  }
  float* zr = z + wave * zrow;
  int32_t* ct = choice + static_cast<int64_t>(t) * rule.top;
  float* wt = weight + static_cast<int64_t>(t) * rule.top;
  if (E <= kWave) route_lanes(ct, wt, zr[lane < E ? lane : 0], lane, E, rule);  // the same for the whole grid
  else route_one(ct, wt, zr, zr, zr + E, zr + 2 * E, lane, E, rule);
}

// One block.  counts -> offsets and tiles (a thread an expert) -> sorted pairs.  `ilds`: [3 E] in LDS.
__device__ __forceinline__ void align_pairs(int32_t* __restrict__ sorted, int32_t* __restrict__ tiles,
                                            int32_t* __restrict__ num_tiles, const int32_t* choice, int pairs, int E,
                                            int max_tiles, int tile_rows, int shared_rows, int32_t* ilds) {
  int32_t* count = ilds;           // [E]
  int32_t* offset = count + E;     // [E]
  int32_t* cursor = offset + E;    // [E]; at first the experts' numbers of tiles
  for (int e = threadIdx.x; e < E; e += blockDim.x) count[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int e = choice[i];
    if (e >= 0 && e < E) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  // an expert's rows in as few tiles as hold them, all of about one size (in sixteens): no tile is left with a few
  const bool wide = tile_rows == kWideTileRows;  // the others are powers of two
  const int shift = 31 - __clz(tile_rows);
  auto rows_each = [&](int n) {
    const int tiles_of = wide ? (n + kWideTileRows - 1) / kWideTileRows : (n + tile_rows - 1) >> shift;
    return tiles_of < 2 ? tile_rows : ((n + tiles_of - 1) / tiles_of + 15) & ~15;
  };
  // the shared expert's tiles come first (its rows fill them), its pairs behind the others
  const int shared_each = rows_each(shared_rows), shared_tiles = (shared_rows + shared_each - 1) / shared_each;
  for (int i = threadIdx.x; i < shared_tiles; i += blockDim.x) {
    const int r = i * shared_each;
    tiles[3 * i] = kSharedExpert;
    tiles[3 * i + 1] = pairs + r;
    tiles[3 * i + 2] = shared_rows - r < shared_each ? shared_rows - r : shared_each;
  }
  for (int i = threadIdx.x; i < shared_rows; i += blockDim.x) sorted[pairs + i] = pairs + i;
  auto list = [&](int e, int n, int each, int at, int nt) {
    offset[e] = at;
    for (int r = 0; r < n && nt < max_tiles; r += each, ++nt) {
      tiles[3 * nt] = e;
      tiles[3 * nt + 1] = at + r;
      tiles[3 * nt + 2] = (n - r < each) ? n - r : each;
    }
  };
  if (E <= kWave) {  // a lane an expert
    if (threadIdx.x < kWave) {
      const int e = threadIdx.x;
      const int n = e < E ? count[e] : 0;
      const int each = rows_each(n), mine = (n + each - 1) / each;
      int at = n, nt = mine;  // running sums over the lanes
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int pa = __shfl_up(at, o, kWave), pt = __shfl_up(nt, o, kWave);
        if (e >= o) {
          at += pa;
          nt += pt;
        }
      }
      nt += shared_tiles;
      if (e == E - 1) *num_tiles = nt < max_tiles ? nt : max_tiles;
      nt -= mine;
      if (wide) {
        // Blocks of tiles of up to 384 rows have a compute unit to themselves: experts with more rows a tile come first (the
        // lower index among equals), each one's tiles side by side, so that the last blocks the chip takes up are the short
        // ones.  Smaller tiles fetch weights in the experts' order (8 rows an expert, 32 gated experts of 2048 x 2048 in
        // tiles of 64 rows: 95.3 us, in the other order 98.3).
        const int key = (n < each ? n : each) * kWave + kWave - 1 - e;
        nt = shared_tiles;
#pragma unroll
        for (int p = 0; p < kWave; ++p) {  // lanes beyond E have no tiles
          if (p == kWave / 2 && E <= kWave / 2) break;  // scalar
          const int pt = __builtin_amdgcn_readlane(mine, p);
          nt += __builtin_amdgcn_readlane(key, p) > key ? pt : 0;
        }
      }
      if (e < E) list(e, n, each, at - n, nt);
    }
  } else {
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      const int each = rows_each(count[e]);
      cursor[e] = (count[e] + each - 1) / each;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      int at = 0, nt = shared_tiles;
      for (int p = 0; p < e; ++p) {
        at += count[p];
        nt += cursor[p];
      }
      list(e, count[e], rows_each(count[e]), at, nt);
      if (e == E - 1) *num_tiles = nt + cursor[e] < max_tiles ? nt + cursor[e] : max_tiles;
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < E; e += blockDim.x) cursor[e] = 0;
  __syncthreads();
  // an expert's pairs take their places in the order in which their threads arrive: a row's sums
  // do not depend on its place
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int e = choice[i];
    if (e < 0 || e >= E) continue;
    const int place = atomicAdd(&cursor[e], 1);
    sorted[offset[e] + place] = i;
  }
}

__global__ __launch_bounds__(1024) void moe_align_kernel(int32_t* __restrict__ sorted, int32_t* __restrict__ tiles,
                                                         int32_t* __restrict__ num_tiles,
                                                         const int32_t* __restrict__ choice, int pairs, int E,
                                                         int max_tiles, int tile_rows, int shared_rows) {
  extern __shared__ int32_t ilds[];
  align_pairs(sorted, tiles, num_tiles, choice, pairs, E, max_tiles, tile_rows, shared_rows, ilds);
}

// The router spread over the chip (at most kRouterSpread tokens and 64 experts), with the arrangement of its pairs.
// One block reads its 260 KB of router and rows at what a compute unit draws (50 GB/s), so the sixteen parts of K
// that moe_router_kernel's waves take go to as many blocks here, which leave their sums in `parts` [16][T][row]
// (the gate's behind the experts'); they are added in the same order by the wave that chooses for a token.  Up to
// kChooseInOne tokens the block that lists the tiles chooses too, a token a wave; with more of them a choice costs
// that one compute unit 0.3 us a token, so a kernel of its own deals the tokens out.  With 32 experts and rows of
// 2,048, 8 tokens 26.4 -> 12.6 us (router and tiles together), 64 tokens
// 23.8 -> 15.7, 300 tokens 23.6 -> 15.7; 2,030 tokens fill the chip either way (27.2 and 26.5).
constexpr int kRouterSpread = 1024;
constexpr int kChooseInOne = 16;
__host__ __device__ __forceinline__ int router_part_row(int E) { return ((E + 3) & ~3) + 4; }

template <typename T, int VEC>
__global__ __launch_bounds__(64) void moe_router_parts_kernel(float* __restrict__ parts, const T* __restrict__ x,
                                                              int64_t x_stride, const float* __restrict__ wr,
                                                              int with_gate_row, int T_, int H, int E) {
  constexpr int NT = kRouterRows / 16;
  const int lane = threadIdx.x, li = lane & 15, lk = lane >> 4;
  const int part = blockIdx.y, e0 = blockIdx.z * kRouterRows, t0 = blockIdx.x * kRouterTokens;
  const T* xr = x + static_cast<int64_t>(t0 + li < T_ ? t0 + li : T_ - 1) * x_stride;  // rows beyond are dropped
  const int ne = (E - e0 < kRouterRows) ? E - e0 : kRouterRows;
  const bool with_gate = with_gate_row && e0 == 0;
  const float* wp[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wp[n] = wr + static_cast<int64_t>(e0 + (16 * n + li < ne ? 16 * n + li : 0)) * H;
  const float* wg = wr + static_cast<int64_t>(with_gate ? E : e0) * H;
  f32x4_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float acc_g = 0.f;
  constexpr int kAhead = 2;  // pieces on their way
  float xn[kAhead][8], wn[kAhead][NT][8], gn[kAhead][8];
  auto fetch = [&](int slot, int k) {  // no branch around the loads: a piece beyond H reads the row's last values
    router_load<VEC>(xr, k + 8 * lk, H, xn[slot]);
#pragma unroll
    for (int n = 0; n < NT; ++n) router_load<VEC>(wp[n], k + 8 * lk, H, wn[slot][n]);
    router_load<VEC>(wg, k + 8 * lk, H, gn[slot]);
  };
#pragma unroll
  for (int s = 0; s < kAhead; ++s) fetch(s, 32 * (part + kRouterWaves * s));
  for (int k0 = 32 * part; k0 < H; k0 += 32 * kRouterWaves * kAhead) {  // scalar
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      const int k = k0 + 32 * kRouterWaves * s;
      if (k >= H) break;  // scalar
      float xc[8], wc[NT][8];
      const bool in = !VEC || k + 8 * lk < H;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        xc[i] = in ? xn[s][i] : 0.f;
#pragma unroll
        for (int n = 0; n < NT; ++n) wc[n][i] = wn[s][n][i];
        if (with_gate) acc_g = fmaf(xc[i], gn[s][i], acc_g);
      }
      fetch(s, k + 32 * kRouterWaves * kAhead);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[n][i], xc[i], acc[n], 0, 0, 0);
    }
  }
  acc_g += __shfl_xor(acc_g, 16, kWave);
  acc_g += __shfl_xor(acc_g, 32, kWave);
  if (t0 + li >= T_) return;
  const int row = router_part_row(E);
  float* dst = parts + (static_cast<int64_t>(part) * T_ + t0 + li) * row;
  // lane holds token li, experts 16 n + 4 lk + i
#pragma unroll
  for (int n = 0; n < NT; ++n)
    if (e0 + 16 * n + 4 * lk < row - 4) *reinterpret_cast<f32x4_t*>(dst + e0 + 16 * n + 4 * lk) = acc[n];
  if (with_gate && lk == 0) dst[row - 4] = acc_g;
}

// One token's choice from the parts of its logits, by one wave.
__device__ __forceinline__ void choose_from_parts(int32_t* choice, float* weight, float* __restrict__ gate,
                                                  const float* __restrict__ parts, int t, int T_, int E, int lane,
                                                  const RouteRule& rule) {
  const int row = router_part_row(E);
  const int64_t step = static_cast<int64_t>(T_) * row;
  const float* p = parts + static_cast<int64_t>(t) * row;
  const int at = lane < E ? lane : 0;
  float v[kRouterWaves], g[kRouterWaves];
#pragma unroll
  for (int w = 0; w < kRouterWaves; ++w) v[w] = p[w * step + at];
  if (gate != nullptr) {  // the same for the whole grid
#pragma unroll
    for (int w = 0; w < kRouterWaves; ++w) g[w] = p[w * step + row - 4];
  }
  float z = 0.f;
#pragma unroll
  for (int w = 0; w < kRouterWaves; ++w) z += v[w];
  if (gate != nullptr) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kRouterWaves; ++w) sum += g[w];
    if (lane == 0) gate[t] = 1.f / (1.f + expf(-sum));
  }
  route_lanes(choice, weight, z, lane, E, rule);
}

__global__ __launch_bounds__(256) void moe_choose_kernel(int32_t* __restrict__ choice, float* __restrict__ weight,
                                                         float* __restrict__ gate, const float* __restrict__ parts, int T_,
                                                         int E, RouteRule rule) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int t = blockIdx.x * 4 + wave;
  if (t >= T_) return;  // scalar
  choose_from_parts(choice + static_cast<int64_t>(t) * rule.top, weight + static_cast<int64_t>(t) * rule.top, gate, parts,
                    t, T_, E, lane, rule);
}

__global__ __launch_bounds__(1024) void moe_choose_align_kernel(
    int32_t* __restrict__ choice, float* __restrict__ weight, float* __restrict__ gate, int32_t* __restrict__ sorted,
    int32_t* __restrict__ tiles, int32_t* __restrict__ num_tiles, const float* __restrict__ parts, int T_, int E,
    int max_tiles, int tile_rows, int shared_rows, RouteRule rule) {
  extern __shared__ int32_t ilds[];  // [T top] choices, then [3 E]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  if (wave < T_)  // scalar
    choose_from_parts(ilds + wave * rule.top, weight + static_cast<int64_t>(wave) * rule.top, gate, parts, wave, T_, E, lane,
                      rule);
  __syncthreads();
  const int pairs = T_ * rule.top;
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) choice[i] = ilds[i];
  align_pairs(sorted, tiles, num_tiles, ilds, pairs, E, max_tiles, tile_rows, shared_rows, ilds + pairs);
}

// bfloat16, few rows: a wave takes one tile of up to 16 rows and 16 columns (gated: of gate and of up).  WK 4: the
// four waves of a block share K: wave w takes the passes w, w + 4, ... of 64 values, four of them on their way, and
// the four sums are added in wave order.  WK 1: each takes all of K of columns of its own.  In a pass lane (li, lk)
// fetches the 16 values from 16 lk of its weight
// row and of its token row (32 contiguous bytes, so that the four lanes of a row read one 128-byte line) and the
// two matrix instructions take its first and its second eight (both operands are dealt the same way, so each
// product still sums over all of K).  Bound by reading the weights of the experts that were chosen: with a whole K
// a wave and 64 columns a block, one token of four experts of 2048 x 2048 had 128 blocks.  Gated and ungated, packed:
// one token 22.0 and 13.4 -> 13.8 and 11.8 us, eight tokens 75 and 46 -> 64 and 34 us (5.6 TB/s).  Where K is a few
// passes long a share of it is one or two, and with many tiles four times the blocks cost more than they bring
// (kvc_moe_gemm has the line): 128 experts of 1024 x 384, 8 rows each, down 37.0 us with WK 4, 20.8 with WK 1
// (two passes on their way: with four 22.6).
// An expert that has one tile has its (packed) matrices read once, with loads that say so (`read8`): eight tokens 64 and 34 ->
// 57 and 30 us (6.0 TB/s), 256 pairs 93 and 49 -> 83 and 46.  Where two tiles share a matrix through the L2 such loads cost
// more than they bring (256 pairs, half of them with few experts, 160 -> 196 us), so those keep the others.
__device__ __forceinline__ bool only_tile(const int32_t* tiles, int tile, int num_tiles) {  // an expert's are side by side
  const int e = tiles[3 * tile];
  return (tile == 0 || tiles[3 * tile - 3] != e) && (tile + 1 >= num_tiles || tiles[3 * tile + 3] != e);
}
// Where a pair's input row lies (in_div 0: the products of its own place), its expert's matrix, and what the expert adds to
// the place at which a block begins its walk along K.
__device__ __forceinline__ int64_t input_row(int pair, int place, int in_div, int e, const SharedExpert& shared) {
  return in_div == 0 ? place : e == kSharedExpert ? pair - shared.first_pair : pair / in_div;
}
template <typename T>
__device__ __forceinline__ const T* expert_weights(const T* w, int e, int64_t elems, const SharedExpert& shared) {
  return e == kSharedExpert ? static_cast<const T*>(shared.w) : w + e * elems;
}
__device__ __forceinline__ int turn_of(int e) { return e == kSharedExpert ? 0 : e * 5; }
template <int GATED, typename TO, int PACKED, int WK>
__global__ __launch_bounds__(256) void moe_gemm_few_kernel(
    TO* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ x, int64_t x_stride,
    const bf16_t* __restrict__ w, const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles,
    const int32_t* __restrict__ num_tiles, int N, int K, int in_div, int out_sorted, float limit, float alpha, float shift,
    int act, const float* __restrict__ row_scale, SharedExpert shared) {
  constexpr int kStages = WK == 1 ? 2 : 4;
  const int tile = blockIdx.z * gridDim.y + blockIdx.y;  // more tiles than a grid's second dimension takes
  if (tile >= *num_tiles) return;
  const int e = tiles[3 * tile], r0 = tiles[3 * tile + 1], nr = tiles[3 * tile + 2];
  const int of_block = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int wave = WK == 1 ? 0 : of_block;  // whose share of K
  const int n0 = (WK == 1 ? blockIdx.x * 4 + of_block : blockIdx.x) * 16;
  if (n0 >= N) return;  // scalar; with WK 4 the whole block
  const int li = lane & 15, lk = lane >> 4;
  // B operand: token row li of the tile; A operand: the expert's row n0 + li
  const bool row_ok = li < nr;
  const int pair = sorted[r0 + (row_ok ? li : 0)];  // a row that is not there reads the tile's first and is dropped
  const int64_t in_row = input_row(pair, r0 + (row_ok ? li : 0), in_div, e, shared);
  // PACKED: w is the copy that `kvc_pack_weight` makes, tiles of 16 rows x 32 values of K in one
  // piece of 1 KB each, so a wave's load of an operand is one contiguous kilobyte instead of 128 bytes
  // from each of 16 rows that lie 2 K bytes apart (which meet in the same memory channels); the lanes
  // then take K in the plain order, 8 values from 8 lk of each 32.
  const bf16_t* xr = x + in_row * x_stride + (PACKED ? 8 : 16) * lk;
  const int wrow = n0 + li < N ? n0 + li : N - 1;
  const int64_t rows_per_expert = GATED ? 2 * static_cast<int64_t>(N) : N;
  const bf16_t* we = expert_weights(w, e, rows_per_expert * K, shared);
  const bf16_t* wr = PACKED ? we + static_cast<int64_t>(n0 >> 4) * (K / 32) * 512 + li * 32 + lk * 8
                            : we + static_cast<int64_t>(wrow) * K + 16 * lk;
  const bf16_t* wr2 = wr + static_cast<int64_t>(N) * K;  // the up rows follow the gate rows (in either order of storage)
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f}, acc2 = {0.f, 0.f, 0.f, 0.f};
  const int passes = K / 64;
  // blocks walk K round from places of their own, as in the kernel for more rows
  const int turn = passes > 0 ? (turn_of(e) + (n0 >> 4) * 3) % passes : 0;
  // ONCE: this tile holds all rows of its expert, so nothing else reads the matrix (see `read8`)
  auto walk = [&](auto once) {
  constexpr bool ONCE = decltype(once)::value;
  bf16x8_t an[kStages][2], a2n[kStages][2], bn[kStages][2];
  auto fetch = [&](int slot, int pass) {  // no branch around the loads: a pass that is not there repeats the last
    int p = pass < passes ? pass + turn : passes - 1 + turn;
    p = p < passes ? p : p - passes;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t wo = PACKED ? static_cast<int64_t>(2 * p + h) * 512 : 64 * p + 8 * h;
      an[slot][h] = read8<ONCE>(wr + wo);
      if (GATED) a2n[slot][h] = read8<ONCE>(wr2 + wo);
      bn[slot][h] = *reinterpret_cast<const bf16x8_t*>(xr + 64 * p + (PACKED ? 32 : 8) * h);
    }
  };
  if (wave < passes) {  // scalar
#pragma unroll
    for (int s = 0; s < kStages; ++s) fetch(s, wave + WK * s);
    for (int p = wave; p < passes; p += WK * kStages) {
#pragma unroll
      for (int s = 0; s < kStages; ++s) {
        if (p + WK * s >= passes) break;  // scalar
        bf16x8_t a[2], a2[2], b[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          a[h] = an[s][h];
          if (GATED) a2[h] = a2n[s][h];
          b[h] = bn[s][h];
        }
        if (p + WK * kStages < passes) fetch(s, p + WK * (s + kStages));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h], b[h], acc, 0, 0, 0);
          if (GATED) acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[h], b[h], acc2, 0, 0, 0);
        }
      }
    }
  }
  };
  if (PACKED && only_tile(tiles, tile, *num_tiles)) walk(std::integral_constant<bool, PACKED != 0>{});
  else walk(std::false_type{});
  const int k_main = 64 * passes;
  if (wave == 0 && k_main < K) {  // a ragged end along K (a multiple of 8): element by element, zeros beyond
    bf16x8_t a[2], a2[2], b[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      a[h] = zero8(); a2[h] = zero8(); b[h] = zero8();
      for (int i = 0; i < 8; ++i) {
        const int off = k_main + 8 * h + i;  // from the lane's own start 16 lk
        if (off + 16 * lk < K) {
          a[h][i] = reinterpret_cast<const __bf16*>(wr)[off];
          if (GATED) a2[h][i] = reinterpret_cast<const __bf16*>(wr2)[off];
          b[h][i] = reinterpret_cast<const __bf16*>(xr)[off];
        }
      }
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h], b[h], acc, 0, 0, 0);
      if (GATED) acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[h], b[h], acc2, 0, 0, 0);
    }
  }
  if constexpr (WK > 1) {
    __shared__ f32x4_t part[(WK - 1) * (GATED ? 2 : 1)][64];
    if (wave > 0) {
      part[wave - 1][lane] = acc;
      if (GATED) part[WK - 2 + wave][lane] = acc2;
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int v = 0; v < WK - 1; ++v) {
      acc += part[v][lane];
      if (GATED) acc2 += part[WK - 1 + v][lane];
    }
  }
  // lane holds column (token) li, rows (features) n0 + 4 * lk + i
  if (!row_ok) return;
  const float scale = row_scale != nullptr ? row_scale[pair] : 1.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    acc[i] = GATED ? clamped_glu(acc[i] * scale, acc2[i] * scale, e == kSharedExpert ? shared.limit : limit, alpha, shift)
                   : plain_act(acc[i] * scale, act);
  const int64_t out_row = out_sorted ? r0 + li : pair;
  const int nf = n0 + 4 * lk;
  if (nf < N) store4<TO>(out + out_row * out_stride + nf, acc, N - nf);
}

// bfloat16, tiles of 64 or 128 rows (NR row blocks of 16; the last ones of a tile may be empty and are not
// multiplied): a block of four waves takes the tile's rows and 128 columns (gated; 256 otherwise).  The rows'
// chunk of 64 values along K goes through LDS (two buffers, one barrier a chunk), which all waves read as the B
// operand; every wave fetches the weight rows of its own columns straight into registers as the A operand
// (NF blocks of 16 columns, for gate and for up), one chunk ahead of the products.  Bound by the weights' way to
// the compute units: a fetched weight meets 16 NR rows, a row 128 or 256 columns, and the blocks that read the
// same weights or the same rows run on one die at the same time (see `place`), so its L2 is asked twice and
// memory once, or, where the expert has no other tile, with loads that say so (`read8`: 256 pairs 94 and 46 -> 86 and 43 us,
// 1,184 pairs 101 and 51.5 -> 90 and 50; 2,880 pairs, two tiles an expert, in that way 121 -> 150).  Packed, 32 experts of 2048 x 2048, gated and ungated: 8,192 pairs 397 and 232 us with tiles of 64
// rows dealt to the dies in turn, 202 and 123 us this way (0.68 PFLOP/s); 1,200 pairs 226 and 143 us in tiles of 16
// rows, 102 and 52 us here (5.3 TB/s of weights); 256 pairs 113 and 61 us, 95 and 46 us (5.8 TB/s), of which
// 14 and 7 us are the turn that every block starts K at.
struct TilePlace {
  int tile, col;
};
// Which row tile and which column block the block `id` takes (tile -1: none).  Blocks are dealt to the eight
// dies in turn, so `id % 8` is the die.  Where the column blocks divide by eight, a die keeps its share of them
// for every tile, its own columns of a tile side by side (they share the rows); otherwise a die takes a run of
// (column, tile) pairs, a column's tiles side by side (an expert's share the weights).
__device__ __forceinline__ TilePlace place(int id, int tiles, int cols) {
  const int die = id & 7, idx = id >> 3;
  if ((cols & 7) == 0) {
    const int own = cols >> 3, tile = idx / own;
    return {tile < tiles ? tile : -1, die * own + (idx - tile * own)};
  }
  const int total = tiles * cols, chunk = (total + 7) >> 3;
  const int at = die * chunk + idx;
  if (idx >= chunk || at >= total) return {-1, 0};
  const int col = at / tiles;
  return {at - col * tiles, col};
}
// The way out of a tile's sums: lane (li, lk) holds NR rows (`row_of`) and of each NF times four columns from n + 16 f on.
// The pairs and scales of all rows are asked for before the first store: a load behind it would wait for the store too,
// which cost a block of 256 rows 9 us.
template <int GATED, int NF, int NR, typename TO, typename RowOf, typename Acc, typename Acc2>
__device__ __forceinline__ void store_tile(TO* out, int64_t out_stride, RowOf row_of, int nr, int n, int N, int r0,
                                           const int32_t* sorted, int out_sorted, const float* row_scale, float limit,
                                           float alpha, float shift, int act, Acc acc_of, Acc2 acc2_of) {
  int pair[NR];
  float scale[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) pair[r] = row_of(r) < nr ? r0 + row_of(r) : r0;
  const bool by_place = out_sorted && row_scale == nullptr;  // the same for the whole grid
  int place_of[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    place_of[r] = pair[r];
    if (!by_place) pair[r] = sorted[pair[r]];
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) scale[r] = row_scale != nullptr ? row_scale[pair[r]] : 1.f;
  constexpr int kBytes = 4 * sizeof(TO);
  const bool whole = N % 4 == 0 && (reinterpret_cast<uintptr_t>(out) % kBytes) == 0 && out_stride % 4 == 0;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (row_of(r) >= nr) continue;
    TO* to = out + static_cast<int64_t>(out_sorted ? place_of[r] : pair[r]) * out_stride + n;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      f32x4_t v = acc_of(f, r);
      const f32x4_t v2 = acc2_of(f, r);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = GATED ? clamped_glu<true>(v[i] * scale[r], v2[i] * scale[r], limit, alpha, shift) : plain_act(v[i] * scale[r], act);
      if (n + 16 * f >= N) continue;
      if (whole) {
        store4_whole(to + 16 * f, v);
      } else {  // rare: kept from becoming a second copy of all of this
#pragma unroll 1
        for (int i = 0; i < 4 && n + 16 * f + i < N; ++i) to[16 * f + i] = from_float<TO>(i == 0 ? v[0] : i == 1 ? v[1] : i == 2 ? v[2] : v[3]);
      }
    }
  }
}

template <int GATED, int NR, typename TO, int PACKED>
__global__ __launch_bounds__(256, 2) void moe_gemm_tiled_kernel(
    TO* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ x, int64_t x_stride,
    const bf16_t* __restrict__ w, const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles,
    const int32_t* __restrict__ num_tiles, int N, int K, int in_div, int out_sorted, float limit, float alpha, float shift,
    int act, const float* __restrict__ row_scale, SharedExpert shared) {
  constexpr int NF = GATED ? 2 : 4;   // column blocks of 16 a wave
  constexpr int KC = 64;              // values of K a pass (two matrix instructions deep)
  constexpr int KROW = KC + 8;        // a row's chunk in LDS, padded against bank conflicts
  constexpr int CH = NR / 2;          // pieces of eight values that a thread stages a pass
  __shared__ __attribute__((aligned(16))) bf16_t x_s[2][16 * NR * KROW];
  const TilePlace at = place(blockIdx.x, *num_tiles, (N + 64 * NF - 1) / (64 * NF));
  if (at.tile < 0) return;
  const int e = tiles[3 * at.tile], r0 = tiles[3 * at.tile + 1];
  const int nr = __builtin_amdgcn_readfirstlane(tiles[3 * at.tile + 2]);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int li = lane & 15, lk = lane >> 4;
  const int n0 = (at.col * 4 + wave) * 16 * NF;
  const bool wave_live = n0 < N;  // the same for the whole wave
  // staging: a thread brings 8 CH values of one row of the tile
  const int srow = threadIdx.x / (8 / CH), spart = threadIdx.x % (8 / CH);
  const bool srow_ok = srow < nr;
  const int srow_safe = srow_ok ? srow : 0;  // a row that is not there reads the tile's first, and is set to zero
  const int64_t in_row = in_div > 0 ? input_row(sorted[r0 + srow_safe], 0, in_div, e, shared) : r0 + srow_safe;
  const bf16_t* xp = x + in_row * x_stride + 8 * CH * spart;
  const int64_t rows_per_expert = GATED ? 2 * static_cast<int64_t>(N) : N;
  const bf16_t* we = expert_weights(w, e, rows_per_expert * K, shared);
  const bf16_t* wp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int wrow = n0 + 16 * f + li < N ? n0 + 16 * f + li : N - 1;
    // PACKED (N a multiple of 16): the copy in pieces of 16 rows x 32 values, one contiguous kilobyte a load
    const int ntile = n0 + 16 * f < N ? n0 + 16 * f : N - 16;
    wp[f] = PACKED ? we + static_cast<int64_t>(ntile >> 4) * (K / 32) * 512 + li * 32 + lk * 8
                   : we + static_cast<int64_t>(wrow) * K + 8 * lk;
  }
  const int64_t up_off = static_cast<int64_t>(N) * K;
  f32x4_t acc[NF][NR], acc2[GATED ? NF : 1][NR];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      acc[f][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (GATED) acc2[f][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  auto walk = [&](auto once) {  // ONCE: loads marked as streaming ones (PACKED 2: see kvc_moe_gemm)
  constexpr bool ONCE = decltype(once)::value;
  uint4 x_next[CH];
  bf16x8_t w_next[2][NF], w2_next[2][GATED ? NF : 1];
  // a pass's second half may lie beyond K (K a multiple of 32 only): the first half is then read
  // again and not multiplied
  auto fetch_x = [&](int k) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int col = 8 * (CH * spart + c);
      x_next[c] = *reinterpret_cast<const uint4*>(xp + k + 8 * c - (k + col < K ? 0 : 32));
    }
  };
  auto fetch_w = [&](int k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kk = k + 32 * h < K ? k + 32 * h : k;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int64_t wo = PACKED ? static_cast<int64_t>(kk / 32) * 512 : kk;
        w_next[h][f] = read8<ONCE>(wp[f] + wo);
        if (GATED) w2_next[h][f] = read8<ONCE>(wp[f] + up_off + wo);
      }
    }
  };
  auto stash = [&](int buffer) {  // the choice word by word: of a whole piece it became a branch that waited for every load
#pragma unroll
    for (int c = 0; c < CH; ++c)
      *reinterpret_cast<uint4*>(x_s[buffer] + srow * KROW + 8 * (CH * spart + c)) =
          uint4{srow_ok ? x_next[c].x : 0u, srow_ok ? x_next[c].y : 0u, srow_ok ? x_next[c].z : 0u, srow_ok ? x_next[c].w : 0u};
  };
  // Every block walks K round from a place of its own (which its expert and columns decide, so a row's sums do
  // not depend on its tile): blocks that start at the same place of rows that lie a power of two apart would ask
  // the same memory channels at the same time.
  const int turn = K % KC == 0 ? (turn_of(e) + at.col * 11) % (K / KC) * KC : 0;
  auto round = [&](int k) { return k + turn < K ? k + turn : k + turn - K; };
  fetch_x(round(0));
  fetch_w(round(0));
  stash(0);
  if (KC < K) fetch_x(round(KC));
  __syncthreads();
  for (int k0 = 0; k0 < K; k0 += 2 * KC) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {  // the chunk is in LDS buffer s
      const int k = k0 + KC * s;
      if (k >= K) break;  // scalar
      const bool two = k + 32 < K;
      bf16x8_t wa[2][NF], wa2[2][GATED ? NF : 1];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          wa[h][f] = w_next[h][f];
          if (GATED) wa2[h][f] = w2_next[h][f];
        }
      fetch_w(round(k + KC < K ? k + KC : k));  // no branch around the loads: the last one repeats
      if (k + KC < K) stash(s ^ 1);  // the chunk after this one, asked for a pass ago
      if (k + 2 * KC < K) fetch_x(round(k + 2 * KC));
      if (wave_live) {  // scalar: matrix instructions are skipped by a branch, never by a lane mask
        const bf16_t* xb = x_s[s] + li * KROW + 8 * lk;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (h == 1 && !two) break;  // scalar
          bf16x8_t b[2][2];
#pragma unroll
          for (int i = 0; i < 2; ++i) b[0][i] = *reinterpret_cast<const bf16x8_t*>(xb + 16 * i * KROW + 32 * h);
#pragma unroll
          for (int g = 0; g < NR / 2; ++g) {  // two row blocks at a time, the next two on their way from LDS
            if (g + 1 < NR / 2)
#pragma unroll
              for (int i = 0; i < 2; ++i)
                b[(g + 1) & 1][i] = *reinterpret_cast<const bf16x8_t*>(xb + 16 * (2 * g + 2 + i) * KROW + 32 * h);
            if (32 * g < nr) {  // scalar
#pragma unroll
              for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                  acc[f][2 * g + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[h][f], b[g & 1][i], acc[f][2 * g + i], 0, 0, 0);
                  if (GATED)
                    acc2[f][2 * g + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa2[h][f], b[g & 1][i], acc2[f][2 * g + i], 0, 0, 0);
                }
            }
          }
        }
      }
      __syncthreads();  // this chunk has been read by every wave, the next one is there
    }
  }
  };
  if constexpr (PACKED == 2) {
    if (only_tile(tiles, at.tile, *num_tiles)) walk(std::true_type{});
    else walk(std::false_type{});
  } else {
    walk(std::false_type{});
  }
  if (!wave_live) return;
  // lane holds row 16 r + li of the tile, columns n0 + 16 f + 4 lk + i
  store_tile<GATED, NF, NR, TO>(
      out, out_stride, [&](int r) { return 16 * r + li; }, nr, n0 + 4 * lk, N, r0, sorted, out_sorted, row_scale,
      e == kSharedExpert ? shared.limit : limit, alpha, shift, act, [&](int f, int r) { return acc[f][r]; },
      [&](int f, int r) { return acc2[GATED ? f : 0][r]; });
}

// bfloat16, tiles of up to 384 rows: a block of eight waves takes the tile's rows and 256 columns (gated: 128 of gate and
// the 128 of up beside them), one block a compute unit.
// Both operands go straight into LDS (`global_load_lds`, 16 bytes a lane) in stages of 32 values of K: one is multiplied, one
// has landed so that its first operands are read before the barrier, the others are on their way (five stages of 32 KB
// up to 256 rows, four of 40 KB above).  A row block's stage is a kilobyte of 16 rows x 64 bytes; a lane's place in LDS is
// fixed, so the lanes swap 16-byte pieces within a row on the way in such that the lanes that read operands together
// meet all banks.  Wave (wr, wc) takes the row blocks of parity wr, so that a tile that is not full is dealt evenly, and 64
// columns.
// Packed, 32 experts of 2048 x 2048, gated and ungated, 8,192 pairs: tiles of 128 rows 202 and 122 us, these 166 and 89 (0.82
// PFLOP/s; the weights alone take 83 and 41 us).  384 rows and not 256: experts of 256 rows in the mean have up to some 330, and
// with tiles of 256 a third of them had two (175 and 115 us).  One expert of 8,192 rows in tiles of 256: 1.0 PFLOP/s, 1.18
// without the way in and out of a block (some 10 us of 60); a stage of 256 rows takes 1,490 cycles at 1.8 GHz, of which the
// matrix instructions are 1,024; without the loads 1,340 at 2.05 GHz: the chip's power, not their latency, is what they cost.
constexpr int kWideBlocks = kWideTileRows / 32;  // row blocks a wave at most
constexpr int kWideLds = 163840;

// 64 lanes x 16 bytes, lane i's to lds + 16 i (a scalar byte address of LDS).  In text: where the compiler sees such a
// load it waits for all of them before the next read of LDS, also of another buffer.  The waits are the kernel's own
// (no register waits for these loads, and waits for others only get stricter).
__device__ __forceinline__ void to_lds16(const void* from, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(from) : "memory", "m0");
}

__device__ __forceinline__ void to_lds16_once(const void* from, uint32_t lds) {  // marked as a streaming load, as `read8`'s
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(from) : "memory", "m0");
}

// The wave's loads but the youngest N have landed; past the barrier that holds for all waves.
template <int N>
__device__ __forceinline__ void landed() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// R: how many row blocks a wave multiplies: the tile has at most 32 R rows.  ONCE: no other block reads these weights
template <int PACKED, int R, bool ONCE>
__device__ __forceinline__ void wide_walk(const char* lds, const char* const (&xp)[3], const char* const (&wp)[2], int wave,
                                          int lane, const int (&wt)[4], int stages, int turn,
                                          f32x4_t (&acc)[4][kWideBlocks]) {
  constexpr int P = (R + 1) / 2;                      // row blocks go two at a time
  constexpr int XL = R > 8 ? 3 : R > 4 ? 2 : 1;       // loads of rows a wave and stage, 8 KB for all waves
  constexpr int LOADS = XL + 2;
  constexpr int kW = XL > 2 ? 24576 : 16384;          // where a stage's weights begin
  constexpr int kStage = kW + 16384;
  constexpr int kStages = XL > 2 ? 4 : 5;
  static_assert(kStage * kStages <= kWideLds, "");
  const int li = lane & 15, lk = lane >> 4, wr = wave & 1;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)lds));
  const int at = li * 64 + 16 * (lk ^ ((li >> 1) & 3));  // the lane's place in a row or column block
  auto round = [&](int s) { return s + turn < stages ? s + turn : s + turn - stages; };
  auto load = [&](int j, int64_t s, uint32_t buffer) {
    if (j < XL) to_lds16(xp[j] + 64 * s, buffer + (wave + 8 * j) * 1024);
    else if (ONCE) to_lds16_once(wp[j - XL] + (PACKED ? 1024 : 64) * s, buffer + kW + (wave + 8 * (j - XL)) * 1024);
    else to_lds16(wp[j - XL] + (PACKED ? 1024 : 64) * s, buffer + kW + (wave + 8 * (j - XL)) * 1024);
  };
  auto x_operand = [&](const char* stage, int r) {
    return *reinterpret_cast<const bf16x8_t*>(stage + (2 * r + wr) * 1024 + at);
  };
  auto w_operand = [&](const char* stage, int f) { return *reinterpret_cast<const bf16x8_t*>(stage + kW + wt[f] + at); };
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    if (s < stages)  // scalar, as all that follow
#pragma unroll
      for (int j = 0; j < LOADS; ++j) load(j, round(s), lds0 + s * kStage);
  if (stages >= kStages - 1) landed<(kStages - 3) * LOADS>();
  else landed<0>();
  bf16x8_t a[4], b[2];
#pragma unroll
  for (int f = 0; f < 4; ++f) a[f] = w_operand(lds, f);
#pragma unroll
  for (int i = 0; i < (R < 2 ? R : 2); ++i) b[i] = x_operand(lds, i);
  int now = 0;  // byte offset of the stage's buffer
  for (int s = 0; s < stages; ++s) {
    const int next = now == (kStages - 1) * kStage ? 0 : now + kStage;
    const int free = now == 0 ? (kStages - 1) * kStage : now - kStage;  // every wave has read it
    const bool more = s + kStages - 1 < stages;
    const int64_t from = round(s + kStages - 1);
    bf16x8_t a_next[4];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      // a load, the operands of the next eight products, the eight products; the loads dealt over the stage, as a wave that
      // asks for all of them at once waits until they are taken
      if (more)
#pragma unroll
        for (int j = p * LOADS / P; j < (p + 1) * LOADS / P; ++j) load(j, from, lds0 + free);
      bf16x8_t b_next[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (p + 1 < P && 2 * p + 2 + i < R) b_next[i] = x_operand(lds + now, 2 * p + 2 + i);
        if (p + 1 == P && i < R) b_next[i] = x_operand(lds + next, i);
      }
      if (p == P - 1)
#pragma unroll
        for (int f = 0; f < 4; ++f) a_next[f] = w_operand(lds + next, f);
#pragma unroll
      for (int i = 0; i < 2 && 2 * p + i < R; ++i)
#pragma unroll
        for (int f = 0; f < 4; ++f)
          acc[f][2 * p + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[f], b[i], acc[f][2 * p + i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i) b[i] = b_next[i];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) a[f] = a_next[f];
    // the stage after the next has landed where only those after it are on their way
    if (more) landed<(kStages - 3) * LOADS>();
    else if (kStages > 4 && s + kStages - 2 < stages) landed<LOADS>();
    else landed<0>();
    now = next;
  }
}

// As `place`, but a tile's column blocks all go to one die, tiles in turn, where experts have a tile each (or up to a quarter
// of all tiles are further ones): the die's L2 holds the tile's rows for them, and no die reads every tile's.  The kernel is bound by
// what it draws through the fabric, and rows read by eight dies are a third of that.  Microseconds of the first and the second
// product, packed, columns dealt to the dies and plain loads / tiles and streaming loads (weights are read once then):
//   32 experts of 2048 x 2048, 245 rows 176 + 93 / 164 + 85, 138 rows 132 + 72 / 120 + 62, every other expert's twice as many
//   176 + 102 / 170 + 98; 25 of them, 240 rows 144 + 73 / 127 + 67; 12 of them 70 + 59 / 68 + 58;
//   64 of 2048 x 1024, 125 rows 127 + 83 / 109 + 66; 16 of 2048 x 2048, 256 rows 89 + 67 / 78 + 66.
// With two tiles an expert (500 rows) the dies would read the weights twice: 296 + 150 / 304 + 157.  Tiles that leave dies idle
// or the fullest die (32 blocks a round) more rounds than an even split stay with it too: 4 experts of 2048 x 2048 61 + 56 /
// 63 + 58, of 2048 x 8192 80 + 181 / 127 + 180.
__device__ __forceinline__ TilePlace place_wide(int id, const int32_t* tiles, int num_tiles, int cols, int lane) {
  const int turns = (num_tiles + 7) / 8;  // tiles of the fullest die
  int again = 0;                          // tiles behind the first of their expert
  for (int t0 = 0; t0 < num_tiles; t0 += kWave) {
    const int t = t0 + lane;
    again += __popcll(__ballot(t + 1 < num_tiles && tiles[3 * t] == tiles[3 * t + 3]));
  }
  if (num_tiles < 8 || (turns * cols + 31) / 32 > (num_tiles * cols + 255) / 256 || 4 * again > num_tiles)
    return place(id, num_tiles, cols);
  const int idx = id >> 3, turn = idx / cols, tile = 8 * turn + (id & 7);
  return {tile < num_tiles ? tile : -1, idx - turn * cols};
}

template <int GATED, typename TO, int PACKED>
__global__ __launch_bounds__(512) void moe_gemm_wide_kernel(
    TO* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ x, int64_t x_stride,
    const bf16_t* __restrict__ w, const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles,
    const int32_t* __restrict__ num_tiles, int N, int K, int in_div, int out_sorted, float limit, float alpha, float shift,
    int act, const float* __restrict__ row_scale, SharedExpert shared) {
  constexpr int COLS = GATED ? 128 : 256;  // a block's columns of the result
  __shared__ __attribute__((aligned(1024))) char lds[kWideLds];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const TilePlace at = place_wide(blockIdx.x, tiles, *num_tiles, (N + COLS - 1) / COLS, lane);
  if (at.tile < 0) return;
  const int e = tiles[3 * at.tile], r0 = tiles[3 * at.tile + 1];
  const int nr = __builtin_amdgcn_readfirstlane(tiles[3 * at.tile + 2]);
  const int li = lane & 15, lk = lane >> 4, wr = wave & 1, wc = wave >> 1;
  const int c0 = at.col * COLS, n0 = c0 + wc * (COLS / 4);
  const int64_t rows_per_expert = GATED ? 2 * static_cast<int64_t>(N) : N;
  // what the lane fetches of row blocks wave, wave + 8 and wave + 16 and of column blocks
  // wave and wave + 8 (gated: the second is up's)
  const int part = 16 * ((lane & 3) ^ ((lane >> 3) & 3));
  const bf16_t* we = expert_weights(w, e, rows_per_expert * K, shared);
  const char *xp[3], *wp[2];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int row = 16 * (wave + 8 * j) + (lane >> 2);
    const int safe = row < nr ? row : 0;  // a row that is not there reads the tile's first and is dropped
    const int64_t in_row = in_div > 0 ? input_row(sorted[r0 + safe], 0, in_div, e, shared) : r0 + safe;
    xp[j] = reinterpret_cast<const char*>(x + in_row * x_stride) + part;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int64_t first = GATED && j == 1 ? N : 0;
    if (PACKED) {  // pieces of 16 rows x 32 values
      const int n = c0 + 16 * (GATED ? wave : wave + 8 * j);
      wp[j] = reinterpret_cast<const char*>(we) + ((first + (n < N ? n : N - 16)) >> 4) * (K / 32) * 1024 + 64 * (lane >> 2) + part;
    } else {
      const int n = c0 + 16 * (GATED ? wave : wave + 8 * j) + (lane >> 2);
      wp[j] = reinterpret_cast<const char*>(we + (first + (n < N ? n : N - 1)) * K) + part;
    }
  }
  int wt[4];  // the wave's column blocks, in bytes
#pragma unroll
  for (int f = 0; f < 4; ++f) wt[f] = 1024 * (GATED ? 8 * (f >> 1) + 2 * wc + (f & 1) : 4 * wc + f);
  f32x4_t acc[4][kWideBlocks];  // gated: [0..1] gate, [2..3] up
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int r = 0; r < kWideBlocks; ++r) acc[f][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // every block walks K round from a place of its own, as in the kernel for tiles of 128 rows, and from the same one
  const int turn = (turn_of(e) + at.col * 11) % (K / 64) * 2;
  // an expert of more tiles than one has some 200 rows in each
  constexpr bool kStream = PACKED != 0;
  const bool alone = kStream && only_tile(tiles, at.tile, *num_tiles);
  switch ((nr + 31) >> 5) {  // scalar
#define KVC_WALK_OF(R, ONCE) wide_walk<PACKED, R, ONCE>(lds, xp, wp, wave, lane, wt, K / 32, turn, acc)
#define KVC_WALK(R) case R: KVC_WALK_OF(R, kStream); break
#define KVC_WALK2(R)                       \
  case R:                                  \
    if (alone) KVC_WALK_OF(R, kStream);    \
    else KVC_WALK_OF(R, false);            \
    break
    KVC_WALK(1); KVC_WALK(2); KVC_WALK(3); KVC_WALK(4); KVC_WALK(5); KVC_WALK2(6); KVC_WALK2(7);
    KVC_WALK2(8); KVC_WALK2(9); KVC_WALK2(10); KVC_WALK2(11); KVC_WALK2(12);
#undef KVC_WALK2
#undef KVC_WALK
#undef KVC_WALK_OF
  }
  if (n0 >= N) return;  // the whole wave
  // lane holds row 16 (2 r + wr) + li of the tile, columns n0 + 16 f + 4 lk + i
  store_tile<GATED, GATED ? 2 : 4, kWideBlocks, TO>(
      out, out_stride, [&](int r) { return 16 * (2 * r + wr) + li; }, nr, n0 + 4 * lk, N, r0, sorted, out_sorted, row_scale,
      e == kSharedExpert ? shared.limit : limit, alpha, shift, act, [&](int f, int r) { return acc[f][r]; },
      [&](int f, int r) { return acc[GATED ? f + 2 : 0][r]; });
}

// Any operand type and any sizes: a thread a (row, column) pair of the tile, float32 sums in index
// order.  The float32 path, and bfloat16 rows that 16-byte loads do not divide.
template <int GATED, typename TI, typename TO>
__global__ __launch_bounds__(256) void moe_gemm_plain_kernel(
    TO* __restrict__ out, int64_t out_stride, const TI* __restrict__ x, int64_t x_stride,
    const TI* __restrict__ w, const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles,
    const int32_t* __restrict__ num_tiles, int N, int K, int in_div, int out_sorted, float limit, float alpha, float shift,
    int act, const float* __restrict__ row_scale, SharedExpert shared) {
  const int tile = blockIdx.x;
  if (tile >= *num_tiles) return;
  const int e = tiles[3 * tile], r0 = tiles[3 * tile + 1], nr = tiles[3 * tile + 2];
  const int li = threadIdx.x & 15, col = threadIdx.x >> 4;  // 16 rows x 16 columns a pass
  if (li >= nr) return;
  const int pair = sorted[r0 + li];
  const int64_t in_row = input_row(pair, r0 + li, in_div, e, shared);
  const TI* xr = x + in_row * x_stride;
  const int64_t rows_per_expert = GATED ? 2 * static_cast<int64_t>(N) : N;
  const int64_t out_row = out_sorted ? r0 + li : pair;
  for (int n = blockIdx.y * 64 + col; n < N && n < (blockIdx.y + 1) * 64; n += 16) {
    const TI* wr = expert_weights(w, e, rows_per_expert * K, shared) + static_cast<int64_t>(n) * K;
    float acc = 0.f, acc2 = 0.f;
    for (int k = 0; k < K; ++k) {
      const float xv = to_float(xr[k]);
      acc = fmaf(xv, to_float(wr[k]), acc);
      if (GATED) acc2 = fmaf(xv, to_float(wr[static_cast<int64_t>(N) * K + k]), acc2);
    }
    const float scale = row_scale != nullptr ? row_scale[pair] : 1.f;
    out[out_row * out_stride + n] = from_float<TO>(
        GATED ? clamped_glu(acc * scale, acc2 * scale, e == kSharedExpert ? shared.limit : limit, alpha, shift)
              : plain_act(acc * scale, act));
  }
}

// VEC columns a thread (4 where rows and pointers allow 16-byte loads): bound by reading the experts' rows.
// 2,030 tokens of 2,048 columns with four choices: 37 us with one column a thread, 21 us.
template <typename TA, int VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ out, const float* __restrict__ y,
                                                          const float* __restrict__ weight, int top,
                                                          const TA* __restrict__ add0, const float* __restrict__ add1,
                                                          const float* __restrict__ add1_gate, int T, int H,
                                                          int accumulate) {
  const int64_t idx = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * VEC;
  if (idx >= static_cast<int64_t>(T) * H) return;
  const int t = static_cast<int>(idx / H), c = static_cast<int>(idx - static_cast<int64_t>(t) * H);
  typedef float vec_t __attribute__((ext_vector_type(VEC)));
  auto load = [](const float* p) { return *reinterpret_cast<const vec_t*>(p); };
  const float* yt = y + static_cast<int64_t>(t) * top * H + c;
  vec_t acc = 0.f;
#pragma unroll 4
  for (int j = 0; j < top; ++j) {
    const float w = weight != nullptr ? weight[static_cast<int64_t>(t) * top + j] : 1.f;
    const vec_t v = load(yt + static_cast<int64_t>(j) * H);
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = fmaf(w, v[i], acc[i]);
  }
  if (add0 != nullptr) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] += to_float(add0[idx + i]);
  }
  if (add1 != nullptr) {
    const vec_t v = load(add1 + idx);
    const float g = add1_gate != nullptr ? add1_gate[t] : 0.f;
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = add1_gate != nullptr ? fmaf(g, v[i], acc[i]) : acc[i] + v[i];
  }
  vec_t* o = reinterpret_cast<vec_t*>(out + idx);
  *o = accumulate ? *o + acc : acc;
}

// The same into the residual stream, a block a token, which has the new row in registers and leaves its norm for the next layer:
// in few rows a launch is all that the norm by itself takes, in many its row read again.  Every sum in the order of the two
// kernels (`add_rmsnorm_vec_kernel` has the norm's), so with their bits.  2,048 columns, four choices and two more rows, float32 to
// bfloat16, in a graph, two kernels / this one: 1 token 5.1 / 3.5 us, 8 5.3 / 3.7, 64 6.2 / 4.1, 300 8.2 / 6.2, 2,048 31.4 / 27.0 (5.6 TB/s).
template <typename TO, int NCH>
__global__ __launch_bounds__(256) void moe_combine_norm_kernel(
    TO* __restrict__ x, float* __restrict__ residual, const float* __restrict__ y, const float* __restrict__ weight, int top,
    const float* __restrict__ add0, const float* __restrict__ add1, const float* __restrict__ add1_gate,
    const float* __restrict__ gain, float eps, int H) {
  __shared__ float scratch[16];
  const int64_t t = blockIdx.x, base = t * H;
  float v[NCH][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int e = (c * 256 + threadIdx.x) * 8;
    if (e >= H) continue;
    const float* yt = y + t * top * H + e;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, u[8];
#pragma unroll 4
    for (int j = 0; j < top; ++j) {
      const float w = weight != nullptr ? weight[t * top + j] : 1.f;
      load8(yt + static_cast<int64_t>(j) * H, u);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = fmaf(w, u[i], acc[i]);
    }
    if (add0 != nullptr) {
      load8(add0 + base + e, u);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += u[i];
    }
    if (add1 != nullptr) {
      load8(add1 + base + e, u);
      const float g = add1_gate != nullptr ? add1_gate[t] : 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = add1_gate != nullptr ? fmaf(g, u[i], acc[i]) : acc[i] + u[i];
    }
    load8(residual + base + e, v[c]);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[c][i] += acc[i];
    store8(residual + base + e, v[c]);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += v[c][i] * v[c][i];
  }
  const float inv = rsqrtf(block_sum(ss, scratch) / static_cast<float>(H) + eps);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int e = (c * 256 + threadIdx.x) * 8;
    if (e >= H) continue;
    float w[8], o[8];
    load8(gain + e, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = w[i] * (v[c][i] * inv);
    store8(x + base + e, o);
  }
}

}  // namespace

extern "C" int kvc_moe_route(int32_t* choice, float* weight, const float* logits, int T, int E, int top,
                             int groups, int keep, int score_fn, const float* bias, const float* correction,
                             int group_best, int renormalize, float weight_scale, kvc_stream stream) {
  if (T < 0 || E <= 0 || top <= 0 || top > E || top > kWave || groups <= 0 || E % groups || keep <= 0 ||
      keep > groups)
    return kvc_fail("kvc_moe_route: bad sizes (at most 64 choices; the experts in equal groups)");
  if (score_fn < 0 || score_fn > 2 || (group_best != 1 && group_best != 2))
    return kvc_fail("kvc_moe_route: scores by softmax (0), sigmoid (1) or logit (2); a group is worth its best 1 or 2");
  const RouteRule rule{top, groups, keep, score_fn, group_best, renormalize, bias, correction, weight_scale};
  const size_t lds = sizeof(float) * 4 * (2 * E + groups);
  if (lds > 60000) return kvc_fail("kvc_moe_route: too many experts for a wave's scores in LDS");
  if (T == 0) return 0;
  hipLaunchKernelGGL(moe_route_kernel, dim3((T + 3) / 4), dim3(256), lds, S(stream), choice, weight, logits, T, E,
                     rule);
  return kvc_check_launch("kvc_moe_route");
}

extern "C" int kvc_moe_router(int32_t* choice, float* weight, const void* x, int64_t x_stride, int x_dtype,
                              const float* router, float* gate, int T, int H, int E, int top, int groups, int keep,
                              int score_fn, const float* bias, const float* correction, int group_best,
                              int renormalize, float weight_scale, kvc_stream stream) {
  if (T < 0 || H <= 0 || E <= 0 || top <= 0 || top > E || top > kWave || groups <= 0 || E % groups || keep <= 0 ||
      keep > groups || x_stride < H)
    return kvc_fail("kvc_moe_router: bad sizes (at most 64 choices; the experts in equal groups)");
  if (score_fn < 0 || score_fn > 2 || (group_best != 1 && group_best != 2))
    return kvc_fail("kvc_moe_router: scores by softmax (0), sigmoid (1) or logit (2); a group is worth its best 1 or 2");
  const RouteRule rule{top, groups, keep, score_fn, group_best, renormalize, bias, correction, weight_scale};
  if (T == 0) return 0;
  const size_t lds = sizeof(float) * (static_cast<size_t>(kRouterWaves) * (kRouterRows * kRouterPad + kRouterTokens) +
                                      static_cast<size_t>(kRouterTokens) * (2 * E + groups));
  if (lds > 160 * 1024) return kvc_fail("kvc_moe_router: too many experts for a block's LDS");
  const dim3 grid((T + kRouterTokens - 1) / kRouterTokens);
  // 16-byte loads where the rows allow
  const bool vectors = H % 8 == 0 && x_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(router) & 15) == 0 &&
                       (reinterpret_cast<uintptr_t>(x) & 15) == 0;
#define KVC_ROUTER(Tp, VEC)                                                                                     \
  do {                                                                                                          \
    if (lds > 64 * 1024) {                                                                                      \
      const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_router_kernel<Tp, VEC>),   \
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)); \
      if (attr != hipSuccess) return kvc_fail("kvc_moe_router: the kernel's LDS size was refused");            \
    }                                                                                                           \
    hipLaunchKernelGGL((moe_router_kernel<Tp, VEC>), grid, dim3(kRouterWaves * kWave), lds, S(stream), choice,  \
                       weight, static_cast<const Tp*>(x), x_stride, router, gate, T, H, E, rule);               \
  } while (0)
  if (x_dtype == 1 && vectors) KVC_ROUTER(bf16_t, 1);
  else if (x_dtype == 1) KVC_ROUTER(bf16_t, 0);
  else if (x_dtype == 0 && vectors) KVC_ROUTER(float, 1);
  else if (x_dtype == 0) KVC_ROUTER(float, 0);
  else return kvc_fail("kvc_moe_router: unknown dtype code");
#undef KVC_ROUTER
  return kvc_check_launch("kvc_moe_router");
}

// how many tiles the rows of an expert that every token runs take at most
static int shared_tiles(int rows, int tile_rows) { return (rows + tile_rows - 1) / tile_rows; }

extern "C" int kvc_moe_router_spread_tokens(void) { return kRouterSpread; }
extern "C" int kvc_moe_router_spread_floats(int T, int E) { return kRouterWaves * T * router_part_row(E); }

extern "C" int kvc_moe_router_spread(int32_t* choice, float* weight, int32_t* sorted, int32_t* tiles, int32_t* num_tiles,
                                  int max_tiles, int tile_rows, int shared_rows, float* parts, int64_t parts_floats, const void* x,
                                  int64_t x_stride, int x_dtype, const float* router, float* gate, int T, int H, int E,
                                  int top, int groups, int keep, int score_fn, const float* bias, const float* correction,
                                  int group_best, int renormalize, float weight_scale, kvc_stream stream) {
  if (T < 0 || H <= 0 || E <= 0 || top <= 0 || top > E || groups <= 0 || E % groups || keep <= 0 || keep > groups ||
      x_stride < H)
    return kvc_fail("kvc_moe_router_spread: bad sizes (the experts in equal groups)");
  if (T > kRouterSpread || E > kWave) return kvc_fail("kvc_moe_router_spread: at most 1024 tokens and 64 experts");
  if (score_fn < 0 || score_fn > 2 || (group_best != 1 && group_best != 2))
    return kvc_fail("kvc_moe_router_spread: scores by softmax (0), sigmoid (1) or logit (2); a group is worth its best 1 or 2");
  if (!known_tile_rows(tile_rows))
    return kvc_fail("kvc_moe_router_spread: tiles of 16, 64, 128 or 384 rows");
  if (shared_rows < 0 || max_tiles < kvc_moe_max_tiles(T * top, E, tile_rows) + shared_tiles(shared_rows, tile_rows))
    return kvc_fail("kvc_moe_router_spread: room for fewer tiles than the routing may need");
  if (parts_floats < kvc_moe_router_spread_floats(T, E) || (reinterpret_cast<uintptr_t>(parts) & 15) != 0)
    return kvc_fail("kvc_moe_router_spread: the workspace is too small or not 16-byte aligned");
  if (x_dtype != 0 && x_dtype != 1) return kvc_fail("kvc_moe_router_spread: unknown dtype code");
  if (T == 0) return 0;
  const RouteRule rule{top, groups, keep, score_fn, group_best, renormalize, bias, correction, weight_scale};
  const dim3 grid((T + kRouterTokens - 1) / kRouterTokens, kRouterWaves, (E + kRouterRows - 1) / kRouterRows);
  // 16-byte loads where the rows allow
  const bool vectors = H % 8 == 0 && x_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(router) & 15) == 0 &&
                       (reinterpret_cast<uintptr_t>(x) & 15) == 0;
#define KVC_PARTS(Tp, VEC)                                                                                       \
  hipLaunchKernelGGL((moe_router_parts_kernel<Tp, VEC>), grid, dim3(kWave), 0, S(stream), parts,                 \
                     static_cast<const Tp*>(x), x_stride, router, gate != nullptr ? 1 : 0, T, H, E)
  if (x_dtype == 1 && vectors) KVC_PARTS(bf16_t, 1);
  else if (x_dtype == 1) KVC_PARTS(bf16_t, 0);
  else if (vectors) KVC_PARTS(float, 1);
  else KVC_PARTS(float, 0);
#undef KVC_PARTS
  if (T <= kChooseInOne) {
    hipLaunchKernelGGL(moe_choose_align_kernel, dim3(1), dim3(1024), sizeof(int32_t) * (T * top + 3 * E), S(stream),
                       choice, weight, gate, sorted, tiles, num_tiles, parts, T, E, max_tiles, tile_rows, shared_rows, rule);
    return kvc_check_launch("kvc_moe_router_spread");
  }
  hipLaunchKernelGGL(moe_choose_kernel, dim3((T + 3) / 4), dim3(256), 0, S(stream), choice, weight, gate, parts, T, E, rule);
  return kvc_moe_align(sorted, tiles, num_tiles, choice, T * top, E, max_tiles, tile_rows, shared_rows, stream);
}

extern "C" int kvc_moe_max_tiles(int pairs, int E, int tile_rows) {
  const int most = (pairs + tile_rows - 1) / tile_rows + E;
  return pairs < most ? pairs : most;  // no tile is empty
}

// How many rows a tile holds, for experts of matrices [I, H] ([2 I, H] if gated) and [H, I], by an estimate of both
// products in us, for tokens that choose their experts at random.  Tiles of 16: the matrices of the experts that are
// chosen at 6.6 TB/s, and again for each further tile, of which there are some from 4.5 rows an expert on.  Tiles of 64:
// one fetch, at 6.1 TB/s gated and 7.2 otherwise (before loads marked as streaming ones, which read a tenth more in
// either kind of tile: 8 rows 129 / 130 us for the first line's 146 / 139, 16 rows 162 / 132), but columns of 128 (ungated 256) a block, so a product is no faster than
// a block's walk along K (1.05 us a pass of 64), and blocks that come out uneven on the units wait for the last.  Both
// products, tiles of 16 / 64, by rows an expert, gated:
//   32 experts of 2048 x 2048     1   90 / 101 us    4  141 / 139    8  146 / 139   16  177 / 145
//   16 experts of 1024 x 1024     4   21 /  27       8   21 /  27   16   27 /  30   32   39 /  34
//   4 experts of 1024 x 2048      8   15 /  36      32   20 /  38   64   33 /  46
//   128 experts of 1024 x 384     4   52 /  60      12   63 /  65   16   74 /  68
// and not gated:
//   32 experts of 2048 x 2048     1   54 /  62       4   97 /  90    8  100 /  91
//   16 experts of 2048 x 2048     8   45 /  56      12   52 /  57   24   87 /  61
// Over 428 such steps of fourteen sizes, gated and not, the tiles it takes are 1.001 x the faster in the mean and 1.09 x
// at most.  Tiles of 128 where experts have that many rows and the blocks still fill the chip (300 in either product if they held
// 64 rows: the second of two blocks a unit keeps the matrix cores busy): 32 experts of 2048 x 2048, 64 rows each,
// 188 / 165 us, 16 experts of 1024 x 1024 41 / 53.  From 104 to 150 rows many an expert has a few more than 128, and two
// tiles of half the size cost more than smaller ones: 128 rows 227 us in tiles of 64, 249 in tiles of 128.
struct TileEstimate {
  double each, used, mb, mid;  // rows an expert, experts with rows, megabytes of an expert, us in tiles of 64
  int first_cols, down_cols;
};
static TileEstimate estimate_tiles(int pairs, int E, int H, int I, int gated) {
  TileEstimate t;
  const double units = kvc_device_compute_units();
  t.each = static_cast<double>(pairs) / E;
  t.used = E * -expm1(-t.each);
  t.first_cols = gated ? (I + 127) / 128 : (I + 255) / 256, t.down_cols = (H + 255) / 256;
  const double down_mb = 2e-6 * H * I, first_mb = gated ? 2 * down_mb : down_mb;
  t.mb = first_mb + down_mb;
  const double mid_tiles = t.used + (t.each > 32 ? (t.each - 32) / 64 * E : 0);
  auto product = [&](double mb, double rate, int k, int cols) {
    const double a_unit = mid_tiles * cols / units;
    const double uneven = a_unit > 1 ? ceil(a_unit) / a_unit : 1;
    return 5 + fmax(1.05 * k / 64, t.used * mb / rate * uneven);
  };
  t.mid = product(first_mb, gated ? 6.1 : 7.2, H, t.first_cols) + product(down_mb, 7.2, I, t.down_cols);
  return t;
}

extern "C" int kvc_moe_tile_rows(int pairs, int E, int H, int I, int gated) {
  if (pairs <= 0 || E <= 0 || H <= 0 || I <= 0) return kTileRows;
  const TileEstimate est = estimate_tiles(pairs, E, H, I, gated);
  const double each = est.each;
  const int first_cols = est.first_cols, down_cols = est.down_cols;
  const double again = each > 4.5 ? (each - 4.5) / 16 * E : 0;
  const double few = 10 + est.mb * (est.used / 6.6 + again / 6.5);
  if (each <= 64 && few <= est.mid) return kTileRows;
  const double blocks = (pairs / 64.0 + E / 2.0) * (first_cols < down_cols ? first_cols : down_cols);
  return blocks >= 300 && (each >= 150 || (each >= 40 && each < 104)) ? kBigTileRows : kMidTileRows;
}

// Whether tiles of up to 384 rows (the answer; otherwise 0) serve such a step better, also where the experts' rows are uneven, which
// no launch knows.  A block of theirs has a compute unit to itself, and the largest one (three times the mean and more rows soon
// make it full) lasts as long as two or three in the mean: with one round of blocks the units wait for it, with two, the
// largest first, they do not.  So the first product needs two blocks a unit and the second one a block, experts wide enough
// that a block's way in and out counts little, and 104 rows an expert; or one block a unit and every other one, where the
// experts' rows fill two thirds of a tile in the mean and K is long; or (an expert has more than one tile only from where nearly all do, as
// rows vary by some three times their root) two tiles an expert.  Both products and the list in us, the best of the smaller tiles /
// these, experts of the same chance, and of chances by which the fullest has 2 to 3, 4 to 5 and 7 to 15 times the mean, gated:
//   32 experts of 2048 x 2048   110  220 / 193  228 / 203  220 / 217  226 / 203    256  324 / 275  337 / 306  334 / 294  337 / 284
//   64 experts of 2048 x 1024   110  234 / 211  230 / 208  228 / 215  219 / 191    256  342 / 297  341 / 328  347 / 313  358 / 319
//   16 experts of 2048 x 2048   256  191 / 160  192 / 183  192 / 170  196 / 176    500  296 / 220  293 / 243  308 / 239  294 / 242
//   64 experts of 1024 x 512    500  209 / 181  208 / 192  208 / 193  208 / 198
// not gated:
//   32 experts of 2048 x 2048   256  243 / 198  245 / 240  244 / 210  232 / 205
// and not taken:
//   16 experts of 2048 x 2048   130  139 / 122  136 / 154  133 / 162  130 / 147    180  133 / 135  138 / 178  146 / 164  140 / 157
//   64 experts of 1024 x 512    130   86 /  76   87 / 114   86 / 124   83 / 121    256  131 / 109  131 / 157  130 / 148  131 / 155
//   64 experts of 1024 x 1024   130  139 / 124  134 / 139  137 / 143  134 / 136    180  149 / 142  154 / 177  154 / 172  151 / 173
//   128 experts of 1024 x 384   130  132 / 136  134 / 156  135 / 161  133 / 160    256  197 / 193  198 / 214  196 / 207  190 / 204
extern "C" int kvc_moe_wide_tile_rows(int pairs, int E, int H, int I, int gated) {
  if (pairs <= 0 || E <= 0 || H <= 0 || I <= 0 || H % 64 || I % 64) return 0;
  const double each = static_cast<double>(pairs) / E, units = kvc_device_compute_units();
  const double of_one = fmax(1.0, ceil((each - 3 * sqrt(each)) / kWideTileRows)), tiles = E * of_one;
  const double first = tiles * (gated ? (I + 127) / 128 : (I + 255) / 256) / units, down = tiles * ((H + 255) / 256) / units;
  const bool two_rounds = first >= 2 && down >= 1 && (H + I >= 3072 || of_one > 1);
  const bool full = first >= 1 && down >= 0.5 && each >= 230 && H >= 2048 && I >= 2048;
  return each >= 104 && (two_rounds || full) ? kWideTileRows : 0;
}

// Tiles of up to 384 rows (the answer; otherwise 0) for fewer rows an expert than the rule above asks for: where the first product
// has two blocks a unit and the second one a block if every expert is one tile, none is waited for, and an expert with more rows
// than its share fetches its weights once, where tiles of 128 rows fetch them again for every tile.  Both products and the
// list in us, the best of the smaller tiles / these, experts of the same chance, and of chances by which the fullest has 2 to 3, and
// 3.5 to 6 times the mean, gated:
//   32 experts of 2048 x 2048    56  153 / 152  167 / 157  164 / 170    72  157 / 155  200 / 174  193 / 199    100  172 / 164  201 / 175  202 / 207
//   64 experts of 2048 x 1024    56  166 / 163  177 / 163  180 / 167    72  173 / 169  206 / 173  196 / 184    100  192 / 175  223 / 189  215 / 192
//   64 experts of 2048 x 2048    56  303 / 294  320 / 296  332 / 302    72  315 / 301  356 / 310  353 / 340    100  346 / 316  387 / 336  383 / 360
//   48 experts of 2048 x 1536    56  193 / 192  189 / 185  204 / 182    72  212 / 201  214 / 197  213 / 197    100  230 / 221  235 / 216  244 / 210
//   32 experts of 4096 x 2048    56  300 / 288  330 / 293  341 / 306    72  314 / 294  368 / 315  361 / 340    100  339 / 306  382 / 319  384 / 361
//   128 experts of 2048 x 1024   56  326 / 310  349 / 323  341 / 331    72  343 / 319  361 / 365  374 / 353    100  371 / 343  408 / 367  414 / 370
// not gated:
//   64 experts of 2048 x 2048    56  209 / 200  223 / 201  239 / 211    72  218 / 204  263 / 213  252 / 233    100  241 / 214  283 / 235  269 / 246
// A step over 15 layers of 32 experts of 2048 x 2048, four a token, beside an expert that every token runs: 450 tokens 4,220 ->
// 4,165 us, 600 4,730 -> 4,565, 700 4,925 -> 4,745, 820 5,830 -> 5,055.
// At 40 rows they are level where experts have the same chance (148 / 148, 155 / 159, 286 / 289), and an expert that every token
// runs costs in them what it does not in tiles of 64 (177 / 193).
extern "C" int kvc_moe_one_tile_rows(int pairs, int E, int H, int I, int gated) {
  if (pairs <= 0 || E <= 0 || H <= 0 || I <= 0 || H % 64 || I % 64) return 0;
  const double each = static_cast<double>(pairs) / E, units = kvc_device_compute_units();
  const double first = E * static_cast<double>(gated ? (I + 127) / 128 : (I + 255) / 256) / units;
  const double down = E * static_cast<double>((H + 255) / 256) / units;
  return each >= 48 && each < 104 && first >= 2 && down >= 1 && H + I >= 3072 ? kWideTileRows : 0;
}

// us that the expert of every one of T tokens takes in tiles of 16 beside the routed ones: its matrices once, at the rate of theirs,
// and again for every further tile (a die's L2 holds less than they are); and in two products of its own, which reach
// the memory's rate where matrices are large (taken for 20 + mb / 2.8 us throughout, 48 tokens of 16 experts of 2048 x 8192 joined in tiles
// of 16 for 360 us a layer, 350 alone).
static double shared_in_few_us(double mb, int T) { return mb / 6.6 + (shared_tiles(T, kTileRows) - 1) * mb / 6.2; }
static double shared_alone_us(double mb, int T) { return T <= 16 ? 8.6 + mb / 6.4 : fmin(20 + mb / 2.8, 28 + mb / 6); }

// Whether the expert that every one of T tokens runs joins the routed experts' launches, and in tiles of how many rows all of
// them then go (0: it stays with products of its own), where tile_rows is what they would take alone.
// In tiles of 16 it is one more expert whose rows fill its tiles, at the rate at which weights stream, where two products of
// its own take 13 us up to 16 tokens and some 30 beyond for 25 MB.  Larger tiles are few blocks a unit: it joins them where the
// launches' blocks a unit, rounded up, stay what they are, as a unit with one block more makes the whole chip wait (32 experts of 2048 x
// 2048, 64 tokens of four, two blocks a unit and 16 more 95 -> 111 us).  So small tiles are worth more with it than without, up to where
// experts of random tokens begin to have more rows than one holds, or its own tiles have read its matrices too often.
// Captured steps, us a layer with it alone / joined in tiles of 16 / of what the others take alone (64 where not said); where this rule
// counted no second reading, it took tiles of 16 up to 128 tokens in all of these:
//   32 of 2048 x 2048, 4 a token  24 tokens 179 / 170 (16)   48 216 / 196 / 203   64 219 / 205 / 207   96 231 / 235 / 231   128 245 / 267 / 241
//   64 of 2048 x 2048, 4 a token  64 tokens 320 / 306 (16)   96 351 / 339 / 332   128 373 / 369 / 355   160 378 / 399 / 375
//   24 of 3072 x 3072, 4 a token  64 tokens 368 / 360 (16)   96 402 / 432 / 354   128 425 / 507 / 371
//   16 of 4096 x 4096, 2 a token  32 tokens 342 / 340 (16)   48 380 / 374 / 374   64 396 / 414 / 404    96 425 / 498 / 441   128 461 / 582 / 456
//   16 of 2048 x 8192, 2 a token  40 tokens 340 / 349 (16)   48 350 / 360 (16)    96 438 / 464 / 412   128 455 / 557 / 423
//   64 of 4096 x 2048, 4 a token  64 tokens 570 / 560 (16)   96 639 / 618 / 597   128 681 / 688 / 651
//   16 of 1024 x 1024, 4 a token  32 tokens 92 / 80 (16)     64 121 / 103 (16)    96 127 / 111 / 103
// A step of 15 layers of 32 experts of 2048 x 2048, four a token, alone / joined in tiles of 64 / of 128 rows, us:
//   300 tokens 4018 / 3883 / 4121   500 4268 / 4267 / 4467
// `beside` another branch's kernels it joins more often, as products of its own come before the branches part: in tiles of 16 wherever these
// cost less than its own products, in larger ones up to 64 MB an expert, or up to 511 tokens.  Steps of eight layers (16 of the first sizes)
// beside mixers, own products / joined, us:
//   32 of 2048 x 2048 (25 MB)    400 tokens 5,620 / 5,230   1,000 6,287 / 6,126   1,500 8,251 / 7,243   2,048 9,385 / 8,889   4,096 17,040 / 16,640
//   64 of 4096 x 1024 (25 MB)    400 tokens 4,135 / 3,940   640 3,840 / 3,745     1,500 5,345 / 5,070   4,096 10,500 / 10,180
//   128 of 2048 x 1024 (13 MB), 8 a token  160 tokens 3,495 / 3,377   640 3,695 / 3,557   2,048 6,097 / 5,920
//   24 of 3072 x 3072 (57 MB)    256 tokens 3,275 / 3,275   640 3,840 / 3,845     1,250 5,300 / 5,350   3,000 11,550 / 11,070
//   16 of 4096 x 4096 (100 MB), 2 a token  64 tokens 3,105 / 3,270   160 3,607 / 3,397   400 4,535 / 4,240   820 5,000 / 4,620   1,000 5,050 / 5,480   1,500 6,270 / 6,600
//   16 of 2048 x 8192 (100 MB), 2 a token  160 tokens 3,977 / 3,537   400 4,810 / 4,560   650 4,885 / 5,050   1,000 6,370 / 6,050   4,096 13,050 / 13,410
extern "C" int kvc_moe_shared_tile_rows(int pairs, int E, int H, int I, int gated, int T, int tile_rows, int beside) {
  if (pairs <= 0 || E <= 0 || H <= 0 || I <= 0 || T <= 0 || !known_tile_rows(tile_rows)) return 0;
  constexpr int kMost = 128;  // tokens up to which tiles of 16 were measured
  const TileEstimate est = estimate_tiles(pairs, E, H, I, gated);
  const double in_few = shared_in_few_us(est.mb, T), own = shared_alone_us(est.mb, T);
  if (tile_rows == kTileRows) return (beside || T <= kMost) && in_few <= own ? kTileRows : 0;
  const double units = kvc_device_compute_units();
  const double tiles = tile_rows == kWideTileRows
                           ? est.used * fmax(1.0, ceil((est.each - 3 * sqrt(est.each)) / kWideTileRows))
                           : est.used + (est.each > tile_rows / 2.0 ? (est.each / tile_rows - 0.5) * E : 0);
  auto room = [&](int cols) {
    return ceil((tiles + shared_tiles(T, tile_rows)) * cols / units) <= ceil(tiles * cols / units);
  };
  // where the last round has but begun, few units wait for it (alone / joined, 32 experts of 2048 x 2048 in tiles of 128 rows, 583
  // tokens 4,520 / 4,600, 650 5,003 / 4,738; tiles of 384 take these numbers of tokens since, but not those of smaller experts)
  const double rounds = tiles * est.first_cols / units;
  const bool begun = rounds - floor(rounds) >= (tile_rows == kMidTileRows ? 0.1 : 0.25);
  const bool joins = begun && room(est.first_cols) && room(est.down_cols);
  if (T <= kMost && est.each <= 16 && tile_rows == kMidTileRows) {
    const double again = 0.5 * E * erfc((16.5 - est.each) / sqrt(2 * est.each));  // experts with more than 16 rows
    const double few = 10 + est.mb * (est.used / 6.6 + again / 6.5) + in_few;
    if (few <= est.mid + (joins ? est.mb / 6.5 : own)) return kTileRows;
  }
  return joins || (beside && (est.mb <= 64 || T < 512)) ? tile_rows : 0;
}

extern "C" int kvc_moe_align(int32_t* sorted, int32_t* tiles, int32_t* num_tiles, const int32_t* choice,
                             int pairs, int E, int max_tiles, int tile_rows, int shared_rows, kvc_stream stream) {
  if (!known_tile_rows(tile_rows)) return kvc_fail("kvc_moe_align: tiles of 16, 64, 128 or 384 rows");
  if (pairs < 0 || E <= 0 || shared_rows < 0 ||
      max_tiles < kvc_moe_max_tiles(pairs, E, tile_rows) + shared_tiles(shared_rows, tile_rows))
    return kvc_fail("kvc_moe_align: bad sizes, or room for fewer tiles than the routing may need");
  const size_t lds = sizeof(int32_t) * 3 * E;
  if (lds > 60000) return kvc_fail("kvc_moe_align: too many experts");
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(1024), lds, S(stream), sorted, tiles, num_tiles, choice,
                     pairs, E, max_tiles, tile_rows, shared_rows);
  return kvc_check_launch("kvc_moe_align");
}

extern "C" int kvc_moe_gemm(void* out, int64_t out_stride, int out_dtype, const void* x, int64_t x_stride,
                            const void* w, int dtype, const int32_t* sorted, const int32_t* tiles,
                            const int32_t* num_tiles, int max_tiles, int tile_rows, int N, int K, int in_div,
                            int out_sorted, int gated, float limit, float alpha, float up_shift, int act,
                            const float* row_scale, const void* w_shared, int shared_first, float shared_limit, int packed,
                            kvc_stream stream) {
  const SharedExpert shared{w_shared, shared_first, shared_limit};
  if (w_shared != nullptr && row_scale != nullptr)
    return kvc_fail("kvc_moe_gemm: no scale a pair beside an expert that every token runs");
  if (max_tiles < 0 || N <= 0 || K <= 0 || x_stride < K || out_stride < N)
    return kvc_fail("kvc_moe_gemm: bad sizes");
  if (!known_tile_rows(tile_rows)) return kvc_fail("kvc_moe_gemm: tiles of 16, 64, 128 or 384 rows");
  if (act < -1 || act > 0 || (gated && act != -1))
    return kvc_fail("kvc_moe_gemm: an ungated product has no activation (-1) or the square of relu (0)");
  if (max_tiles == 0) return 0;
  dim3 grid(max_tiles, (N + 63) / 64);
  if (grid.y > 65535u) return kvc_fail("kvc_moe_gemm: too many columns");
#define KVC_MOE_ARGS sorted, tiles, num_tiles, N, K, in_div, out_sorted, limit, alpha, up_shift, act, row_scale, shared
#define KVC_MOE_LAUNCH(KERNEL, TI, TO)                                                                          \
  hipLaunchKernelGGL(KERNEL, grid, dim3(256), 0, S(stream), static_cast<TO*>(out), out_stride,                   \
                     static_cast<const TI*>(x), x_stride, static_cast<const TI*>(w), KVC_MOE_ARGS)
  if (out_dtype != 0 && out_dtype != 1) return kvc_fail("kvc_moe_gemm: unknown dtype code");
  if (dtype == 1) {
    // the matrix cores read 16 bytes at a time: rows of a multiple of 8 values, 16-byte aligned
    const bool vectors = K % 8 == 0 && x_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
                         ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(w_shared)) & 15) == 0;
    if (tile_rows != kTileRows) {
      if (!vectors || K % 32) return kvc_fail("kvc_moe_gemm: tiles of 64 rows and more need K to be a multiple of 32");
      if (tile_rows == kWideTileRows && K % 64) return kvc_fail("kvc_moe_gemm: tiles of 384 rows need K to be a multiple of 64");
      if (packed && (N % 16 || K % 64))
        return kvc_fail("kvc_moe_gemm: a packed matrix has experts of a multiple of 16 rows of a multiple of 64");
      const int64_t cols = gated ? (N + 127) / 128 : (N + 255) / 256;
      // every die gets its share of the pairs, or (384 rows) of the tiles
      const int64_t blocks = tile_rows == kWideTileRows ? 8 * (cols * ((static_cast<int64_t>(max_tiles) + 7) / 8))
                                                        : 8 * ((cols * max_tiles + 7) / 8);
      if (blocks > 0x7fffffff) return kvc_fail("kvc_moe_gemm: too many tiles for one launch");
      grid = dim3(static_cast<unsigned>(blocks));
      // Streaming loads have a kernel of their own with a second walk for experts of more tiles, which takes some registers more
      // (tiles of 64 rows 172, and so two blocks a unit for three): where most experts have more, all take the kernel without (4
      // experts of 2048 x 2048, 200 rows each, down 31.0 us, 29.4 so, 28.9 before there were such loads).  Short walks are not faster with
      // such loads (128 experts of 1024 x 384, 44 rows each, down 31.0 us with and 28.4 without).
      const bool stream_tiles = packed == 2 && K >= 512;
#define KVC_MOE_TILED(NR, PACKED)                                                                               \
  do {                                                                                                          \
    if (gated && out_dtype == 1) KVC_MOE_LAUNCH((moe_gemm_tiled_kernel<1, NR, bf16_t, PACKED>), bf16_t, bf16_t); \
    else if (gated) KVC_MOE_LAUNCH((moe_gemm_tiled_kernel<1, NR, float, PACKED>), bf16_t, float);               \
    else if (out_dtype == 1) KVC_MOE_LAUNCH((moe_gemm_tiled_kernel<0, NR, bf16_t, PACKED>), bf16_t, bf16_t);    \
    else KVC_MOE_LAUNCH((moe_gemm_tiled_kernel<0, NR, float, PACKED>), bf16_t, float);                          \
  } while (0)
      if (tile_rows == kWideTileRows) {
#define KVC_MOE_WIDE(GATED, TO, PACKED)                                                                           \
  hipLaunchKernelGGL((moe_gemm_wide_kernel<GATED, TO, PACKED>), grid, dim3(512), 0, S(stream),                     \
                     static_cast<TO*>(out), out_stride, static_cast<const bf16_t*>(x), x_stride,                  \
                     static_cast<const bf16_t*>(w), KVC_MOE_ARGS)
#define KVC_MOE_WIDE_OF(PACKED)                                  \
  do {                                                           \
    if (gated && out_dtype == 1) KVC_MOE_WIDE(1, bf16_t, PACKED); \
    else if (gated) KVC_MOE_WIDE(1, float, PACKED);              \
    else if (out_dtype == 1) KVC_MOE_WIDE(0, bf16_t, PACKED);    \
    else KVC_MOE_WIDE(0, float, PACKED);                         \
  } while (0)
        if (packed) KVC_MOE_WIDE_OF(1);
        else KVC_MOE_WIDE_OF(0);
#undef KVC_MOE_WIDE_OF
#undef KVC_MOE_WIDE
      } else if (tile_rows == kBigTileRows) {
        if (stream_tiles) KVC_MOE_TILED(8, 2);
        else if (packed) KVC_MOE_TILED(8, 1);
        else KVC_MOE_TILED(8, 0);
      } else {
        if (stream_tiles) KVC_MOE_TILED(4, 2);
        else if (packed) KVC_MOE_TILED(4, 1);
        else KVC_MOE_TILED(4, 0);
      }
#undef KVC_MOE_TILED
    } else if (vectors) {
      if (packed && (N % 16 || K % 64))
        return kvc_fail("kvc_moe_gemm: a packed matrix has experts of a multiple of 16 rows of a multiple of 64");
      // A whole K a wave where a share of it is at most two passes and there are waves enough without: one a compute unit
      // up to K of 256, three up to 512.  Shares / whole: 64 experts of 2048 x 512 down, 8 rows each, 36.7 / 26.2 us; 8
      // experts of 512 x 512 gated, 1 row each (256 waves), 5.4 / 6.6 us, 32 rows (768 waves) 9.5 / 8.3; 4 experts of
      // 256 x 384 gated, 48 rows (384 waves), 7.1 / 5.8; 16 experts of 1024 x 1024 (sixteen passes), 64 rows, 27 / 33 us.
      const int64_t waves = static_cast<int64_t>(max_tiles) * ((N + 15) / 16);
      const bool whole = K <= 512 && waves >= (K <= 256 ? 1 : 3) * static_cast<int64_t>(kvc_device_compute_units());
      kvc_note_variant(kVariantMoeGemm, whole ? "moe_gemm_few_kernel, whole K" : "moe_gemm_few_kernel, shares of K");
      const int layers = (max_tiles + 65534) / 65535;
      grid = dim3(whole ? (N + 63) / 64 : (N + 15) / 16, (max_tiles + layers - 1) / layers, layers);
#define KVC_MOE_FEW(PACKED, WK)                                                                                  \
  do {                                                                                                          \
    if (gated && out_dtype == 1) KVC_MOE_LAUNCH((moe_gemm_few_kernel<1, bf16_t, PACKED, WK>), bf16_t, bf16_t);   \
    else if (gated) KVC_MOE_LAUNCH((moe_gemm_few_kernel<1, float, PACKED, WK>), bf16_t, float);                 \
    else if (out_dtype == 1) KVC_MOE_LAUNCH((moe_gemm_few_kernel<0, bf16_t, PACKED, WK>), bf16_t, bf16_t);      \
    else KVC_MOE_LAUNCH((moe_gemm_few_kernel<0, float, PACKED, WK>), bf16_t, float);                            \
  } while (0)
      if (packed && whole) KVC_MOE_FEW(1, 1);
      else if (packed) KVC_MOE_FEW(1, 4);
      else if (whole) KVC_MOE_FEW(0, 1);
      else KVC_MOE_FEW(0, 4);
#undef KVC_MOE_FEW
    } else if (packed) {
      return kvc_fail("kvc_moe_gemm: a packed matrix has experts of a multiple of 16 rows of a multiple of 64");
    } else {
      if (gated && out_dtype == 1) KVC_MOE_LAUNCH((moe_gemm_plain_kernel<1, bf16_t, bf16_t>), bf16_t, bf16_t);
      else if (gated) KVC_MOE_LAUNCH((moe_gemm_plain_kernel<1, bf16_t, float>), bf16_t, float);
      else if (out_dtype == 1) KVC_MOE_LAUNCH((moe_gemm_plain_kernel<0, bf16_t, bf16_t>), bf16_t, bf16_t);
      else KVC_MOE_LAUNCH((moe_gemm_plain_kernel<0, bf16_t, float>), bf16_t, float);
    }
  } else if (dtype == 0) {
    if (out_dtype != 0) return kvc_fail("kvc_moe_gemm: float32 operands give float32 rows");
    if (tile_rows != kTileRows || packed) return kvc_fail("kvc_moe_gemm: float32 operands take tiles of 16 rows of a row-major matrix");
    if (gated) KVC_MOE_LAUNCH((moe_gemm_plain_kernel<1, float, float>), float, float);
    else KVC_MOE_LAUNCH((moe_gemm_plain_kernel<0, float, float>), float, float);
  } else {
    return kvc_fail("kvc_moe_gemm: unknown dtype code");
  }
#undef KVC_MOE_LAUNCH
#undef KVC_MOE_ARGS
  return kvc_check_launch("kvc_moe_gemm");
}

extern "C" int kvc_moe_combine(float* out, const float* y, const float* weight, int top, const void* add0,
                               int add0_dtype, const float* add1, const float* add1_gate, int T, int H,
                               int accumulate, kvc_stream stream) {
  if (T < 0 || H <= 0 || top < 0) return kvc_fail("kvc_moe_combine: bad sizes");
  if (T == 0) return 0;
  const int64_t n = static_cast<int64_t>(T) * H;
  const bool vec = H % 4 == 0 && ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(y) |
                                   reinterpret_cast<uintptr_t>(add1) | reinterpret_cast<uintptr_t>(add0)) & 15) == 0;
  const dim3 grid(static_cast<unsigned>((n / (vec ? 4 : 1) + 255) / 256));
#define KVC_COMBINE(TA, VEC)                                                                                \
  hipLaunchKernelGGL((moe_combine_kernel<TA, VEC>), grid, dim3(256), 0, S(stream), out, y, weight, top,     \
                     static_cast<const TA*>(add0), add1, add1_gate, T, H, accumulate)
  if (add0_dtype == 1) {
    if (vec) KVC_COMBINE(bf16_t, 4);
    else KVC_COMBINE(bf16_t, 1);
  } else {
    if (vec) KVC_COMBINE(float, 4);
    else KVC_COMBINE(float, 1);
  }
#undef KVC_COMBINE
  return kvc_check_launch("kvc_moe_combine");
}

extern "C" int kvc_moe_combine_norm(void* x, int x_dtype, float* residual, const float* y, const float* weight, int top,
                                    const float* add0, const float* add1, const float* add1_gate, const float* gain,
                                    float eps, int T, int H, kvc_stream stream) {
  if (T < 0 || H <= 0 || top < 0) return kvc_fail("kvc_moe_combine_norm: bad sizes");
  if (x_dtype != 0 && x_dtype != 1) return kvc_fail("kvc_moe_combine_norm: unknown dtype code");
  if (T == 0) return 0;
  const uintptr_t places = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(residual) |
                           reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(add0) |
                           reinterpret_cast<uintptr_t>(add1) | reinterpret_cast<uintptr_t>(gain);
  if (H % 8 || H > 8 * 2048 || (places & 15)) {  // no vectors, or more than a block's registers hold: one after the other
    const int bad = kvc_moe_combine(residual, y, weight, top, add0, 0, add1, add1_gate, T, H, 1, stream);
    return bad ? bad : kvc_add_rmsnorm(x, residual, nullptr, gain, eps, T, H, x_dtype, stream);
  }
  const int nch = (H + 2047) / 2048;
#define KVC_COMBINE_NORM(TO, NCH)                                                                              \
  hipLaunchKernelGGL((moe_combine_norm_kernel<TO, NCH>), dim3(T), dim3(256), 0, S(stream), static_cast<TO*>(x), \
                     residual, y, weight, top, add0, add1, add1_gate, gain, eps, H)
#define KVC_COMBINE_NORM_OF(TO)               \
  do {                                        \
    if (nch <= 1) KVC_COMBINE_NORM(TO, 1);      \
    else if (nch <= 2) KVC_COMBINE_NORM(TO, 2); \
    else if (nch <= 4) KVC_COMBINE_NORM(TO, 4); \
    else KVC_COMBINE_NORM(TO, 8);               \
  } while (0)
  if (x_dtype == 1) KVC_COMBINE_NORM_OF(bf16_t);
  else KVC_COMBINE_NORM_OF(float);
#undef KVC_COMBINE_NORM_OF
#undef KVC_COMBINE_NORM
  return kvc_check_launch("kvc_moe_combine_norm");
}
