// Paged attention for single tokens (decode), bfloat16, on the matrix cores, with the
// rotation of the token's query and key and the write of its key and value into the cache
// done by the same kernel, where the layer has one behind a norm of every query and key head.
// Value heads are as wide as the keys or half as wide, or the key heads themselves as projected.
//
// One block of W waves per (token, kv head, split of the key range); the waves take the
// 32-key units of the range in turn.  The query heads that share the kv head are the
// columns of one 16-wide MFMA tile, so every key and value is fetched once for the whole
// group, straight from global memory:
//
//   S^T[2 x 16 keys, 16 heads] = K[2 x 16 keys, d]   * Q^T[d, 16 heads]      (16x16x32, two chains)
//   O^T[dv, 16 heads]         += V^T[dv, 32 keys]    * P^T[32 keys, 16 heads] (16x16x32)
//
// K pages are [page_size, d] (d contiguous) and V pages are [dv, page_size] (keys
// contiguous), which are exactly the A-operand layouts of the two products.  Which key is
// which row of the two score tiles is free, and chosen so that a lane's eight scores are
// of eight neighbouring keys: the accumulators are then the B operand of the second
// product, the probabilities never leave registers, and a lane takes 16 bytes of a row of V
// at once.  (With units of 16 keys it took 8, and a wave gave 24 loads for what are 16 now.)
// The probabilities go into the product as two bfloat16 parts.  Softmax state (max, sum) is
// float32, one per head, kept redundantly by the four lanes that hold a head's column.
// Against 64 bits the float32 results are off by 4.0e-6 to 4.8e-6 of their norm over 60 to 1,500
// keys of random numbers (6e-4 to 8e-4 with probabilities rounded to one bfloat16).
//
// What bounds it: at 8 tokens of 512 keys of 8 kv heads of 128 (16.8 MB) in four splits, 7.2 us
// from a block's start to its end are 0.9 until the token's row is known, 0.5 for its pages, 3.2 for
// the burst of keys and values of all blocks (a unit's loads are all in flight together), 0.6 for the
// rotation behind them, 0.5 for scores and values, 0.8 for the merge; 64 tokens of 450 keys read
// 118 MB at 4.4 TB/s.  A compute unit draws some 45 GB/s, so few blocks of many keys are the slower
// ones.  Every load is asked for as early as its address is known and waits for nothing else: the
// queries before the pages, units only where there are some, and barriers that do not wait for
// global memory.  Before (units of 16 keys, barriers that did, the merge's reads one by one) and now,
// in a graph: 8 tokens x 512 keys of 128 in four splits 14.2 -> 11.7 us, of 64 11.7 -> 9.7; one token, 512 keys of
// 64 in eight splits 10.5 -> 8.8; 64 tokens x 450 keys of 128 34.9 -> 29.7, of 64 21.8 -> 18.5; 4 tokens x 1,024 of
// 256 in eight splits 19.9 -> 15.3.
//
// The block first rotates the group's query heads into LDS.  The block whose range holds
// the token's own position also rotates the key, stores key and value in their cache slot
// and keeps both in LDS; the wave that meets the position's unit takes them from
// there, so nothing is read back from global memory in the kernel that wrote it.
//
// The waves' partial results (max, sum, output) are merged through LDS in wave order.
// With more than one split each block writes an unnormalised partial and a second kernel
// combines them; split boundaries depend on the request's length only.  (Letting the last
// block to finish do that combination needs a device-wide fence per block, which costs
// more than the second kernel.)

#include <hip/hip_runtime.h>

#include <type_traits>

#include "attention_combine.h"
#include "device_utils.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kMaxWaves = 8;
constexpr int kUnit = 32;   // keys a wave takes at once
constexpr int kQPad = 8;    // bf16 elements between query rows in LDS beyond d
constexpr int kOPad = 16;   // floats between output rows in LDS beyond d
constexpr size_t kLdsLimit = 64 * 1024;

struct DecodeArgs {
  bf16_t* out;
  int out_f32;  // out receives float32 values (the sums as they are) instead of bfloat16
  float* part_o;
  float* part_ml;
  const bf16_t* qkv;  // rows [nh q heads of d | nkv k heads of d], nkv v heads of dv from v_begin on
  int64_t qkv_stride;
  bf16_t* k_cache;
  bf16_t* v_cache;
  const int32_t* table;
  int table_stride;
  const int32_t* positions;
  const int32_t* token_req;
  const int32_t* slots;
  const int32_t* token_rows;  // [T] block-table row of each token (-1: padding), or null
  const float* cos_tab;  // [T, rot_dim / 2]
  const float* sin_tab;
  int rot_dim;
  int interleaved;
  const float* q_gain;  // [d] or null: every q head (and the k head, with k_gain) is first divided by
  const float* k_gain;  // its root mean square, norm_eps inside the root, and multiplied by the gain
  float norm_eps;
  int write_kv;  // store the token's key and value (and attend to them from LDS)
  int nh, nkv, page_size, num_pages;
  float scale_log2e;
  float cap_rate, cap_log2e;  // cap_rate > 0: a score is cap_log2e * capped_unit(raw score, cap_rate)
  int window;
  const float* slopes;  // [nh] or null: slope * (position - key position) comes off the score
  int chunk;            // > 0: only the keys of the token's own chunk of so many positions
  const float* sinks;   // [nh] or null: exp(sink) joins the softmax's denominator and brings no value along
  GateRows gate;        // sigmoid of these rows multiplies the result, element by element
  unsigned page_magic;  // 16-key blocks to pages: 0 where a page is a block, else ceil(2^32 / blocks a page)
  int v_begin;          // column of the first value head in a row of qkv
  int nsplit;
  int lds_pages;  // page ids of a block's range that fit in LDS
};

__host__ __device__ inline size_t lds_q_bytes(int g, int d) {
  return (static_cast<size_t>(g) * (d + kQPad) * 2 + 15) / 16 * 16;
}
__host__ __device__ inline size_t lds_kv_bytes(int d) { return static_cast<size_t>(2) * d * 2; }
__host__ __device__ inline size_t lds_ml_bytes(int waves) { return static_cast<size_t>(waves) * 16 * 8; }
__host__ __device__ inline size_t lds_o_bytes(int waves, int g, int d) {
  return static_cast<size_t>(waves) * g * (d + kOPad) * 4;
}
constexpr int kMaxLdsPages = 1024;  // what the choice of waves per block leaves room for
inline size_t lds_total(int waves, int g, int d, int lds_pages) {
  return lds_q_bytes(g, d) + lds_kv_bytes(d) + lds_ml_bytes(waves) + lds_o_bytes(waves, g, d) +
         static_cast<size_t>(lds_pages) * 4;
}

// wide heads keep more registers per lane, so fewer waves fit in a block
template <int D>
constexpr int max_waves() { return D > 128 ? 4 : kMaxWaves; }

// whether a wave's registers hold two units of keys and values beside queries and results
// (128 / 128 with two spills: 8 tokens of 512 keys 15.4 us unsplit, with one 13.4; 64 tokens of 1,024 keys 70 us and 57)
template <int D, int DV>
constexpr bool two_units() {
  return 2 * (D / 4 + DV / 4) + DV / 4 + D / 8 <= (max_waves<D>() == 4 ? 270 : 140);
}

// A barrier for what the block's waves exchange through LDS alone: __syncthreads would also wait for every load and
// store in flight to global memory, here the first keys and values and the cache's new entries.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// D: the size of a query and key head; DV: the size of a value head.
template <int D, int DV>
__global__ __launch_bounds__(max_waves<D>() * 64) void decode_attention_kernel(const DecodeArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int t = blockIdx.x;
  const int hk = blockIdx.y;
  const int split = blockIdx.z;
  const int tid = threadIdx.x;
  const int nthreads = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = nthreads >> 6;
  const int lane = tid & 63;
  const int col = lane & 15;   // head within the group (B/C column)
  const int quad = lane >> 4;  // 0..3
  const int nh = a.nh, nkv = a.nkv, nsplit = a.nsplit, page_size = a.page_size;
  const int g = nh / nkv;
  const bool head_live = col < g;
  constexpr int NJ = DV / 16;  // output row blocks
  constexpr int NC = D / 32;  // 32-wide chunks of the head for Q.K

  bf16_t* sq = reinterpret_cast<bf16_t*>(lds);                       // [g][D + kQPad]
  bf16_t* sk = reinterpret_cast<bf16_t*>(lds + lds_q_bytes(g, D));   // [D] key, then [DV] value
  bf16_t* sv = sk + D;
  float* sml = reinterpret_cast<float*>(lds + lds_q_bytes(g, D) + lds_kv_bytes(D));  // [2][16][waves]: m, then l
  float* so = sml + 2 * 16 * waves;                              // [waves][g][DV + kOPad]
  int32_t* spage = reinterpret_cast<int32_t*>(so + static_cast<int64_t>(waves) * g * (DV + kOPad));  // [lds_pages]

  // which row of the block table: one load if the caller resolved it, else two in a chain
  const int pos = __builtin_amdgcn_readfirstlane(a.positions[t]);
  int trow_idx;
  if (a.token_rows != nullptr) {
    trow_idx = a.token_rows[t];
  } else {
    const int req = a.token_req[t];
    trow_idx = req < 0 ? -1 : a.slots[req];
  }
  trow_idx = __builtin_amdgcn_readfirstlane(trow_idx);

  // A pair of elements of a head that turn together (beyond rot_dim: two neighbours).  The first pair of every
  // thread is asked for here, before the chain from the token to its pages.
  const bf16_t* trow = a.qkv + static_cast<int64_t>(t) * a.qkv_stride;
  const int rot_dim = a.rot_dim, half = rot_dim / 2;
  auto pair_of = [&](int idx, int& hh, int& e0, int& e1) {
    hh = idx / (D / 2);
    const int j = idx - hh * (D / 2);
    e0 = j < half && !a.interleaved ? j : j < half ? 2 * j : rot_dim + 2 * (j - half);
    e1 = j < half && !a.interleaved ? j + half : e0 + 1;
    return j;
  };
  auto head_row = [&](int hh) { return trow + static_cast<int64_t>(hh < g ? hk * g + hh : nh + hk) * D; };
  const float* cs = a.cos_tab + static_cast<int64_t>(t) * half;
  const float* sn = a.sin_tab + static_cast<int64_t>(t) * half;
  const int most_heads = a.write_kv ? g + 1 : g;  // the key is one more head to rotate
  float pre_x0 = 0.f, pre_x1 = 0.f, pre_c = 1.f, pre_s = 0.f;
  if (tid < most_heads * (D / 2)) {
    int hh, e0, e1;
    const int j = pair_of(tid, hh, e0, e1);
    const bf16_t* src = head_row(hh);
    pre_x0 = to_float(src[e0]);
    pre_x1 = to_float(src[e1]);
    if (j < half) {
      pre_c = cs[j];
      pre_s = sn[j];
    }
  }

  if (trow_idx < 0) {  // padding token
    if (nsplit == 1) {
      for (int idx = tid; idx < g * DV; idx += nthreads)
        store_result(a.out, (static_cast<int64_t>(t) * nh + hk * g) * DV + idx, 0.f, a.out_f32);
    } else if (tid < g) {
      float* ml = a.part_ml + ((static_cast<int64_t>(t) * nh + hk * g + tid) * nsplit + split) * 2;
      ml[0] = -INFINITY;
      ml[1] = 0.f;
    }
    return;
  }
  const int window = a.window;
  int first = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  if (a.chunk > 0 && (pos / a.chunk) * a.chunk > first) first = (pos / a.chunk) * a.chunk;
  const int32_t* row = a.table + static_cast<int64_t>(trow_idx) * a.table_stride;

  // the units of 32 keys this block owns: [u0, u1) of the range that holds keys first..pos
  const int unit_first = first / kUnit;
  const int unit_end = pos / kUnit + 1;
  const int per = (unit_end - unit_first + nsplit - 1) / nsplit;
  const int u0 = unit_first + split * per;
  const int u1 = (u0 + per < unit_end) ? u0 + per : unit_end;
  const int unit_own = unit_end - 1;  // the unit of the token's own key
  const int blk_own = pos / 16;
  const bool owner = a.write_kv && u0 <= unit_own && unit_own < u1;
  // page that holds 16-key block b; the host keeps b below 2^27 and the division exact
  auto page_index = [&](int b) {
    return a.page_magic == 0 ? b : static_cast<int>(__umulhi(static_cast<unsigned>(b), a.page_magic));
  };
  const int blocks_per_page = page_size / 16;

  // the page ids of the range go to LDS, where the walk below reads them
  const int page_lo = page_index(2 * u0);
  const int n_range_pages = (u1 > u0) ? page_index(2 * u1 - 1) - page_lo + 1 : 0;
  for (int i = tid; i < n_range_pages && i < a.lds_pages; i += nthreads)
    spage[i] = (page_lo + i < a.table_stride) ? row[page_lo + i] : 0;

  // A unit of 32 keys.  Row 4q + i of the first product's tile of keys is key 8q + i of the unit, of its second tile key
  // 8q + 4 + i: a lane's eight scores (quad q) are then of keys 8q .. 8q + 7, in the order in which 16 bytes of a row of
  // V^T hold their values.  K rows as A operands: elements 32c + 8 * quad .. +8 of the lane's two keys, both in the same
  // half of the unit; V^T rows: element 16j + col, keys 8 * quad .. +8.  A half whose page is not there (behind the
  // window, or past the token) reads the null page and its keys are masked.
  struct Unit {
    bf16x8_t k[2][NC];
    bf16x8_t v[NJ];
    int page[2];
  };
  const int key_row = 8 * ((col >> 2) & 1) + (col & 3);  // within a half of 16 keys; the second tile: + 4
  // scalar: where a half's page begins for this kv head (in keys), and the first of its keys there
  auto half_of = [&](int u, int h, int page, int64_t& base, int& sub) {
    const int b = 2 * u + h;
    const bool real = page > 0;
    base = real ? static_cast<int64_t>(page) * nkv + hk : 0;
    sub = real ? (b - page_index(b) * blocks_per_page) * 16 : 0;
  };
  auto set_pages = [&](Unit& un, int u, int page0, int page1) {  // 0: not there
    un.page[0] = page0 > 0 && page0 < a.num_pages ? page0 : 0;
    un.page[1] = 2 * u + 1 <= blk_own && page1 > 0 && page1 < a.num_pages ? page1 : 0;
  };
  auto issue_keys = [&](Unit& un, int u) {
    int64_t base[2];
    int sub[2];
    half_of(u, 0, un.page[0], base[0], sub[0]);
    half_of(u, 1, un.page[1], base[1], sub[1]);
    const int64_t k0 = (base[0] * page_size + sub[0]) * D, k1 = (base[1] * page_size + sub[1]) * D;
    const bf16_t* krow = a.k_cache + (col >= 8 ? k1 : k0) + (key_row * D + 8 * quad);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < NC; ++c) un.k[h][c] = *reinterpret_cast<const bf16x8_t*>(krow + h * 4 * D + 32 * c);
  };
  auto issue_values = [&](Unit& un, int u) {
    int64_t base[2];
    int sub[2];
    half_of(u, 0, un.page[0], base[0], sub[0]);
    half_of(u, 1, un.page[1], base[1], sub[1]);
    const int64_t v0 = base[0] * DV * page_size + sub[0], v1 = base[1] * DV * page_size + sub[1];
    const bf16_t* vrow = a.v_cache + (quad >= 2 ? v1 : v0) + (col * page_size + 8 * (quad & 1));
#pragma unroll
    for (int j = 0; j < NJ; ++j) un.v[j] = *reinterpret_cast<const bf16x8_t*>(vrow + j * 16 * page_size);
  };

  // the first unit of this wave is asked for at once, before anything else waits
  const int u_wave = u0 + wave;
  const bool has_work = u_wave < u1;
  Unit ua;
  if (has_work) {
    const int i0 = page_index(2 * u_wave), i1 = page_index(2 * u_wave + 1);
    const int p0 = __builtin_amdgcn_readfirstlane(i0 < a.table_stride ? row[i0] : 0);
    const int p1 = __builtin_amdgcn_readfirstlane(i1 < a.table_stride ? row[i1] : 0);
    set_pages(ua, u_wave, p0, p1);
    issue_keys(ua, u_wave);
    issue_values(ua, u_wave);
  }

  // ---- norm and rotation of the group's queries (and the key) into LDS; key and value into the cache
  {
    int64_t k_off = -1, v_off = -1;
    if (owner) {
      const int page = (page_index(blk_own) < a.table_stride) ? row[page_index(blk_own)] : 0;
      if (page > 0 && page < a.num_pages) {
        const int off = pos - page_index(blk_own) * page_size;
        k_off = ((static_cast<int64_t>(page) * nkv + hk) * page_size + off) * D;
        v_off = (static_cast<int64_t>(page) * nkv + hk) * DV * page_size + off;
      }
    }
    const int n_heads = owner ? g + 1 : g;
    if (a.q_gain != nullptr) {  // a wave a head: its scale factor, into what will hold the waves' sums
      for (int hh = wave; hh < n_heads; hh += waves) {
        const bf16_t* src = head_row(hh);
        float ss = 0.f;
        for (int e = lane; e < D; e += 64) {
          const float x = to_float(src[e]);
          ss = fmaf(x, x, ss);
        }
        ss = wave_sum(ss);
        if (lane == 0) sml[hh] = 1.f / sqrtf(ss / static_cast<float>(D) + a.norm_eps);
      }
      lds_barrier();
    }
    for (int idx = tid; idx < n_heads * (D / 2); idx += nthreads) {
      int hh, e0, e1;
      const int j = pair_of(idx, hh, e0, e1);
      float x0 = pre_x0, x1 = pre_x1, c = pre_c, s_ = pre_s;
      if (idx != tid) {
        const bf16_t* src = head_row(hh);
        x0 = to_float(src[e0]);
        x1 = to_float(src[e1]);
        if (j < half) {
          c = cs[j];
          s_ = sn[j];
        }
      }
      const float* gain = (hh < g) ? a.q_gain : a.k_gain;
      if (gain != nullptr) {
        const float norm = sml[hh];
        x0 = x0 * norm * gain[e0];
        x1 = x1 * norm * gain[e1];
      }
      bf16_t y0, y1;
      if (j < half) {
        y0 = from_float<bf16_t>(rotate_first(x0, x1, c, s_));
        y1 = from_float<bf16_t>(rotate_second(x0, x1, c, s_));
      } else {  // as they are (bfloat16 values come out unchanged) or normalised
        y0 = from_float<bf16_t>(x0);
        y1 = from_float<bf16_t>(x1);
      }
      if (hh < g) {
        sq[hh * (D + kQPad) + e0] = y0;
        sq[hh * (D + kQPad) + e1] = y1;
      } else {
        sk[e0] = y0;
        sk[e1] = y1;
        if (k_off >= 0) {
          a.k_cache[k_off + e0] = y0;
          a.k_cache[k_off + e1] = y1;
        }
      }
    }
    if (owner) {
      const bf16_t* vsrc = trow + a.v_begin + static_cast<int64_t>(hk) * DV;
      for (int e = tid; e < DV; e += nthreads) {
        const bf16_t v = vsrc[e];
        sv[e] = v;
        if (v_off >= 0) a.v_cache[v_off + static_cast<int64_t>(e) * page_size] = v;
      }
    }
  }
  lds_barrier();

  // Q^T as B operand: lane holds head `col`, elements 32c + 8*quad .. +8
  bf16x8_t bq[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (head_live) {
      bq[c] = *reinterpret_cast<const bf16x8_t*>(sq + col * (D + kQPad) + 32 * c + 8 * quad);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) bq[c][e] = static_cast<__bf16>(0.f);
    }
  }

  const float slope_l2e = (a.slopes != nullptr && head_live) ? a.slopes[hk * g + col] * kLog2e : 0.f;
  f32x4_t o[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) o[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  f32x4_t s[2];  // s[h][i] belongs to key 32u + 8*quad + 4h + i and head `col`
  auto scores = [&](int u, Unit& un) {
    if (owner && u == unit_own) {
      // the token's own key comes from LDS, not from the cache line just written
      const int kk = pos & (kUnit - 1);
      const bool mine = (col >> 2) == (kk >> 3) && (col & 3) == (kk & 3);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (mine && ((kk >> 2) & 1) == h) {
#pragma unroll
          for (int c = 0; c < NC; ++c) un.k[h][c] = *reinterpret_cast<const bf16x8_t*>(sk + 32 * c + 8 * quad);
        }
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) s[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) s[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(un.k[h][c], bq[c], s[h], 0, 0, 0);
  };
  auto join_values = [&](int u, Unit& un, int page0, int page1) {
    const int key0 = kUnit * u + 8 * quad;
    const bool half_real = quad >= 2 ? page1 > 0 : page0 > 0;
    float p[8];
    bool ok[8];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = key0 + i;
      const float raw = s[i >> 2][i & 3];
      ok[i] = half_real && key >= first && key <= pos;
      const float score = a.cap_rate > 0.f ? a.cap_log2e * capped_unit(raw, a.cap_rate)  // scalar
                                           : __builtin_fmaf(raw, a.scale_log2e, -slope_l2e * static_cast<float>(pos - key));
      p[i] = ok[i] ? score : -INFINITY;
      mx = fmaxf(mx, p[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
    float ps = 0.f;
    // P^T as B operand: k = key 8*quad + i, column = head.  In two parts whose sum holds 16 bits of p and more, both
    // above zero where p is (the upper one is cut, a little below p), so that infinite values stay what they are.
    bf16x8_t pb, pl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = __builtin_amdgcn_exp2f(p[i] - m_safe);  // exp2(-inf) = 0 for masked keys
      ps += p[i];
      const uint32_t upper = __float_as_uint(p[i] * 0.998046875f) & 0xffff0000u;  // 1 - 2^-9
      pb[i] = __builtin_bit_cast(__bf16, static_cast<uint16_t>(upper >> 16));
      pl[i] = static_cast<__bf16>(p[i] - __uint_as_float(upper));
    }
    ps += __shfl_xor(ps, 16, 64);
    ps += __shfl_xor(ps, 32, 64);
    l = l * alpha + ps;
    m = m_new;

    if (owner && u == unit_own) {  // the token's own value, as its key
      const int kk = pos & (kUnit - 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if ((kk & 7) == i && quad == (kk >> 3)) {
#pragma unroll
          for (int j = 0; j < NJ; ++j) un.v[j][i] = __builtin_bit_cast(__bf16, sv[16 * j + col].bits);
        }
      }
    }
    // values of masked keys may be anything (a reused page, NaN): they must not meet the
    // product even with weight zero
    const bool edge = (kUnit * u + kUnit - 1 > pos) || (kUnit * u < first) || page0 == 0 || page1 == 0;
    if (edge) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) un.v[j][i] = ok[i] ? un.v[j][i] : static_cast<__bf16>(0.f);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      o[j] = o[j] * alpha;
      o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(un.v[j], pl, o[j], 0, 0, 0);
      o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(un.v[j], pb, o[j], 0, 0, 0);
    }
  };

  // The wave's units u_wave, u_wave + waves, ...: while one is worked on, the next loads.  A unit is asked for only
  // where there is one, and every path counts its own loads, so no wait is for more than it needs.  Where two units do
  // not fit the registers the next unit's keys take the place of the scored ones and its values that of the joined ones.
  if (has_work) {
    auto next_pages = [&](Unit& un, int u) {
      set_pages(un, u, __builtin_amdgcn_readfirstlane(spage[page_index(2 * u) - page_lo]),
                __builtin_amdgcn_readfirstlane(spage[page_index(2 * u + 1) - page_lo]));
    };
    int u = u_wave;
    if constexpr (two_units<D, DV>()) {
      Unit ub;
      auto work = [&](int w, Unit& un) {
        scores(w, un);
        join_values(w, un, un.page[0], un.page[1]);
      };
      auto issue = [&](int w, Unit& un) {
        next_pages(un, w);
        issue_keys(un, w);
        issue_values(un, w);
      };
      for (;; u += 2 * waves) {
        if (u + waves >= u1) {
          work(u, ua);
          break;
        }
        issue(u + waves, ub);
        work(u, ua);
        if (u + 2 * waves >= u1) {
          work(u + waves, ub);
          break;
        }
        issue(u + 2 * waves, ua);
        work(u + waves, ub);
      }
    } else {
      for (; u + waves < u1; u += waves) {
        const int page0 = ua.page[0], page1 = ua.page[1];
        scores(u, ua);
        next_pages(ua, u + waves);
        issue_keys(ua, u + waves);
        join_values(u, ua, page0, page1);
        issue_values(ua, u + waves);
      }
      scores(u, ua);
      join_values(u, ua, ua.page[0], ua.page[1]);
    }
  }

  // ---- merge the waves' partials in wave order
  // o[j][i] = O^T[element 16j + 4*quad + i, head col]
  if (head_live) {
    float* wo = so + (static_cast<int64_t>(wave) * g + col) * (DV + kOPad) + 4 * quad;
#pragma unroll
    for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4_t*>(wo + 16 * j) = o[j];
    if (quad == 0) {
      sml[col * waves + wave] = m;
      sml[(16 + col) * waves + wave] = l;
    }
  }
  lds_barrier();
  auto merge = [&](auto count) {  // the count of waves is a constant: all reads are asked for at once
    constexpr int W = decltype(count)::value;
    for (int idx = tid; idx < g * DV; idx += nthreads) {
      const int h = idx / DV;
      const int e = idx - h * DV;
      const int64_t th = static_cast<int64_t>(t) * nh + hk * g + h;
      const float raw_gate = a.gate.gate != nullptr && nsplit == 1  // scalar
                                 ? to_float(a.gate.gate[t * a.gate.stride + static_cast<int64_t>(hk * g) * DV + idx])
                                 : 0.f;
      // the sink counts once for a row: the first split takes it, as one more partial sum without values
      const float sink_l2e = (a.sinks != nullptr && split == 0) ? a.sinks[hk * g + h] * kLog2e : -INFINITY;
      float wm[W], wl[W], wo[W];
#pragma unroll
      for (int w = 0; w < W; ++w) {
        wm[w] = sml[h * W + w];
        wl[w] = sml[(16 + h) * W + w];
        wo[w] = so[(static_cast<int64_t>(w) * g + h) * (DV + kOPad) + e];
      }
      float mmax = sink_l2e;
#pragma unroll
      for (int w = 0; w < W; ++w) mmax = fmaxf(mmax, wm[w]);
      const float m_safe = (mmax == -INFINITY) ? 0.f : mmax;
      float denom = __builtin_amdgcn_exp2f(sink_l2e - m_safe), acc = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float wgt = __builtin_amdgcn_exp2f(wm[w] - m_safe);
        denom = wgt > 0.f ? denom + wgt * wl[w] : denom;
        acc = wgt > 0.f ? acc + wgt * wo[w] : acc;
      }
      if (nsplit == 1) {
        const float gain = a.gate.gate != nullptr ? sigmoid_of(raw_gate) : 1.f;
        store_result(a.out, th * DV + e, denom > 0.f ? acc / denom * gain : 0.f, a.out_f32);
      } else {
        a.part_o[(th * nsplit + split) * DV + e] = acc;
        if (e == 0) {
          a.part_ml[(th * nsplit + split) * 2] = mmax;
          a.part_ml[(th * nsplit + split) * 2 + 1] = denom;
        }
      }
    }
  };
  if (waves == 8) merge(std::integral_constant<int, 8>{});
  else if (waves == 4) merge(std::integral_constant<int, 4>{});
  else if (waves == 2) merge(std::integral_constant<int, 2>{});
  else merge(std::integral_constant<int, 1>{});
}

// out[t, head, :] = sum_s w_s * part_o[s] / sum_s w_s * l_s with w_s = exp2(m_s - max m).
// Every wave works the weights out for itself (lane s holds split s), so nothing waits on
// another wave; the partial outputs are asked for before the weights are known.
constexpr int kMaxSplits = kMaxAttentionSplits;
__global__ void decode_combine_kernel(bf16_t* __restrict__ out, const float* __restrict__ part_o,
                                      const float* __restrict__ part_ml, int D, int nsplit, int out_f32,
                                      GateRows gate) {
  const int64_t th = blockIdx.x;  // token * nh + head
  const int lane = threadIdx.x & 63;
  const float* ml = part_ml + th * nsplit * 2;
  const float* po = part_o + th * nsplit * D;
  float m_s = -INFINITY, l_s = 0.f;
  if (lane < nsplit) {
    m_s = ml[2 * lane];
    l_s = ml[2 * lane + 1];
  }
  for (int e0 = 0; e0 < D; e0 += blockDim.x) {
    const int e = e0 + threadIdx.x;
    const bool live = e < D;
    float acc = 0.f;
    float raw_gate = 0.f;
    if (gate.gate != nullptr && live) {  // asked for before the sums are known
      const int64_t t = th / gate.nh;
      raw_gate = to_float(gate.gate[t * gate.stride + (th - t * gate.nh) * D + e]);
    }
    float mmax = wave_max(m_s);
    const float m_safe = (mmax == -INFINITY) ? 0.f : mmax;
    const float w_lane = __builtin_amdgcn_exp2f(m_s - m_safe);  // 0 for lanes beyond nsplit
    const float denom = wave_sum(w_lane * l_s);
    for (int s0 = 0; s0 < nsplit; s0 += 4) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = (live && s0 + i < nsplit) ? po[static_cast<int64_t>(s0 + i) * D + e] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w = __shfl(w_lane, (s0 + i) & 63, 64);
        if (s0 + i < nsplit && w > 0.f) acc += w * v[i];
      }
    }
    const float gain = gate.gate != nullptr ? sigmoid_of(raw_gate) : 1.f;
    if (live) store_result(out, th * D + e, denom > 0.f ? acc / denom * gain : 0.f, out_f32);
  }
}

int decode_waves(int g, int d) {
  int waves = d > 128 ? 4 : kMaxWaves;
  while (waves > 1 && lds_total(waves, g, d, kMaxLdsPages) > kLdsLimit) waves /= 2;
  return waves;
}

template <int D, int DV>
int launch_decode(DecodeArgs& args, int T, hipStream_t stream) {
  const int g = args.nh / args.nkv;
  // a split's range of pages always fits: the table's width cut into nsplit parts, and slack, as a split is whole
  // units of two blocks; all of them may end one page behind the table
  args.lds_pages = (args.table_stride + args.nsplit - 1) / args.nsplit + 4;
  if (args.lds_pages > args.table_stride + 1) args.lds_pages = args.table_stride + 1;
  int waves = decode_waves(g, D);
  // more blocks than compute units: smaller blocks pack better
  if (static_cast<int64_t>(T) * args.nkv * args.nsplit > kvc_device_compute_units() && waves > 4) waves = 4;
  while (waves > 1 && lds_total(waves, g, D, args.lds_pages) > kLdsLimit) waves /= 2;
  if (lds_total(waves, g, D, args.lds_pages) > kLdsLimit)
    return kvc_fail("kvc_decode_attention: the block table is wider than kvc_decode_attention_max_table "
                    "allows for one split");
  hipLaunchKernelGGL((decode_attention_kernel<D, DV>), dim3(T, args.nkv, args.nsplit), dim3(waves * 64),
                     lds_total(waves, g, D, args.lds_pages), stream, args);
  if (args.nsplit > 1)
    hipLaunchKernelGGL(decode_combine_kernel, dim3(T * args.nh), dim3((DV + 63) / 64 * 64), 0, stream,
                       args.out, args.part_o, args.part_ml, DV, args.nsplit, args.out_f32, args.gate);
  return kvc_check_launch("kvc_decode_attention");
}

}  // namespace

int kvc::launch_attention_combine(bf16_t* out, const float* part_o, const float* part_ml, int64_t rows,
                                  int d, int nsplit, int out_f32, const GateRows& gate, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (rows > 0x7fffffff || nsplit < 1 || nsplit > kMaxAttentionSplits)
    return kvc_fail("attention combine: bad sizes");
  hipLaunchKernelGGL(decode_combine_kernel, dim3(static_cast<unsigned>(rows)), dim3((d + 63) / 64 * 64), 0,
                     stream, out, part_o, part_ml, d, nsplit, out_f32, gate);
  return kvc_check_launch("attention combine");
}

extern "C" int kvc_decode_attention_supported(int nh, int nkv, int d, int dv, int page_size, int dtype) {
  if (dtype != 1) return 0;
  if (dv != d && 2 * dv != d) return 0;
  if (nkv <= 0 || nh % nkv || nh / nkv > 16) return 0;
  if (page_size % 16) return 0;
  return d == 32 || d == 64 || d == 96 || d == 128 || d == 160 || d == 192 || d == 224 || d == 256;
}

extern "C" int kvc_decode_attention_max_table(int nh, int nkv, int d) {
  if (nkv <= 0 || nh % nkv || d <= 0) return 0;
  const size_t fixed = lds_total(1, nh / nkv, d, 0);
  if (fixed >= kLdsLimit) return 0;
  // launch_decode keeps two entries of slack beyond a split's share of the table
  return static_cast<int>((kLdsLimit - fixed) / 4) - 2;
}

extern "C" int kvc_decode_attention_waves(int nh, int nkv, int d) {
  if (nkv <= 0 || nh % nkv || d <= 0) return 0;
  return decode_waves(nh / nkv, d);
}

extern "C" int kvc_decode_attention(void* out, void* part_o, void* part_ml, const void* qkv,
                                    int64_t qkv_stride, void* k_cache, void* v_cache,
                                    const int32_t* table, int table_stride,
                                    const int32_t* positions, const int32_t* token_req,
                                    const int32_t* slots, const int32_t* token_rows,
                                    const float* cos_tab, const float* sin_tab, int rot_dim, int interleaved,
                                    const float* q_gain, const float* k_gain, float norm_eps, int write_kv, int T, int nh,
                                    int nkv, int d, int dv, int page_size, int num_pages, float scale,
                                    int window, const float* slopes, int chunk, const float* sinks, float softcap,
                                    const void* gate, int64_t gate_stride, int values_are_keys,
                                    int nsplit, int out_f32, kvc_stream stream) {
  if (!kvc_decode_attention_supported(nh, nkv, d, dv, page_size, 1))
    return kvc_fail("kvc_decode_attention: unsupported shape (bfloat16, head size a multiple of 32 "
                    "up to 256, values as wide or half as wide, at most 16 query heads per kv head, page size a multiple of 16)");
  if (T < 0 || nsplit < 1 || nsplit > kMaxSplits || nkv > 65535 || table_stride <= 0 || num_pages <= 0)
    return kvc_fail("kvc_decode_attention: bad sizes (at most 64 splits)");
  if (values_are_keys && dv != d) return kvc_fail("kvc_decode_attention: values that are the keys have the keys' size");
  if (softcap < 0.f || (softcap > 0.f && slopes != nullptr))
    return kvc_fail("kvc_decode_attention: a soft cap is positive and does not go with distance slopes");
  if (gate != nullptr && gate_stride < static_cast<int64_t>(nh) * dv)
    return kvc_fail("kvc_decode_attention: gate rows too short");
  if (qkv_stride % 8 || qkv_stride < static_cast<int64_t>(nh) * d + (write_kv ? static_cast<int64_t>(nkv) * (values_are_keys ? d : d + dv) : 0))
    return kvc_fail("kvc_decode_attention: token rows must be 16-byte aligned and hold q (and k, v)");
  if (rot_dim < 0 || rot_dim > d || rot_dim % 2)
    return kvc_fail("kvc_decode_attention: the rotated width must be even and at most the head size");
  if (rot_dim > 0 && (cos_tab == nullptr || sin_tab == nullptr))
    return kvc_fail("kvc_decode_attention: rotation needs its cos and sin tables");
  if (nsplit > 1 && (part_o == nullptr || part_ml == nullptr))
    return kvc_fail("kvc_decode_attention: splits need a workspace");
  if ((k_gain != nullptr && q_gain == nullptr) || (q_gain != nullptr && k_gain == nullptr && write_kv))
    return kvc_fail("kvc_decode_attention: a norm of the heads has gains for the queries and for the keys it writes");
  if (T == 0) return 0;
  DecodeArgs args;
  args.out = static_cast<bf16_t*>(out);
  args.out_f32 = out_f32;
  args.part_o = static_cast<float*>(part_o);
  args.part_ml = static_cast<float*>(part_ml);
  args.qkv = static_cast<const bf16_t*>(qkv);
  args.qkv_stride = qkv_stride;
  args.k_cache = static_cast<bf16_t*>(k_cache);
  args.v_cache = static_cast<bf16_t*>(v_cache);
  args.table = table;
  args.table_stride = table_stride;
  const unsigned blocks = page_size / 16;
  args.page_magic = blocks == 1 ? 0u : static_cast<unsigned>(((1ull << 32) + blocks - 1) / blocks);
  args.positions = positions;
  args.token_req = token_req;
  args.slots = slots;
  args.token_rows = token_rows;
  args.cos_tab = cos_tab;
  args.sin_tab = sin_tab;
  args.rot_dim = rot_dim;
  args.interleaved = interleaved;
  args.q_gain = q_gain;
  args.k_gain = k_gain;
  args.norm_eps = norm_eps;
  args.write_kv = write_kv;
  args.nh = nh;
  args.nkv = nkv;
  args.page_size = page_size;
  args.num_pages = num_pages;
  args.scale_log2e = scale * kLog2e;
  args.cap_rate = softcap > 0.f ? 2.f * kLog2e * scale / softcap : 0.f;
  args.cap_log2e = softcap * kLog2e;
  args.gate = GateRows{static_cast<const bf16_t*>(gate), gate_stride, nh};
  args.v_begin = values_are_keys ? nh * d : (nh + nkv) * d;
  args.window = window;
  args.slopes = slopes;
  args.chunk = chunk;
  args.sinks = sinks;
  args.nsplit = nsplit;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  kvc_note_variant(kVariantDecodeAttention, nsplit > 1 ? "decode_attention_kernel with splits" : "decode_attention_kernel");
#define KVC_DECODE(D_) \
  case D_: return dv == d ? launch_decode<D_, D_>(args, T, s) : launch_decode<D_, D_ / 2>(args, T, s)
  switch (d) {
    KVC_DECODE(32);
    KVC_DECODE(64);
    KVC_DECODE(96);
    KVC_DECODE(128);
    KVC_DECODE(160);
    KVC_DECODE(192);
    KVC_DECODE(224);
    KVC_DECODE(256);
  }
#undef KVC_DECODE
  return kvc_fail("kvc_decode_attention: unsupported head size");
}
