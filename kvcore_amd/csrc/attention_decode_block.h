// Attention of one token over its cached keys and values, bfloat16 on the matrix cores: the work of one block.  The kernel
// for single tokens (attention_decode.hip, which says how it works) is made of it, and the kernel for portions of prompts
// gives it the requests that bring one token.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "attention_combine.h"
#include "device_utils.h"
#include "gemm_common.h"

namespace kvc {
namespace decode {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kMaxWaves = 8;
constexpr int kUnit = 32;   // keys a wave takes at once
constexpr int kQPad = 8;    // bf16 elements between query rows in LDS beyond d
constexpr int kOPad = 16;   // floats between output rows in LDS beyond d

struct DecodeArgs {
  bf16_t* out;
  int out_f32;  // out receives float32 values (the sums as they are) instead of bfloat16
  float* part_o;
  float* part_ml;
  const bf16_t* qkv;  // rows [nh q heads of d | nkv k heads of d], nkv v heads of dv from v_begin on
  int64_t qkv_stride;
  bf16_t* k_cache;
  bf16_t* v_cache;
  const bf16_t* v_second;  // the other half of every value head, where it is twice as wide as a key head (not written)
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

// 16-key blocks to pages by a multiplication: exact as long as blocks times blocks a page stay below 2^32
inline unsigned page_magic_of(int page_size) {
  const unsigned blocks = page_size / 16;
  return blocks == 1 ? 0u : static_cast<unsigned>(((1ull << 32) + blocks - 1) / blocks);
}

__host__ __device__ inline size_t lds_q_bytes(int g, int d) {
  return (static_cast<size_t>(g) * (d + kQPad) * 2 + 15) / 16 * 16;
}
__host__ __device__ inline size_t lds_kv_bytes(int d) { return static_cast<size_t>(2) * d * 2; }
__host__ __device__ inline size_t lds_ml_bytes(int waves) { return static_cast<size_t>(waves) * 16 * 8; }
__host__ __device__ inline size_t lds_o_bytes(int waves, int g, int d) {
  return static_cast<size_t>(waves) * g * (d + kOPad) * 4;
}
inline size_t lds_total(int waves, int g, int d, int lds_pages) {
  return lds_q_bytes(g, d) + lds_kv_bytes(d) + lds_ml_bytes(waves) + lds_o_bytes(waves, g, d) +
         static_cast<size_t>(lds_pages) * 4;
}

// wide heads keep more registers per lane, so fewer waves fit in a block
template <int D>
constexpr int max_waves() { return D > 128 ? 4 : kMaxWaves; }

// Whether a wave has two units of keys and values on their way.  Two bring 1 to 2% of a launch of few blocks of 64 / 64 (one
// token of 100 keys 6.4 us, with one unit 6.5); their registers cost a place on the unit, or spill, wherever heads are wider and where
// values are half as wide: one, two and one again, 64 requests of 40 keys, 16 heads of 128 / 64 16.1, 14.8 and 10.1 us; 128 requests of 8 keys, 3
// of 224 / 112 9.1, 14.1 and 8.6, 16 of 96 20.0, 26.2 and 17.5, 12 of 64 / 32 9.9, 12.0 and 11.3 (units of 16 keys, of 32, and now).
template <int D, int DV>
constexpr bool two_units() { return D == 64 && DV >= 64; }

// A barrier for what the block's waves exchange through LDS alone: __syncthreads would also wait for every load and
// store in flight to global memory, here the first keys and values and the cache's new entries.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One block's work: token t (its row of the block table: trow_idx), kv head hk, one split of the keys; lds: lds_total()
// bytes of it, 16-byte aligned.  D: the size of a query and key head; DV: the size of a value head, at most D, or 2 D in two
// planes.  STREAM: keys and values come by loads marked as streaming ones (`read8`).  They bring more where blocks fill
// the chip, and take longer where a block walks many keys with few beside it (one token's 2,048 keys of 128, unsplit, 25 -> 32 us;
// kvc_decode_attention has the line).
template <int D, int DV, bool STREAM>
__device__ __forceinline__ void decode_block(const DecodeArgs& a, int t, int hk, int split, int trow_idx, unsigned char* lds) {
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
  constexpr int DVP = DV > D ? D : DV;  // a plane's share of a value head
  constexpr int NC = D / 32;  // 32-wide chunks of the head for Q.K

  bf16_t* sq = reinterpret_cast<bf16_t*>(lds);                       // [g][D + kQPad]
  bf16_t* sk = reinterpret_cast<bf16_t*>(lds + lds_q_bytes(g, D));   // [D] key, then [DV] value
  bf16_t* sv = sk + D;
  float* sml = reinterpret_cast<float*>(lds + lds_q_bytes(g, D) + lds_kv_bytes(D));  // [2][16][waves]: m, then l
  float* so = sml + 2 * 16 * waves;                              // [waves][g][DV + kOPad]
  int32_t* spage = reinterpret_cast<int32_t*>(so + static_cast<int64_t>(waves) * g * (DV + kOPad));  // [lds_pages]

  const int pos = __builtin_amdgcn_readfirstlane(a.positions[t]);
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
  // page that holds 16-key block b (exact: see page_magic_of)
  auto page_index = [&](int b) {
    return a.page_magic == 0 ? b : static_cast<int>(__umulhi(static_cast<unsigned>(b), a.page_magic));
  };
  const int blocks_per_page = page_size / 16;

  // the page ids of the range go to LDS, where the walk below reads them
  const int page_lo = page_index(2 * u0);
  // of a unit's second half only where the token sees it, so that no page behind the token's own has a place
  auto second_page = [&](int u) { return page_index(2 * u + 1 < blk_own ? 2 * u + 1 : blk_own) - page_lo; };
  const int n_range_pages = (u1 > u0) ? second_page(u1 - 1) + 1 : 0;
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
    // keys and values are read once (see read8); rows of wide heads are several loads' way from whole lines: 8 tokens x 1,024
    // keys of 128 14.4 -> 13.6 us marked (values alone 14.1), of 256 16.0 -> 16.6 (values alone 15.8)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < NC; ++c) un.k[h][c] = read8<(STREAM && D <= 128)>(krow + h * 4 * D + 32 * c);
  };
  auto issue_values = [&](Unit& un, int u) {
    int64_t base[2];
    int sub[2];
    half_of(u, 0, un.page[0], base[0], sub[0]);
    half_of(u, 1, un.page[1], base[1], sub[1]);
    const int64_t v0 = base[0] * DVP * page_size + sub[0], v1 = base[1] * DVP * page_size + sub[1];
    const int64_t at = (quad >= 2 ? v1 : v0) + (col * page_size + 8 * (quad & 1));
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      un.v[j] = read8<STREAM>((j < DVP / 16 ? a.v_cache : a.v_second) + at + j % (DVP / 16) * 16 * page_size);
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
                __builtin_amdgcn_readfirstlane(spage[second_page(u)]));
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

}  // namespace decode
}  // namespace kvc
