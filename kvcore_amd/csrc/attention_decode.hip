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
// 118 MB at 4.8 TB/s.  A compute unit draws some 45 GB/s, so few blocks of many keys are the slower
// ones.  Every load is asked for as early as its address is known and waits for nothing else: the
// queries before the pages, units only where there are some, and barriers that do not wait for
// global memory.  Before (units of 16 keys, barriers that did, the merge's reads one by one) and now,
// in a graph: 8 tokens x 512 keys of 128 in four splits 14.2 -> 11.0 us, of 64 11.7 -> 9.6; one token, 512 keys of
// 64 in eight splits 10.5 -> 9.0; 64 tokens x 450 keys of 128 34.9 -> 27.9, of 64 21.8 -> 17.3; 4 tokens x 1,024 of
// 256 in eight splits 19.9 -> 15.8 (with loads marked as streaming ones, `read8`: 11.7, 9.7, 8.8, 29.7, 18.5 and 15.3 without).
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

#include "attention_combine.h"
#include "attention_decode_block.h"
#include "device_utils.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

using namespace kvc::decode;

constexpr size_t kLdsLimit = 64 * 1024;
constexpr int kMaxLdsPages = 1024;  // what the choice of waves per block leaves room for

template <int D, int DV, bool STREAM>
__global__ __launch_bounds__(max_waves<D>() * 64) void decode_attention_kernel(const DecodeArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int t = blockIdx.x;
  // which row of the block table: one load if the caller resolved it, else two in a chain
  int trow_idx;
  if (a.token_rows != nullptr) {
    trow_idx = a.token_rows[t];
  } else {
    const int req = a.token_req[t];
    trow_idx = req < 0 ? -1 : a.slots[req];
  }
  decode_block<D, DV, STREAM>(a, t, blockIdx.y, blockIdx.z, __builtin_amdgcn_readfirstlane(trow_idx), lds);
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
int launch_decode(DecodeArgs& args, int T, bool stream_keys, hipStream_t stream) {
  const int g = args.nh / args.nkv;
  // a split's range of pages always fits: the table's width cut into nsplit parts, and slack, as a split is whole
  // units of 32 keys (not more than two pages, also where a page is half a unit, as none behind the token's own counts)
  args.lds_pages = (args.table_stride + args.nsplit - 1) / args.nsplit + 2;
  if (args.lds_pages > args.table_stride) args.lds_pages = args.table_stride;
  int waves = decode_waves(g, D);
  // more blocks than compute units: smaller blocks pack better
  if (static_cast<int64_t>(T) * args.nkv * args.nsplit > kvc_device_compute_units() && waves > 4) waves = 4;
  while (waves > 1 && lds_total(waves, g, D, args.lds_pages) > kLdsLimit) waves /= 2;
  if (lds_total(waves, g, D, args.lds_pages) > kLdsLimit)
    return kvc_fail("kvc_decode_attention: the block table is wider than kvc_decode_attention_max_table "
                    "allows for one split");
  const dim3 grid(T, args.nkv, args.nsplit), block(waves * 64);
  const size_t lds = lds_total(waves, g, D, args.lds_pages);
  if (stream_keys) hipLaunchKernelGGL((decode_attention_kernel<D, DV, true>), grid, block, lds, stream, args);
  else hipLaunchKernelGGL((decode_attention_kernel<D, DV, false>), grid, block, lds, stream, args);
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
                                    int nsplit, int longest, int out_f32, kvc_stream stream) {
  if (!kvc_decode_attention_supported(nh, nkv, d, dv, page_size, 1))
    return kvc_fail("kvc_decode_attention: unsupported shape (bfloat16, head size a multiple of 32 "
                    "up to 256, values as wide or half as wide, at most 16 query heads per kv head, page size a multiple of 16)");
  if (T < 0 || nsplit < 1 || nsplit > kMaxSplits || longest < 0 || nkv > 65535 || table_stride <= 0 || num_pages <= 0)
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
  args.v_second = nullptr;
  args.table = table;
  args.table_stride = table_stride;
  args.page_magic = page_magic_of(page_size);
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
  // Streaming loads, but not where few blocks walk many keys each: they give a block some 10% fewer keys a second, which counts
  // where blocks do not fill the chip.  Steps of 16 layers with them and without, one token, 8 heads over 1 of 128 in 32
  // parts: 8,000 tokens 815 and 820 us, 32,000 972 and 938, 60,000 1,174 and 1,151, 120,000 1,576 and 1,480; 16 over 4 of
  // 128 / 64 32,000 1,391 and 1,448, 60,000 1,577 and 1,558, 120,000 1,948 and 1,847; 256 blocks of 4,096 keys 1,438 and 1,532.
  // (The kernel by itself, over and over on keys that the caches hold, is up to 12% faster without at any length.)
  const bool stream_keys = static_cast<int64_t>(T) * nkv * nsplit >= kvc_device_compute_units() || longest / nsplit < 2048;
  kvc_note_variant(kVariantDecodeAttention, !stream_keys ? "decode_attention_kernel, plain loads"
                                            : nsplit > 1 ? "decode_attention_kernel with splits" : "decode_attention_kernel");
#define KVC_DECODE(D_) \
  case D_: return dv == d ? launch_decode<D_, D_>(args, T, stream_keys, s) : launch_decode<D_, D_ / 2>(args, T, stream_keys, s)
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
