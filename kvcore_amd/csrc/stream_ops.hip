// Kernels on rows of the residual stream that are not an RMS norm: layer norm with the
// residual sum, the mean of several branches that are each divided by their root mean
// square, two float32 row sets side by side as one operand of a product, a vector added to
// every row.  All arithmetic is float32; storage is float32 or bfloat16.

#include <hip/hip_runtime.h>

#include "device_utils.h"
#include "kvcore_hip.h"

using namespace kvc;

namespace {

inline hipStream_t S(kvc_stream s) { return reinterpret_cast<hipStream_t>(s); }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// One block per row.  residual += delta; mean; mean of the squared deviations; then
// (x - mean) / sqrt(var + eps) * weight + bias.  Three passes over a row that stays in cache.
template <typename T>
__global__ __launch_bounds__(256) void add_layernorm_kernel(T* __restrict__ out,
                                                            float* __restrict__ residual,
                                                            const T* __restrict__ delta,
                                                            const float* __restrict__ weight,
                                                            const float* __restrict__ bias,
                                                            float eps, int H) {
  __shared__ float scratch[16];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * H;
  float* r = residual + base;
  float sum = 0.f;
  if (delta != nullptr) {
    const T* dl = delta + base;
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
      const float v = r[i] + to_float(dl[i]);
      r[i] = v;
      sum += v;
    }
  } else {
    for (int i = threadIdx.x; i < H; i += blockDim.x) sum += r[i];
  }
  const float mean = block_sum(sum, scratch) / static_cast<float>(H);
  float ss = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float dv = r[i] - mean;
    ss = fmaf(dv, dv, ss);
  }
  const float var = block_sum(ss, scratch) / static_cast<float>(H);
  const float inv = 1.f / sqrtf(var + eps);
  T* o = out + base;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float b = bias != nullptr ? bias[i] : 0.f;
    o[i] = from_float<T>(fmaf((r[i] - mean) * inv, weight[i], b));
  }
}

// The same for rows of up to 256 * NV values, which a thread keeps in registers: residual and
// delta are read once and everything else is arithmetic and two block sums.
template <typename T, int NV>
__global__ __launch_bounds__(256) void add_layernorm_regs_kernel(T* __restrict__ out,
                                                                 float* __restrict__ residual,
                                                                 const T* __restrict__ delta,
                                                                 const float* __restrict__ weight,
                                                                 const float* __restrict__ bias,
                                                                 float eps, int H) {
  __shared__ float scratch[16];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * H;
  float* r = residual + base;
  float v[NV], w[NV], sh[NV];  // gain and shift come with the row: one trip to memory in all
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * 256;
    v[i] = w[i] = sh[i] = 0.f;
    if (c < H) {
      v[i] = r[c];
      w[i] = weight[c];
      if (bias != nullptr) sh[i] = bias[c];
      if (delta != nullptr) {
        v[i] += to_float(delta[base + c]);
        r[c] = v[i];
      }
      sum += v[i];
    }
  }
  const float mean = block_sum(sum, scratch) / static_cast<float>(H);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < H) {
      v[i] -= mean;
      ss = fmaf(v[i], v[i], ss);
    }
  }
  const float inv = 1.f / sqrtf(block_sum(ss, scratch) / static_cast<float>(H) + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < H) out[base + c] = from_float<T>(fmaf(v[i] * inv, w[i], sh[i]));
  }
}

__device__ __forceinline__ void load4(const float* p, float* v) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void store4(float* p, const float* v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}

// The same for rows of a multiple of 8 values up to 2048 * NCH, 16-byte aligned: a thread takes eight neighbouring values, or,
// of float32, two fours 1,024 apart, so that every load of a wave is a kilobyte in one piece.
// Bound by its bytes: 2,048 rows of 2,048, bfloat16 (50 MB), value by value 13.4 us, 12.1 this way; float32 (67 MB) 10.6, 12.1 with
// eight neighbours and 9.9 so.
template <typename T, int NCH>
__global__ __launch_bounds__(256) void add_layernorm_vec_kernel(T* __restrict__ out, float* __restrict__ residual,
                                                                const T* __restrict__ delta, const float* __restrict__ weight,
                                                                const float* __restrict__ bias, float eps, int H) {
  __shared__ float scratch[16];
  constexpr bool kFours = sizeof(T) == 4;
  constexpr int kParts = kFours ? 2 * NCH : NCH, kWide = kFours ? 4 : 8;  // pieces of a thread, and values in each
  const int64_t base = static_cast<int64_t>(blockIdx.x) * H;
  auto load = [](const auto* p, float* v) {
    if constexpr (kFours) load4(p, v);
    else load8(p, v);
  };
  auto store = [](auto* p, const float* v) {
    if constexpr (kFours) store4(p, v);
    else store8(p, v);
  };
  float v[kParts][kWide], w[kParts][kWide], sh[kParts][kWide];  // gain and shift come with the row: one trip to memory in all
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < kParts; ++c) {
    const int e = (c * 256 + threadIdx.x) * kWide;
#pragma unroll
    for (int i = 0; i < kWide; ++i) v[c][i] = w[c][i] = sh[c][i] = 0.f;
    if (e < H) {
      load(residual + base + e, v[c]);
      load(weight + e, w[c]);
      if (bias != nullptr) load(bias + e, sh[c]);
      if (delta != nullptr) {
        float d[kWide];
        load(delta + base + e, d);
#pragma unroll
        for (int i = 0; i < kWide; ++i) v[c][i] += d[i];
        store(residual + base + e, v[c]);
      }
#pragma unroll
      for (int i = 0; i < kWide; ++i) sum += v[c][i];
    }
  }
  const float mean = block_sum(sum, scratch) / static_cast<float>(H);
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < kParts; ++c) {
    if ((c * 256 + threadIdx.x) * kWide < H)
#pragma unroll
      for (int i = 0; i < kWide; ++i) {
        v[c][i] -= mean;
        ss = fmaf(v[c][i], v[c][i], ss);
      }
  }
  const float inv = 1.f / sqrtf(block_sum(ss, scratch) / static_cast<float>(H) + eps);
#pragma unroll
  for (int c = 0; c < kParts; ++c) {
    const int e = (c * 256 + threadIdx.x) * kWide;
    if (e < H) {
#pragma unroll
      for (int i = 0; i < kWide; ++i) v[c][i] = fmaf(v[c][i] * inv, w[c][i], sh[c][i]);
      store(out + base + e, v[c]);
    }
  }
}

constexpr int kMaxBranches = 4;
struct Branches {
  const float* x[kMaxBranches];
  const float* gain[kMaxBranches];
};

// out[t] = (1 / n) * sum_b gain_b * x_b[t] / sqrt(mean(x_b[t]^2) + eps).  One block per row.
// REGS: the rows (up to 256 * 8 values) and the gains are fetched once, all at the start, and
// kept in registers; otherwise a row is read twice.  VEC (with REGS): a multiple of 8 values, 16-byte aligned, eight
// neighbouring ones a thread (2,048 rows of 2,048, two branches, 40 MB: 13.4 us value by value, 10.8 so).
template <typename T, bool REGS, bool VEC>
__global__ __launch_bounds__(256) void rms_branches_mean_kernel(T* __restrict__ out, Branches br,
                                                                int n, float eps, int H) {
  __shared__ float scratch[16];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * H;
  const float share = 1.f / static_cast<float>(n);
  if constexpr (REGS) {
    constexpr int NV = 8;
    float x[kMaxBranches][NV], gn[kMaxBranches][NV], ss[kMaxBranches];
#pragma unroll
    for (int b = 0; b < kMaxBranches; ++b) {
      ss[b] = 0.f;
      if constexpr (VEC) {
        const int c = threadIdx.x * 8;
#pragma unroll
        for (int i = 0; i < NV; ++i) x[b][i] = gn[b][i] = 0.f;
        if (b < n && c < H) {
          load8(br.x[b] + base + c, x[b]);
          load8(br.gain[b] + c, gn[b]);
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) ss[b] = fmaf(x[b][i], x[b][i], ss[b]);
      } else {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const int c = threadIdx.x + i * 256;
          const bool ok = b < n && c < H;
          x[b][i] = ok ? br.x[b][base + c] : 0.f;
          gn[b][i] = ok ? br.gain[b][c] : 0.f;
          ss[b] = fmaf(x[b][i], x[b][i], ss[b]);
        }
      }
    }
    float acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.f;
#pragma unroll
    for (int b = 0; b < kMaxBranches; ++b) {
      if (b < n) {  // uniform
        const float inv = 1.f / sqrtf(block_sum(ss[b], scratch) / static_cast<float>(H) + eps);
#pragma unroll
        for (int i = 0; i < NV; ++i) acc[i] = fmaf(x[b][i] * inv, gn[b][i], acc[i]);
      }
    }
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NV; ++i) acc[i] *= share;
      if (threadIdx.x * 8 < H) store8(out + base + threadIdx.x * 8, acc);
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = threadIdx.x + i * 256;
        if (c < H) out[base + c] = from_float<T>(acc[i] * share);
      }
    }
  } else {
    float inv[kMaxBranches];
    for (int b = 0; b < n; ++b) {
      const float* x = br.x[b] + base;
      float ss = 0.f;
      for (int i = threadIdx.x; i < H; i += blockDim.x) ss = fmaf(x[i], x[i], ss);
      inv[b] = 1.f / sqrtf(block_sum(ss, scratch) / static_cast<float>(H) + eps);
    }
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
      float acc = 0.f;
      for (int b = 0; b < n; ++b) acc = fmaf(br.x[b][base + i] * inv[b], br.gain[b][i], acc);
      out[base + i] = from_float<T>(acc * share);
    }
  }
}

// out[t] = [a[t] | b[t]] rounded to T.
template <typename T>
__global__ void concat2_kernel(T* __restrict__ out, const float* __restrict__ a,
                               const float* __restrict__ b, int H, int64_t n) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int64_t t = idx / (2 * H);
  const int c = static_cast<int>(idx - t * 2 * H);
  out[idx] = from_float<T>(c < H ? a[t * H + c] : b[t * H + (c - H)]);
}

__global__ void add_row_kernel(float* __restrict__ x, const float* __restrict__ v, int H, int64_t n) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  x[idx] += v[idx % H];
}

}  // namespace

extern "C" int kvc_add_layernorm(void* out, float* residual, const void* delta, const float* weight,
                                 const float* bias, float eps, int T, int H, int dtype,
                                 kvc_stream stream) {
  if (T < 0 || H <= 0) return kvc_fail("kvc_add_layernorm: bad sizes");
  if (T == 0) return 0;
  if (H % 8 == 0 && H <= 2048 * 4 && aligned16(out) && aligned16(residual) && aligned16(weight) && aligned16(bias) && aligned16(delta)) {
#define KVC_LAYERNORM(NCH)                                                                                            \
  KVC_DISPATCH_DTYPE(dtype, Tp, hipLaunchKernelGGL((add_layernorm_vec_kernel<Tp, NCH>), dim3(T), dim3(256), 0, S(stream), \
                                                   static_cast<Tp*>(out), residual, static_cast<const Tp*>(delta),    \
                                                   weight, bias, eps, H))
    if (H <= 2048) KVC_LAYERNORM(1);
    else if (H <= 4096) KVC_LAYERNORM(2);
    else KVC_LAYERNORM(4);
#undef KVC_LAYERNORM
    return kvc_check_launch("kvc_add_layernorm");
  }
  if (H <= 256 * 8) {
    KVC_DISPATCH_DTYPE(dtype, Tp,
                       hipLaunchKernelGGL((add_layernorm_regs_kernel<Tp, 8>), dim3(T), dim3(256), 0, S(stream),
                                          static_cast<Tp*>(out), residual,
                                          static_cast<const Tp*>(delta), weight, bias, eps, H));
    return kvc_check_launch("kvc_add_layernorm");
  }
  if (H <= 256 * 32) {
    KVC_DISPATCH_DTYPE(dtype, Tp,
                       hipLaunchKernelGGL((add_layernorm_regs_kernel<Tp, 32>), dim3(T), dim3(256), 0, S(stream),
                                          static_cast<Tp*>(out), residual,
                                          static_cast<const Tp*>(delta), weight, bias, eps, H));
    return kvc_check_launch("kvc_add_layernorm");
  }
  KVC_DISPATCH_DTYPE(dtype, Tp,
                     hipLaunchKernelGGL(add_layernorm_kernel<Tp>, dim3(T), dim3(256), 0, S(stream),
                                        static_cast<Tp*>(out), residual,
                                        static_cast<const Tp*>(delta), weight, bias, eps, H));
  return kvc_check_launch("kvc_add_layernorm");
}

extern "C" int kvc_rms_branches_mean(void* out, const float* const* host_x,
                                     const float* const* host_gain, int n, float eps, int T, int H,
                                     int dtype, kvc_stream stream) {
  if (T < 0 || H <= 0 || n <= 0 || n > kMaxBranches)
    return kvc_fail("kvc_rms_branches_mean: bad sizes (one to four branches)");
  if (T == 0) return 0;
  Branches br{};
  bool vec = H % 8 == 0 && aligned16(out);
  for (int b = 0; b < n; ++b) {
    br.x[b] = host_x[b];
    br.gain[b] = host_gain[b];
    vec = vec && aligned16(host_x[b]) && aligned16(host_gain[b]);
  }
  if (H <= 256 * 8 && vec)
    KVC_DISPATCH_DTYPE(dtype, Tp,
                       hipLaunchKernelGGL((rms_branches_mean_kernel<Tp, true, true>), dim3(T), dim3(256), 0,
                                          S(stream), static_cast<Tp*>(out), br, n, eps, H));
  else if (H <= 256 * 8)
    KVC_DISPATCH_DTYPE(dtype, Tp,
                       hipLaunchKernelGGL((rms_branches_mean_kernel<Tp, true, false>), dim3(T), dim3(256), 0,
                                          S(stream), static_cast<Tp*>(out), br, n, eps, H));
  else
    KVC_DISPATCH_DTYPE(dtype, Tp,
                       hipLaunchKernelGGL((rms_branches_mean_kernel<Tp, false, false>), dim3(T), dim3(256), 0,
                                          S(stream), static_cast<Tp*>(out), br, n, eps, H));
  return kvc_check_launch("kvc_rms_branches_mean");
}

extern "C" int kvc_concat2(void* out, const float* a, const float* b, int T, int H, int dtype,
                           kvc_stream stream) {
  if (T < 0 || H <= 0) return kvc_fail("kvc_concat2: bad sizes");
  const int64_t n = static_cast<int64_t>(T) * 2 * H;
  if (n == 0) return 0;
  const unsigned blocks = static_cast<unsigned>((n + 255) / 256);
  KVC_DISPATCH_DTYPE(dtype, Tp,
                     hipLaunchKernelGGL(concat2_kernel<Tp>, dim3(blocks), dim3(256), 0, S(stream),
                                        static_cast<Tp*>(out), a, b, H, n));
  return kvc_check_launch("kvc_concat2");
}

extern "C" int kvc_add_row(float* x, const float* v, int T, int H, kvc_stream stream) {
  if (T < 0 || H <= 0) return kvc_fail("kvc_add_row: bad sizes");
  const int64_t n = static_cast<int64_t>(T) * H;
  if (n == 0) return 0;
  const unsigned blocks = static_cast<unsigned>((n + 255) / 256);
  hipLaunchKernelGGL(add_row_kernel, dim3(blocks), dim3(256), 0, S(stream), x, v, H, n);
  return kvc_check_launch("kvc_add_row");
}
