// Elementwise quantisation kernels, bit-exact with the reference's scalar definitions:
//   quantize_linear_f32_to_i8_scalar     crates/yscv-kernels/src/ops/quantize.rs:242-254
//   requant_scalar                       crates/yscv-kernels/src/ops/int8_requant.rs:143-169
//   requant_i8_per_channel_scalar        crates/yscv-kernels/src/ops/int8_requant.rs:537-555
//   exec_dynamic_quantize_linear         crates/yscv-onnx/src/runner/misc.rs:241-289
// All of them are one pass over HBM; the arithmetic uses explicitly rounded single
// operations (no FMA contraction, IEEE division) because the Rust source never fuses.
#include <type_traits>

#include "int4_common.hpp"
#include "kernels.hpp"

namespace yscv {

__device__ __forceinline__ float round_half_away_f(float v) {
  float t = truncf(v);
  float d = fabsf(__fsub_rn(v, t));
  return (d >= 0.5f) ? __fadd_rn(t, copysignf(1.0f, v)) : t;
}

// clamp that keeps NaN, then the saturating NaN->0 integer cast of Rust's `as`
__device__ __forceinline__ int clamp_cast(float r, float lo, float hi) {
  if (r != r) return 0;
  return (int)fminf(fmaxf(r, lo), hi);
}

__global__ void quantize_linear_i8_kernel(const float *__restrict__ x, size_t len, float scale, float zp,
                                          int8_t *__restrict__ out) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < len;
       i += (size_t)gridDim.x * blockDim.x) {
    float v = __fadd_rn(__fdiv_rn(x[i], scale), zp);
    out[i] = (int8_t)clamp_cast(rintf(v), -128.0f, 127.0f);
  }
}

int32_t launch_quantize_linear_i8(const float *x, size_t len, float scale, float zp, int8_t *out,
                                  hipStream_t s) {
  size_t blocks = ceil_div(len, (size_t)256);
  if (blocks > 16384) blocks = 16384;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(quantize_linear_i8_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, len, scale,
                     zp, out);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// quantize_f32_to_int4 (crates/yscv-kernels/src/ops/quantize.rs:69-95): q = clamp(round_ties_even(x * inv_scale) as
// i32 + zp, -8, 7) with inv_scale = 1 / scale, or 0 when |scale| <= f32::EPSILON; element 2i in the low nibble, the
// high nibble of an odd tail is 0.  `as i32` saturates and maps NaN to 0; the addition of zp wraps.
__device__ __forceinline__ int quant_int4_one(float x, float inv_scale, int zp) {
  const float r = rintf(__fmul_rn(x, inv_scale));
  int32_t q;
  if (r != r) q = 0;
  else if (r >= 2147483648.0f) q = INT32_MAX;
  else if (r <= -2147483648.0f) q = INT32_MIN;
  else q = (int32_t)r;
  q = (int32_t)((uint32_t)q + (uint32_t)zp);
  return q < -8 ? -8 : (q > 7 ? 7 : q);
}
__global__ void quantize_int4_kernel(const float *__restrict__ x, size_t len, float inv_scale, int zp,
                                     uint8_t *__restrict__ out) {
  const size_t n_out = (len + 1) / 2;
  for (size_t o = blockIdx.x * (size_t)blockDim.x + threadIdx.x; o < n_out; o += (size_t)gridDim.x * blockDim.x) {
    const int q0 = quant_int4_one(x[2 * o], inv_scale, zp);
    const int q1 = (2 * o + 1 < len) ? quant_int4_one(x[2 * o + 1], inv_scale, zp) : 0;
    out[o] = (uint8_t)((q0 & 0x0F) | ((q1 & 0x0F) << 4));
  }
}

int32_t launch_quantize_f32_to_int4(const float *x, size_t len, float scale, int zp, uint8_t *out, hipStream_t s) {
  if (len == 0) return YSCV_HIP_OK;
  const float inv_scale = fabsf(scale) > 1.1920929e-7f ? 1.0f / scale : 0.0f;  // host IEEE division, as the reference's
  size_t blocks = ceil_div((len + 1) / 2, (size_t)256);
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(quantize_int4_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, len, inv_scale, zp, out);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

__global__ void requant_kernel(const int32_t *__restrict__ acc, size_t len, size_t c,
                               const int32_t *__restrict__ corr, const float *__restrict__ composite_v,
                               float composite, float y_zp, int round_mode, float lo, float hi, int relu,
                               uint8_t *__restrict__ out) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < len;
       i += (size_t)gridDim.x * blockDim.x) {
    size_t ch = i % c;
    int32_t a = acc[i];
    if (corr) a = (int32_t)((uint32_t)a + (uint32_t)corr[ch]);
    float comp = composite_v ? composite_v[ch] : composite;
    float v = __fadd_rn(__fmul_rn((float)a, comp), y_zp);
    float r = round_mode == YSCV_HIP_ROUND_HALF_AWAY ? round_half_away_f(v) : rintf(v);
    int q = clamp_cast(r, lo, hi);
    if (relu && q < 0) q = 0;
    out[i] = (uint8_t)q;
  }
}

int32_t launch_requant(const int32_t *acc, size_t len, size_t c, const int32_t *corr,
                       const float *composite_v, float composite, float y_zp, int round_mode, int lo,
                       int hi, int relu, void *out, hipStream_t s) {
  size_t blocks = ceil_div(len, (size_t)256);
  if (blocks > 16384) blocks = 16384;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(requant_kernel, dim3((unsigned)blocks), dim3(256), 0, s, acc, len, c, corr,
                     composite_v, composite, y_zp, round_mode, (float)lo, (float)hi, relu,
                     static_cast<uint8_t *>(out));
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// ---- DynamicQuantizeLinear ---------------------------------------------------------------
// Pass 1: every workgroup writes its min / max to minmax[2*block].  Pass 2: every workgroup
// re-reduces those few hundred partials (cheaper than a third launch), derives scale and
// zero point exactly as the reference does, and quantises its share.
// Both passes take four values per load where x allows it, four loads ahead (VEC): a loop of single values waits for each of
// them in turn.  With the GEMM behind them, 1024 x 4096 values 41.5 -> 37.7 us, 1000 x 8192 107.6 -> 98.5.
constexpr int DQL_BLOCKS = 1024;
// values that a workgroup goes through for itself: with the GEMM behind it, 18 000 values 10.5 -> 9.4 and
// 11.4 -> 10.8 us, 37 000 11.7 -> 11.8
constexpr size_t kDqlOwn = 24576;

// four values each at i, i + step, ...: requests past the end repeat the last ones, and there are none where a grid step covers them all
template <int BATCH>
__device__ __forceinline__ void dql_batch(const float *__restrict__ x, size_t n4, size_t i, size_t step, float4_t (&v)[BATCH]) {
  v[0] = reinterpret_cast<const float4_t *>(x)[i];
  if (n4 > step) {
#pragma unroll
    for (int u = 1; u < BATCH; u++) v[u] = reinterpret_cast<const float4_t *>(x)[min(i + u * step, n4 - 1)];
  }
}

// minimum and maximum of a workgroup, neither of them a NaN
__device__ __forceinline__ void dql_reduce(float &mn, float &mx, float (&smin)[4], float (&smax)[4]) {
  mn = -wave_max(-mn);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) {
    smin[threadIdx.x >> 6] = mn;
    smax[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  mn = fminf(fminf(smin[0], smin[1]), fminf(smin[2], smin[3]));
  mx = fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3]));
}

// the values of x this thread takes, f(index, value) for each of them, in batches of four loads
template <bool VEC, int BATCH = 4, typename F>
__device__ __forceinline__ void dql_each(const float *__restrict__ x, size_t len, int block, int blocks, F f) {
  const size_t step = (size_t)blocks * 256, first = block * (size_t)256 + threadIdx.x;
  if constexpr (VEC) {
    const size_t n4 = len / 4;
    if (n4 <= step) {  // one each at most
      if (first < n4) f(first, reinterpret_cast<const float4_t *>(x)[first]);
      return;
    }
    // (no test around loads in here: behind one the four are waited for together: the whole operator, 26 M values 55.4 us,
    // 54.5 so, 33 M 67.6 and 62.8)
    for (size_t i = first; i < n4; i += BATCH * step) {
      float4_t v[BATCH];
#pragma unroll
      for (int u = 0; u < BATCH; u++) v[u] = reinterpret_cast<const float4_t *>(x)[min(i + u * step, n4 - 1)];
#pragma unroll
      for (int u = 0; u < BATCH; u++)
        if (i + u * step < n4) f(i + u * step, v[u]);
    }
  } else {
    for (size_t i = first; i < len; i += step) f(i, x[i]);
  }
}

template <bool VEC>
__global__ void __launch_bounds__(256) dql_minmax_kernel(const float *__restrict__ x, size_t len,
                                                         float *__restrict__ minmax, int blocks) {
  __shared__ float smin[4], smax[4];
  float mn = 3.40282347e+38f, mx = -3.40282347e+38f;
  auto take = [&](float v) {
    if (v < mn) mn = v;  // comparisons, not fmin: NaN never wins, as in misc.rs:250-256
    if (v > mx) mx = v;
  };
  dql_each<VEC>(x, len, (int)blockIdx.x, blocks, [&](size_t, const auto &v) {
    if constexpr (VEC) {
#pragma unroll
      for (int e = 0; e < 4; e++) take(v[e]);
    } else {
      take(v);
    }
  });
  dql_reduce(mn, mx, smin, smax);
  if (threadIdx.x == 0) {
    minmax[2 * blockIdx.x] = mn;
    minmax[2 * blockIdx.x + 1] = mx;
  }
}

// OWN: few values (kDqlOwn): every workgroup takes the minimum and maximum of all of them itself, from L2, instead of a launch in front
template <typename T, bool VEC, bool OWN>
__global__ void __launch_bounds__(256) dql_quantize_kernel(const float *__restrict__ x, size_t len,
                                                           const float *__restrict__ minmax, int nparts,
                                                           T *__restrict__ y, float *__restrict__ scale_out,
                                                           float *__restrict__ zp_out) {
  __shared__ float smin[4], smax[4];
  float mn = 3.40282347e+38f, mx = -3.40282347e+38f;
  // The first four loads of x go out behind the partials' and arrive while those are reduced: one memory round trip instead of two, and
  // the reduction is DPP moves.  us a launch: 2^20 values 5.8 -> 4.5 (the ranges in front 3.0 -> 2.8), 131072 3.4 -> 3.0 (2.6 -> 2.4); with
  // the GEMM against 1024 columns 1024 x 1024 15.5 -> 13.6, 300 x 4096 17.1 -> 16.2, 1000 x 8192 35.1 -> 34.4; up to 131072 values the host's
  // three launches take as long (11.5).
  constexpr bool AHEAD = VEC && !OWN;
  constexpr int BATCH = 4;
  const size_t n4 = len / 4, step = (size_t)nparts * 256, first = blockIdx.x * (size_t)256 + threadIdx.x;
  float4_t v[BATCH];
  if constexpr (OWN) {
    dql_each<VEC, 8>(x, len, 0, 1, [&](size_t, const float4_t &v) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (v[e] < mn) mn = v[e];
        if (v[e] > mx) mx = v[e];
      }
    });
  } else {
    // (at most DQL_BLOCKS parts; repeats of the last one change nothing)
    typedef float float2_t __attribute__((ext_vector_type(2)));
    float2_t part[DQL_BLOCKS / 256];
#pragma unroll
    for (int u = 0; u < DQL_BLOCKS / 256; u++)
      if (u == 0 || nparts > 256) part[u] = reinterpret_cast<const float2_t *>(minmax)[min((int)threadIdx.x + 256 * u, nparts - 1)];
    if constexpr (VEC) {
      if (first < n4) dql_batch(x, n4, first, step, v);
    }
#pragma unroll
    for (int u = 0; u < DQL_BLOCKS / 256; u++) {
      if (u == 0 || nparts > 256) {
        mn = fminf(mn, part[u][0]);
        mx = fmaxf(mx, part[u][1]);
      }
    }
  }
  dql_reduce(mn, mx, smin, smax);
  mn = fminf(mn, 0.0f);  // f32::min / f32::max: range always contains 0 (misc.rs:260-261)
  mx = fmaxf(mx, 0.0f);
  const float range = __fsub_rn(mx, mn);
  const float scale = (fabsf(range) < 1.1920929e-7f) ? 1.0f : __fdiv_rn(range, 255.0f);
  float zp = round_half_away_f(__fsub_rn(0.0f, __fdiv_rn(mn, scale)));
  if (zp == zp) zp = fminf(fmaxf(zp, 0.0f), 255.0f);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *scale_out = scale;
    *zp_out = zp;
  }
  auto one = [&](float v) { return (uint8_t)clamp_cast(round_half_away_f(__fadd_rn(__fdiv_rn(v, scale), zp)), 0.0f, 255.0f); };
  auto put = [&](size_t i, const auto &w) {
    if constexpr (VEC) {
      typedef T vec4 __attribute__((ext_vector_type(4)));
      reinterpret_cast<vec4 *>(y)[i] = vec4{(T)one(w[0]), (T)one(w[1]), (T)one(w[2]), (T)one(w[3])};
    } else {
      y[i] = (T)one(w);
    }
  };
  if constexpr (AHEAD) {
#pragma unroll
    for (int u = 0; u < BATCH; u++)
      if (first + u * step < n4) put(first + u * step, v[u]);
  }
  dql_each<VEC>(x, len, (int)blockIdx.x + (AHEAD ? BATCH * nparts : 0), nparts, put);
}

static int dql_blocks(size_t len) {
  const size_t blocks = ceil_div(len, (size_t)1024);
  return blocks > DQL_BLOCKS ? DQL_BLOCKS : (blocks < 1 ? 1 : (int)blocks);
}
size_t dql_partial_bytes(size_t len) { return sizeof(float) * 2 * dql_blocks(len); }

int32_t launch_dynamic_quantize_linear(const float *x, size_t len, void *y, bool y_f32, float *scale_out, float *zp_out,
                                       float *partial, hipStream_t s) {
  const int blocks = dql_blocks(len);
  Scratch own;
  if (!partial) {
    YSCV_TRY(own.take(dql_partial_bytes(len), s));
    partial = own.as<float>();
  }
  const bool vec = len % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
  auto quantize = [&](auto VEC, auto OWN) -> int32_t {
    constexpr bool V = decltype(VEC)::value, O = decltype(OWN)::value;
    if (y_f32)
      hipLaunchKernelGGL((dql_quantize_kernel<float, V, O>), dim3(blocks), dim3(256), 0, s, x, len, partial, blocks, static_cast<float *>(y), scale_out, zp_out);
    else
      hipLaunchKernelGGL((dql_quantize_kernel<uint8_t, V, O>), dim3(blocks), dim3(256), 0, s, x, len, partial, blocks, static_cast<uint8_t *>(y), scale_out, zp_out);
    YSCV_HIP_TRY(hipGetLastError());
    return YSCV_HIP_OK;
  };
  // (one launch reads what another workgroup may already have written, were y to lie on x)
  const uintptr_t xa = reinterpret_cast<uintptr_t>(x), ya = reinterpret_cast<uintptr_t>(y);
  const bool apart = ya + len * (y_f32 ? 4 : 1) <= xa || xa + len * 4 <= ya;
  if (vec && apart && len > 0 && len <= kDqlOwn) return quantize(std::true_type(), std::true_type());
  if (vec) hipLaunchKernelGGL(dql_minmax_kernel<true>, dim3(blocks), dim3(256), 0, s, x, len, partial, blocks);
  else hipLaunchKernelGGL(dql_minmax_kernel<false>, dim3(blocks), dim3(256), 0, s, x, len, partial, blocks);
  YSCV_HIP_TRY(hipGetLastError());
  return vec ? quantize(std::true_type(), std::false_type()) : quantize(std::false_type(), std::false_type());
}

// ---- KV-cache int8 storage: per-row symmetric quantisation (crates/yscv-onnx/src/runner/kv_cache.rs:45-61) ----
// One wavefront per appended row: abs-max (f32::max ignores NaN), scale = abs_max / 127 (1.0 when abs_max <=
// EPSILON), q = clamp(round_half_away(v * (1 / scale)), -127, 127) as i8.
__global__ void __launch_bounds__(256) kv_i8_quantize_rows_kernel(const float *__restrict__ src, size_t rows, size_t kv_dim,
                                                                  int8_t *__restrict__ data, float *__restrict__ scales) {
  const size_t row = blockIdx.x * (size_t)(blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const float *x = src + row * kv_dim;
  float amax = 0.0f;
  for (size_t i = lane; i < kv_dim; i += 64) amax = fmaxf(amax, fabsf(x[i]));  // fmaxf drops NaN like f32::max
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  const float scale = (amax <= 1.1920929e-7f) ? 1.0f : __fdiv_rn(amax, 127.0f);
  const float inv = __fdiv_rn(1.0f, scale);
  if (lane == 0) scales[row] = scale;
  for (size_t i = lane; i < kv_dim; i += 64)
    data[row * kv_dim + i] = (int8_t)clamp_cast(round_half_away_f(__fmul_rn(x[i], inv)), -127.0f, 127.0f);
}

// LayerStorage::dequantise_to_vec (kv_cache.rs:64-79): q as f32 * scale of its row
__global__ void kv_i8_dequantize_rows_kernel(const int8_t *__restrict__ data, const float *__restrict__ scales, size_t rows,
                                             size_t kv_dim, float *__restrict__ out) {
  const size_t total = rows * kv_dim;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x)
    out[i] = __fmul_rn((float)data[i], scales[i / kv_dim]);
}

int32_t launch_kv_i8_quantize_rows(const float *src, size_t rows, size_t kv_dim, int8_t *data, float *scales, hipStream_t s) {
  hipLaunchKernelGGL(kv_i8_quantize_rows_kernel, dim3((unsigned)ceil_div(rows, (size_t)4)), dim3(256), 0, s, src, rows, kv_dim,
                     data, scales);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

int32_t launch_kv_i8_dequantize_rows(const int8_t *data, const float *scales, size_t rows, size_t kv_dim, float *out,
                                     hipStream_t s) {
  size_t blocks = ceil_div(rows * kv_dim, (size_t)256);
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(kv_i8_dequantize_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, s, data, scales, rows, kv_dim, out);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

}  // namespace yscv
