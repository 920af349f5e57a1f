// Shared by the int8 GEMM kernels (i8_gemm.hip, i8_ksplit.hip, i8_gemm_wide.hip): arguments and the per-element epilogue arithmetic.
#pragma once

#include "int4_common.hpp"
#include "kernels.hpp"

namespace yscv {

// ---- rounding helpers (bit-exact with the reference's two rules) -----------------------
// f32::round: half away from zero.  v - trunc(v) is exact, so the comparison is too.
__device__ __forceinline__ float round_half_away(float v) {
  float t = truncf(v);
  float d = fabsf(__fsub_rn(v, t));
  return (d >= 0.5f) ? __fadd_rn(t, copysignf(1.0f, v)) : t;
}

// Towards zero, a NaN as 0 (`as i8`).  The instruction does that; of a cast it is undefined, and where the compiler knows of the NaN it
// drops the result and what is done with it.  (A select in front of the cast costs two instructions a value.)
__device__ __forceinline__ int nan_to_zero_int(float v) {
  int r;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// clamp(round(a * comp + y_zp), lo, hi) as an int, a NaN as 0 (clamp keeps it, `as i8` makes it 0).  Rounding is monotonic and leaves lo and hi
// as they are, so the clamp comes first: what is rounded is then finite or a NaN, and half away from zero is trunc(v) + trunc(2 (v - trunc(v))).
template <bool HALF_AWAY>
__device__ __forceinline__ int requant_int(int32_t a, float comp, float y_zp, float lo, float hi) {
  float v = __fadd_rn(__fmul_rn((float)a, comp), y_zp);  // two roundings, never an FMA
  v = __builtin_elementwise_minimum(__builtin_elementwise_maximum(v, lo), hi);  // (these keep a NaN)
  if constexpr (HALF_AWAY) {
    const float t = truncf(v), d = __fsub_rn(v, t);
    v = __fadd_rn(t, truncf(__fadd_rn(d, d)));
  } else {
    v = rintf(v);
  }
  return nan_to_zero_int(v);
}

__device__ __forceinline__ int requant_one(int32_t acc, int32_t corr, float comp, float y_zp, int round_mode,
                                           float lo, float hi) {
  const int32_t a = (int32_t)((uint32_t)acc + (uint32_t)corr);  // wrapping_add
  return round_mode == YSCV_HIP_ROUND_HALF_AWAY ? requant_int<true>(a, comp, y_zp, lo, hi) : requant_int<false>(a, comp, y_zp, lo, hi);
}

// requantise, then DequantizeLinear of the quantised value: (q - y_zp) * dq_scale (crates/yscv-onnx/src/runner/misc.rs:124-128)
__device__ __forceinline__ int32_t requant_dequant_bits(int32_t acc, int32_t corr, float comp, float y_zp, int round_mode,
                                                        float lo, float hi, float dq_scale) {
  const int q = requant_one(acc, corr, comp, y_zp, round_mode, lo, hi);
  return __float_as_int(__fmul_rn(__fsub_rn((float)q, y_zp), dq_scale));
}

// requantise and keep the value as an f32 carrier, the form exec_qlinear_matmul returns (crates/yscv-onnx/src/runner/
// linear.rs:481-485): clamp keeps a NaN
__device__ __forceinline__ int32_t requant_f32_bits(int32_t acc, int32_t corr, float comp, float y_zp, int round_mode,
                                                    float lo, float hi) {
  int32_t a = (int32_t)((uint32_t)acc + (uint32_t)corr);
  float v = __fadd_rn(__fmul_rn((float)a, comp), y_zp);
  float r = round_mode == YSCV_HIP_ROUND_HALF_AWAY ? round_half_away(v) : rintf(v);
  if (r == r) r = fminf(fmaxf(r, lo), hi);
  return __float_as_int(r);
}

struct I8Args {
  const uint8_t *a;   // [m][k]
  const int8_t *frag; // packed B
  const int32_t *col_sum;
  void *out;
  const int32_t *corr;
  const float *composite_v;
  float composite, y_zp, dq_scale;
  int lo, hi, how;  // how: I8Epilogue's mode, its round_mode from bit 8 on.  (Whole words: with 16 bits each the arguments came in more
                    // fetches, some of them behind the main loop; 197 x 3072 x 768 requantised 5.9 -> 6.2 us)
  int m, n;
  int lda;          // row stride of a in bytes (k, or kp for a padded copy)
  int ksteps;       // kp / 64
  int a_xor;        // 0x80808080 for uint8 activations, 0 for int8
  int zp_mul;       // multiplies col_sum in the epilogue
  const float *a_zp_dev;  // null, or the uint8 zero point of A as an f32 in device memory (then zp_mul = 128 - that)
  __host__ __device__ int mode() const { return how & 255; }
  __host__ __device__ int round_mode() const { return how >> 8; }
};

static_assert(sizeof(I8Args) + 2 * sizeof(int) <= kCheapArgs, "arguments of a launch");

// The matrix kernels, on 16-byte aligned a with an lda that is a multiple of 64, m * lda below 2 GiB, and the us that a launch is
// estimated to take: small tiles whose waves split K (i8_ksplit.hip; the tiles that all run at once, 1e30 where none do), and large ones
// (i8_gemm_wide.hip).
double i8_ksplit_us(size_t m, size_t n, size_t ksteps, size_t cus);
int32_t launch_i8_ksplit(const I8Args &p, int num_cus, hipStream_t s);
enum : int { IW_64x128, IW_128x256 };
double i8_wide_us(int tile, size_t m, size_t n, size_t ksteps, int mode, size_t cus);
int32_t launch_i8_gemm_wide(const I8Args &p, int tile, hipStream_t s);

}  // namespace yscv
