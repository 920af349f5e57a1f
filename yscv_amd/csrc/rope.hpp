// The rotary embedding of one pair, for every kernel that rotates.
#pragma once

#include <hip/hip_runtime.h>

namespace yscv {

// sin and cos of the angle of pair i at position pos: inv_freq[i] = 1 / theta^(2i / d)
struct SinCos {
  float sn, cs;
};
__device__ __forceinline__ SinCos rope_sincos(float theta, int i, int d, int pos) {
  const float inv_freq = 1.0f / powf(theta, (float)(2 * i) / (float)d);
  SinCos r;
  sincosf(inv_freq * (float)pos, &r.sn, &r.cs);
  return r;
}

// rotate-half of one pair, written with explicit fused multiply-adds so that every kernel that rotates rounds alike
__device__ __forceinline__ void rope_pair_f32(float x0, float x1, float cs, float sn, float &y0, float &y1) {
  y0 = fmaf(x0, cs, -(x1 * sn));
  y1 = fmaf(x0, sn, x1 * cs);
}
// f32 -> fp16 of a value that exists as an f32 first.  Without the empty asm the compiler may merge the conversion
// into the multiply-add that produced the value (a mixed-precision fma that rounds once, straight to fp16), in one
// kernel and not in another: one rotated q element in a few thousand then differs by an fp16 ulp between them.
__device__ __forceinline__ _Float16 f16_of_f32(float v) {
  asm volatile("" : "+v"(v));
  return (_Float16)v;
}
__device__ __forceinline__ void rope_pair(float x0, float x1, float cs, float sn, _Float16 &y0, _Float16 &y1) {
  float f0, f1;
  rope_pair_f32(x0, x1, cs, sn, f0, f1);
  y0 = f16_of_f32(f0);
  y1 = f16_of_f32(f1);
}

}  // namespace yscv
