// Exchange of small vectors between resident workgroups, as decode_layers.hip and decode_wide.hip use it: 8-byte {payload,
// tag} entries written with agent-scope stores and polled with coherent loads.
#pragma once

#include <hip/hip_runtime.h>

#include "decode_layers.hpp"
#include "int4_common.hpp"

namespace yscv {

namespace {

typedef unsigned long long u64;

constexpr unsigned POLL_LIMIT = 1u << 24;  // a failed poll takes 0.3 us and more: several seconds

// the eight weights of a word: {1024 + q, 1024 + q, 64 + q, 64 + q, ...} less these is q - 8, exactly
__device__ __forceinline__ half8_t decode_q8(uint32_t s, const NibbleConsts &nc, uint32_t magic_hi) {
  const half8_t off = {(_Float16)1032.0f, (_Float16)1032.0f, (_Float16)72.0f, (_Float16)72.0f,
                       (_Float16)1032.0f, (_Float16)1032.0f, (_Float16)72.0f, (_Float16)72.0f};
  return extract8(s, nc, magic_hi) - off;
}

__device__ __forceinline__ void put_entry(u64 *p, uint32_t payload, uint32_t tag) {
  __hip_atomic_store(p, ((u64)tag << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// two entries, coherent; valid behind landed()
__device__ __forceinline__ uint4_t get2(const u64 *p) {
  uint4_t v;
  asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v) : "v"(p) : "memory");
  return v;
}
template <int N>
__device__ __forceinline__ void landed(uint4_t (&v)[N]) {
  static_assert(N == 1 || N == 2 || N == 4 || N == 8, "operands of the wait");
  if constexpr (N == 1)
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(v[0])::"memory");
  else if constexpr (N == 2)
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(v[0]), "+v"(v[1])::"memory");
  else if constexpr (N == 4)
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])::"memory");
  else
    asm volatile("s_waitcnt vmcnt(0)"
                 : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])::"memory");
}
__device__ __forceinline__ bool both(const uint4_t &v, uint32_t tag) { return v[1] == tag && v[3] == tag; }

// a poll came back incomplete: false when the wait is over without a result
struct Patience {
  unsigned left;
  uint32_t *flag;
  __device__ __forceinline__ bool again() {
    __builtin_amdgcn_s_sleep(1);
    if (left <= 1) return false;
    left--;
    const bool out = left == 1;
    if (out) __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (out || ((left & 1023u) == 0 && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0)) {
      left = 1;
      return false;
    }
    return true;
  }
};

__device__ __forceinline__ uint32_t pack2(_Float16 a, _Float16 b) {
  U32H2 u;
  u.h = half2_t{a, b};
  return u.u;
}
// entry of channels row, row + 1 (row even) of q / k / v: eight in a 128-byte line per block of 16 rows
__device__ __forceinline__ int qkv_entry(int row) { return (row >> 4) * 16 + ((row & 15) >> 1); }
__device__ __forceinline__ float as_f(uint32_t v) { return __uint_as_float(v); }
// f32 -> fp16 of a value that exists as an f32 first (no conversion merged into the multiply-add before it)
__device__ __forceinline__ _Float16 narrow(float v) {
  asm volatile("" : "+v"(v));
  return (_Float16)v;
}
// LDS written by some lanes of a wave and read by others of the same wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

typedef __attribute__((address_space(4))) LayersLayer LayerAt;  // scalar loads

// the layer's gate/up blocks go to the workgroups in runs; entries of the SwiGLU output of block b (four) start at
__device__ __forceinline__ int act_entry(int b, int base, int rem) {
  const int first = rem * (base + 1);
  const int w = b < first ? b / (base + 1) : rem + (b - first) / base;
  const int o = b < first ? b % (base + 1) : (b - first) % base;
  return w * kLayersActSlots + 4 * o;
}

}  // namespace

}  // namespace yscv
