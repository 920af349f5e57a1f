// Packed-int4 matrix x one activation row: packed_int4_gemv_dispatch (crates/yscv-kernels/src/ops/int4_matmul.rs:310) for one
// row where the skinny kernel's workgroups, made for up to 16 rows and many blocks each, start slowly.
//
// A wave takes 16 weight rows x 512 k: every load it needs is requested at once (four 1 KiB tiles, one load of scales, one or two
// of activations) and nothing passes through LDS on the way to the matrix cores.  The 16 rows of the MFMA's activation
// operand carry the wave's 16 blocks of 32 k, so a lane's operand is eight consecutive activations, as they lie in memory, and
// it serves all sixteen MFMAs of the slice; of the result of block j = 4t + q only row j counts: register q of the lanes 16 t ..
// 16 t + 15, which also hold the scales of tile t.  f32 and bf16 activations are brought to 2^14 .. 2^15 by a power of two per
// slice, f32 split into fp16 hi + lo (22 bits), as in the skinny kernel; weights are exact (q - 8); a zero point enters as
// (8 - zp) * sum of the block's activations, one more MFMA against ones for all sixteen blocks.
// K above 4096 takes sixteen waves, so that few of them have a second or third slice behind the first (4096 x 14336 fp16 with
// eight waves 8.9 us, with sixteen 7.8).  Residual updates, SwiGLU and a folded norm (NormFold in kernels.hpp) are done by the threads
// that hold the sums, with their operands requested ahead of the weights.
// Bound: below a few MB of weights the launch and one round trip to memory each for arguments, loads and sums (4096 x 4096 f32 8.5
// -> 4.4 us, fp16 4.95 -> 4.05, bf16 6.3 -> 4.0; 4096 x 14336 f32 28 -> 9.3; 16384 x 1024 with zero points 8.4 -> 4.5; the weights
// alone are 1 - 4 us of HBM); above that the 4.5 - 5 TB/s that loads of this kind reach behind decode and MFMA (151936 x 1024
// fp16 27.7 -> 16.5, f32 42.0 -> 17.5; 128256 x 4096 51 - 53 and 58.5 - 59 in both).  All captured, weights from HBM, the skinny
// kernel -> this one.  A graph step of the 7B-shape decoder at batch 1: 1619 -> 1376 us (q/k/v 7.3 -> 5.5, o 6.2 -> 4.7, gate/up 14.5 ->
// 13.6, down with its second pass 14.5 -> 8.6, traced), of the 24-layer one 692 -> 630.
// Relative error against 64 bits over those shapes and a dozen others: f32 0.99e-7 .. 1.29e-7 -> 0.80e-7 .. 0.90e-7; fp16 and bf16
// 5e-6 .. 1.3e-5 (0.5e-7 .. 0.9e-7 with zero points) -> 0.47e-7 .. 0.49e-7, as no 1024 stays in the weights here and the sums of
// more than 128 products are in 64 bits.  The low product is added behind the high one: the other order costs up to half as
// much again.
#include <type_traits>

#include "int4_common.hpp"
#include "kernels.hpp"

namespace yscv {

namespace {

__device__ __forceinline__ double sum_xor16_xor32(double v) {  // v + v[lane ^ 16], then the same over lane ^ 32
  float xl, yl, xh, yh;
  xor16_pair(__int_as_float(__double2loint(v)), xl, yl);
  xor16_pair(__int_as_float(__double2hiint(v)), xh, yh);
  v = __hiloint2double(__float_as_int(xh), __float_as_int(xl)) + __hiloint2double(__float_as_int(yh), __float_as_int(yl));
  xor32_pair(__int_as_float(__double2loint(v)), xl, yl);
  xor32_pair(__int_as_float(__double2hiint(v)), xh, yh);
  return __hiloint2double(__float_as_int(xh), __float_as_int(xl)) + __hiloint2double(__float_as_int(yh), __float_as_int(yl));
}

struct GemvRowArgs {
  const uint8_t *tiles;
  const void *tscales;
  const uint8_t *tzps;
  const void *x;
  void *y;
  int n, k, nt, ktp, chunks, chunk_div;
  int groups;              // groups of rows, waves / split blocks of 16 each
  int slices, split_log2;  // 512-k slices of K; waves of a workgroup that share a block of 16 rows (1, 2, 4, 8 or 16)
  int y_dtype, epi;
  // a norm folded into this call (NormFold in kernels.hpp); null / 0 when unused
  const float *gamma_next, *pre;
  _Float16 *xg;
  float *ss_out;
  const float *ss_in, *pre_in;
  float *pre_next;
  int ss_in_count;
  float inv_d, eps;
};

// XD: type of the activations; f32 takes two MFMA operands, the others one.
// KEEP: a wave has one slice of K (K <= 4096).  Its activations stay in registers while the workgroup goes through its groups of
// rows; without it a workgroup has one group and the waves go through their slices.
template <int XD, int GM, bool SF16, bool HAS_ZP, bool KEEP>
__global__ void __launch_bounds__(KEEP ? 512 : 1024, 4) int4_gemv_kernel(GemvRowArgs p) {
  constexpr int WAVES = KEEP ? 8 : 16;
  constexpr int SPT = GM == GM32 ? 4 : (GM == GM64 ? 2 : 1);
  constexpr bool F32 = XD == YSCV_HIP_F32;
  typedef typename std::conditional<SF16, _Float16, float>::type elem_t;
  typedef elem_t scale_t __attribute__((ext_vector_type(SPT)));
  typedef uint8_t zp_t __attribute__((ext_vector_type(SPT)));
  __shared__ double part[2][WAVES][16];
  __shared__ float norm_factor;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const int split = 1 << p.split_log2, sub = wave >> p.split_log2, ks = wave & (split - 1);  // block of the group, first slice
  const int blocks = WAVES >> p.split_log2;
  NibbleConsts nc;
  nc.init();
  uint32_t magic_hi = 0x54005400u;
  asm volatile("" : "+v"(magic_hi));
  const half8_t off8 = {(_Float16)1032.0f, (_Float16)1032.0f, (_Float16)72.0f, (_Float16)72.0f,
                        (_Float16)1032.0f, (_Float16)1032.0f, (_Float16)72.0f, (_Float16)72.0f};
  const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};

  struct Weights {
    uint4_t w[4];
    scale_t s;
    zp_t z;
  };
  struct Acts {
    half8_t hi, lo;
    float4_t sum;  // zero points: the sums of the blocks of tile c
    float down;
  };
  struct Raw {
    float4_t x[2];  // f32: eight values; fp16 and bf16: the first four words
  };
  auto load = [&](int group, int sl) {
    Weights v;
    const int nt = min(group * blocks + sub, p.nt - 1);
    const uint8_t *t0 = p.tiles + ((size_t)nt * p.ktp + (size_t)sl * 4) * kTileBytes + lane * 16;
#pragma unroll
    for (int t = 0; t < 4; t++) v.w[t] = *reinterpret_cast<const uint4_t *>(t0 + t * kTileBytes);
    const int chunk = GM == GM128 ? min((sl * 4 + c) / p.chunk_div, p.chunks - 1) : sl * 4 + c;
    const size_t at = (((size_t)nt * p.chunks + chunk) * 16 + r) * SPT;
    v.s = *reinterpret_cast<const scale_t *>(reinterpret_cast<const elem_t *>(p.tscales) + at);
    if constexpr (HAS_ZP) v.z = *reinterpret_cast<const zp_t *>(p.tzps + at);
    return v;
  };
  auto load_x = [&](int sl) {
    Raw v;
    const int k0 = sl * 512 + 32 * r + 8 * c;  // K is a multiple of 32: a lane's eight values exist or do not
    const bool in = k0 < p.k;
    const int kk = in ? k0 : 0;
    if constexpr (F32) {
      const float *src = static_cast<const float *>(p.x) + kk;
      v.x[0] = *reinterpret_cast<const float4_t *>(src);
      v.x[1] = *reinterpret_cast<const float4_t *>(src + 4);
    } else {
      v.x[0] = *reinterpret_cast<const float4_t *>(static_cast<const _Float16 *>(p.x) + kk);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v.x[0][e] = in ? v.x[0][e] : 0.0f;
      if constexpr (F32) v.x[1][e] = in ? v.x[1][e] : 0.0f;
    }
    return v;
  };
  auto times = [&](const Acts &x, half8_t b) {
    float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.hi, b, zero, 0, 0, 0);
    if constexpr (F32) d = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.lo, b, d, 0, 0, 0);
    return d;
  };
  auto prepare = [&](const Raw &v) {
    Acts x;
    x.down = 1.0f;
    if constexpr (XD == YSCV_HIP_F16) {
      union {
        float4_t f;
        half8_t h;
      } u;
      u.f = v.x[0];
      x.hi = u.h;
    } else {
      float f[8], mx = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint32_t two = __float_as_uint(v.x[0][e >> 1]);
        f[e] = F32 ? v.x[e >> 2][e & 3] : __uint_as_float((e & 1) ? two & 0xffff0000u : two << 16);
        mx = fmaxf(mx, fabsf(f[e]));
      }
      const uint32_t top = (__float_as_uint(wave_max(mx)) >> 23) & 255u, ex = min(268u - top, 253u);
      const float up = __uint_as_float(ex << 23);
      x.down = __uint_as_float((254u - ex) << 23);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float t = f[e] * up;
        x.hi[e] = (_Float16)t;
        if constexpr (F32) x.lo[e] = (_Float16)(t - (float)x.hi[e]);
      }
    }
    if constexpr (HAS_ZP) {
      const half8_t ones = {(_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f,
                            (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f};
      x.sum = times(x, ones);
    }
    return x;
  };
  auto multiply = [&](const Weights &v, const Acts &x) {
    float sel[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float4_t d = times(x, extract8(v.w[t][q], nc, magic_hi) - off8);
        sel[q] = t == 0 ? d[q] : (c == t ? d[q] : sel[q]);
      }
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = GM == GM32 ? q : (GM == GM64 ? q >> 1 : 0);
      if constexpr (HAS_ZP) sel[q] = fmaf(8.0f - (float)v.z[e], x.sum[q], sel[q]);
      acc = fmaf((float)v.s[e], sel[q], acc);
    }
    return acc * x.down;
  };
  // What the folded norm needs, requested ahead of everything else: the partial sums of squares (the last wave adds them up), and
  // the residuals of the first group in the threads that will update them
  float ss[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ss_pre = 1.0f, h_old = 0.0f, h_mul = 0.0f;
  if (p.ss_in && wave == 7) {
#pragma unroll
    for (int i = 0; i < 4; i++) ss[i] = p.ss_in[min(lane * 4 + i, p.ss_in_count - 1)];
    ss_pre = p.pre_in[0];
  }
  if (p.epi == EPI_ADD_F32 && wave < 2) {  // 16 * blocks threads at most
    const int row = min((int)blockIdx.x * blocks * 16 + tid, p.n - 1);
    h_old = static_cast<const float *>(p.y)[row];
    if (p.xg) h_mul = p.gamma_next[row] * p.pre[0];
  }
  auto norm_sum = [&] {  // before the barrier of the first group
    if (p.ss_in && wave == 7) {
#pragma unroll
      for (int i = 0; i < 4; i++) ss[i] = lane * 4 + i < p.ss_in_count ? ss[i] : 0.0f;
      const float inv_rms = 1.0f / sqrtf(wave_sum((ss[0] + ss[1]) + (ss[2] + ss[3])) * p.inv_d + p.eps);
      if (lane == 0) {
        norm_factor = inv_rms / ss_pre;
        if (p.pre_next && blockIdx.x == 0) p.pre_next[0] = norm_fold_prescale(inv_rms);
      }
    }
  };
  auto store_row = [&](int group, int b, int row, float v) {
    if (p.ss_in) v *= norm_factor;
    const bool live = row < p.n;
    if (p.epi == EPI_ADD_F32) {
      float *h = static_cast<float *>(p.y) + row;
      const bool first = group == (int)blockIdx.x;
      const float hn = live ? (first ? h_old : *h) + v : 0.0f;
      if (live) *h = hn;
      if (p.xg) {  // the sixteen lanes of a block leave one sum of squares
        const float mul = first ? h_mul : (live ? p.gamma_next[row] * p.pre[0] : 0.0f);
        if (live) p.xg[row] = (_Float16)fminf(fmaxf(hn * mul, -65504.0f), 65504.0f);
        const float sq = row_sum16(hn * hn);
        if ((tid & 15) == 0 && live) p.ss_out[group * blocks + b] = sq;
      }
    } else if (p.epi == EPI_SWIGLU) {  // rows 2i and 2i + 1 of the weight are gate i and up i
      const float up = dpp_move<DPP_XOR1>(v);
      if (live && !(row & 1)) store_out(p.y, (size_t)(row >> 1), silu(v) * up, p.y_dtype);
    } else if (live) {
      store_out(p.y, (size_t)row, v, p.y_dtype);
    }
  };
  // from the 128 k of a lane on the sums are in 64 bits; the waves' meet in LDS; only LDS is waited for, the loads ahead stay in flight
  auto finish = [&](int group, int buf, double total) {
    total = sum_xor16_xor32(total);
    if (lane < 16) part[buf][wave][lane] = total;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid < 16 * blocks) {
      const int b = tid >> 4, row = (group * blocks + b) * 16 + (tid & 15);
      double v = 0.0;
      for (int w = 0; w < split; w++) v += part[buf][b * split + w][tid & 15];
      store_row(group, b, row, (float)v);
    }
  };

  if constexpr (KEEP) {  // two buffers: a wave past the barrier of group i + 1 has read the sums of group i
    const int sl = min(ks, p.slices - 1), step = (int)gridDim.x;
    const bool in = ks < p.slices;
    int group = (int)blockIdx.x, buf = 0;
    const Raw xr = load_x(sl);
    Weights v = load(group, sl);
    const Acts x = prepare(xr);
    norm_sum();
    for (; group + step < p.groups; group += step, buf ^= 1) {
      const Weights nx = load(group + step, sl);
      finish(group, buf, in ? (double)multiply(v, x) : 0.0);
      v = nx;
    }
    finish(group, buf, in ? (double)multiply(v, x) : 0.0);
  } else {
    int sl = ks;
    double total = 0.0;
    if (sl < p.slices) {  // uniform in the wave
      Raw xr = load_x(sl);
      Weights v = load((int)blockIdx.x, sl);
      for (; sl + split < p.slices; sl += split) {
        const Raw xn = load_x(sl + split);
        const Weights nx = load((int)blockIdx.x, sl + split);
        total += (double)multiply(v, prepare(xr));
        xr = xn;
        v = nx;
      }
      total += (double)multiply(v, prepare(xr));
    }
    norm_sum();
    finish((int)blockIdx.x, 0, total);
  }
}

template <int XD, int GM, bool SF16>
int32_t gemv_go(const GemvRowArgs &a, unsigned grid, hipStream_t s) {
  const bool keep = a.slices <= 8;
  if (keep && a.tzps) hipLaunchKernelGGL((int4_gemv_kernel<XD, GM, SF16, true, true>), dim3(grid), dim3(512), 0, s, a);
  else if (keep) hipLaunchKernelGGL((int4_gemv_kernel<XD, GM, SF16, false, true>), dim3(grid), dim3(512), 0, s, a);
  else if (a.tzps) hipLaunchKernelGGL((int4_gemv_kernel<XD, GM, SF16, true, false>), dim3(grid), dim3(1024), 0, s, a);
  else hipLaunchKernelGGL((int4_gemv_kernel<XD, GM, SF16, false, false>), dim3(grid), dim3(1024), 0, s, a);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}
template <int XD>
int32_t gemv_gm(const GemvRowArgs &a, unsigned grid, int gm, bool sf16, hipStream_t s) {
  if (gm == GM32) return sf16 ? gemv_go<XD, GM32, true>(a, grid, s) : gemv_go<XD, GM32, false>(a, grid, s);
  if (gm == GM64) return sf16 ? gemv_go<XD, GM64, true>(a, grid, s) : gemv_go<XD, GM64, false>(a, grid, s);
  return sf16 ? gemv_go<XD, GM128, true>(a, grid, s) : gemv_go<XD, GM128, false>(a, grid, s);
}

}  // namespace

bool int4_gemv_takes(const yscv_hip_int4_weight *w, const void *x, int x_dtype, size_t m) {
  if (!w->tiled || m != 1 || (reinterpret_cast<uintptr_t>(x) & 15) != 0 || w->k % 32 != 0) return false;
  return w->n < ((size_t)1 << 31) && w->k < ((size_t)1 << 30);
}

int32_t launch_int4_gemv(const yscv_hip_int4_weight *w, const void *x, int x_dtype, void *y, int y_dtype, int epi, const NormFold *nf,
                         int num_cus, hipStream_t s) {
  if (epi == EPI_ADD_F32 && y_dtype != YSCV_HIP_F32)
    return set_error(YSCV_HIP_ERR_INVALID_ARG, "residual accumulation needs an f32 output");
  if (epi == EPI_SWIGLU && (w->n & 1)) return set_error(YSCV_HIP_ERR_INVALID_ARG, "SwiGLU epilogue needs an even row count");
  GemvRowArgs a = {};
  a.tiles = w->tiles;
  a.tscales = w->tscales;
  a.tzps = w->has_zp ? w->tzps : nullptr;
  a.x = x;
  a.y = y;
  a.n = (int)w->n;
  a.k = (int)w->k;
  a.nt = (int)w->nt;
  a.ktp = (int)w->ktp;
  a.chunks = (int)w->chunks;
  a.chunk_div = w->gm == GM128 ? (int)(w->g / 128) : 1;
  a.slices = (int)(w->ktp / 4);
  a.split_log2 = a.slices > 8 ? 4 : a.slices >= 5 ? 3 : (a.slices >= 3 ? 2 : a.slices - 1);
  a.y_dtype = y_dtype;
  a.epi = epi;
  if (nf && nf->ss_in) {
    if (nf->ss_in_count < 1 || nf->ss_in_count > 256 || !nf->pre_in)
      return set_error(YSCV_HIP_ERR_INVALID_ARG, "folded norm: %d partial sums of the row", nf->ss_in_count);
    a.ss_in = nf->ss_in;
    a.pre_in = nf->pre_in;
    a.pre_next = nf->pre_next;
    a.ss_in_count = nf->ss_in_count;
    a.inv_d = nf->inv_d;
    a.eps = nf->eps;
  }
  if (nf && nf->xg) {
    if (epi != EPI_ADD_F32 || !nf->gamma_next || !nf->ss_out || !nf->ss_out_count || !nf->pre || nf->ss_out_stride < (int)w->nt)
      return set_error(YSCV_HIP_ERR_INVALID_ARG, "folded norm: the producing call is a residual update with gamma and a place for the sums");
    a.gamma_next = nf->gamma_next;
    a.pre = nf->pre;
    a.xg = nf->xg;
    a.ss_out = nf->ss_out;
    *nf->ss_out_count = (int)w->nt;
  }
  const int blocks = (a.slices > 8 ? 16 : 8) >> a.split_log2;
  a.groups = (a.nt + blocks - 1) / blocks;
  unsigned grid = (unsigned)a.groups;
  if (a.slices <= 8) {
    // Groups of a workgroup, where it may have several.  From 16 per CU, as many as keep all workgroups on the chip together:
    // 128256 x 4096 58.6 us with f32 activations and 51.6 with fp16, one group each 67.9 and 54.4.  Below that the 16-bit types are
    // best with one (28672 x 4096 14.0 against 14.8 us, 151936 x 1024 15.8 against 17.1), and f32, which splits its activations anew in
    // each workgroup, with two (16.2 against 16.9, 18.5 against 20.0) once there are more than four per CU.
    const int rounds = a.groups >= 16 * num_cus ? (a.groups + 2 * num_cus - 1) / (2 * num_cus)
                                                : (x_dtype == YSCV_HIP_F32 && a.groups > 4 * num_cus ? 2 : 1);
    grid = (unsigned)((a.groups + rounds - 1) / rounds);
  }
  const bool sf16 = w->scale_dtype == YSCV_HIP_F16;
  if (x_dtype == YSCV_HIP_F32) return gemv_gm<YSCV_HIP_F32>(a, grid, w->gm, sf16, s);
  if (x_dtype == YSCV_HIP_BF16) return gemv_gm<YSCV_HIP_BF16>(a, grid, w->gm, sf16, s);
  return gemv_gm<YSCV_HIP_F16>(a, grid, w->gm, sf16, s);
}

}  // namespace yscv
